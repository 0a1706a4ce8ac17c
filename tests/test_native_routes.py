"""Which calls the native call layer may take, decided in Python before any launch: the layer is replaced by a recorder and the
packs stand on the CPU, so every test here asks only which path a call takes."""
import copy
import io
import pickle
import weakref

import pytest
import torch

from mortar_amd import _lib, synth
from mortar_amd.engine import MortarDecodeMLP
from mortar_amd.mlp import _SwiGLUMortar


class _Native:
    """Answers every entry point of the native layer with TAKEN."""
    TAKEN = torch.full((1,), 7.0)

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*a):
            self.calls.append((name, a))
            return self.TAKEN
        return call


@pytest.fixture
def native(monkeypatch):
    n = _Native()
    monkeypatch.setattr(_lib, "_native", n)
    monkeypatch.setattr(_SwiGLUMortar, "native_pair", lambda self: (self.gate_up._cms._pack, self.down._cms._pack))
    return n


def _mlp(cls=_SwiGLUMortar):
    mlp = synth.mlp_module(synth.synth_mlp(64, 128, 0.5, seed=1), torch.device("cpu"))
    mlp.__class__ = cls
    return mlp


X = torch.zeros(2, 64, dtype=torch.bfloat16)


class _Adapter(_SwiGLUMortar):
    def forward(self, x, **kw):
        return x + 1


def _instance_forward():
    mlp = _mlp()
    mlp.forward = lambda x, **kw: x + 1
    return mlp


def test_decode_call_of_the_plain_module_is_native(native):
    assert MortarDecodeMLP(_mlp())(X) is native.TAKEN


@pytest.mark.parametrize("make", [lambda: _mlp(_Adapter), _instance_forward])
def test_decode_call_runs_an_overridden_forward(native, make):
    y = MortarDecodeMLP(make())(X)
    assert torch.equal(y, torch.ones(2, 1, 64, dtype=torch.bfloat16)) and not native.calls


class _Host:
    """What MortarDecodeMLP reads of its host, without being a module."""
    def __init__(self, mlp):
        self.gate_up, self.down, self.d_ff, self.router = mlp.gate_up, mlp.down, mlp.d_ff, None

    def __call__(self, x, iter_idx=0, gates=None, norm=None):
        return x + 2


def test_decode_call_serves_a_host_that_is_no_module(native):
    y = MortarDecodeMLP(_Host(_mlp()))(X)
    assert torch.equal(y, torch.full((2, 1, 64), 2, dtype=torch.bfloat16)) and not native.calls


class _Router:
    """A router that is no module: the MLP only calls it."""
    def __call__(self, x, iter_idx=0):
        return torch.zeros(x.shape[0], 4), None

    def route(self, x, iter_idx=0):
        return torch.zeros(x.shape[0], 4), None


def test_a_router_that_is_no_module_is_not_left_out(native):
    mlp = _mlp()
    dec = MortarDecodeMLP(mlp)
    mlp.router = _Router()
    for call in (mlp, dec):
        with pytest.raises(RuntimeError, match="ROCm device"):       # the general path, which needs the GPU
            call(X)
    assert not native.calls


def test_decode_call_keeps_the_packs_it_was_built_with(native):
    """Where the general path multiplies with the packs of the constructor (no router, but a norm in its own launch; or a
    router), so does the native one: not with those of weights that were loaded since."""
    mlp = _mlp()
    dec = MortarDecodeMLP(mlp)
    mlp.to(torch.device("cpu"))                      # drops the packs
    mlp.gate_up._cms.mortar_pack(), mlp.down._cms.mortar_pack()
    dec._general = lambda x, gates: "general"
    assert dec(X) == "general" and not native.calls


@pytest.fixture
def pair_of(monkeypatch):
    """native_pair() as on a GPU: the packs of a CPU module taken for resident ones."""
    from mortar_amd.pack import MortarPack
    monkeypatch.setattr(MortarPack, "on_gpu", True)
    monkeypatch.setattr(_lib, "_native", _Native())

    def build(cls=_SwiGLUMortar):
        mlp = _mlp(cls)
        mlp.gate_up._cms.mortar_pack(), mlp.down._cms.mortar_pack()
        assert mlp.native_pair() is not None
        return mlp
    return build


def test_a_module_copies_and_saves_after_a_native_call(pair_of):
    mlp = pair_of()
    mlp.to(torch.device("cpu"))                      # (a move drops the packs, which hold device addresses)
    again = copy.deepcopy(mlp)
    torch.save(mlp, io.BytesIO())
    pickle.dumps(mlp)
    assert again.native_pair() is None
    again.gate_up._cms.mortar_pack(), again.down._cms.mortar_pack()
    assert again.native_pair() == (again.gate_up._cms._pack, again.down._cms._pack)


@pytest.mark.parametrize("layer", ["gate_up", "down"])
def test_a_dropped_pack_is_freed(pair_of, layer):
    mlp = pair_of()
    packs = [weakref.ref(m._cms._pack) for m in (mlp.gate_up, mlp.down)]
    getattr(mlp, layer).to(torch.device("cpu"))
    assert mlp.native_pair() is None
    assert [p() is None for p in packs] == [layer == "gate_up", layer == "down"]


def test_a_copied_pack_hands_out_its_own_addresses(pair_of):
    """clone_weights() copies the pack's attributes: not what was found out for the original's pair."""
    mlp = pair_of()
    cms = mlp.gate_up._cms
    old, cms._pack = cms._pack, cms._pack.clone_weights()
    new = mlp.native_pair()
    assert new[0] is cms._pack and new[0].address != old.address and new[0]._handle.sched2 != old._handle.sched2


def test_flags_of_the_native_layer_are_read_by_their_truth():
    """numpy.True_, 1 and other true objects are true: the layer asks them, it does not look for the object True."""
    class Flag:
        asked = 0

        def __bool__(self):
            Flag.asked += 1
            return True

    n, x = _lib.native(), torch.zeros(2, 64)               # a CPU tensor: declined, once the arguments are read
    assert n.gemv_f32(x, 0, x[0, :1], Flag(), Flag(), None, None, None) is None and Flag.asked == 2
    assert n.mlp(x, 0, 0, Flag(), Flag(), None, 0.0, None) is None and Flag.asked == 4
    with pytest.raises(ValueError, match="ambiguous"):
        n.gemv_f32(x, 0, x[0, :1], torch.zeros(2).numpy(), False, None, None, None)


def _instance_forward_of(router, called):
    def forward(x, iter_idx=0):
        called.append(1)
        return None, None
    router.forward = forward


@pytest.mark.parametrize("change", [lambda r, called: torch.nn.modules.module.register_module_forward_pre_hook(lambda m, a: called.append(1)),
                                    lambda r, called: r.register_forward_hook(lambda m, a, o: called.append(1)), _instance_forward_of])
def test_the_modules_router_is_called_where_a_call_is_more_than_its_forward(monkeypatch, change):
    mlp = _mlp()
    mlp.enable_routing(n_clusters=4)
    monkeypatch.setattr(type(mlp.router), "forward_native", lambda self, x, iter_idx=0: ("native", None))
    called = []
    handle = change(mlp.router, called)
    try:
        mlp._routed(X, 0)
        assert called == [1]
    finally:
        if handle is not None:
            handle.remove()


def test_the_modules_router_is_left_to_the_native_layer_otherwise(monkeypatch):
    mlp = _mlp()
    mlp.enable_routing(n_clusters=4)
    monkeypatch.setattr(type(mlp.router), "forward_native", lambda self, x, iter_idx=0: ("native", None))
    assert mlp._routed(X, 0)[0] == "native"


@pytest.mark.parametrize("on_instance", [False, True])
def test_an_overridden_route_is_called(native, monkeypatch, on_instance):
    """TileRouter.forward goes through route() for the calls that the kernels cover: a route() of a subclass or of the
    instance is what runs, from the router's forward, the module and the decode call alike."""
    from mortar_amd.routing import TileRouter
    called = []

    def route(self, x_flat, iter_idx=0):
        called.append(1)
        return torch.zeros(x_flat.shape[0], 4), torch.zeros(x_flat.shape[0], 4, dtype=torch.uint8)

    mlp = _mlp()
    mlp.enable_routing(n_clusters=4)
    if on_instance:
        mlp.router.route = route.__get__(mlp.router)
    else:
        mlp.router.__class__ = type("Router", (TileRouter,), {"route": route})
    monkeypatch.setattr(TileRouter, "forward_native", lambda self, x, iter_idx=0: ("native", None))
    monkeypatch.setattr(TileRouter, "_fused_ok", lambda self, x: True)
    mlp.router(X)
    assert len(called) == 1
    mlp._routed(X, 0)
    assert len(called) == 2
    dec = MortarDecodeMLP(mlp)
    dec._general = lambda x, gates: "general"
    assert dec(X) == "general" and not native.calls


class _Wrapped(torch.nn.Module):
    """A carved linear layer inside another module, which hands on what the MLP reads of it."""
    def __init__(self, layer):
        super().__init__()
        self.inner = layer

    @property
    def _cms(self):
        return self.inner._cms


def test_wrapped_layers_take_the_general_path(monkeypatch):
    monkeypatch.setattr(_lib, "_native", _Native())
    mlp = _mlp()
    mlp.down = _Wrapped(mlp.down)
    dec = MortarDecodeMLP(mlp)
    for call in (mlp, dec):
        with pytest.raises(RuntimeError, match="ROCm device"):
            call(X)
    assert not _lib._native.calls


def test_a_bad_eps_is_a_type_error():
    """Read before anything else, as float(eps) would: no result may be returned with an exception pending."""
    n, x = _lib.native(), torch.zeros(2, 64)
    with pytest.raises(TypeError):
        n.mlp(x, 0, 0, False, True, None, "1e-6", None)


def test_iteration_index_and_k_are_taken_as_integers(native, monkeypatch):
    """int() of whatever number the caller holds, as the general path takes them."""
    mlp = _mlp()
    mlp.enable_routing(n_clusters=4)
    mlp.router.activation_k = 2.0
    assert MortarDecodeMLP(mlp, iter_idx=1.0)(X) is native.TAKEN
    args = native.calls[-1][1]
    assert type(args[-1]) is int and all(type(v) is int for v in args[-3])
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    mlp.router._native_route(X, 1.0, False)
    args = native.calls[-1][1]
    assert type(args[6]) is int and all(type(v) is int for v in args[4])


@pytest.mark.parametrize("fails", ["forward", "step_pack", "declined", None])
def test_packs_are_fresh_only_behind_a_training_forward_that_ended(native, monkeypatch, fails):
    """A native training forward that raises (out of memory before its re-pack, an error code) or declines leaves both layers to
    re-encode at their next use, whatever key they had before; one that returns leaves them fresh."""
    from mortar_amd import mlp as M
    from mortar_amd.pack import MortarPack
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    encoded = []
    monkeypatch.setattr(MortarPack, "requantize", lambda self, v, **kw: (encoded.append(self), torch.ones(1))[1])
    mlp = synth.qat_mlp_module(synth.synth_mlp(64, 128, 0.5, seed=1), torch.device("cpu"), seed=2)
    layers = [mlp.gate_up._cms, mlp.down._cms]
    packs = [m.mortar_pack() for m in layers]
    assert encoded == packs and [m.mortar_pack() for m in layers] == packs and len(encoded) == 2
    scales = torch.ones(1), torch.ones(1)
    if fails == "forward":
        def train_forward(*a):
            raise RuntimeError("out of memory")
    else:
        def train_forward(*a):
            return None if fails == "declined" else (1, 2, 3, *scales)
    native.train_forward = train_forward
    if fails == "step_pack":
        monkeypatch.setattr(packs[1], "sched", lambda n: (_ for _ in ()).throw(RuntimeError("out of memory")))
    x = torch.zeros(2, 64, dtype=torch.bfloat16)
    if fails in ("forward", "step_pack"):
        with pytest.raises(RuntimeError, match="out of memory"):
            M._native_step(x, *layers, True, True)
    else:
        assert M._native_step(x, *layers, True, True) == (None if fails else (1, 2, 3))
    encoded.clear()
    assert [m.mortar_pack() for m in layers] == packs
    assert encoded == ([] if fails is None else packs)
    forms = [(P.uniform_scale, P.one_scale) for W in packs for P in (W, W._transposed) if P is not None]
    assert forms == [(0.0, 1 if fails is None else 0)] * len(forms)
    assert [W.scales_f32 is s for W, s in zip(packs, scales)] == [fails is None] * 2


def test_packs_are_stale_behind_a_re_pack_that_failed(monkeypatch):
    from mortar_amd.block_sparse import CMSBlockLinear
    from mortar_amd.pack import MortarPack
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    mlp = synth.qat_mlp_module(synth.synth_mlp(64, 128, 0.5, seed=1), torch.device("cpu"), seed=2)
    encoded = []
    monkeypatch.setattr(MortarPack, "requantize", lambda self, v, **kw: (encoded.append(self), torch.ones(1))[1])
    cms = mlp.gate_up._cms
    W = cms.mortar_pack()

    def failing(jobs):
        raise RuntimeError("launch failed")
    monkeypatch.setattr(MortarPack, "requantize_pairs", staticmethod(failing))
    with pytest.raises(RuntimeError, match="launch failed"):
        CMSBlockLinear.repack_for_step([(cms, True)])
    assert cms.mortar_pack() is W and encoded == [W, W]


def test_a_declined_training_step_leaves_deployed_packs_alone(monkeypatch):
    """One matrix deployed, the other trainable: the deployed pack keeps the form it was built with."""
    from mortar_amd import mlp as M
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    spec = dict(synth.synth_mlp(64, 128, 0.5, seed=1), gate_up=synth.synth_matrix(256, 64, 0.5, seed=3, per_tensor_scale=True))
    mlp = synth.mlp_module(spec, torch.device("cpu"))
    cms = mlp.gate_up._cms
    W = cms.mortar_pack()
    assert W.uniform_scale != 0
    form = W.uniform_scale
    cms.__dict__.pop("_step_key", None)                # as in a module saved by an earlier version
    assert M._native_step(torch.zeros(2, 64, dtype=torch.bfloat16), cms, mlp.down._cms, True, True) is None
    assert cms.mortar_pack() is W and (W.uniform_scale, W.struct.uniform_scale, W.one_scale) == (form, form, 0)


def test_a_topology_copies_and_pickles():
    """By copy, deepcopy, pickle and torch.save, before and after its transposed form was made; every copy hands out the addresses of
    its own arrays."""
    from mortar_amd.pack import BcsrTopology
    m = synth.synth_matrix(16 * 5, 16 * 400, 0.2, seed=1)              # wide enough for per-segment row pointers
    T = BcsrTopology(m["offsets"], m["col_idx"], 16 * 5, 16 * 400, "cpu")
    assert T.seg_ptr is not None

    def saved(t):
        f = io.BytesIO()
        torch.save(t, f)
        return torch.load(io.BytesIO(f.getvalue()), weights_only=False)
    for _ in range(2):
        for make in (copy.copy, copy.deepcopy, lambda t: pickle.loads(pickle.dumps(t)), saved):
            t = make(T)
            assert t.address != T.address and (t.Rb, t.Cb, t.nnz, t.nseg, t.seg_cb) == (T.Rb, T.Cb, T.nnz, T.nseg, T.seg_cb)
            for name in ("row_ptr", "col", "seg_ptr"):
                assert torch.equal(getattr(t, name), getattr(T, name)) and getattr(t._handle, name) == getattr(t, name).data_ptr()
            (a, src), (b, want) = t.transposed(), T.transposed()
            assert torch.equal(src, want) and a._handle.src == src.data_ptr() != want.data_ptr() and torch.equal(a.col, b.col)
