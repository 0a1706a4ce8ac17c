"""The native training calls (stk_dds with its autograd node, the QAT step of the MLP) against the general paths they leave out: same
bits, same gradients, same refusals, and the general path wherever something looks on."""
import pytest
import torch

import mortar_amd
from mortar_amd import _lib, synth

pytestmark = pytest.mark.gpu


class _Declines:
    """A native layer that takes nothing."""
    def __getattr__(self, name):
        return lambda *a: None


class general:
    """The operator as it is without the native layer, in forward and backward: general(f)() runs f so."""
    def __init__(self, f):
        self.f = f

    def __call__(self):
        kept, _lib._native = _lib._native, _Declines()
        try:
            return self.f()
        finally:
            _lib._native = kept


def both(f):
    """f() through the native layer and through the general path."""
    return f(), general(f)()


def _operands(dev, M, s0, s1, tb, seed=0, pad=0):
    rows, cols = (s1, s0) if tb else (s0, s1)
    m = synth.synth_matrix(rows, cols, 0.3, seed=seed + 1)
    sd = synth.carved_state(m)
    index = [sd["mortar_" + k].to(dev) for k in ("offsets", "row_indices", "column_indices", "offsets_t", "column_indices_t", "block_offsets_t")]
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(M, s0 + pad, generator=g, device=dev).to(torch.bfloat16)[:, :s0]
    data = (torch.randn(m["col_idx"].size, 16, 16, generator=g, device=dev) * 0.1).to(torch.bfloat16)
    dy = torch.randn(M, s1, generator=g, device=dev).to(torch.bfloat16)
    return x, data, dy, (*index, s0, s1, tb)


@pytest.fixture
def took(monkeypatch):
    """The names of the native calls that returned a result."""
    n, names = _lib.native(), []

    class Recorder:
        def __getattr__(self, name):
            f = getattr(n, name)

            def call(*a):
                r = f(*a)
                if r is not None:
                    names.append(name)
                return r
            return call
    monkeypatch.setattr(_lib, "_native", Recorder())
    return names


@pytest.mark.parametrize("M,s0,s1", [(1, 16, 16), (65, 96, 160), (130, 2800, 64), (513, 64, 2800)])
@pytest.mark.parametrize("tb", [True, False])
@pytest.mark.parametrize("need", [(True, True), (True, False), (False, True), (False, False)])
def test_dds_native_is_the_operator(dev, took, M, s0, s1, tb, need):
    x, data, dy, rest = _operands(dev, M, s0, s1, tb, pad=8)

    def step():
        a, b = x.detach().requires_grad_(need[0]), data.detach().requires_grad_(need[1])
        y = mortar_amd.stk_dds(a, b, *rest)
        assert y.requires_grad == any(need)
        if any(need):
            y.backward(dy)
        return y.detach(), a.grad, b.grad
    res = both(step)
    assert took == ["dds"]
    for got, want in zip(*res):
        assert (got is None) == (want is None) and (got is None or torch.equal(got, want))


def test_dds_native_gradients_of_other_kinds(dev, took):
    """Expanded, strided and fp32 gradients, a retained graph, hooks on the saved tensors and in-place changes of them."""
    x, data, dy, rest = _operands(dev, 33, 64, 96, True)
    for grad in (torch.ones((), device=dev, dtype=torch.bfloat16).expand(33, 96), dy.t().contiguous().t()):
        def step():
            a, b = x.detach().requires_grad_(), data.detach().requires_grad_()
            y = mortar_amd.stk_dds(a, b, *rest)
            y.backward(grad, retain_graph=True)
            y.backward(grad)
            return a.grad, b.grad
        res = both(step)
        assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(1), t.clone())[1], lambda t: t):
        a, b = x.detach().requires_grad_(), data.detach().requires_grad_()
        y = mortar_amd.stk_dds(a, b, *rest)
    y.backward(dy)
    assert len(packed) == 8 and b.grad is not None
    a, b = x.detach().clone().requires_grad_(), data.detach().clone().requires_grad_()
    y = mortar_amd.stk_dds(a * 1, b, *rest)
    with torch.no_grad():
        b.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy)


def test_dds_native_second_order(dev, took):
    """A gradient that autograd records again goes through the operators: dx is differentiable in dy, as the operator's is."""
    x, data, dy, rest = _operands(dev, 20, 64, 96, True)
    def step():
        a, v = x.detach().requires_grad_(), dy.detach().requires_grad_()
        (dx,) = torch.autograd.grad(mortar_amd.stk_dds(a, data, *rest), a, v, create_graph=True)
        (dv,) = torch.autograd.grad(dx, v, x)
        return dx.detach(), dv
    res = both(step)
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])


def test_dds_general_path_where_something_looks_on(dev, took):
    from torch.utils._python_dispatch import TorchDispatchMode
    x, data, dy, rest = _operands(dev, 20, 64, 96, True)
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    want = general(lambda: mortar_amd.stk_dds(x, data, *rest))()
    with Mode():
        y = mortar_amd.stk_dds(x, data, *rest)
    assert torch.equal(y, want) and any("mortar_amd.dds" in s for s in seen) and not took
    compiled = torch.compile(lambda a, b: mortar_amd.stk_dds(a, b, *rest) * 2, backend="aot_eager", fullgraph=True)
    a, b = x.detach().requires_grad_(), data.detach().requires_grad_()
    y = compiled(a, b)
    assert torch.equal(y, want * 2) and not took
    y.backward(dy)
    assert a.grad is not None and b.grad is not None
    for bad in (lambda: mortar_amd.stk_dds(x, data, *rest[:1], rest[1].int(), *rest[2:]), lambda: mortar_amd.stk_dds(x[:, :48], data, *rest)):
        with pytest.raises((ValueError, AssertionError)):
            bad()
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level():
        dual = fwAD.make_dual(x, torch.ones_like(x))
        try:
            mortar_amd.stk_dds(dual, data, *rest)
        except Exception:
            pass
    assert not took
    with torch.inference_mode():
        assert torch.equal(mortar_amd.stk_dds(x, data, *rest), want)
    assert took == ["dds"]
    assert torch.equal(mortar_amd.stk_dds(x.float(), data, *rest).bfloat16(), want) and took == ["dds"]


@pytest.mark.parametrize("M", [1, 70, 600])
@pytest.mark.parametrize("need", [(True, True, True), (False, True, True), (True, False, False), (False, False, True), (False, True, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_train_step_native_is_the_general_one(dev, took, monkeypatch, M, need, dtype):
    spec = synth.synth_mlp(64, 176, 0.3, seed=3)
    g = torch.Generator(device=dev).manual_seed(1)
    x0 = torch.randn(M, 64, generator=g, device=dev).to(torch.bfloat16)
    dy = torch.randn(M, 64, generator=g, device=dev).to(torch.bfloat16)
    res = []
    for native in (True, False):
        mlp = synth.qat_mlp_module(spec, dev, seed=5).to(dtype)
        data = [mlp.gate_up._cms.mortar_data, mlp.down._cms.mortar_data]
        for p, r in zip(data, need[1:]):
            p.requires_grad_(r)
        if not native:
            monkeypatch.setattr("mortar_amd.mlp._native_step", lambda *a: None)
            monkeypatch.setattr("mortar_amd.mlp._native_step_backward", lambda *a: None)
        out = []
        for step in range(2):                     # the second one on values written through .data
            x = x0.detach().requires_grad_(need[0])
            y = mlp(x.view(1, M, 64)).view(M, 64)
            y.backward(dy, retain_graph=True)
            out += [y.detach(), x.grad] + [p.grad for p in data]
            for p in data:
                p.grad = None
                p.data.mul_(-1.5)
        res.append(out)
    assert took == ["train_forward", "train_backward"] * 2
    for got, want in zip(*res):
        assert (got is None) == (want is None) and (got is None or torch.equal(got, want))


def test_train_step_after_the_values_have_changed(dev, took):
    """Values that change between forward and backward (version counter) are re-packed by the general backward, as before."""
    mlp = synth.qat_mlp_module(synth.synth_mlp(64, 176, 0.3, seed=3), dev, seed=5)
    x = torch.randn(70, 64, device=dev).to(torch.bfloat16).requires_grad_()
    y = mlp(x)
    with torch.no_grad():
        mlp.down._cms.mortar_data.neg_()
    y.sum().backward()
    assert took == ["train_forward"]
    want = mlp(x.detach().requires_grad_())
    assert torch.equal(want, -y) and x.grad is not None


def test_train_step_that_failed_leaves_no_stale_weights(dev, took):
    """The re-pack refuses a negative threshold, behind the point where the step's packs were handed out: the next inference call
    multiplies the values as they are, not those of the last pack, and the next step is a native one again."""
    mlp = synth.qat_mlp_module(synth.synth_mlp(64, 176, 0.3, seed=3), dev, seed=5)
    x = torch.randn(70, 64, device=dev).to(torch.bfloat16)
    layers = [mlp.gate_up._cms, mlp.down._cms]
    mlp(x.requires_grad_()).sum().backward()
    for m in layers:
        m._values_threshold = -1.0
    with torch.no_grad():
        mlp.down._cms.mortar_data.neg_()
    with pytest.raises(ValueError, match="threshold"):
        mlp(x)
    for m in layers:
        m._values_threshold = 0.5
        m.mortar_data.requires_grad_(False)           # an inference call re-packs by the key alone
    with torch.no_grad():
        y = mlp(x)
    for m in layers:
        m.invalidate_pack()
    with torch.no_grad():
        assert torch.equal(y, mlp(x))
    for m in layers:
        m.mortar_data.requires_grad_(True)
    assert mlp(x).requires_grad and took.count("train_forward") == 2


def test_the_scales_of_a_step_stay_as_they_were(dev, took):
    """Every step hands out scale tensors of its own: what a caller kept of step N does not change in step N + 1."""
    mlp = synth.qat_mlp_module(synth.synth_mlp(64, 176, 0.3, seed=3), dev, seed=5)
    layers = [mlp.gate_up._cms, mlp.down._cms]
    x = torch.randn(70, 64, device=dev).to(torch.bfloat16).requires_grad_()
    kept = []
    for step in range(3):
        mlp(x)
        kept.append([m._pack.scales_f32 for m in layers])
        for m, s in zip(layers, kept[-1]):
            assert m._pack_scale is s is m._pack._transposed.scales_f32
            m.mortar_data.data.mul_(2)
    assert took == ["train_forward"] * 3
    for step in (1, 2):
        for first, s in zip(kept[0], kept[step]):
            assert torch.equal(s, first * 2 ** step)           # a power of two scales every sum exactly
