"""Decode calls of wide models: the RMSNorm inside gate_up beyond 2048 values, the stand-alone norm with its rows in registers, and `down`
rows that fit no 8-token tile."""
import numpy as np
import pytest
import torch

import mortar_amd
from mortar_amd import _lib, ops, synth
from oracle import mortar_oracle as O
from util import assert_close_bf16, oracle_spmm, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,d", [(1, 8), (5, 1016), (3, 1024), (1025, 1032), (2, 2056), (1, 4096), (3, 4104), (2, 8192), (2, 8200)])
def test_rmsnorm_widths(dev, M, d):
    x = O.bf16_round(synth.synth_x(M, d, 90) * 3)
    w = O.bf16_round(1.0 + 0.1 * synth.synth_x(1, d, 91)[0])
    assert_close_bf16(to_np(ops.rmsnorm(to_dev(x, dev), to_dev(w, dev))), O.rmsnorm(x, w), "rmsnorm", ulps=2)


@pytest.mark.parametrize("M,d", [(1100, 512), (1030, 504), (4096, 2048), (6200, 1024), (8703, 1024), (4099, 1536), (4500, 2048), (4096, 2056)])
@pytest.mark.parametrize("weight", [False, True])
def test_rmsnorm_of_many_rows_has_the_bits_of_few(dev, M, d, weight):
    """Calls of 12 to 17 MB run another form than smaller and larger ones, and calls of few rows."""
    g = torch.Generator(device=dev).manual_seed(d)
    x = (torch.randn(M, d, device=dev, generator=g) * 2).bfloat16()
    w = torch.randn(d, device=dev, generator=g).bfloat16() if weight else None
    want = torch.cat([ops.rmsnorm(c, w) for c in x.split(500)])
    assert torch.equal(ops.rmsnorm(x, w), want)


# d_ff / 16 units: one or two per workgroup with the parts in chunks, four, eight (from 9 rows)
@pytest.mark.parametrize("d,units", [(2512, 24), (2560, 300), (4096, 30), (4096, 560), (3072, 512)])
@pytest.mark.parametrize("one_scale", [False, True])
def test_wide_norm_has_the_bits_of_the_separate_one(dev, d, units, one_scale):
    spec = synth.synth_mlp(d, 16 * units, 0.1, seed=d + units, zipf_s=1.2)
    if one_scale:
        for k in ("gate_up", "down"):
            spec[k]["scales"][:] = spec[k]["scales"][0]
    mlp = synth.mlp_module(spec, dev)
    W = mlp.gate_up._cms.mortar_pack()
    assert not ops.norm_fusable(W)
    w = to_dev(O.bf16_round(1.0 + 0.1 * synth.synth_x(1, d, 3)[0]), dev)
    for nw in (w, None):
        call = mortar_amd.MortarDecodeMLP(mlp, norm_weight=nw)
        for M in (1, 3, 4, 5, 8, 9, 16, 17, 40, 64):
            x = to_dev(O.bf16_round(synth.synth_x(M, d, M) * 2.5), dev)
            xn = ops.rmsnorm(x, nw, call.eps)
            assert torch.equal(call(x).view(M, d), ops.mlp(xn, W, mlp.down._cms.mortar_pack())), (M, nw is None)
            h = torch.full((M + 1, 16 * units), float("nan"), device=dev, dtype=torch.bfloat16)
            rc = _lib.lib().mortar_norm_gateup_decode_bf16(W.ref, W.sched(2).data_ptr(), x.data_ptr(), M, d, nw.data_ptr() if nw is not None else None,
                                                           call.eps, h.data_ptr(), 16 * units, torch.cuda.current_stream().cuda_stream)
            assert rc == 0 if M <= 16 else rc in (0, -100)
            if rc == 0:
                assert torch.equal(h[:M], ops.gateup_swiglu(xn, W)) and torch.isnan(h[M].float()).all()


@pytest.mark.parametrize("M", [17, 32, 33, 49, 64])
@pytest.mark.parametrize("masked", [False, True])
def test_down_of_a_wide_model(dev, M, masked):
    # (256 rows of blocks: from 33 rows on more 4-token tiles than are worth it)
    m = synth.synth_matrix(4096, 16 * 620, 0.1, seed=M, zipf_s=1.2)
    W = synth.to_pack(m, dev)
    x = synth.synth_x(M, 9920, seed=M)
    active = None
    if masked:
        on = np.random.default_rng(M).random((M, 155)) < 0.4
        x = x * np.repeat(on, 64, axis=1)
        active = torch.from_numpy(on.astype(np.uint8)).to(dev)
    buf = torch.full((M + 1, 4096), float("nan"), device=dev, dtype=torch.bfloat16)
    ops.spmm(to_dev(x, dev), W, out=buf[:M], **({"active": active} if masked else {}))
    assert torch.isnan(buf[M].float()).all()
    assert_close_bf16(to_np(buf[:M]), oracle_spmm(x, m), "down")


# K beyond an 8-token tile of all of it: 4-token tiles and, from more of them than are worth it, the two-buffer kernel
@pytest.mark.parametrize("Rb,M", [(256, 16), (256, 32), (256, 33), (256, 64), (320, 25), (520, 17)])
@pytest.mark.parametrize("one_scale", [False, True])
@pytest.mark.parametrize("masked", [False, True])
def test_post_write_of_a_wide_down_has_the_bits_of_the_product(dev, Rb, M, one_scale, masked):
    m = synth.synth_matrix(16 * Rb, 16 * 688, 0.25, seed=Rb + M, zipf_s=1.2)      # rows long enough for another order of additions to show
    if one_scale:
        m["scales"][:] = m["scales"][0]
    W = synth.to_pack(m, dev)
    x = to_dev(synth.synth_x(M, 11008, seed=M), dev)
    g = torch.Generator(device=dev).manual_seed(M)
    kw = {"active": (torch.rand(M, 172, device=dev, generator=g) < 0.4).to(torch.uint8)} if masked else {}
    y = ops.spmm(x, W, **kw).float()
    for n, dt in ((1, torch.bfloat16), (4, torch.float32)):
        h = torch.randn(M, n, 16 * Rb, device=dev, generator=g).to(dt)
        one, zero = torch.ones(M, n, device=dev), torch.zeros(M, n, n, device=dev)
        out = ops.spmm_hc_post(x, W, h, zero, one, **kw)
        assert torch.equal(out.float(), y[:, None, :].expand(M, n, 16 * Rb))
        res, post = torch.randn(M, n, n, device=dev, generator=g), torch.randn(M, n, device=dev, generator=g)
        got = ops.spmm_hc_post(x, W, h, res, post, h[:, 0].contiguous(), **kw).double()
        terms = (res.double()[..., None] * h.double()[:, None]).sum(2), post.double()[..., None] * y.double()[:, None], h.double()[:, :1]
        size = (res.double().abs()[..., None] * h.double().abs()[:, None]).sum(2) + terms[1].abs() + terms[2].abs()
        # six roundings to fp32 of sums no larger than `size`, and the one of the result
        assert ((got - sum(terms)).abs() <= size * 6 * 2.0 ** -24 + got.abs() * (2.0 ** -8 if dt == torch.bfloat16 else 0.0)).all()
