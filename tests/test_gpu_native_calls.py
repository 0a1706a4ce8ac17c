"""The native call layer (csrc/mortar_torch.cpp) against the general Python path of the same modules: same bits where both
serve a call, and the general path where the layer declines."""
import numpy as np
import pytest
import torch

import mortar_amd
from mortar_amd import _lib, ops, synth
from mortar_amd.engine import MortarDecodeMLP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d_model,d_ff", [(256, 16 * 44), (16 * 160, 16 * 20)])         # norm fused into gate_up / in its own launch
@pytest.mark.parametrize("M", [1, 4, 16, 17, 64, 65, 203])
def test_module_and_decode_calls_equal_the_general_path(dev, d_model, d_ff, M):
    mlp = synth.mlp_module(synth.synth_mlp(d_model, d_ff, 0.25, seed=3), dev)
    x = torch.randn(M, d_model, device=dev).to(torch.bfloat16)
    w = torch.rand(d_model, device=dev).to(torch.bfloat16)
    assert mlp.native_pair() is None                                       # nothing packed yet: the first call packs
    first = mlp(x)
    assert mlp.native_pair() is not None
    h = ops.gateup_swiglu(x, mlp.gate_up._cms.mortar_pack())
    y = ops.spmm(h, mlp.down._cms.mortar_pack())
    assert torch.equal(first, y) and torch.equal(mlp(x), y)
    assert torch.equal(mlp(x.view(1, M, d_model)), y.view(1, M, d_model))
    strided = torch.zeros(M, d_model + 8, device=dev, dtype=torch.bfloat16)
    strided[:, :d_model] = x
    assert torch.equal(mlp(strided[:, :d_model]), y)                       # declined (not contiguous)
    xf = x.float()
    assert torch.equal(mlp(xf), y.float())                                 # declined (another dtype)
    xn = ops.rmsnorm(x, w, 1e-5)
    yn = ops.spmm(ops.gateup_swiglu(xn, mlp.gate_up._cms.mortar_pack()), mlp.down._cms.mortar_pack())
    assert torch.equal(mlp(x, norm=(w, 1e-5)), yn)
    dec = MortarDecodeMLP(mlp, norm_weight=w, eps=1e-5)
    assert torch.equal(dec(x), yn.view(M, 1, -1)) and torch.equal(dec._general(x), yn.view(M, 1, -1))
    mlp.to(dev)                                                            # drops the packs: the next call builds new ones
    assert mlp.native_pair() is None and torch.equal(mlp(x), y)


@pytest.mark.parametrize("B", [1, 5, 64, 65])
@pytest.mark.parametrize("n_clusters", [4, 44])
def test_routed_decode_call_equals_the_general_path(dev, B, n_clusters):
    mlp = synth.mlp_module(synth.synth_mlp(256, 16 * 44, 0.25, seed=4), dev)
    torch.manual_seed(1)
    mlp.enable_routing(n_clusters=n_clusters, activation_ratio=0.5, n_iters=2)
    with torch.no_grad():
        mlp.router.iter_embed.normal_()
    dec = MortarDecodeMLP(mlp, norm_weight=torch.rand(256, device=dev).to(torch.bfloat16), iter_idx=1)
    x = torch.randn(B, 256, device=dev).to(torch.bfloat16)
    y, ref = dec(x), dec._general(x)
    assert torch.allclose(y.float(), ref.float(), rtol=1e-2, atol=1e-2 * ref.float().abs().max().item())
    with torch.no_grad():
        mlp.router.query_proj.weight = torch.nn.Parameter(mlp.router.query_proj.weight.flip(0).contiguous())      # a replaced parameter is seen
    y2, ref2 = dec(x), dec._general(x)
    assert torch.allclose(y2.float(), ref2.float(), rtol=1e-2, atol=1e-2 * ref2.float().abs().max().item())


@pytest.mark.parametrize("K_blocks,seg", [(3, None), (48, None), (352, None), (352, 40), (704, None), (1376, None)])   # every token tile, 1 .. 9 parts
@pytest.mark.parametrize("B", [1, 2, 4, 5, 6, 11])
def test_one_launch_fp32_decode_product(dev, K_blocks, seg, B):
    """mortar_gemv on a one-scale matrix against float64: plain and SwiGLU-on-load products with per-stream flags, and the
    gated gate_up form."""
    m = synth.synth_matrix(16 * 10, 16 * K_blocks, 0.25, seed=K_blocks, per_tensor_scale=True)
    W = mortar_amd.MortarPack(synth.flat_pack(m["codes"]), m["scales"], m["col_idx"], m["offsets"], *m["shape"], dev, seg_cb=seg)
    dense = torch.zeros(10, K_blocks, 16, 16, dtype=torch.float64, device=dev)
    dense[torch.from_numpy(m["row_idx"]).long(), torch.from_numpy(m["col_idx"]).long()] = torch.from_numpy(m["codes"]).to(dev).double()
    dense = dense.permute(0, 2, 1, 3).reshape(160, -1) * float(m["scales"][0])
    g = torch.Generator(device=dev).manual_seed(B)
    K = 16 * K_blocks
    x2 = torch.randn(B, 2 * K, device=dev, generator=g)
    x = x2[:, :K].contiguous()
    ca = (torch.rand(B, K_blocks, device=dev, generator=g) < 0.6).int()
    ra = (torch.rand(B, 10, device=dev, generator=g) < 0.6).int()
    ra[:, 3] = 0                                                             # off for every stream

    def close(got, want):
        assert (got.double() - want).abs().max() <= 3e-6 * want.abs().max().clamp(min=1e-30) + 1e-12

    close(mortar_amd.mortar_gemv(x, W), x.double() @ dense.t())
    on = ca.repeat_interleave(16, 1).double()
    want = (x.double() * on) @ dense.t() * ra.repeat_interleave(16, 1)
    close(mortar_amd.mortar_gemv(x, W, row_act=ra, col_act=ca), want)
    h = torch.nn.functional.silu(x2[:, :K].double()) * x2[:, K:].double()
    close(mortar_amd.mortar_gemv(x2, W, swiglu_x=True), h @ dense.t())
    gates = torch.relu(torch.randn(B, 5, device=dev, generator=g))
    gates[:, 2] = 0
    gu = x.double() @ dense.t()
    want = torch.nn.functional.silu(gu[:, :80]) * gu[:, 80:] * gates.double().repeat_interleave(16, 1)
    got = mortar_amd.mortar_gemv(x, W, swiglu_out=True, gates=gates)
    assert torch.allclose(got.double(), want, rtol=1e-4, atol=1e-5 * want.abs().max().item() + 1e-12)


@pytest.mark.parametrize("flag", [1, np.True_, torch.tensor(True)])
def test_fp32_decode_product_takes_any_true_flag(dev, flag):
    m = synth.synth_matrix(16 * 4, 16 * 8, 0.5, seed=9, per_tensor_scale=True)
    W = synth.to_pack(m, dev)
    x = torch.randn(3, 256, device=dev)
    assert torch.equal(mortar_amd.mortar_gemv(x, W, swiglu_x=flag), mortar_amd.mortar_gemv(x, W, swiglu_x=True))
    x = x[:, :128].contiguous()
    h = mortar_amd.mortar_gemv(x, W, swiglu_out=flag)
    assert h.shape == (3, 32) and torch.equal(h, mortar_amd.mortar_gemv(x, W, swiglu_out=True))


@pytest.mark.parametrize("out_b,K_blocks,B,better", [(10, 1700, 1, 0), (10, 1700, 5, 0), (10, 1700, 22, 0),      # no tile of all K
                                                     (256, 688, 32, 1), (256, 688, 33, 0),                     # four rounds of workgroups, five
                                                     (512, 192, 60, 1), (512, 192, 61, 0), (512, 192, 64, 0)])  # SwiGLU form: three rounds, four
def test_fp32_decode_product_on_either_side_of_the_one_launch_form(dev, out_b, K_blocks, B, better):
    """mortar_gemv of one-scale matrices where the three launches on the SpMM kernels take over from the one: against float64."""
    swiglu = out_b == 512
    m = synth.synth_matrix(16 * out_b, 16 * K_blocks, 0.1, seed=K_blocks, per_tensor_scale=True)
    W = synth.to_pack(m, dev)
    assert _lib.lib().mortar_gemv_f32_one_better(W.ref, int(swiglu), B) == better
    dense = torch.zeros(out_b, K_blocks, 16, 16, dtype=torch.float64, device=dev)
    dense[torch.from_numpy(m["row_idx"]).long(), torch.from_numpy(m["col_idx"]).long()] = torch.from_numpy(m["codes"]).to(dev).double()
    dense = dense.permute(0, 2, 1, 3).reshape(16 * out_b, -1) * float(m["scales"][0])
    g = torch.Generator(device=dev).manual_seed(B)
    K = 16 * K_blocks
    x2 = torch.randn(B, 2 * K, device=dev, generator=g)
    x = x2[:, :K].contiguous()
    ca = (torch.rand(B, K_blocks, device=dev, generator=g) < 0.6).int()
    ra = (torch.rand(B, out_b, device=dev, generator=g) < 0.6).int()

    def close(got, want):
        assert (got.double() - want).abs().max() <= 3e-6 * want.abs().max()

    on = (x.double() * ca.repeat_interleave(16, 1)) @ dense.t() * ra.repeat_interleave(16, 1)
    if not swiglu:
        close(mortar_amd.mortar_gemv(x, W), x.double() @ dense.t())
        close(mortar_amd.mortar_gemv(x, W, row_act=ra, col_act=ca), on)
        close(mortar_amd.mortar_gemv(x2, W, swiglu_x=True), (torch.nn.functional.silu(x2[:, :K].double()) * x2[:, K:].double()) @ dense.t())
        return
    gates = torch.relu(torch.randn(B, 16, device=dev, generator=g))
    f = 8 * out_b
    want = torch.nn.functional.silu(on[:, :f]) * on[:, f:] * gates.double().repeat_interleave(f // 16, 1)
    close(mortar_amd.mortar_gemv(x, W, swiglu_out=True, gates=gates, row_act=ra, col_act=ca), want)


@pytest.mark.parametrize("units,in_b,density", [(37, 128, 0.3), (257, 128, 0.3), (511, 128, 0.05), (513, 128, 0.3),     # one, two, two, four units a workgroup
                                                (37, 352, 0.3), (259, 352, 0.03)])
@pytest.mark.parametrize("B", [1, 5, 9])
def test_fp32_decode_products_of_few_units(dev, units, in_b, density, B):
    """Row parts cut over many waves, odd numbers of units, parts of less than an octet: plain and SwiGLU forms against float64."""
    x = torch.randn(B, 16 * in_b, device=dev, generator=torch.Generator(device=dev).manual_seed(B))
    for rows in (units, 2 * units):
        m = synth.synth_matrix(16 * rows, 16 * in_b, density, seed=63, per_tensor_scale=True)
        W = synth.to_pack(m, dev)
        dense = torch.zeros(rows, in_b, 16, 16, dtype=torch.float64, device=dev)
        dense[torch.from_numpy(m["row_idx"]).long(), torch.from_numpy(m["col_idx"]).long()] = torch.from_numpy(m["codes"]).to(dev).double()
        want = x.double() @ (dense.permute(0, 2, 1, 3).reshape(16 * rows, -1) * float(m["scales"][0])).t()
        assert (mortar_amd.mortar_gemv(x, W).double() - want).abs().max() <= 3e-6 * want.abs().max()      # fp32 sums of up to 1700 exact terms
        if rows == 2 * units:
            f = 16 * units
            h = torch.nn.functional.silu(want[:, :f]) * want[:, f:]
            assert torch.allclose(mortar_amd.mortar_gemv(x, W, swiglu_out=True).double(), h, rtol=1e-4, atol=1e-5 * h.abs().max().item())


@pytest.mark.parametrize("units,in_b,density,zipf", [(1, 2, 1.0, None), (5, 9, 0.3, None), (37, 128, 0.25, None), (37, 128, 0.2, 1.3), (130, 200, 0.05, None),
                                                     (9, 352, 0.25, 1.2), (64, 352, 0.02, None), (3, 620, 0.25, None),
                                                     (350, 100, 0.04, None), (128, 48, 0.25, None)])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 33])
@pytest.mark.parametrize("one_scale", [False, True])
def test_decode_products_of_few_units(dev, units, in_b, density, zipf, M, one_scale):
    """Row parts cut into chunks over many waves: one to four K segments, parts of less than an octet and ragged ones, odd numbers of
    units, rows past the tile, both scale forms, clusters that are off, against float64."""
    K = 16 * in_b
    x = synth.synth_x(M, K, 61)
    xd = torch.from_numpy(x).to(torch.bfloat16).to(dev)
    xf = xd.double().cpu()

    def product(m):
        w = np.zeros((m["shape"][0], K))
        s = m["scales"].astype(np.float64) if m["scales"].size > 1 else np.full(m["col_idx"].size, float(m["scales"][0]))
        s = torch.from_numpy(s).to(torch.bfloat16).double().numpy()
        for j, (r, c) in enumerate(zip(m["row_idx"], m["col_idx"])):
            w[16 * r:16 * r + 16, 16 * c:16 * c + 16] = m["codes"][j] * s[j]
        return xf @ torch.from_numpy(w).t()
    for rows in (units, 2 * units):
        m = synth.synth_matrix(16 * rows, K, density, seed=62, zipf_s=zipf)
        if one_scale:
            m["scales"] = m["scales"][:1]
        W = synth.to_pack(m, dev)
        want = product(m)
        # fp32 sums of K products, rounded once: half a bf16 ulp, and a few ulps of fp32 of the row's largest
        tol = 2.0 ** -8 * want.abs() + 2.0 ** -18 * want.abs().max()
        assert ((ops.spmm(xd, W).double().cpu() - want).abs() <= tol).all()
        if rows == 2 * units:
            gates = torch.rand(M, units, device=dev) * (torch.rand(M, units, device=dev) < 0.4)
            gates[:, 0] = 0
            for g in (None, gates):
                h = ops.gateup_swiglu(xd, W, gates=g)
                gu = ops.spmm(xd, W)
                ref = ops.swiglu(gu).float()
                if g is not None:
                    ref = (ref * g.to(torch.bfloat16).float().repeat_interleave(16, 1)).to(torch.bfloat16).float()
                assert torch.allclose(h.float(), ref, rtol=2.0 ** -6, atol=2.0 ** -7 * float(ref.abs().max()))      # gate, up one ulp apart
            if ops.norm_fusable(W):
                nw = (1 + 0.1 * torch.randn(K, device=dev)).to(torch.bfloat16)
                for w in (nw, None):
                    assert torch.equal(ops.gateup_swiglu(xd, W, norm=(w, 1e-6)), ops.gateup_swiglu(ops.rmsnorm(xd, w, 1e-6), W))


@pytest.mark.parametrize("units,in_b,density", [(1, 3, 1.0), (5, 48, 0.25), (37, 128, 0.25), (48, 128, 0.05), (130, 155, 0.1),
                                                (1, 156, 1.0), (70, 180, 0.2), (37, 352, 0.25), (130, 311, 0.03), (9, 700, 0.1)])
@pytest.mark.parametrize("M", [65, 96, 97, 250, 512, 700])
@pytest.mark.parametrize("one_scale", [False, True])
def test_mid_sized_products(dev, units, in_b, density, M, one_scale):
    """Up to 155 block-columns: 32-token tiles with a unit on one, two or four waves (65 rows up to one round of the chip); beyond: several K
    segments through two buffers (up to 512 rows).  Remainders of tiles, segments and units, parts of less than an octet, the widest tile
    and segment, both scale forms, gates, input mask and norm, against float64."""
    K = 16 * in_b
    xd = torch.from_numpy(synth.synth_x(M, K, 71)).to(torch.bfloat16).to(dev)
    for rows in (units, 2 * units):
        m = synth.synth_matrix(16 * rows, K, density, seed=72, zipf_s=1.1)
        if one_scale:
            m["scales"] = m["scales"][:1]
        W = synth.to_pack(m, dev)
        w = torch.zeros(16 * rows, K, dtype=torch.float64)
        s = torch.from_numpy(np.broadcast_to(m["scales"], m["col_idx"].shape).copy()).to(torch.bfloat16).double()
        for j, (r, c) in enumerate(zip(m["row_idx"], m["col_idx"])):
            w[16 * r:16 * r + 16, 16 * c:16 * c + 16] = torch.from_numpy(m["codes"][j]).double() * s[j]
        want = (xd.double() @ w.to(dev).t())
        tol = 2.0 ** -8 * want.abs() + 2.0 ** -18 * want.abs().max()       # one bf16 rounding of an fp32 sum
        assert ((ops.spmm(xd, W).double() - want).abs() <= tol).all()
        act = torch.randint(0, 2, (M, in_b), dtype=torch.uint8, device=dev)
        assert torch.equal(ops.spmm(xd, W, active=act), ops.spmm(xd * act.repeat_interleave(16, 1).to(xd.dtype), W))
        if rows == 2 * units:
            gates = torch.rand(M, units, device=dev) * (torch.rand(M, units, device=dev) < 0.4)
            gu = want.float().to(torch.bfloat16).float()
            ref = (torch.nn.functional.silu(gu[:, :16 * units]) * gu[:, 16 * units:])
            for g in (None, gates):
                r = ref if g is None else ref * g.repeat_interleave(16, 1)
                # four bf16 roundings (gate_up, silu, product, gated product) of 2^-9 each, silu's slope up to 1.1
                assert torch.allclose(ops.gateup_swiglu(xd, W, gates=g).float(), r, rtol=2.0 ** -6, atol=2.0 ** -9 * float(r.abs().max()))
            if ops.norm_fusable(W):
                nw = (1 + 0.1 * torch.randn(K, device=dev)).to(torch.bfloat16)
                assert torch.equal(ops.gateup_swiglu(xd, W, norm=(nw, 1e-6)), ops.gateup_swiglu(ops.rmsnorm(xd, nw, 1e-6), W))


@pytest.mark.parametrize("d,nsk,n", [(8, 2, 4), (264, 4, 16), (1024, 4, 16), (1032, 19, 352), (2048, 4, 16), (2056, 4, 16)])      # one wave's piece, ragged, both widths, too wide
@pytest.mark.parametrize("B", [1, 2, 4, 5, 16, 17, 33, 64])
@pytest.mark.parametrize("weight", [True, False])
def test_router_with_the_norm_inside_gives_the_bits_of_both_launches(dev, d, nsk, n, B, weight):
    g = torch.Generator(device=dev).manual_seed(B)
    rand = lambda *s: torch.randn(*s, device=dev, generator=g)
    x = (3 * rand(B, d)).to(torch.bfloat16)
    nw = (1 + 0.1 * rand(d)).to(torch.bfloat16) if weight else None
    wq, it, lnw, lnb, bias = rand(d, d) / d ** 0.5, rand(d), rand(d), rand(d), rand(n)
    ka, kb = rand(nsk, d // 2), rand(nsk, d // 2)
    want_x = ops.rmsnorm(x, nw, 1e-5)
    outs = []
    for fused in (False, True):
        xn = torch.full((B + 1, d), 7.0, dtype=torch.bfloat16, device=dev)
        qv, gates = torch.empty(B, d, device=dev), torch.empty(B, n, device=dev)
        p = lambda t: None if t is None else t.data_ptr()
        tail = (p(wq), p(it), p(lnw), p(lnb), 1e-5, p(ka), p(kb), nsk, p(bias), n, max(1, n // 4), p(qv), None, p(gates), None,
                torch.cuda.current_stream().cuda_stream)
        if fused:
            _lib.check(_lib.lib().mortar_norm_router_bf16(p(x), B, d, d, p(nw), 1e-5, p(xn), *tail), "norm_router")
            assert torch.equal(xn[:B], want_x) and (xn[B] == 7).all()
        else:
            _lib.check(_lib.lib().mortar_router_bf16(p(want_x), 0, B, d, d, *tail), "router")
        outs.append((qv, gates))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
