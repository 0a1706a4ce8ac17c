"""The prefill router's own kernels: projection on the matrix cores, score and rank launches, load statistics."""
import pytest
import torch

from mortar_amd import _lib, ops
from mortar_amd.routing import TileRouter

pytestmark = pytest.mark.gpu


def _project(x, w):
    qv = torch.full((x.shape[0], w.shape[0]), float("nan"), device=x.device)
    _lib.check(_lib.lib().mortar_router_project_bf16(x.data_ptr(), x.shape[0], x.shape[1], x.stride(0), w.data_ptr(), w.shape[0], qv.data_ptr(),
                                                     qv.stride(0), torch.cuda.current_stream().cuda_stream), "project")
    return qv


@pytest.mark.parametrize("M", [1, 63, 65, 129, 257, 1000, 4097])          # each token tile of the dispatch, whole and ragged
@pytest.mark.parametrize("d_in,d_out", [(8, 4), (72, 136), (256, 260), (2048, 2048)])
def test_projection_has_fp32_accuracy(dev, M, d_in, d_out):
    g = torch.Generator(device=dev).manual_seed(M + d_in)
    x = torch.randn(M, d_in, device=dev, generator=g).to(torch.bfloat16)
    w = torch.randn(d_out, d_in, device=dev, generator=g) * 0.05
    qv = _project(x, w).double()
    ref = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * 2.0 ** -22           # fp32 sums of exact products
    assert ((qv - ref).abs() <= bound).all(), (qv - ref).abs().max().item()


@pytest.mark.parametrize("M", [65, 129, 300])                             # the kernel that shares K: whole and ragged K, outputs, token groups
@pytest.mark.parametrize("d_in,d_out", [(1000, 1024), (1032, 260), (2040, 2044)])
def test_shared_k_projection_has_fp32_accuracy(dev, M, d_in, d_out):
    test_projection_has_fp32_accuracy(dev, M, d_in, d_out)


@pytest.mark.parametrize("B", [5, 16, 17, 33, 64])
@pytest.mark.parametrize("d", [8, 136, 1032, 2040])
def test_decode_projection_on_the_matrix_cores(dev, B, d):
    g = torch.Generator(device=dev).manual_seed(B + d)
    x = torch.randn(B, d + 8, device=dev, generator=g).to(torch.bfloat16)[:, :d]
    w, iv = torch.randn(d, d, device=dev, generator=g) * 0.05, torch.randn(d, device=dev, generator=g)
    qv, gates = torch.full((B, d), float("nan"), device=dev), torch.empty(B, 4, device=dev)
    one, keys = torch.ones(d, device=dev), torch.randn(2, 2, d // 2, device=dev, generator=g)
    for bias in (None, iv):
        rc = _lib.lib().mortar_router_bf16(x.data_ptr(), 0, B, d, x.stride(0), w.data_ptr(), bias.data_ptr() if bias is not None else None,
                                           one.data_ptr(), one.data_ptr(), 1e-5, keys[0].data_ptr(), keys[1].data_ptr(), 2, one.data_ptr(), 4, 2,
                                           qv.data_ptr(), None, gates.data_ptr(), None, torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "router")
        ref = x.double() @ w.double().t() + (0 if bias is None else iv.double())
        bound = (x.double().abs() @ w.double().abs().t() + iv.double().abs()) * 2.0 ** -22
        assert ((qv.double() - ref).abs() <= bound).all(), (qv.double() - ref).abs().max().item()


def test_projection_is_exact_on_small_integers(dev):
    x = torch.randint(-8, 9, (300, 128), device=dev).to(torch.bfloat16)
    w = torch.randint(-2 ** 15, 2 ** 15, (96, 128), device=dev).float()       # needs two of the three terms; every sum fits 24 bits
    assert torch.equal(_project(x, w).double(), x.double() @ w.double().t())


@pytest.mark.parametrize("M,n", [(1, 2), (31, 16), (65, 352), (4097, 1024)])
def test_load_statistics(dev, M, n):
    gates = torch.relu(torch.randn(M, n, device=dev))
    ema = torch.rand(n, device=dev)
    want = ema * 0.99 + (gates > 0).float().mean(0) * 0.01
    aux = torch.empty((), device=dev)
    L = _lib.lib()
    ws = torch.empty(L.mortar_router_stats_workspace_bytes(M, n), dtype=torch.uint8, device=dev)
    _lib.check(L.mortar_router_stats(gates.data_ptr(), M, n, 0.99, 0.01, 0.5, ema.data_ptr(), aux.data_ptr(), ws.data_ptr(),
                                     torch.cuda.current_stream().cuda_stream), "stats")
    assert torch.allclose(ema, want, rtol=1e-6, atol=1e-7)
    assert torch.allclose(aux.double(), 0.5 * gates.double().mean(0).var(), rtol=1e-4, atol=1e-9)


@pytest.mark.parametrize("N,d,nsk,n", [(65, 8, 4, 16), (66, 136, 4, 13), (100, 1032, 16, 256), (130, 2048, 17, 300), (77, 4096, 32, 1024),
                                       (70, 256, 4, 8), (70, 256, 4, 7)])       # (last: fewer groups than scores, the one-launch form)
@pytest.mark.parametrize("iter_vec", [False, True])
def test_tail_against_float64(dev, N, d, nsk, n, iter_vec):
    g = torch.Generator(device=dev).manual_seed(N + d)
    qv = torch.randn(N, d, device=dev, generator=g)
    iv = torch.randn(d, device=dev, generator=g) if iter_vec else None
    lw, lb = torch.rand(d, device=dev, generator=g) + 0.5, torch.randn(d, device=dev, generator=g) * 0.1
    ka, kb = (torch.randn(nsk, d // 2, device=dev, generator=g) * (d // 2) ** -0.5 for _ in range(2))
    bias, k = torch.randn(n, device=dev, generator=g) * 0.1, max(1, n // 3)
    gates, active, logits = ops.router_tail(qv, iv, lw, lb, 1e-5, ka, kb, bias, k, want_logits=True)
    q = torch.nn.functional.layer_norm((qv + iv if iter_vec else qv).double(), (d,), lw.double(), lb.double(), 1e-5)
    ps = ((q[:, :d // 2] @ ka.double().t()).unsqueeze(2) + (q[:, d // 2:] @ kb.double().t()).unsqueeze(1)).reshape(N, -1)
    ref = (ps.topk(n, dim=-1).values if nsk * nsk > n else ps[:, torch.arange(n, device=dev) % (nsk * nsk)]) + bias.double()
    assert torch.allclose(logits.double(), ref, rtol=0, atol=2e-5)
    want = torch.relu(logits - logits.topk(k, dim=-1).values[:, -1:])
    want = want * (k / want.sum(-1, keepdim=True).clamp(min=1e-6))
    assert torch.allclose(gates, want, rtol=1e-4, atol=1e-5)
    assert torch.equal(active.bool(), gates > 0)


@pytest.mark.parametrize("N,d,nsk,n", [(512, 2048, 20, 390), (513, 2048, 20, 390), (2048, 136, 4, 13), (2049, 136, 4, 13), (600, 1032, 16, 256),
                                       (65, 2048, 4, 16), (65, 2056, 4, 16), (66, 768, 21, 441)])     # either side of the one-token workgroups
@pytest.mark.parametrize("iter_vec", [False, True])
def test_tail_dispatch_against_float64(dev, N, d, nsk, n, iter_vec):
    test_tail_against_float64(dev, N, d, nsk, n, iter_vec)


@pytest.mark.parametrize("M", [64, 65, 600])
def test_router_module_call_equals_the_torch_ops(dev, M):
    torch.manual_seed(2)
    rt = TileRouter(44, 256, activation_ratio=0.25, n_iters=2).to(dev)
    with torch.no_grad():
        rt.iter_embed.normal_()
        x = torch.randn(2, M // 2, 256, device=dev).to(torch.bfloat16) if M % 2 == 0 else torch.randn(M, 256, device=dev).to(torch.bfloat16)
        flat = x.reshape(-1, 256)
        want, act = ops.remoe_gates(rt.group_logits(flat, 1), rt.activation_k)
        ema = rt.group_load_ema * 0.99 + act.float().mean(0) * (1 - 0.99)
        gates, aux = rt.forward_native(x, iter_idx=1)
    assert gates.shape == (flat.shape[0], 44) and torch.allclose(gates.reshape(-1, 44), want, rtol=1e-3, atol=1e-4)
    assert torch.allclose(rt.group_load_ema, ema, rtol=1e-3, atol=1e-4) and rt.last_active.shape == (flat.shape[0], 44)
    assert torch.allclose(aux, rt.aux_loss_coeff * want.mean(0).var(), rtol=1e-2)


@pytest.mark.parametrize("M", [3, 300])
def test_load_statistics_are_an_in_place_update_for_torch(dev, M):
    rt = TileRouter(16, 256).to(dev)
    x = torch.randn(M, 256, device=dev).to(torch.bfloat16)
    before = rt.group_load_ema._version
    with torch.no_grad():
        assert rt.forward_native(x) is not None
    assert rt.group_load_ema._version > before
    with torch.inference_mode():
        rt = TileRouter(16, 256).to(dev)
        x = x.clone()
        assert rt.forward_native(x) is not None
    with torch.no_grad(), pytest.raises(RuntimeError, match="[Ii]nference"):      # as any in-place operator on such a buffer
        rt(x)


@pytest.mark.parametrize("M,d_in,d_out", [(65, 136, 260), (300, 1032, 1024), (129, 2048, 136), (1000, 2056, 260), (4097, 72, 132)])
def test_projection_keeps_non_finite_values_to_their_row_and_output(dev, M, d_in, d_out):
    """An infinity or NaN of x makes its row non-finite and no other, one of the weights its output and no other (ragged K
    and tiles included: what is staged past the end must not come in); weights up to the largest float are exact."""
    g = torch.Generator(device=dev).manual_seed(M)
    x = torch.randn(M, d_in, device=dev, generator=g).to(torch.bfloat16)
    w = torch.randn(d_out, d_in, device=dev, generator=g) * 0.05
    ref = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * 2.0 ** -22
    rows, outs = torch.zeros(M, dtype=torch.bool, device=dev), torch.zeros(d_out, dtype=torch.bool, device=dev)
    for r, k, v in ((0, 0, float("inf")), (M - 1, d_in - 1, float("nan")), (M // 2, 0, float("-inf"))):
        x[r, k], rows[r] = v, True
    for o, k, v in ((0, d_in - 1, float("inf")), (d_out - 1, 0, float("nan")), (d_out // 2, 0, float("-inf"))):
        w[o, k], outs[o] = v, True
    qv = _project(x, w)
    hit = rows[:, None] | outs[None, :]
    assert not qv[hit].isfinite().any()
    assert ((qv.double() - ref).abs() <= bound)[~hit].all()
    x = torch.zeros(M, d_in, device=dev, dtype=torch.bfloat16)
    x[:, d_in - 1] = 2.0 ** -8
    w = torch.full((d_out, d_in), torch.finfo(torch.float32).max, device=dev)
    assert torch.equal(_project(x, w), (w[:, -1] * 2.0 ** -8).expand(M, -1))


@pytest.mark.parametrize("nsk", [2, 11, 12, 16, 17, 19, 20, 22, 23, 32])       # 2, 4, 6, 8 and 16 keys per lane, the smallest and largest of each
@pytest.mark.parametrize("N", [3, 530])                                      # a workgroup per token, a wave per token
def test_ranked_products_are_the_sorted_direct_ones(dev, nsk, N):
    """The logits of P - 1 groups under P = nsk^2 product keys against those of P groups, sorted: the same sums, bit for bit."""
    d, P = 64, nsk * nsk
    g = torch.Generator(device=dev).manual_seed(nsk)
    qv = torch.randn(N, d, device=dev, generator=g)
    qv[0] = 0                                                                # exact ties
    ka, kb = (torch.randn(nsk, d // 2, device=dev, generator=g) for _ in range(2))
    one, zero = torch.ones(d, device=dev), torch.zeros(max(d, P), device=dev)

    def logits(n):
        out, gates = torch.empty(N, n, device=dev), torch.empty(N, n, device=dev)
        _lib.check(_lib.lib().mortar_router_tail_f32(qv.data_ptr(), N, d, d, None, one.data_ptr(), zero.data_ptr(), 1e-5, ka.data_ptr(), kb.data_ptr(), nsk,
                                                     zero.data_ptr(), n, 1, out.data_ptr(), gates.data_ptr(), None,
                                                     torch.cuda.current_stream().cuda_stream), "tail")
        return out
    assert torch.equal(logits(P - 1), logits(P).sort(-1, descending=True).values[:, :P - 1])


@pytest.mark.parametrize("n", [1, 2, 3, 16, 31, 32, 33, 64])
def test_gates_of_few_groups_with_ties(dev, n):
    g = torch.Generator(device=dev).manual_seed(n)
    logits = torch.randint(-3, 4, (67, n), device=dev, generator=g).float()
    logits[1] = torch.randn(n, device=dev, generator=g)
    for k in range(1, n + 1):
        gates = torch.empty(67, n, device=dev)
        _lib.check(_lib.lib().mortar_remoe_gates(logits.data_ptr(), 67, n, k, gates.data_ptr(), None, torch.cuda.current_stream().cuda_stream), "gates")
        kth = logits.topk(k, -1).values[:, -1:] if k < n else torch.zeros(67, 1, device=dev)
        r = torch.relu(logits - kth).double()
        want = r * k / r.sum(-1, keepdim=True).clamp(min=1e-6)
        assert torch.equal(gates > 0, want > 0) and torch.allclose(gates.double(), want, rtol=64 * 2.0 ** -24)      # a sum of up to 64, a quotient, a product
