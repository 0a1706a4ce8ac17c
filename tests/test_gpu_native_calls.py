"""The native call layer (csrc/mortar_torch.cpp) against the general Python path of the same modules: same bits where both
serve a call, and the general path where the layer declines."""
import pytest
import torch

import mortar_amd
from mortar_amd import ops, synth
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
