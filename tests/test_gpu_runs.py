"""Prefill launches whose workgroups take runs of units across token tiles: row counts that whole tiles per workgroup would spread badly over
the chip.  Every row is written, nothing past the last one, and a sample of rows (both ends of tiles, the last partial one) equals the oracle."""
import numpy as np
import pytest
import torch

from mortar_amd import ops, synth
from oracle import mortar_oracle as O
from util import assert_close_bf16, oracle_spmm, to_dev, to_np

pytestmark = pytest.mark.gpu


def _sample(M):
    rows = {0, M - 1, M - 2} | set(range(31, M, 997)) | set(range(32, M, 1013)) | set(range(M - M % 32, M, 5))
    return np.array(sorted(rows))


def _call(f, M, cols, dev):
    out = torch.full((M + 1, cols), float("nan"), device=dev, dtype=torch.bfloat16)
    f(out[:M])
    assert torch.isfinite(out[:M].float()).all() and torch.isnan(out[M].float()).all()
    return out


@pytest.mark.parametrize("Rb,Cb,M", [(64, 3, 64 * 257 - 7),          # 64-token tiles, all of K in one
                                     (70, 80, 32 * 257 - 9),         # 32-token tiles
                                     (77, 200, 32 * 141 - 15)])      # K segments, a row of units left over
@pytest.mark.parametrize("one_scale", [False, True])
def test_spmm_runs(dev, Rb, Cb, M, one_scale):
    m = synth.synth_matrix(Rb * 16, Cb * 16, 0.25, seed=Rb, zipf_s=1.2 if Cb == 80 else None)
    if one_scale:
        m["scales"][:] = m["scales"][0]
    W = synth.to_pack(m, dev)
    x = synth.synth_x(M, Cb * 16, seed=M)
    out = _call(lambda y: ops.spmm(to_dev(x, dev), W, out=y), M, Rb * 16, dev)
    rows = _sample(M)
    assert_close_bf16(to_np(out[torch.from_numpy(rows).to(dev)]), oracle_spmm(x[rows], m), f"{Rb}x{Cb}")


@pytest.mark.parametrize("norm,gated", [(False, False), (True, False), (False, True)])
def test_mlp_runs(dev, norm, gated):
    d, f, M = 1280, 3200, 32 * 141 - 19                              # gate_up: one tile of all K; down: K segments from tile order
    spec = synth.synth_mlp(d, f, 0.2, seed=5)
    G, D = synth.to_pack(spec["gate_up"], dev), synth.to_pack(spec["down"], dev)
    x = synth.synth_x(M, d, seed=6)
    rows = _sample(M)
    xo, kw, gates = x[rows], {}, None
    if norm:
        w = O.bf16_round(np.linspace(0.5, 1.5, d, dtype=np.float32))
        kw["norm"] = (to_dev(w, dev), 1e-5)
        xo = O.rmsnorm(xo, w, 1e-5)
    if gated:
        gates = np.random.default_rng(1).random((M, 40), dtype=np.float32)
        gates[gates < 0.6] = 0.0
        kw["gates"] = torch.from_numpy(gates).to(dev)
        gates = gates[rows]
    ref = O.swiglu_mlp(xo, spec["gate_up"], spec["down"], gates)["y"]
    out = _call(lambda y: ops.mlp(to_dev(x, dev), G, D, out=y, **kw), M, d, dev)
    assert_close_bf16(to_np(out[torch.from_numpy(rows).to(dev)]), ref, "mlp", ulps=8)


@pytest.mark.parametrize("units,M", [(200, 1300), (688, 1300), (40, 97)])      # runs of one, of two units per wave, whole groups
@pytest.mark.parametrize("one_scale", [False, True])
def test_gateup_of_an_odd_width(dev, units, M, one_scale):
    """K segments of an odd number of block-columns, copied in pairs; a partial last tile; the module's hidden activations in tile order."""
    d = 16 * 161
    spec = synth.synth_mlp(d, 16 * units, 0.1, seed=units, zipf_s=1.2)
    if one_scale:
        for k in ("gate_up", "down"):
            spec[k]["scales"][:] = spec[k]["scales"][0]
    G, D = synth.to_pack(spec["gate_up"], dev), synth.to_pack(spec["down"], dev)
    x = synth.synth_x(M, d, seed=M)
    rows = _sample(M)
    idx = torch.from_numpy(rows).to(dev)
    ref = O.swiglu_mlp(x[rows], spec["gate_up"], spec["down"])
    h = _call(lambda y: ops.gateup_swiglu(to_dev(x, dev), G, out=y), M, 16 * units, dev)
    assert_close_bf16(to_np(h[idx]), ref["h"], "h", ulps=8)
    y = _call(lambda out: ops.mlp(to_dev(x, dev), G, D, out=out), M, d, dev)
    assert_close_bf16(to_np(y[idx]), ref["y"], "mlp", ulps=8)
