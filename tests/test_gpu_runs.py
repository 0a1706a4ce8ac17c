"""Prefill launches whose workgroups take runs of units across token tiles: row counts that whole tiles per workgroup would spread badly over
the chip.  Every row is written, nothing past the last one, and a sample of rows (both ends of tiles, the last partial one) equals the oracle."""
import numpy as np
import pytest
import torch

from mortar_amd import ops, synth
from oracle import mortar_oracle as O
from util import assert_close_bf16, oracle_spmm, prefill_form, to_dev, to_np

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
@pytest.mark.parametrize("one_scale,prefill_stream", [(False, True), (True, True), (False, False)])
def test_spmm_runs(dev, Rb, Cb, M, one_scale, prefill_stream):
    upw, span = prefill_form(0, M, Rb, Cb)
    assert span > 0 and upw == (3 if Cb == 200 else 0)
    m = synth.synth_matrix(Rb * 16, Cb * 16, 0.25, seed=Rb, zipf_s=1.2 if Cb == 80 else None)
    if one_scale:
        m["scales"][:] = m["scales"][0]
    W = synth.to_pack(m, dev, prefill_stream=prefill_stream)
    x = synth.synth_x(M, Cb * 16, seed=M)
    out = _call(lambda y: ops.spmm(to_dev(x, dev), W, out=y), M, Rb * 16, dev)
    rows = _sample(M)
    assert_close_bf16(to_np(out[torch.from_numpy(rows).to(dev)]), oracle_spmm(x[rows], m), f"{Rb}x{Cb}")


# gate_up: one 32-token tile of all K, `down`: K segments from tile order; gate_up in 64-token tiles; gate_up in K segments
@pytest.mark.parametrize("d,f,M,norm,gated", [(1280, 3200, 32 * 141 - 19, False, False), (1280, 3200, 32 * 141 - 19, True, False),
                                              (1280, 3200, 32 * 141 - 19, False, True), (768, 2048, 9000, False, False), (768, 2048, 9000, True, True),
                                              (16 * 161, 16 * 688, 1300, False, True)])
def test_mlp_runs(dev, d, f, M, norm, gated):
    upw, span = prefill_form(2 if norm else 1, M, f // 16, d // 16)
    assert span > 0 and upw == (2 if d > 2048 else 0)
    if d == 1280:
        assert prefill_form(0, M, d // 16, f // 16, tiled=True) == (4, 3)
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
        gates = np.random.default_rng(1).random((M, f // 16 // (8 if d > 768 else 4)), dtype=np.float32)
        gates[gates < 0.6] = 0.0
        kw["gates"] = torch.from_numpy(gates).to(dev)
        gates = gates[rows]
    ref = O.swiglu_mlp(xo, spec["gate_up"], spec["down"], gates)["y"]
    out = _call(lambda y: ops.mlp(to_dev(x, dev), G, D, out=y, **kw), M, d, dev)
    assert_close_bf16(to_np(out[torch.from_numpy(rows).to(dev)]), ref, "mlp", ulps=8)


@pytest.mark.parametrize("units,M,form", [(200, 1300, (3, 0)), (688, 1300, (2, 7)), (40, 97, None)])      # whole groups of three, runs of groups of two, small tiles
@pytest.mark.parametrize("one_scale", [False, True])
def test_gateup_of_an_odd_width(dev, units, M, form, one_scale):
    """K segments of an odd number of block-columns, copied in pairs; a partial last tile; the module's hidden activations in tile order."""
    d = 16 * 161
    assert form is None or prefill_form(1, M, units, d // 16) == form
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


@pytest.mark.parametrize("Rb,M,form", [(128, 2103, (3, 0)), (128, 1000, (1, 0)), (128, 4094, (4, 0))])
def test_masked_product_of_several_segments(dev, Rb, M, form):
    assert prefill_form(3, M, Rb, 200) == form
    m = synth.synth_matrix(Rb * 16, 3200, 0.2, seed=M, zipf_s=1.2)
    on = np.random.default_rng(M).random((M, 50)) < 0.4
    x = synth.synth_x(M, 3200, seed=M)
    out = _call(lambda y: ops.spmm(to_dev(x, dev), synth.to_pack(m, dev), out=y, active=torch.from_numpy(on.astype(np.uint8)).to(dev)), M, Rb * 16, dev)
    rows = _sample(M)
    assert_close_bf16(to_np(out[torch.from_numpy(rows).to(dev)]), oracle_spmm(x[rows] * np.repeat(on[rows], 64, axis=1), m), "masked")


@pytest.mark.parametrize("M", [2103, 32 * 141 - 15])                     # whole groups, runs
def test_rows_of_x_apart(dev, M):
    """A leading dimension beyond the row: the copied pieces come from the rows, and nothing between them is looked at."""
    d, Rb = 16 * 161, 77
    assert (prefill_form(0, M, Rb, 161)[1] > 0) == (M > 4000)
    W = synth.to_pack(synth.synth_matrix(Rb * 16, d, 0.2, seed=1), dev)
    x = to_dev(synth.synth_x(M, d, seed=M), dev)
    wide = torch.full((M, d + 24), float("nan"), device=dev, dtype=torch.bfloat16)
    wide[:, 8:8 + d] = x
    assert torch.equal(ops.spmm(wide[:, 8:8 + d], W), ops.spmm(x, W))


@pytest.mark.parametrize("col", [79, 80, 160])          # segments of 81 and 80 columns: the last pair of the first one holds its last column twice
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_non_finite_activations_reach_the_blocks_of_their_column(dev, col, value):
    """... and no other output of the token, and no other token.  (Not so the first column of a segment, which padding multiplies by zero.)"""
    Rb, Cb, M, tok = 77, 161, 2103, 1234
    m = synth.synth_matrix(Rb * 16, Cb * 16, 0.2, seed=col)
    W = synth.to_pack(m, dev)
    assert W.seg_cb == 81 and prefill_form(0, M, Rb, Cb) == (2, 0)
    x = to_dev(synth.synth_x(M, Cb * 16, seed=3), dev)
    want = ops.spmm(x, W)
    x[tok, col * 16 + 5] = value
    got = ops.spmm(x, W)
    holds = np.zeros((Rb, 16), bool)
    holds[np.repeat(np.arange(Rb), np.diff(m["offsets"]))[m["col_idx"] == col]] = True
    hit = torch.from_numpy(holds.reshape(-1)).to(dev)
    assert hit.any() and not hit.all()
    assert torch.equal(got[:tok], want[:tok]) and torch.equal(got[tok + 1:], want[tok + 1:])
    assert torch.equal(got[tok][~hit], want[tok][~hit]) and not torch.isfinite(got[tok][hit].float()).any()
