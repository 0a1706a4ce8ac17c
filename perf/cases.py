"""Workloads of the sparse-MLP runtime as its users run them, one pass each through the public entry points.

Every case is one kind of call over a range of widths, row counts, densities and scale formats:

  decode         a serving engine's MLP call, one to 64 single-token rows, launched eagerly (MortarDecodeMLP)
  decode_graph   the MLPs of a few consecutive blocks as an engine replays them, from a captured graph
  decode_routed  the same eager call with a ReMoE router in front
  decode_fp32    the reference engine's own arithmetic (fp32 activations, one scale per matrix) through mortar_gemv
  prefill        the module's forward on a prompt (or a batch of prompts)
  prefill_routed the same with the module's own router
  looped         the looped core: shared blocks run several times, activations normalised in front of each
  train          one training step of the MLP with trainable ternarised block values (forward and backward)
  values         one training step of the stored-values operator stk_dds (forward, dx and dW)

Activations are N(0, 1) in bf16; a kept block holds {-1, 0, +1} with probability (0.3, 0.4, 0.3) and a scale from
U(0.01, 0.1); the topology is drawn per block-row, with equal or power-law counts.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import mortar_amd
from mortar_amd import synth

#: (d_model, d_ff) of the repository's configurations and of the wider models its tests and tables go through.
WIDTHS = {768: 2048, 1024: 2816, 1536: 4096, 2048: 5632, 3072: 8192, 4096: 11008}
BLOCK = 16
MAX_ROWS = 16384
MAX_FLOPS = 2.0e11          # of a drawn case: less than the largest listed one


def _case(name, kind, d, rows, density=0.25, scale="block", topology="uniform", clusters=0, ratio=0.25, blocks=1, iters=1):
    return {"name": name, "kind": kind, "d_model": d, "d_ff": WIDTHS[d], "rows": rows, "density": density, "scale": scale,
            "topology": topology, "clusters": clusters, "ratio": ratio, "blocks": blocks, "iters": iters}


def listed():
    return [
        # one token of one stream through one block's MLP, at the benchmark's width: what a chat session decodes with
        _case("decode_1", "decode", 2048, 1),
        # an odd batch of streams through four consecutive blocks, replayed from a graph as a serving engine does
        _case("decode_graph_13", "decode_graph", 2048, 13, blocks=4),
        # a small batch with the router of the deployed routed model: 16 clusters, half of them active
        _case("decode_routed_4", "decode_routed", 2048, 4, clusters=16, ratio=0.5),
        # a batch in the reference engine's arithmetic and deploy format (one scale per matrix)
        _case("decode_fp32_8", "decode_fp32", 2048, 8, scale="matrix"),
        # a short prompt of odd length through the base-width model
        _case("prefill_base_203", "prefill", 768, 203),
        # the benchmark's prompt: 4096 tokens at its width
        _case("prefill_4096", "prefill", 2048, 4096),
        # a training-sized batch of prompts (4 x 4096) at base width
        _case("prefill_base_16384", "prefill", 768, 16384),
        # a prompt of odd length through a wide model whose rows do not fit one on-chip tile
        _case("prefill_wide_1999", "prefill", 4096, 1999),
        # the benchmark's routed prompt: 352 clusters of one block-row, a quarter of them active per token
        _case("prefill_routed_4096", "prefill_routed", 2048, 4096, clusters=352, ratio=0.25),
        # two shared blocks, two iterations, power-law rows (more calls in a row amplify rounding beyond any comparison)
        _case("looped_4096", "looped", 2048, 4096, topology="zipf", blocks=2, iters=2),
        # one step of ternary-values training at the benchmark's width
        _case("train_4096", "train", 2048, 4096),
        # the stored-values operator at base width on 16384 tokens (one 768 -> 4096 layer), forward and backward
        _case("values_16384", "values", 768, 16384),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode_graph", "decode_routed", "decode_fp32", "prefill", "prefill", "prefill_routed", "looped",
                       "train", "values"])
    wide = kind in ("decode", "decode_graph", "prefill")
    d = rng.choice(sorted(WIDTHS) if wide else [w for w in sorted(WIDTHS) if w <= 2048])
    density = rng.choice([0.125, 0.25, 0.25, 0.25, 0.5]) if d <= 2048 else rng.choice([0.125, 0.25])
    scale = "matrix" if kind == "decode_fp32" else rng.choice(["block", "block", "matrix"])
    c = _case("", kind, d, 1, density, scale, rng.choice(["uniform", "uniform", "zipf"]))
    del c["name"]
    if kind.startswith("decode"):
        c["rows"] = _log(rng, 1, 64)
        c["blocks"] = rng.randint(2, 4) if kind == "decode_graph" else 1
    else:
        if kind == "looped":
            c["blocks"], c["iters"] = rng.choice([(2, 2), (4, 1), (1, 4), (2, 1), (3, 1), (1, 2)])
        top = int(MAX_ROWS * MAX_FLOPS / work(dict(c, rows=MAX_ROWS))["flops"])
        c["rows"] = _log(rng, 65, max(66, min(MAX_ROWS if kind in ("prefill", "values") else 8192, top)))
    if "routed" in kind:
        c["clusters"], c["ratio"] = rng.choice([(16, 0.5), (16, 0.25), (WIDTHS[d] // BLOCK, 0.25)])
    return c


def _rng(seed, tag):
    return np.random.Generator(np.random.PCG64([seed & 0xffffffff, tag]))


def _matrix(case, out_f, in_f, rng):
    """One carved ternary matrix in the layout of a checkpoint: numpy arrays as synth.synth_matrix returns them."""
    rb, cb = out_f // BLOCK, in_f // BLOCK
    counts = synth.row_counts(rb, cb, case["density"], rng, 1.2 if case["topology"] == "zipf" else None)
    keep = np.argsort(rng.random((rb, cb), dtype=np.float32), axis=1)
    cols = [np.sort(keep[r, :n]) for r, n in enumerate(counts)]
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    nnz = int(offsets[-1])
    ternary = np.array([-1, -1, -1, 0, 0, 0, 0, 1, 1, 1], dtype=np.int8)
    codes = ternary[rng.integers(0, 10, size=(nnz, BLOCK, BLOCK), dtype=np.uint8)]
    scales = rng.uniform(0.01, 0.1, size=1 if case["scale"] == "matrix" else nnz).astype(np.float32)
    return {"codes": codes, "scales": scales, "col_idx": np.concatenate(cols).astype(np.int16),
            "row_idx": np.repeat(np.arange(rb), counts).astype(np.int16), "offsets": offsets, "shape": (out_f, in_f)}


def _spec(case, rng):
    d, f = case["d_model"], case["d_ff"]
    return {"gate_up": _matrix(case, 2 * f, d, rng), "down": _matrix(case, d, f, rng), "d_model": d, "d_ff": f}


def _randn(shape, seed, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _norm_weight(d, seed):
    return (1.0 + 0.1 * _randn((d,), seed, torch.float32)).to(torch.bfloat16)


def _router(mlp, case, seed):
    """A router as a trained model has it: no zero biases, one iteration embedding."""
    torch.manual_seed(seed)
    mlp.enable_routing(n_clusters=case["clusters"], activation_ratio=case["ratio"])
    with torch.no_grad():
        mlp.router.group_bias.normal_(0.0, 0.02)
        mlp.router.iter_embed.normal_(0.0, 0.02)


def _packed(mlp):
    """The weights in the runtime's device format, as a serving program has them before its first request."""
    mlp.gate_up._cms.mortar_pack(), mlp.down._cms.mortar_pack()
    return mlp


def prepare(case, seed):
    kind, d, f, rows = case["kind"], case["d_model"], case["d_ff"], case["rows"]
    dev = torch.device("cuda")
    rng = _rng(seed, 1)
    state = {"kind": kind, "case": case}
    if kind == "values":
        m = _matrix(case, 2 * f, d, rng)
        sd = synth.carved_state(m)
        state["index"] = [sd["mortar_" + k].to(dev) for k in ("offsets", "row_indices", "column_indices", "offsets_t", "column_indices_t",
                                                             "block_offsets_t")]
        state["shape"] = (d, 2 * f)
        state["data"] = (_randn((m["codes"].shape[0], BLOCK, BLOCK), seed + 1, torch.float32) * 0.05).to(torch.bfloat16).requires_grad_(True)
        state["x"] = _randn((rows, d), seed + 2).requires_grad_(True)
        state["dy"] = _randn((rows, 2 * f), seed + 3)
        return state
    if kind == "train":
        state["mlp"] = synth.qat_mlp_module(_spec(case, rng), dev, seed=seed)
        state["x"] = _randn((rows, d), seed + 2).requires_grad_(True)
        state["dy"] = _randn((rows, d), seed + 3)
        return state
    if kind == "decode_fp32":
        mlp = _packed(synth.mlp_module(_spec(case, rng), dev))
        state["gate_up"], state["down"] = (mortar_amd.mortar_pack_strips(m._cms) for m in (mlp.gate_up, mlp.down))
        state["x"] = _randn((rows, d), seed + 2, torch.float32)
        return state
    mlps = [_packed(synth.mlp_module(_spec(case, rng), dev)) for _ in range(case["blocks"])]
    state["x"] = _randn((rows, d), seed + 2)
    state["norms"] = [_norm_weight(d, seed + 10 + i) for i in range(len(mlps))]
    if case["clusters"]:
        _router(mlps[0], case, seed + 4)
    state["mlps"] = mlps
    if kind in ("decode", "decode_routed"):
        state["call"] = mortar_amd.MortarDecodeMLP(mlps[0], norm_weight=state["norms"][0])
    if kind == "decode_graph":
        calls = [mortar_amd.MortarDecodeMLP(m, norm_weight=w) for m, w in zip(mlps, state["norms"])]

        def step():
            y = state["x"]
            for call in calls:
                y = call(y)
            return y

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["y"] = step()
    return state


def run(state):
    kind = state["kind"]
    if kind == "decode":
        return state["call"](state["x"])
    if kind == "decode_graph":
        state["graph"].replay()
        return state["y"]
    if kind == "decode_routed":
        return state["call"](state["x"])
    if kind == "decode_fp32":
        h = mortar_amd.mortar_gemv(state["x"], state["gate_up"], swiglu_out=True)
        return mortar_amd.mortar_gemv(h, state["down"])
    if kind == "prefill":
        with torch.no_grad():
            return state["mlps"][0](state["x"])
    if kind == "prefill_routed":
        mlp = state["mlps"][0]
        with torch.no_grad():
            y = mlp(state["x"])
        return {"y": y, "aux_loss": mlp._last_aux_loss, "load": mlp.router.group_load_ema}
    if kind == "looped":
        return mortar_amd.looped_core_forward(state["mlps"], state["x"], state["case"]["iters"], norm_weights=state["norms"])
    if kind == "train":
        mlp, x = state["mlp"], state["x"]
        x.grad = None
        for p in mlp.parameters():
            p.grad = None
        y = mlp(x)
        y.backward(state["dy"])
        return {"y": y.detach(), "dx": x.grad, "gate_up": mlp.gate_up._cms.mortar_data.grad, "down": mlp.down._cms.mortar_data.grad}
    x, data = state["x"], state["data"]
    x.grad = data.grad = None
    y = mortar_amd.stk_dds(x, data, *state["index"], *state["shape"], True)
    y.backward(state["dy"])
    return {"y": y.detach(), "dx": x.grad, "data": data.grad}


def _blocks(case, out_f, in_f):
    return out_f // BLOCK * max(1, round(case["density"] * (in_f // BLOCK)))


def work(case):
    """Each input read once and each output written once: a ternary block is 64 bytes of codes, a 2-byte column and (with a
    scale per block) 4 bytes of scale, a block-row 4 bytes of index.  Products count kept blocks, and with a router those of
    the active clusters only."""
    kind, d, f, rows = case["kind"], case["d_model"], case["d_ff"], case["rows"]
    gu, dn = _blocks(case, 2 * f, d), _blocks(case, d, f)
    if kind == "values":
        return {"bytes": 3 * gu * 512.0 + gu * 2 + 8 * f / BLOCK + rows * (2.0 * d + 2 * f + d) * 2, "flops": 3 * 2.0 * rows * 256 * gu}
    if kind == "train":
        return {"bytes": 2 * (gu + dn) * 514.0 + rows * 4.0 * d * 2, "flops": 3 * 2.0 * rows * 256 * (gu + dn)}
    weights = (gu + dn) * (70.0 if case["scale"] == "block" else 66.0) + 4 * (2 * f + d) / BLOCK
    act = 4 if kind == "decode_fp32" else 2
    bytes_, flops = weights * case["blocks"] + rows * 2.0 * d * act, 2.0 * rows * 256 * (gu + dn)
    if case["clusters"]:
        nsk = max(4, math.ceil(math.sqrt(case["clusters"])))
        flops = flops * case["ratio"] + 2.0 * rows * d * d + 2.0 * rows * nsk * d
        bytes_ += 4.0 * d * d + 4.0 * nsk * d
    return {"bytes": bytes_, "flops": flops * case["blocks"] * case["iters"]}


def tolerance(case):
    if case["kind"] == "decode_fp32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["blocks"] * case["iters"] > 1:
        return {"rel": 0.03, "max": 0.5}        # bf16 rounding of one MLP grows about twofold with every further one
    return {"rel": 1e-2, "max": 0.25}
