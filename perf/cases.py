"""The calls this framework is used for, as cases that can be timed and compared.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)` another one of the same ranges,
`prepare(case, seed)` what a user's program holds before the call (weights loaded, inputs on the GPU), `run(state)` one
pass through the public entry points, `work(case)` the bytes and operations a pass cannot do without and
`tolerance(case)` how far the results of two correct implementations may lie apart.

Kinds of case:

    linear   one QVBandLinearV8 called on M rows: decode (M = 1), draft verification (a few to 64), prefill chunks
    step     the projections of a few decoder layers at decode, replayed as one HIP graph: fused q+k+v, o, and the MLP
             block (gate+up, SiLU, down)
    moe      one QVBandExpertsV8 block, routed tokens from one (decode) to a prompt chunk
    qvb8r    one QVBandLinearV8R (the entropy-coded format) called on M rows
    attn     attention of a few query tokens over the banded KV cache of one layer
    band     what happens to a filled segment of that cache: keys and values banded, their id layout built

Shapes are those of the decoder layers in bench.py: hidden 4096 / FFN 12288 and hidden 5120 / FFN 17408 with 1024-row
k and v, the 128-expert stack of hidden 2048 / 768 with top-8 routing, 24 query heads over 4 kv heads of 256 channels.
Weights are N(0, 0.02) at tau = 1e-3 (2e-3 for expert stacks and the entropy-coded format), as there.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from qvb8_amd.formats.qvb8 import pack as PK
from qvb8_amd.formats.qvb8.backends_experts import QVBandExpertsV8
from qvb8_amd.formats.qvb8.fuse import concat_linears
from qvb8_amd.formats.qvb8.mlp import QVBandMLPV8
from qvb8_amd.formats.qvb8.module import QVBandLinearV8
from qvb8_amd.formats.qvb8r import pack as RP
from qvb8_amd.formats.qvb8r.module import QVBandLinearV8R
from qvb8_amd.kv import codec as KC
from qvb8_amd.kv import fused_attn as FA

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIGMA = 0.02                        # weights: N(0, SIGMA)
TAU, TAU_COARSE = 1e-3, 2e-3        # certified bound of dense packs; of expert stacks and of the entropy-coded format
BITS, BITS_COARSE, BITS_CODED = 7.0, 5.9, 4.55      # stored bits per weight these give
SEGMENT = 4096                      # keys per segment of the banded cache
BAND_BITS, BAND_TAU = 7, 0.25       # its least width, which always certifies the bound for the values drawn here
BASE_ROWS = 512                     # rows an entropy-coded tensor is built from, see _coded
LARGEST = 1999 * 4096 * 12288       # multiply-adds of the largest listed linear: no drawn case has more


def listed():
    return [
        # the smallest call: one token through one square projection, called as a module (no graph): launch and host latency
        dict(name="linear_m1", kind="linear", M=1, Q=4096, P=4096, x="bf16", escapes=0, restore="fp16"),
        # a decode step as a serving loop runs it: every projection of four layers, one token, one graph replay
        dict(name="step_m1", kind="step", M=1, layers=4, hidden=4096, kv=1024, inter=12288, x="bf16"),
        # verification of a 16-token draft against a pack with escapes (outlier weights kept exactly)
        dict(name="linear_m16_escapes", kind="linear", M=16, Q=34816, P=5120, x="bf16", escapes=3000, restore="fp16"),
        # verification of a wide draft tree / a small batch, in the pack's other activation type
        dict(name="linear_m64", kind="linear", M=64, Q=24576, P=4096, x="fp16", escapes=0, restore="fp16"),
        # the last chunk of a prompt: a ragged number of rows well past the fused kernels
        dict(name="linear_m1999", kind="linear", M=1999, Q=4096, P=12288, x="bf16", escapes=0, restore="fp16"),
        # routed experts: one token (decode), a batch of eight, a prompt chunk
        dict(name="moe_t1", kind="moe", T=1, E=128, k=8, hidden=2048, inter=768, x="bf16"),
        dict(name="moe_t8", kind="moe", T=8, E=128, k=8, hidden=2048, inter=768, x="bf16"),
        dict(name="moe_t509", kind="moe", T=509, E=128, k=8, hidden=2048, inter=768, x="bf16"),
        # the entropy-coded format at decode
        dict(name="qvb8r_m1", kind="qvb8r", M=1, Q=17408, P=5120, x="bf16"),
        # attention of one new token over a long cache; of a prompt chunk over the cache so far
        dict(name="attn_t1", kind="attn", T=1, n=32768, heads=24, kv_heads=4, dim=256, x="bf16"),
        dict(name="attn_t120", kind="attn", T=120, n=16001, heads=24, kv_heads=4, dim=256, x="bf16"),
        # a filled segment of one layer's cache goes into bands
        dict(name="band_4096", kind="band", n=4096, kv_heads=4, dim=256, x="bf16"),
    ]


def _log(rng, lo, hi):
    """A whole number in lo..hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "step", "moe", "moe", "qvb8r", "attn", "attn", "band"])
    x = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "linear":
        Q, P = _log(rng, 1000, 36000), 128 * _log(rng, 8, 136)
        if rng.random() < 0.15:                     # columns no matrix-core tile covers
            P -= 8 * rng.randint(1, 15)
        M = _log(rng, 1, min(2048, max(1, LARGEST // (Q * P))))
        if rng.random() < 0.15:
            x = "fp32"
        return dict(kind=kind, M=M, Q=Q, P=P, x=x, escapes=rng.choice([0, 0, rng.randint(1, 4000)]),
                    restore=rng.choice(["fp16", "fp16", "fp16+bf16"]))
    if kind == "step":
        hidden = 128 * rng.randint(16, 40)
        return dict(kind=kind, M=_log(rng, 1, 16), layers=rng.randint(2, 4), hidden=hidden, kv=rng.choice([512, 1024]),
                    inter=128 * rng.randint(hidden // 64, hidden // 36), x=x)
    if kind == "moe":
        return dict(kind=kind, T=_log(rng, 1, 512), E=rng.choice([32, 64, 128]), k=rng.choice([4, 8]), hidden=128 * rng.randint(8, 16),
                    inter=128 * rng.randint(4, 8), x=x)
    if kind == "qvb8r":
        Q, P = _log(rng, 1000, 17408), 128 * _log(rng, 8, 136)
        return dict(kind=kind, M=_log(rng, 1, 512), Q=max(BASE_ROWS, min(Q, 17408 * 5120 // P)), P=P, x=x)
    if kind == "attn":
        T, kv_heads, dim = _log(rng, 1, 128), rng.choice([2, 4, 8]), rng.choice([128, 256])
        n = _log(rng, 1000, 32768 * 1024 // (kv_heads * dim) // (1 if T < 16 else 2))
        return dict(kind=kind, T=min(T, n), n=n, heads=kv_heads * rng.choice([4, 6, 8]), kv_heads=kv_heads, dim=dim, x=x)
    return dict(kind=kind, n=_log(rng, 200, 4096), kv_heads=rng.choice([2, 4]), dim=rng.choice([64, 128, 256]), x=x)


# ---- what a program holds before the call -----------------------------------------------------------------------------

def _weight(Q, P, gen):
    return (SIGMA * torch.randn(Q, P, device=gen.device, generator=gen)).to(torch.bfloat16)


def _linear(Q, P, gen, escapes=0, restore="fp16"):
    forced = torch.randperm(Q * P, device=gen.device, generator=gen)[:escapes].sort().values if escapes else None
    return QVBandLinearV8.from_encoded(PK.encode_tensor(_weight(Q, P, gen), TAU, restore=restore, force_escapes=forced)).prepare()


def _experts(n, Q, P, gen):
    """n packed experts of (Q, P): encoded as one matrix, then cut apart (rows of a pack are independent)."""
    enc = PK.encode_tensor(_weight(n * Q, P, gen), TAU_COARSE)
    assert enc["esc_idx"].numel() == 0
    first = enc["bit_off"][::Q].tolist() + [8 * (enc["ids"].numel() - 8)]
    mods = []
    for e in range(n):
        rows = slice(e * Q, (e + 1) * Q)
        ids = torch.zeros((first[e + 1] - first[e]) // 8 + 8, dtype=torch.uint8, device=gen.device)
        ids[:-8] = enc["ids"][first[e] // 8:first[e + 1] // 8]
        part = dict(enc, Q=Q, ids=ids, bit_off=enc["bit_off"][rows] - first[e], **{name: enc[name][rows].clone() for name in ("min_s", "tau_s", "nbits")})
        mods.append(QVBandLinearV8.from_encoded(part))
    return mods


def _coded(Q, P, gen):
    """An entropy-coded (Q, P) tensor.  Coding a tensor of full size on the host takes longer than everything else here, so
    BASE_ROWS rows are coded and their streams repeated class by class, each repeat with its own row origins."""
    base = RP.transcode(PK.encode_tensor(_weight(BASE_ROWS, P, gen), TAU_COARSE, keep_ids=True))
    assert len(base["esc_idx"]) == 0
    reps = -(-Q // BASE_ROWS)
    words = [base["words"][base["tile_off"][t]:base["tile_off"][t + 1]] for t in range(len(base["tiles"]))]
    perm, tiles, parts, states, row = [], [], [], [], 0
    for cls in range(base["K"]):
        for r in range(reps):
            for t in np.flatnonzero(base["tiles"][:, 0] == cls):
                _, first, count = base["tiles"][t]
                rows = base["perm"][first:first + count] + r * BASE_ROWS
                if rows.max() >= Q:
                    continue                            # (one row per tile for rows of more than 2048 columns: see below)
                perm.append(rows)
                tiles.append((cls, row, count))
                parts.append(words[t])
                states.append(base["states"][t])
                row += int(count)
    perm = np.concatenate(perm)
    used = np.sort(perm)                                # a tile across the last row was left out: close the gaps it made
    new_name = np.zeros(int(used[-1]) + 1, np.int64)
    new_name[used] = np.arange(len(used))
    origin = np.tile(base["min_s"], reps)[used] + (SIGMA / 16) * torch.randn(len(used), device=gen.device, generator=gen).cpu().numpy()
    return dict(base, Q=len(used), P=P, perm=new_name[perm].astype(np.int32), tiles=np.array(tiles, np.int32), words=np.concatenate(parts),
                tile_off=np.concatenate([[0], np.cumsum([len(p) for p in parts])]).astype(np.uint32), states=np.stack(states),
                min_s=origin.astype(np.float32), tau_s=np.tile(base["tau_s"], reps)[used], drow=np.tile(base["drow"], reps)[used])


def _keys_and_values(case, gen):
    """(kv heads, n, channels) as a model writes them: channels of different scale and offset in K, plain ones in V."""
    h, n, d = case["kv_heads"], case["n"], case["dim"]
    dt = DTYPES[case["x"]]
    scale = torch.exp(0.4 * torch.randn(h, 1, d, device=gen.device, generator=gen))
    k = torch.randn(h, n, d, device=gen.device, generator=gen) * scale + torch.randn(h, 1, d, device=gen.device, generator=gen)
    return k.to(dt), torch.randn(h, n, d, device=gen.device, generator=gen).to(dt)


def _banded(k, v):
    return KC.band_kv_heads(k, k.dtype, BAND_BITS, tau=BAND_TAU), KC.band_kv_heads(v, v.dtype, BAND_BITS, tau=BAND_TAU)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    randn = lambda *shape: torch.randn(*shape, device=gen.device, generator=gen)       # noqa: E731
    dt = DTYPES[case["x"]]
    kind = case["kind"]
    if kind == "linear":
        mod = _linear(case["Q"], case["P"], gen, case["escapes"], case["restore"])
        return dict(call=mod, args=(randn(case["M"], case["P"]).to(dt),))
    if kind == "qvb8r":
        mod = QVBandLinearV8R(_coded(case["Q"], case["P"], gen), device="cuda")
        return dict(call=mod, args=(randn(case["M"], case["P"]).to(dt),))
    if kind == "moe":
        E, H, I = case["E"], case["hidden"], case["inter"]
        mod = QVBandExpertsV8(_experts(E, 2 * I, H, gen), _experts(E, H, I, gen), num_experts=E).prepare()
        w, idx = torch.softmax(randn(case["T"], E), -1).topk(case["k"], -1)
        return dict(call=mod, args=(randn(case["T"], H).to(dt), idx, w / w.sum(-1, keepdim=True)))
    if kind == "step":
        return _step(case, gen, dt)
    k, v = _keys_and_values(case, gen)
    if kind == "band":
        return dict(call=_band, args=(k, v))
    lens = [min(SEGMENT, case["n"] - at) for at in range(0, case["n"], SEGMENT)]
    segs = [_banded(k[:, i * SEGMENT:i * SEGMENT + m].contiguous(), v[:, i * SEGMENT:i * SEGMENT + m].contiguous()) for i, m in enumerate(lens)]
    lay = FA.layout_from_segments([s[0] for s in segs], [s[1] for s in segs], lens, k.device, allow_wide=True)
    q = randn(case["T"], case["heads"], case["dim"]).to(dt)
    return dict(call=FA.attend, args=(q, lay, case["n"] - case["T"], case["dim"] ** -0.5))


def _step(case, gen, dt):
    """The launches of a decode step, captured once as a serving loop does (capture needs one eager call first)."""
    M, H, I = case["M"], case["hidden"], case["inter"]
    layers = []
    for _ in range(case["layers"]):
        qkv = concat_linears([_linear(n, H, gen) for n in (H, case["kv"], case["kv"])])[0].prepare()
        o = _linear(H, H, gen)
        mlp = QVBandMLPV8(_linear(I, H, gen), _linear(I, H, gen), _linear(H, I, gen))
        layers.append((qkv, o, mlp, [torch.randn(M, H, device=gen.device, generator=gen).to(dt) for _ in range(3)]))

    def step():
        return [(qkv(a), o(b), mlp(c)) for qkv, o, mlp, (a, b, c) in layers]

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        out = step()
    return dict(call=lambda: (graph.replay(), out)[1], args=(), keep=layers)


def _band(k, v):
    seg_k, seg_v = _banded(k, v)
    lay = FA.layout_from_segments([seg_k], [seg_v], [k.shape[1]], k.device, allow_wide=True)
    heads = [(b.packed, b.min_s, b.tau_s) for b in seg_k + seg_v]
    return heads, (lay.ki, lay.vi, lay.kmin, lay.kstep, lay.vmin, lay.vstep, lay.kc, lay.vc)


def run(state):
    with torch.no_grad():
        return state["call"](*state["args"])


# ---- what a pass cannot do without, and how exact it is ------------------------------------------------------------------

def work(case):
    kind, b = case["kind"], 4 if case["x"] == "fp32" else 2
    if kind in ("linear", "qvb8r"):
        M, Q, P = case["M"], case["Q"], case["P"]
        per_weight = (BITS if kind == "linear" else BITS_CODED) / 8
        return dict(bytes=Q * P * per_weight + 17 * Q + 12 * case.get("escapes", 0) + b * M * (P + Q), flops=2 * M * Q * P)
    if kind == "step":
        M, H, I = case["M"], case["hidden"], case["inter"]
        weights = case["layers"] * (2 * H * H + 2 * case["kv"] * H + 3 * H * I)
        rows = case["layers"] * (3 * H + 2 * case["kv"] + 2 * I)
        return dict(bytes=weights * BITS / 8 + 17 * rows + b * M * case["layers"] * (6 * H + 2 * case["kv"]), flops=2 * M * weights)
    if kind == "moe":
        T, E, k, H, I = (case[n] for n in ("T", "E", "k", "hidden", "inter"))
        chosen = E * (1 - (1 - k / E) ** T)
        return dict(bytes=chosen * (3 * H * I * BITS_COARSE / 8 + 17 * (2 * I + H)) + 2 * b * T * H, flops=2 * T * k * 3 * H * I)
    n, h, d = case["n"], case["kv_heads"], case["dim"]
    if kind == "attn":
        T, hq = case["T"], case["heads"]
        return dict(bytes=2 * n * h * d + (b + 4) * T * hq * d, flops=4 * T * hq * d * (n - T / 2))
    # band: keys and values in; bits packed, and a byte per id of the layout out; a few operations per value
    return dict(bytes=2 * n * h * d * (b + BAND_BITS / 8 + 1), flops=2 * n * h * d * 8)


def tolerance(case):
    # Four times what the same product in float64 over the restored values differs by:
    #   linear, qvb8r  1.7e-3 where results are rounded to bf16, 2.1e-4 .. 2.9e-4 to fp16; fp32 results of more than 8 rows
    #                  may be products of the fp16-rounded weight (2e-4)
    #   moe            as those up to 64 tokens (3.0e-4 in fp16); a prompt chunk's experts are added up in the activations'
    #                  type: 5.8e-3 in bf16, 7.2e-4 in fp16
    #   attn           7.4e-4: keys, values and probabilities are rounded to fp16
    kind, x = case["kind"], case["x"]
    if kind == "band":
        return "exact"
    if kind == "attn":
        return {"rel": 3e-3}
    if kind == "moe" and case["T"] > QVBandExpertsV8.FUSED_MAX_TOKENS:
        return {"rel": 2.3e-2 if x == "bf16" else 3e-3}
    return {"rel": 7e-3 if x == "bf16" else 1.2e-3}
