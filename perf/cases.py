"""The calls whose speed matters to a program that serves the model with this package, over the
range such a program meets: decode steps of one sequence and of batches, prompt chunks from a few
hundred to 16,384 tokens, the synthetic and the shipped artifact's weight widths, plain and fused
with the post-attention norm and residual add, the block with every stage output, and the untied
lm_head.

A block case names: T tokens, the number of decoder layers run in the pass (each on its own input,
as the mixers between two MoE blocks hand it over), the weight widths, the activation type, whether
routing is Zipf-skewed, whether the norm and residual add are fused in, and whether the pass is a
captured HIP graph (a decode loop of fixed batch) or eager calls (prompts).
"""
from __future__ import annotations

import math

import torch

from __graft_entry__ import load_package

H, I, IS, E, K = 2048, 512, 512, 256, 8
V = 248320
MAX_T = 16384
GRAPH_MAX_T = 64

# name -> (down, split gate/up with f32 router and scalar gate, Q8_0 shared expert)
WIDTHS = {
    "q4k": ("q4k", False, False),        # Q4_K experts, bf16 router and shared expert
    "q6k_down": ("q6k", False, False),   # the same with Q6_K down
    "artifact": ("q5k", True, True),     # the shipped file's: Q5_K down, f32 router, Q8_0 shared
}
BLOCK_BYTES = {"q4k": 144, "q5k": 176, "q6k": 210}      # per 256 elements
TABLE_BYTES = {"q6k": H // 256 * 210, "q8_0": H // 32 * 34, "bf16": H * 2}


def _block(name, T, widths="q4k", dtype="f32", layers=1, norm=False, zipf=False, graph=False,
           stages=False):
    return {"name": name, "op": "block", "T": T, "widths": widths, "dtype": dtype, "layers": layers,
            "norm": norm, "zipf": zipf, "graph": graph, "stages": stages}


def _head(name, B, fmt="q6k", dtype="f32", rows=0):
    return {"name": name, "op": "lm_head", "B": B, "fmt": fmt, "dtype": dtype, "rows": rows}


def listed():
    return [
        # one sequence being decoded: four consecutive layers of a token, norm and residual fused,
        # the next layer named, replayed from the graph a decode loop keeps
        _block("decode_1", 1, layers=4, norm=True, graph=True),
        # the same with the weights as the shipped file stores them
        _block("decode_1_artifact", 1, "artifact", layers=4, norm=True, graph=True),
        # a few sequences (or one sequence's speculated tokens) per step
        _block("decode_3", 3, layers=2, norm=True, graph=True),
        # a small serving batch on the artifact's widths
        _block("decode_16_artifact", 16, "artifact", layers=2, norm=True, graph=True),
        # a full serving batch with skewed expert load, the bare block
        _block("decode_64_zipf", 64, zipf=True, graph=True),
        # a short prompt on the artifact's widths, as the decoder layer calls it
        _block("prompt_200_artifact", 200, "artifact", norm=True),
        # a ragged prompt through the reference's block call, every stage returned (parity checks)
        _block("stages_333", 333, dtype="bf16", stages=True),
        # a prompt chunk on the artifact's widths, as the decoder layer calls it
        _block("prompt_1000_artifact", 1000, "artifact", norm=True),
        # the headline prefill: a 4096-token prompt in bf16 activations
        _block("prompt_4096", 4096, dtype="bf16"),
        # the largest prefill: mixed quantization, skewed expert load
        _block("prompt_16384_q6k_zipf", 16384, "q6k_down", dtype="bf16", zipf=True),
        # logits of one decoded token over the whole vocabulary, the artifact's table
        _head("lm_head_1_q6k", 1),
        # logits of a small batch over a Q8_0 table
        _head("lm_head_6_q8_0", 6, "q8_0", dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    if rng.random() < 0.2:
        rows = 0 if rng.random() < 0.6 else _log_int(rng, 1000, V)
        c = _head("", rng.randint(1, 8), rng.choice(sorted(TABLE_BYTES)), rng.choice(["f32", "bf16"]),
                  rows)
    else:
        T = _log_int(rng, 1, MAX_T)
        graph = T <= GRAPH_MAX_T
        norm = rng.random() < 0.6
        # the decoder layer's residual stream is f32
        dtype = "f32" if norm else rng.choice(["f32", "bf16"])
        c = _block("", T, rng.choice(sorted(WIDTHS)), dtype, 2 if graph else 1, norm,
                   rng.random() < 0.4, graph, not norm and not graph and T <= 1024 and rng.random() < 0.5)
    del c["name"]
    return c


# ------------------------------------------------------------------------------------- inputs ---
def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _layers(case, seed):
    """Weights, input rows and norm weight of each layer of the pass."""
    pkg = load_package()
    Q, synth = pkg.quant, pkg.synth
    down, split, q8 = WIDTHS[case["widths"]]
    wide = torch.float32 if split else torch.bfloat16
    out = []
    for l in range(case["layers"]):
        s = 1000 * seed + l
        lw = synth.make_layer(
            s, "cuda", down_fmt={"q4k": Q.FMT_Q4_K, "q5k": Q.FMT_Q5_K, "q6k": Q.FMT_Q6_K}[down],
            zipf=case["zipf"], router_dtype=wide, scalar_gate_dtype=wide, split_gate_up=split,
            shared_fmt=Q.FMT_Q8_0 if q8 else Q.FMT_BF16)
        x = synth.make_input(case["T"], s, "cuda", _dtype(case))
        out.append((lw, x, synth.make_norm_weight(s, "cuda") if case["norm"] else None))
    return out


def _head_inputs(case, seed):
    pkg = load_package()
    L, Q = pkg._lib, pkg.quant
    fmt = {"q6k": L.MOE_FMT_Q6_K, "q8_0": L.MOE_FMT_Q8_0, "bf16": L.MOE_FMT_BF16}[case["fmt"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    h = torch.randn(case["B"], H, generator=g, device="cuda").to(_dtype(case))
    parts = []
    for r0 in range(0, V, 1 << 16):
        w = torch.randn(min(1 << 16, V - r0), H, generator=g, device="cuda") * 0.02
        parts.append(w.to(torch.bfloat16) if case["fmt"] == "bf16" else Q.quantize(w, fmt))
    table = torch.cat(parts)
    ids = None
    if case["rows"]:
        ids = torch.randperm(V, generator=g, device="cuda")[:case["rows"]].to(torch.int32)
    return h, table, fmt, ids


def prepare(case, seed):
    if case["op"] == "lm_head":
        h, table, fmt, ids = _head_inputs(case, seed)
        return {"case": case, "h": h, "table": table, "fmt": fmt, "ids": ids}
    pkg = load_package()
    layers = _layers(case, seed)
    st = {"case": case, "layers": layers, "cfg": pkg.load_geometry(),
          "outs": [torch.empty(case["T"], H, device="cuda") for _ in layers]}
    if case["graph"]:
        _capture(st)
    torch.cuda.synchronize()
    return st


def _capture(st):
    """The pass as a HIP graph, recorded on a stream of its own after one eager run on it; the
    workspace that the graph uses is kept with it."""
    abi = load_package().abi
    T = st["case"]["T"]
    g, cap = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    cap.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(cap):
        st["ws"] = abi.workspace(torch.device("cuda", torch.cuda.current_device()),
                                 abi.workspace_bytes(T, H, I, E, K, IS))
        _layer_calls(st)
    cap.synchronize()
    with torch.cuda.stream(cap), torch.cuda.graph(g, stream=cap):
        _layer_calls(st)
    torch.cuda.current_stream().wait_stream(cap)
    st["graph"] = g


def _layer_calls(st):
    abi = load_package().abi
    n = len(st["layers"])
    for l, (lw, x, nw) in enumerate(st["layers"]):
        nlw, _, nnw = st["layers"][(l + 1) % n]
        hint = {"next_layer": nlw, "next_norm_w": nnw} if n > 1 else {}
        abi.block_forward(x, lw, out=st["outs"][l], norm_w=nw, residual=None if nw is None else x, **hint)


def run(st):
    case, pkg = st["case"], load_package()
    if case["op"] == "lm_head":
        return pkg.abi.lm_head(st["h"], st["table"], st["fmt"], st["ids"])
    if case["stages"]:
        lw, x, _ = st["layers"][0]
        return pkg.block.moe_block(x, lw, st["cfg"])
    if case["graph"]:
        st["graph"].replay()
    else:
        _layer_calls(st)
    return st["outs"]


# --------------------------------------------------------------------------------------- work ---
def _zipf_bias(s=1.1):
    r = torch.arange(1, E + 1, dtype=torch.float64).pow(-s)
    return torch.log(r / r.sum())


def _experts_hit(case):
    """Distinct experts of one layer's T x 8 routed pairs, from simulated router logits."""
    g = torch.Generator().manual_seed(1)
    logits = 0.02 * math.sqrt(H) * torch.randn(case["T"], E, generator=g, dtype=torch.float64)
    if case["zipf"]:
        logits += _zipf_bias()
    return int(torch.unique(logits.topk(K, dim=-1).indices).numel())


def work(case):
    act = 2 if case["dtype"] == "bf16" else 4
    if case["op"] == "lm_head":
        rows = case["rows"] or V
        return {"bytes": rows * TABLE_BYTES[case["fmt"]] + 4 * case["rows"] + case["B"] * (H * act + rows * 4),
                "flops": 2 * case["B"] * rows * H}
    T, n = case["T"], case["layers"]
    down, split, q8 = WIDTHS[case["widths"]]
    expert = 2 * I * H // 256 * BLOCK_BYTES["q4k"] + H * I // 256 * BLOCK_BYTES[down]
    shared = 3 * IS * H // 32 * 34 if q8 else 3 * IS * H * 2
    router = (E * H + H) * (4 if split else 2) + (E * 4 if case["zipf"] else 0)
    rows = T * H * (act + 4) + (H * 4 if case["norm"] else 0)
    if case["stages"]:
        rows += T * (2 * E + K * (8 + 2 + 4) + 2 * H * 4 + 4 + K * H * 4)
    return {"bytes": n * (_experts_hit(case) * expert + shared + router + rows),
            "flops": n * 2 * T * (K * 3 * I * H + 3 * IS * H + E * H)}


# ---------------------------------------------------------------------------------- tolerances ---
def tolerance(case):
    # about four times the distance from exact() below, measured on the listed and drawn cases
    if case["op"] == "lm_head":
        return {"rel": 1e-6}                   # f32 sums of 2048 products
    if case["T"] <= 6:
        return {"rel": 2e-6}                   # f32 sums throughout
    if case["stages"]:
        return {"rel": 5e-3, "differ": 0.0}    # f16 operands, the expert rows held in f16
    # f16 matrix-core operands in the routed experts; with the norm, added to an f32 residual
    return {"rel": 5e-4} if case["norm"] else {"rel": 4e-3}


# --------------------------------------------------------------------------------------- exact ---
def _f16(b):
    """f16 values of byte pairs [..., 2]."""
    return b.contiguous().view(torch.float16).squeeze(-1).double()


def _scale_min(s):
    """The eight 6-bit scales and mins of packed bytes [n, 12]."""
    s = s.to(torch.int32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    return sc, mn


def _dequant(raw, fmt, cols):
    """Super-block bytes -> f64 [rows, cols]."""
    size = 34 if fmt == "q8_0" else BLOCK_BYTES[fmt]
    b = raw.reshape(-1, size)
    n = b.shape[0]
    if fmt == "q8_0":
        v = _f16(b[:, :2])[:, None] * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "q6k":
        ql = b[:, :128].reshape(n, 2, 2, 32).to(torch.int32)
        qh = b[:, 128:192].reshape(n, 2, 1, 32).to(torch.int32)
        low = torch.stack([ql & 15, ql >> 4], 2).reshape(n, 2, 4, 32)
        shift = torch.arange(0, 8, 2, device=b.device, dtype=torch.int32).view(1, 1, 4, 1)
        q = (low | (((qh >> shift) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = _f16(b[:, 208:210])[:, None, None] * sc[:, :, None] * q.reshape(n, 16, 16).double()
    else:
        d, dmin = _f16(b[:, 0:2]), _f16(b[:, 2:4])
        sc, mn = _scale_min(b[:, 4:16])
        qs = b[:, -128:].reshape(n, 4, 32).to(torch.int32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if fmt == "q5k":
            bit = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 8, 1)
            q = q + (((b[:, 16:48].to(torch.int32)[:, None, :] >> bit) & 1) << 4)
        v = (d[:, None] * sc)[:, :, None] * q - (dmin[:, None] * mn)[:, :, None]
    return v.reshape(-1, cols)


def _round_bf16(v):
    """f64 -> bf16 with one rounding (to nearest, ties to even)."""
    f = v.float()
    half = (f.view(torch.int32) & 0xFFFF) == 0x8000
    inf = torch.full_like(f, float("inf"))
    f = torch.where(half & (v > f.double()), torch.nextafter(f, inf), f)
    f = torch.where(half & (v < f.double()), torch.nextafter(f, -inf), f)
    return f.to(torch.bfloat16)


def _route(x, lw):
    """The block's definition of its routing: logits rounded once to bf16, f32 softmax, the CPU's
    topk, renormalised weights in f32 and rounded to bf16."""
    logits = x @ lw.router.double().T
    if lw.router_bias is not None:
        logits = logits + lw.router_bias.double()
    logits = _round_bf16(logits)
    p, ids = torch.topk(torch.softmax(logits.float().cpu(), -1), K, dim=-1)
    w = p / p.sum(-1, keepdim=True)
    return logits, ids.to(x.device), w.to(x.device)


def _mlp(x, gate, up, down):
    return (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T


def _exact_block(case, lw, x0, nw):
    down, split, q8 = WIDTHS[case["widths"]]
    x = x0.double()
    if nw is not None:
        # the norm's own result is f32: its scale, then the product, rounded
        r = (1.0 / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)).float()
        x = ((x0.float() * r) * nw).double()
    logits, ids, w = _route(x, lw)
    wb = w.to(torch.bfloat16)
    raw = torch.zeros(x.shape[0], K, H, dtype=torch.float64, device=x.device) if case["stages"] else None
    routed = torch.zeros_like(x)
    for e in torch.unique(ids).tolist():
        t, k = (ids == e).nonzero(as_tuple=True)
        gu = _dequant(lw.gate_up_q[e], "q4k", H)
        gate, up = (gu, _dequant(lw.up_q[e], "q4k", H)) if split else (gu[:I], gu[I:])
        y = _mlp(x[t], gate, up, _dequant(lw.down_q[e], down, I))
        routed.index_add_(0, t, wb[t, k].double()[:, None] * y)
        if raw is not None:
            raw[t, k] = y
    s = [_dequant(m, "q8_0", m.shape[1] // 34 * 32) if q8 else m.double()
         for m in (lw.shared_gate, lw.shared_up, lw.shared_down)]
    prob = torch.sigmoid(x @ lw.shared_scalar_gate.double().T)
    shared = prob * _mlp(x, *s)
    out = routed + shared
    if case["stages"]:
        return {"router_logits": logits, "topk_ids": ids, "topk_weights": wb, "topk_weights_f32": w,
                "routed_sum": routed, "shared_out": shared, "shared_gate_prob": prob,
                "expert_raw": raw, "combined_out": out}
    return out if nw is None else x0.double() + out


def exact(case, seed):
    if case["op"] == "lm_head":
        h, table, _, ids = _head_inputs(case, seed)
        rows = table if ids is None else table[ids.long()]
        h = h.double()
        step = 1 << 15
        deq = (lambda r: r.double()) if case["fmt"] == "bf16" else (lambda r: _dequant(r, case["fmt"], H))
        return torch.cat([h @ deq(rows[r:r + step]).T for r in range(0, rows.shape[0], step)], 1)
    outs = [_exact_block(case, lw, x, nw) for lw, x, nw in _layers(case, seed)]
    return outs[0] if case["stages"] else outs
