"""The measured work of this library: what an engine that runs a
DeepSeek-V4-Flash decoder layer by layer has it do, through the public entry
points of the Python binding (python/dsv4_gpu.py over include/dsv4_gpu.h).

Kinds of case (one field "kind"):

  matvec     dsv4g_gemv_fp8_float: the public FP8 matvec with float block
             scales on an fp32 activation, one call per layer of a stack
  expert     dsv4g_expert_forward: single FP4 experts at one token (an engine
             that walks the experts itself)
  proj       the four FP8 attention projections of a layer, each after the
             E4M3 quantisation of its input (dsv4g_quant_fp8_act,
             dsv4g_gemv_fp8_batch_q): one token, a speculative draft, the
             largest batch that the drop-in entry takes
  head       the BF16 vocabulary head and the greedy token per row
             (dsv4g_gemv_bf16, dsv4g_argmax)
  ffn_step   the FFN half of decoder layers on the residual state of a few
             tokens (dsv4g_ffn_step: hyper-connection pre-mix, RMSNorm, MoE
             layer, post-mix), the state as the attention half left it
  moe        the decode MoE layer of a few tokens (dsv4g_moe_forward and its
             tolerance mode dsv4g_moe_forward_fast)
  moe_batch  the batched MoE layer (dsv4g_moe_forward_batch): speculative
             verify and prefill
  ffn_batch  the FFN half of a layer for a prompt (dsv4g_hc_pre with the
             RMSNorm, dsv4g_moe_forward_batch, dsv4g_hc_post)

The decode kinds (matvec, expert, proj up to 8 tokens, ffn_step, moe) are
captured once into a HIP graph and replayed, as a decode loop does; the
others are called one by one. Weights are N(0, 0.02) in the checkpoint's own
formats, activations N(0, 1) BF16 values. Decode kinds walk several layers,
so their weights come from HBM and not from the last-level cache, as in a
model of 43 layers.

The decode-path entries document results equal, bit for bit, to the scalar
loop order of the engine they serve, so their tolerance is "exact"; the
batched MoE path documents exact routing and fp32 accumulation in any order.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "deepseek-v4-flash-0731-in-c_amd", "python"))

H, I, E, K = 4096, 2048, 256, 6        # hidden, expert width, routed experts, routes per token
MULT = 4                               # hyper-connection streams
MIX = (2 + MULT) * MULT
VOCAB = 129280
LIMIT, ROUTE_SCALE, EPS = 10.0, 1.5, 1e-6
EXPERT_BYTES = 3 * H * I // 2 + 3 * H * I // 32
SHARED_BYTES = 3 * (H * I + H * I // (128 * 128))
# rows x columns of one layer's attention projections
PROJ = (("wq_a", 1024, 4096), ("wq_b", 32768, 1024), ("wkv", 512, 4096), ("wo_b", 4096, 8192))


def listed():
    return [
        # the FP8 matvec that the CPU engine's own kernel benchmark is built
        # around, over a stack of layers
        {"name": "matvec_2048x4096", "kind": "matvec", "rows": 2048, "cols": 4096, "layers": 8},
        # single experts at one token: the smallest unit an engine schedules
        {"name": "expert_1_token", "kind": "expert", "experts": 8},
        # attention projections of plain decode, of a speculative draft of
        # five, and of the largest batch that the drop-in entry allows
        {"name": "proj_1_token", "kind": "proj", "tokens": 1, "layers": 4},
        {"name": "proj_5_tokens", "kind": "proj", "tokens": 5, "layers": 4},
        {"name": "proj_33_tokens", "kind": "proj", "tokens": 33, "layers": 1},
        # the FFN half of decode, one sequence: the path of every generated token
        {"name": "ffn_decode_1_token", "kind": "ffn_step", "tokens": 1, "layers": 4},
        # the decode MoE layer for a few sequences (or drafts) at once
        {"name": "moe_decode_4_tokens", "kind": "moe", "tokens": 4, "layers": 2,
         "fast": False, "hash": False},
        # speculative verify: uneven expert loads
        {"name": "moe_verify_64", "kind": "moe_batch", "tokens": 64, "zipf": True,
         "hash": False},
        # a prompt of ordinary, ragged length through the FFN half of a layer
        {"name": "ffn_prefill_777", "kind": "ffn_batch", "tokens": 777, "zipf": True},
        # the largest prefill chunk
        {"name": "moe_prefill_4096", "kind": "moe_batch", "tokens": 4096, "zipf": True,
         "hash": False},
        # logits of one sequence, and of a verify batch
        {"name": "head_1_token", "kind": "head", "tokens": 1, "vocab": VOCAB},
        {"name": "head_64_tokens", "kind": "head", "tokens": 64, "vocab": VOCAB},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("matvec", "expert", "proj", "ffn_step", "moe", "moe_batch", "moe_batch",
                       "ffn_batch", "head"))
    if kind == "matvec":
        # rows and widths of the model's matrices and odd ones between
        cols = rng.choice((512, 1024, 2048, 4096, 16 * rng.randint(24, 256)))
        return {"kind": kind, "rows": _log(rng, 192, 4096), "cols": cols,
                "layers": rng.randint(4, 12)}
    if kind == "expert":
        return {"kind": kind, "experts": rng.randint(2, 40)}
    if kind == "proj":
        return {"kind": kind, "tokens": _log(rng, 1, 33), "layers": rng.randint(2, 4)}
    if kind == "ffn_step":
        return {"kind": kind, "tokens": rng.randint(1, 6), "layers": rng.randint(2, 4)}
    if kind == "moe":
        return {"kind": kind, "tokens": rng.randint(1, 7), "layers": rng.randint(2, 3),
                "fast": rng.random() < 0.4, "hash": rng.random() < 0.3}
    if kind == "moe_batch":
        return {"kind": kind, "tokens": _log(rng, 8, 4000), "zipf": rng.random() < 0.7,
                "hash": rng.random() < 0.2}
    if kind == "ffn_batch":
        return {"kind": kind, "tokens": _log(rng, 8, 2200), "zipf": rng.random() < 0.7}
    return {"kind": kind, "tokens": _log(rng, 1, 64), "vocab": _log(rng, 16384, VOCAB)}


# ------------------------------------------------------------------ inputs

def _lib():
    import dsv4_gpu
    return dsv4_gpu.lib()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _bf16(t):
    """BF16 values held as fp32, the form that the entries take."""
    return t.to(torch.bfloat16).to(torch.float32).contiguous()


def _bits16(t):
    return t.to(torch.bfloat16).view(torch.int16).contiguous()


def _tokens(g, n, width):
    return _bf16(torch.randn(n, width, generator=g, device="cuda"))


def _zipf_bias(seed):
    """Router bias of Zipf(1.2) expert popularity over a random permutation:
    0.15 * (log p_rank - mean)."""
    rng = np.random.default_rng(seed)
    p = np.arange(1, E + 1, dtype=np.float64) ** -1.2
    b = np.empty(E)
    b[rng.permutation(E)] = np.log(p / p.sum())
    return (0.15 * (b - b.mean())).astype(np.float32)


def _layer(seed, zipf=False, hash_vocab=0):
    import synth
    layer = synth.device_layer(seed=seed, hidden=H, inter=I, n_experts=E, topk=K)
    extra = {}
    if zipf:
        extra["bias"] = torch.from_numpy(_zipf_bias(seed)).cuda()
    if hash_vocab:
        g = _gen(seed + 1)
        # K different experts per token id
        extra["tid2eid"] = torch.rand(hash_vocab, E, generator=g, device="cuda").topk(K)[1] \
            .to(torch.int64).contiguous()
    return type(layer)(dict(layer.tensors, **extra), layer.meta) if extra else layer


def _fp8_matrix(g, rows, cols, mode):
    w = torch.randn(rows, cols, generator=g, device="cuda") * 0.02
    codes = torch.empty(rows, cols, dtype=torch.uint8, device="cuda")
    scales = torch.empty((rows + 127) // 128, (cols + 127) // 128, device="cuda",
                         dtype=torch.float32 if mode else torch.uint8)
    _lib().quant_fp8_blocks(w, codes, scales, mode=mode)
    return codes, scales


def _hc(g):
    """One layer's hyper-connection parameters and its FFN norm."""
    return {"fn": torch.randn(MIX, MULT * H, generator=g, device="cuda") * 0.01,
            "scale": torch.rand(3, generator=g, device="cuda") + 0.5,
            "base": torch.randn(MIX, generator=g, device="cuda") * 0.5,
            "norm": _bits16(1 + 0.1 * torch.randn(H, generator=g, device="cuda"))}


def _captured(call):
    """call() run once and then captured: (graph, the captured call's outputs).
    Every buffer that call() names is kept by the caller's state, since the
    graph holds bare addresses."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


def _inputs(case, seed):
    """The case's weights and activations, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    s = {}
    if kind == "matvec":
        s["x"] = torch.randn(case["layers"], case["cols"], generator=g, device="cuda")
        s["w"] = [_fp8_matrix(g, case["rows"], case["cols"], 1) for _ in range(case["layers"])]
    elif kind == "expert":
        s["x"] = _tokens(g, 1, H)
        s["layer"] = _expert_pool(seed, case["experts"])
    elif kind == "proj":
        n = case["tokens"]
        s["layers"] = [{name: (_tokens(g, n, cols), *_fp8_matrix(g, rows, cols, 0))
                        for name, rows, cols in PROJ} for _ in range(case["layers"])]
    elif kind == "head":
        s["x"] = _tokens(g, case["tokens"], H)
        s["w"] = _bits16(torch.randn(case["vocab"], H, generator=g, device="cuda") * 0.02)
    else:
        n = case["tokens"]
        count = case.get("layers", 1)
        vocab = 4096 if case.get("hash") else 0
        s["layers"] = [_layer(16 * seed + l, case.get("zipf", False), vocab)
                       for l in range(count)]
        if vocab:
            s["ids"] = torch.randint(0, vocab, (n,), generator=g, device="cuda",
                                     dtype=torch.int32)
        if kind in ("ffn_step", "ffn_batch"):
            s["hc"] = [_hc(g) for _ in range(count)]
            # what the attention halves left: one residual state per layer (the
            # layers of a case do not feed each other, so that a rounding in
            # one is not carried through the routing of the next)
            s["attended"] = _bf16(torch.randn(count, n, MULT * H, generator=g, device="cuda")
                                  * 0.5)
            s["state"] = torch.empty_like(s["attended"])
        else:
            s["x"] = [_tokens(g, n, H) for _ in range(count)]
    return s


def _expert_pool(seed, count):
    import synth
    return synth.device_layer(seed=seed, hidden=H, inter=I, n_experts=count, topk=1)


# ------------------------------------------------------------------- calls

def prepare(case, seed):
    lib, s = _lib(), _inputs(case, seed)
    kind = case["kind"]
    s["kind"] = kind
    if kind == "matvec":
        rows, cols = case["rows"], case["cols"]
        s["graph"], s["out"] = _captured(lambda: [
            lib.gemv_fp8_float(s["x"][l], w, ws, cols, rows, 128, 0)
            for l, (w, ws) in enumerate(s["w"])])
    elif kind == "expert":
        m, experts = s["layer"].meta, s["layer"].tensors["experts"]
        ws = s["ws"] = torch.empty(lib.expert_workspace_bytes(I), dtype=torch.uint8,
                                   device="cuda")
        stride = m["expert_stride"]

        def call():
            qx, qs = lib.quant_fp8_act(s["x"])
            return [lib.expert_forward(torch.empty(H, device="cuda"), qx[0], qs[0],
                                       experts[e * stride:(e + 1) * stride], m["scale_run"],
                                       H, I, LIMIT, None, ws) for e in range(case["experts"])]
        s["graph"], s["out"] = _captured(call)
    elif kind == "proj":
        if case["tokens"] <= 8:
            s["graph"], s["out"] = _captured(lambda: _proj(lib, s["layers"]))
    elif kind == "ffn_step":
        ws = s["ws"] = torch.zeros(
            lib.ffn_step_workspace_bytes(s["layers"][0], MULT, case["tokens"]),
            dtype=torch.uint8, device="cuda")

        def call():
            s["state"].copy_(s["attended"])
            return [lib.ffn_step(state, hc["fn"], hc["scale"], hc["base"], hc["norm"], layer,
                                 MULT, workspace=ws, check=False)
                    for state, layer, hc in zip(s["state"], s["layers"], s["hc"])]
        s["graph"], s["out"] = _captured(call)
    elif kind == "moe":
        ws = s["ws"] = lib.new_moe_workspace(s["layers"][0], case["tokens"], "cuda")
        s["graph"], s["out"] = _captured(lambda: [
            lib.moe_forward(layer, x, s.get("ids"), workspace=ws, fast=case["fast"],
                            check=False) for layer, x in zip(s["layers"], s["x"])])
    elif kind != "head":
        s["ws"] = torch.empty(lib.moe_batch_workspace_bytes(s["layers"][0], case["tokens"]),
                              dtype=torch.uint8, device="cuda")
    return s


def _proj(lib, layers):
    out = []
    for layer in layers:
        for name, rows, cols in PROJ:
            x, w, ws = layer[name]
            qx, qs = lib.quant_fp8_act(x)
            out.append(lib.gemv_fp8_batch_q(qx, qs, w, ws, cols, rows))
    return out


def run(s):
    lib, kind = _lib(), s["kind"]
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    if kind == "proj":
        return _proj(lib, s["layers"])
    if kind == "head":
        logits = lib.gemv_bf16(s["x"], s["w"], H, s["w"].shape[0])
        return logits, lib.argmax(logits)
    layer = s["layers"][0]
    if kind == "moe_batch":
        return lib.moe_forward_batch(layer, s["x"][0], s.get("ids"), workspace=s["ws"])
    state, hc = s["state"][0], s["hc"][0]
    s["state"].copy_(s["attended"])
    x, post, comb = lib.hc_pre(state, hc["fn"], hc["scale"], hc["base"], MULT, hc["norm"])
    branch, idx, wt = lib.moe_forward_batch(layer, x, workspace=s["ws"])
    lib.hc_post(state, branch, post, comb, MULT)
    return state, idx, wt


# -------------------------------------------------------------- what it costs

def _experts_hit(tokens, zipf, hash_):
    """Different experts that so many tokens reach (a routing drawn on the host
    with the case's router statistics)."""
    rng = np.random.default_rng(5)
    if hash_:
        choice = rng.random((tokens, E))
    else:
        z = rng.standard_normal((tokens, E))
        choice = np.sqrt(np.log1p(np.exp(z))) + (_zipf_bias(1)[None] if zipf else 0.0)
    return len(np.unique(np.argpartition(-choice, K - 1, axis=1)[:, :K]))


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        r, c, n = case["rows"], case["cols"], case["layers"]
        blocks = ((r + 127) // 128) * ((c + 127) // 128)
        return {"bytes": n * (r * c + 4 * (blocks + r + c)), "flops": 2 * n * r * c}
    if kind == "expert":
        n = case["experts"]
        return {"bytes": n * (EXPERT_BYTES + 4 * H) + 4 * H, "flops": 6 * n * H * I}
    if kind == "head":
        n, v = case["tokens"], case["vocab"]
        return {"bytes": 2 * v * H + 4 * n * (H + v + 1), "flops": 2 * n * v * H}
    n = case["tokens"]
    if kind == "proj":
        b = sum(r * c + (r // 128) * (c // 128) + 4 * n * (r + c) for _, r, c in PROJ)
        f = sum(2 * n * r * c for _, r, c in PROJ)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    hit = _experts_hit(n, case.get("zipf", False), case.get("hash", False))
    b = hit * EXPERT_BYTES + SHARED_BYTES + 2 * E * H + 8 * n * K
    f = 6 * H * I * n * (K + 1) + 2 * E * H * n
    if kind in ("ffn_step", "ffn_batch"):
        b += 4 * MIX * MULT * H + 2 * H + 8 * n * MULT * H
        f += 2 * MIX * MULT * H * n + 2 * n * MULT * H * (MULT + 2)
    else:
        b += 8 * n * H
    count = case.get("layers", 1)
    return {"bytes": count * b, "flops": count * f}


def tolerance(case):
    """The decode-path entries give the scalar loop's bits. The batched MoE
    layer sums in fp32 in any order between BF16 and E4M3 roundings of its
    intermediate values, so a last-bit difference of a sum moves some of them
    by one step: 1e-4 to 3e-4 in the 2-norm against the same in 64 bits."""
    if case["kind"] in ("moe_batch", "ffn_batch") or case.get("fast"):
        return {"rel": 1e-3, "max": 0.06, "differ": 0.0}
    return "exact"


# ------------------------------------------------------- the same in 64 bits

def _r16(t):
    """BF16 rounding of 64-bit values, kept in 64 bits."""
    return t.to(torch.float32).to(torch.bfloat16).to(torch.float64)


def _quant64(x):
    """E4M3 quantisation per 128 columns with a power-of-two scale: the values."""
    n, width = x.shape
    g = x.view(n, width // 128, 128)
    amax = g.abs().amax(-1, keepdim=True).clamp(min=1e-4)
    scale = torch.exp2(torch.ceil(torch.log2(amax / 448.0)))
    q = (g / scale).clamp(-448.0, 448.0)
    step = torch.exp2(torch.floor(torch.log2(q.abs().clamp(min=2.0 ** -6))) - 3)
    return (torch.round(q / step) * step * scale).view(n, width)


def _fp4_64(packed, scales, rows, cols):
    mag = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64,
                       device="cuda")
    values = torch.cat([mag, -mag])
    b = packed.view(rows, cols // 2)
    w = torch.stack([values[(b & 15).long()], values[(b >> 4).long()]], -1).view(rows, cols)
    s = torch.exp2(scales.view(rows, cols // 32).to(torch.float64) - 127)
    return w * s.repeat_interleave(32, 1)


def _fp8_64(codes, scales, rows, cols):
    w = codes.view(torch.float8_e4m3fn).to(torch.float32).to(torch.float64)
    s = scales.to(torch.float64) if scales.dtype == torch.float32 \
        else torch.exp2(scales.to(torch.float64) - 127)
    return w * s.repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :cols]


def _swiglu64(g, u, weight):
    g, u = _r16(g).clamp(max=LIMIT), _r16(u).clamp(-LIMIT, LIMIT)
    return _quant64(_r16(g / (1 + torch.exp(-g)) * u * weight))


def _expert64(experts, meta, e, xq, weight):
    slot = experts[e * meta["expert_stride"]:(e + 1) * meta["expert_stride"]]
    scales, w = slot[:meta["scale_run"]], slot[meta["scale_run"]:]
    ns, nw = H * I // 32, H * I // 2
    w1, w2, w3 = (_fp4_64(w[k * nw:(k + 1) * nw], scales[k * ns:(k + 1) * ns], r, c)
                  for k, (r, c) in enumerate(((I, H), (H, I), (I, H))))
    return _r16(_swiglu64(xq @ w1.T, xq @ w3.T, weight) @ w2.T)


def _moe64(layer, x, ids=None):
    t, x = layer.tensors, x.to(torch.float64)
    z = x @ t["gate_w"].view(torch.bfloat16).to(torch.float64).T
    score = torch.sqrt(torch.nn.functional.softplus(z, threshold=100.0))
    if ids is not None:
        idx = t["tid2eid"][ids.long()]
    else:
        bias = t.get("bias")
        idx = (score if bias is None else score + bias.to(torch.float64)).topk(K)[1]
    idx = idx.sort(-1)[0]
    wt = score.gather(1, idx)
    wt = wt * (ROUTE_SCALE / wt.sum(-1, keepdim=True))
    xq = _quant64(x)
    out = torch.zeros_like(x)
    for e in idx.unique().tolist():
        tok, slot = (idx == e).nonzero(as_tuple=True)
        out[tok] += _expert64(t["experts"], layer.meta, e, xq[tok], wt[tok, slot][:, None])
    sh = [_fp8_64(t[n], t[n + "_s"], *t[n].shape) for n in ("sh1", "sh3", "sh2")]
    out += _r16(_swiglu64(xq @ sh[0].T, xq @ sh[1].T, 1.0) @ sh[2].T)
    return _r16(out), idx.to(torch.int32), wt


def _hc_pre64(state, hc):
    n = state.shape[0]
    rs = 1 / torch.sqrt((state * state).mean(-1, keepdim=True) + EPS)
    mixes = (state @ hc["fn"].to(torch.float64).T) * rs
    sc, base = hc["scale"].to(torch.float64), hc["base"].to(torch.float64)
    pre = torch.sigmoid(mixes[:, :MULT] * sc[0] + base[:MULT]) + EPS
    post = 2 * torch.sigmoid(mixes[:, MULT:2 * MULT] * sc[1] + base[MULT:2 * MULT])
    c = (mixes[:, 2 * MULT:] * sc[2] + base[2 * MULT:]).view(n, MULT, MULT)
    c = torch.softmax(c, -1) + EPS
    c = c / (c.sum(1, keepdim=True) + EPS)
    for _ in range(19):
        c = c / (c.sum(2, keepdim=True) + EPS)
        c = c / (c.sum(1, keepdim=True) + EPS)
    x = _r16((pre[:, :, None] * state.view(n, MULT, H)).sum(1))
    r = 1 / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return _r16(x * r * hc["norm"].view(torch.bfloat16).to(torch.float64)), post, c


def _ffn64(state, hc, layer):
    x, post, comb = _hc_pre64(state, hc)
    branch, idx, wt = _moe64(layer, x)
    n = state.shape[0]
    new = post[:, :, None] * branch[:, None, :] + comb @ state.view(n, MULT, H)
    return _r16(new).view(n, MULT * H), idx, wt


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "matvec":
        return [_fp8_64(w, ws, case["rows"], case["cols"]) @ s["x"][l].to(torch.float64)
                for l, (w, ws) in enumerate(s["w"])]
    if kind == "expert":
        layer, xq = s["layer"], _quant64(s["x"].to(torch.float64))
        return [_expert64(layer.tensors["experts"], layer.meta, e, xq, 1.0)[0]
                for e in range(case["experts"])]
    if kind == "proj":
        return [_r16(_quant64(layer[name][0].to(torch.float64))
                     @ _fp8_64(layer[name][1], layer[name][2], rows, cols).T)
                for layer in s["layers"] for name, rows, cols in PROJ]
    if kind == "head":
        x = s["x"].to(torch.float64)
        logits = torch.cat([x @ w.view(torch.bfloat16).to(torch.float64).T
                            for w in s["w"].split(8192)], 1)
        return logits, logits.argmax(-1).to(torch.int32)
    if kind == "moe":
        return [_moe64(layer, x, s.get("ids")) for layer, x in zip(s["layers"], s["x"])]
    if kind == "moe_batch":
        return _moe64(s["layers"][0], s["x"][0], s.get("ids"))
    out = [_ffn64(state.to(torch.float64), hc, layer)
           for state, layer, hc in zip(s["attended"], s["layers"], s["hc"])]
    return out if kind == "ffn_step" else out[0]
