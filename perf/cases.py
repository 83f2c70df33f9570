"""Performance cases of the butterquant library: what a serving program has it do.

A case is one pass of one block of the 128-expert decoder (hidden 2816, dense MLP
2112, experts 704 wide with top-8 routing, 16 query heads) or of a single call, through
the calls of the `bq` package:

  attn    the attention block: norm-quant with the q/k/v projections, the head
          prep into the paged int8 cache, flash attention, block-quant and the
          output projection.  "sliding" layers have 8 kv heads of 256 and a
          1024-position window over a ring of two 1024-row pages; "full" layers
          have 2 kv heads of 512, one projection for k and v, and every position
  ffn     the feed-forward block: router logits, the combined prep, gate/up and
          down calls with the dense MLP beside the experts
  moe     the expert block alone, from given router logits
  linear  norm-quant and one per-row linear
  head    the vocabulary head: head prep and flash sampling
  load    one weight quantized from bf16 and laid out for the device

Decode steps ("graph") are captured once and replayed, as a serving loop does with
buffers that it keeps; everything else is called directly with kept outputs.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mojo-gemma4-cpu_amd"))
import bq  # noqa: E402

HIDDEN, DENSE, INTER = 2816, 2112, 704
MOE = dict(experts=128, topk=8)
NUM_Q, PAGE, WINDOW, VOCAB = 16, 1024, 1024, 262144
LAYER = {"sliding": dict(nkv=8, hd=256, window=WINDOW, rope=128),
         "full": dict(nkv=2, hd=512, window=0, rope=64)}
DEV = "cuda"


def _decode(n, ctx):
    """n sequences of one new token each, their lengths spread below ctx."""
    return ",".join("%d:1" % (ctx - 1 - (37 * i) % max(1, ctx // 2)) for i in range(n))


def listed():
    return [
        # one chat stream: the attention block of one token, 1500 positions in
        dict(name="attn_decode_1_sliding", kind="attn", layer="sliding", seqs="1499:1", graph=True),
        # a full batch of a serving loop, in a layer that sees all 4096 positions
        dict(name="attn_decode_16_full", kind="attn", layer="full", seqs=_decode(16, 4096), graph=True),
        # a long prompt's first chunk
        dict(name="attn_prefill_2048_sliding", kind="attn", layer="sliding", seqs="0:2048", graph=False),
        # a ragged prefill step: a fresh prompt and a later chunk of another
        dict(name="attn_prefill_1111_full", kind="attn", layer="full", seqs="0:700,1500:411", graph=False),
        # one chat stream: the feed-forward block of one token
        dict(name="ffn_decode_1", kind="ffn", tokens=1, **MOE, graph=True),
        # the feed-forward block of a continuous batch of 16
        dict(name="ffn_decode_16", kind="ffn", tokens=16, **MOE, graph=True),
        # a short ragged prompt
        dict(name="ffn_prefill_333", kind="ffn", tokens=333, **MOE, graph=False),
        # the expert block at a large decode batch and at a prefill chunk
        dict(name="moe_decode_32", kind="moe", tokens=32, **MOE, graph=True),
        dict(name="moe_prefill_2048", kind="moe", tokens=2048, **MOE, graph=False),
        # a single projection of a prefill chunk
        dict(name="linear_prefill_512", kind="linear", tokens=512, k=4096, n=4096, graph=False),
        # sampling the next token of a batch over the whole vocabulary
        dict(name="head_8", kind="head", rows=8, vocab=VOCAB, graph=True),
        # loading: an output projection's weight
        dict(name="load_2816x4096", kind="load", rows=2816, k=4096, graph=False),
    ]


def _logint(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "ffn", "ffn", "moe", "linear", "head", "load"])
    if kind == "attn":
        layer = rng.choice(["sliding", "full"])
        if rng.random() < 0.5:  # decode
            n, ctx = rng.randint(1, 32), _logint(rng, 40, 6000)
            seqs = ",".join("%d:1" % rng.randint(ctx // 2, ctx) for _ in range(n))
            return dict(kind=kind, layer=layer, seqs=seqs, graph=True)
        n = _logint(rng, 48, 1400)
        base = rng.choice([0, 0, rng.randint(1, 600 if layer == "sliding" else 900)])
        seqs = "%d:%d" % (base, n)
        if rng.random() < 0.4:
            seqs += ",0:%d" % _logint(rng, 20, 500)
        return dict(kind=kind, layer=layer, seqs=seqs, graph=False)
    if kind in ("ffn", "moe"):
        t = _logint(rng, 1, 2000 if kind == "moe" else 1500)
        # the model's routing most of the time, else a smaller expert set
        experts, topk = rng.choice([(128, 8), (128, 8), (128, 8), (128, 4), (96, 6), (64, 8), (32, 4)])
        return dict(kind=kind, tokens=t + (t in (1, 16, 32)), experts=experts, topk=topk, graph=t <= 32)
    if kind == "linear":
        t = _logint(rng, 1, 2048)
        return dict(kind=kind, tokens=t, k=128 * rng.randint(8, 40), n=16 * rng.randint(60, 400),
                    graph=t <= 32)
    if kind == "head":
        return dict(kind=kind, rows=rng.randint(1, 32), vocab=16 * _logint(rng, 1000, VOCAB // 16),
                    graph=True)
    return dict(kind=kind, rows=16 * _logint(rng, 32, 500), k=128 * rng.randint(4, 44), graph=False)


# ---------------------------------------------------------------------------
# inputs: everything below is a function of (seed, tag), so exact() makes the
# same row-major codes that prepare() lays out
# ---------------------------------------------------------------------------

def _gen(seed, tag):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + sum(ord(c) * 131 ** i for i, c in
                                                                         enumerate(tag))) % (1 << 62))


def _codes(seed, tag, n, k):
    """Row-major int8 codes of a rotated weight: near-normal, the row's largest about 127."""
    g = _gen(seed, tag)
    out = torch.empty(n, k, dtype=torch.int8, device=DEV)
    step = max(16, (1 << 26) // k)
    for r in range(0, n, step):
        w = torch.empty(min(step, n - r), k, device=DEV).normal_(0.0, 35.0, generator=g)
        out[r:r + step] = w.round_().clamp_(-127, 127).to(torch.int8)
    return out


def _scales(seed, tag, *shape):
    """The scales (largest value over 127) of weights of deviation 0.02."""
    return (0.02 / 35) * (0.9 + 0.2 * torch.rand(*shape, device=DEV, generator=_gen(seed, tag + ".scale")))


def _weight(seed, tag, n, k):
    return bq.ButterquantWeight(bq.retile(_codes(seed, tag, n, k), n, k), _scales(seed, tag, n), n, k)


def _normal(seed, tag, *shape, mean=0.0, std=1.0):
    return mean + std * torch.randn(*shape, device=DEV, generator=_gen(seed, tag))


def _bf(t):
    return t.to(torch.bfloat16)


def _e(*shape, dt=torch.bfloat16):
    return torch.empty(*shape, dtype=dt, device=DEV)


def _seqs(case):
    return [tuple(int(v) for v in s.split(":")) for s in case["seqs"].split(",")]


def _attn_inputs(case, seed):
    """Hidden rows, gains, RoPE tables and a paged cache that holds each
    sequence's earlier positions."""
    L, seqs = LAYER[case["layer"]], _seqs(case)
    nkv, hd, sliding = L["nkv"], L["hd"], L["window"] > 0
    T = sum(n for _, n in seqs)
    pages = [2 if sliding else (b + n + PAGE - 1) // PAGE for b, n in seqs]
    perm = np.random.RandomState(seed % (1 << 31)).permutation(sum(pages))
    runs, buf, off = [], 0, 0
    for (b, n), p in zip(seqs, pages):
        runs.append((buf, b, off, p))
        buf, off = buf + n, off + p
    slots, kvs = sum(pages) * PAGE, nkv * hd
    maxpos = max(b + n for b, n in seqs)
    ang = (torch.arange(maxpos, device=DEV, dtype=torch.float64)[:, None] *
           10000.0 ** (-torch.arange(L["rope"], device=DEV, dtype=torch.float64) / L["rope"]))
    return dict(
        T=T, seqs=seqs, nkv=nkv, hd=hd, window=L["window"], rope=L["rope"], slots=slots,
        page_mask=1 if sliding else -1, max_kv=L["window"] if sliding else maxpos,
        x=_bf(_normal(seed, "x", T, HIDDEN)), gamma=_bf(_normal(seed, "gamma", HIDDEN, mean=1, std=0.1)),
        qn=_bf(_normal(seed, "qn", hd, mean=0.35, std=0.03)),
        kn=_bf(_normal(seed, "kn", hd, mean=0.35, std=0.03)),
        cos=ang.cos().float(), sin=ang.sin().float(),
        kc=_codes(seed, "kc", slots, kvs), vc=_codes(seed, "vc", slots, kvs),
        ks=0.35 * (3 + torch.rand(slots, nkv, device=DEV, generator=_gen(seed, "ks"))),
        vs=3 + torch.rand(slots, nkv, device=DEV, generator=_gen(seed, "vs")),
        runs=torch.tensor(runs, dtype=torch.int32, device=DEV),
        rows=torch.tensor([int(p) * PAGE for p in perm], dtype=torch.int32, device=DEV))


def _params(rows, seed):
    """Sampling parameters as a server's requests mix them."""
    r = np.random.RandomState(seed % (1 << 31))
    p = np.zeros(rows, np.dtype([("temperature", "<f4"), ("min_p", "<f4"), ("top_k", "<i8"),
                                 ("seed", "<u8"), ("n_keep", "<i8"), ("greedy", "u1"), ("pad", "u1", 7)]))
    p["temperature"] = r.choice([0.7, 1.0, 1.3], rows)
    p["min_p"], p["top_k"] = r.choice([0.0, 0.05], rows), r.choice([0, 64], rows)
    p["seed"], p["n_keep"], p["greedy"] = r.randint(0, 1 << 30, rows), 256, r.rand(rows) < 0.2
    return p


def prepare(case, seed):
    kind, s = case["kind"], {}
    if kind == "attn":
        s = _attn_inputs(case, seed)
        T, nkv, hd = s["T"], s["nkv"], s["hd"]
        s["wq"], s["wk"] = _weight(seed, "wq", NUM_Q * hd, HIDDEN), _weight(seed, "wk", nkv * hd, HIDDEN)
        if s["window"]:
            s["wv"] = _weight(seed, "wv", nkv * hd, HIDDEN)
        s["wo"] = _weight(seed, "wo", HIDDEN, NUM_Q * hd)
        s["q"], s["k"] = _e(T, NUM_Q * hd), _e(T, nkv * hd)
        s["v"] = _e(T, nkv * hd) if s["window"] else s["k"]
        s["act"] = (_e(T, HIDDEN, dt=torch.int8), _e(T, dt=torch.float32))
        s["heads"] = (_e(T, NUM_Q * hd, dt=torch.int8), _e(T, NUM_Q, dt=torch.float32),
                      _e(T, NUM_Q, dt=torch.float32))
        s["splits"] = bq.attention_splits(T, nkv, s["max_kv"])
        s["ws"] = bq.attention_workspace(T, NUM_Q, hd, s["splits"])
        s["o"], s["y"] = _e(T, NUM_Q * hd), _e(T, HIDDEN)
        s["oq"] = (_e(T, NUM_Q * hd, dt=torch.int8), _e(T, NUM_Q, dt=torch.float32))
        s["geo"] = (NUM_Q, nkv, hd)
        s["paging"] = (int(math.log2(PAGE)), PAGE - 1, s["page_mask"])
    elif kind in ("ffn", "moe"):
        T, E, K = case["tokens"], case["experts"], case["topk"]
        s = dict(T=T, E=E, K=K, x=_bf(_normal(seed, "x", T, HIDDEN)),
                 gamma=_bf(_normal(seed, "gamma", HIDDEN, mean=1, std=0.1)),
                 pes=_bf(_normal(seed, "pes", E, mean=1, std=0.1)),
                 wgu=_weight(seed, "wgu", E * 2 * INTER, HIDDEN),
                 wd=_weight(seed, "wd", E * HIDDEN, INTER),
                 route=(_e(T, K, dt=torch.int32), _e(T, K, dt=torch.float32), _e(E + 1, dt=torch.int32),
                        torch.zeros(T * K, 2, dtype=torch.int32, device=DEV)),
                 act=(_e(T, HIDDEN, dt=torch.int8), _e(T, dt=torch.float32)),
                 bucket=(_e(T * K, INTER, dt=torch.int8), _e(T * K, INTER // 64, dt=torch.float32)),
                 ws=_e(max(bq.moe_phase2_workspace_size(T, K, HIDDEN), 256), dt=torch.uint8),
                 accum=_e(T, HIDDEN, dt=torch.float32), out=_e(T, HIDDEN))
        if kind == "ffn":
            s.update(dgamma=_bf(_normal(seed, "dgamma", HIDDEN, mean=1, std=0.1)),
                     proj=_bf(_normal(seed, "proj", E, HIDDEN, std=0.02)),
                     rscale=_bf(_normal(seed, "rscale", HIDDEN, mean=1, std=0.1)),
                     logits=_e(T, E, dt=torch.float32),
                     dg=_weight(seed, "dg", DENSE, HIDDEN), du=_weight(seed, "du", DENSE, HIDDEN),
                     dd=_weight(seed, "dd", HIDDEN, DENSE),
                     dact=(_e(T, HIDDEN, dt=torch.int8), _e(T, dt=torch.float32)),
                     dq=(_e(T, DENSE, dt=torch.int8), _e(T, DENSE // 64, dt=torch.float32)),
                     dout=_e(T, HIDDEN))
        else:
            s["logits"] = _normal(seed, "logits", T, E)
    elif kind == "linear":
        T, k, n = case["tokens"], case["k"], case["n"]
        s = dict(x=_bf(_normal(seed, "x", T, k)), gamma=_bf(_normal(seed, "gamma", k, mean=1, std=0.1)),
                 w=_weight(seed, "w", n, k), out=_e(T, n),
                 act=(_e(T, k, dt=torch.int8), _e(T, dt=torch.float32)))
    elif kind == "head":
        R, V = case["rows"], case["vocab"]
        s = dict(x=_bf(_normal(seed, "x", R, HIDDEN)),
                 gamma=_bf(_normal(seed, "gamma", HIDDEN, mean=1, std=0.1)),
                 w=_weight(seed, "w", V, HIDDEN), wscales=_scales(seed, "blocks", V, HIDDEN // 128),
                 params=torch.from_numpy(_params(R, seed).view(np.uint8).reshape(R, -1)).to(DEV),
                 act=(_e(R, HIDDEN, dt=torch.int8), _e(R, HIDDEN // 128, dt=torch.float32)),
                 ws=_e(max(bq.flash_sample_workspace_size(R, V), 256), dt=torch.uint8),
                 out=_e(R, bq.OUTCOME_BYTES, dt=torch.uint8))
    elif kind == "load":
        s = dict(w=_bf(_normal(seed, "w", case["rows"], case["k"], std=0.02)))
    s["kind"] = kind
    if case["graph"]:
        _pass(s)  # the first call loads the kernels, outside the capture
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            s["outputs"] = _pass(s)
        s["graph"] = g
    return s


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    return _pass(state)


def _pass(s):
    kind = s["kind"]
    if kind == "attn":
        if s["window"]:
            bq.norm_qkv(s["x"], s["gamma"], s["wq"], s["wk"], s["wv"], outs=(s["q"], s["k"], s["v"]),
                        act_out=s["act"])
        else:
            bq.norm_linear_pair(s["x"], s["gamma"], s["wq"], s["wk"], outs=(s["q"], s["k"]),
                                act_out=s["act"])
        cache = (s["kc"], s["ks"], s["vc"], s["vs"])
        bq.attn_prep(s["q"], s["k"], s["v"], s["qn"], s["kn"], *cache, s["cos"], s["sin"], s["runs"],
                     s["rows"], *s["geo"], s["rope"], s["hd"] // 2, *s["paging"], out=s["heads"])
        bq.attention(*s["heads"], *cache, s["runs"], s["rows"], *s["geo"], s["window"], *s["paging"],
                     s_max=s["splits"], workspace=s["ws"], out=s["o"])
        bq.block_quant(s["o"], s["hd"], False, out=s["oq"])
        bq.block_linear(*s["oq"], s["wo"], s["hd"], out=s["y"])
        return dict(y=s["y"], o=s["o"], q=s["heads"][0], k_cache=s["kc"], k_scale=s["ks"],
                    v_cache=s["vc"], v_scale=s["vs"])
    if kind == "ffn":
        T, E, K = s["T"], s["E"], s["K"]
        bq.router_logits(s["x"], s["proj"], s["rscale"], out=s["logits"])
        idx, w, eo, routes, *_ = bq.ffn_prep(s["logits"], s["x"], s["gamma"], s["dgamma"], K, s["pes"],
                                             out=s["route"] + s["act"] + s["dact"])
        bq.ffn_gate_up(*s["act"], eo, routes, s["wgu"], E, T, K, INTER, *s["dact"], s["dg"],
                       s["du"], out=s["bucket"] + s["dq"])
        bq.ffn_down(*s["bucket"], eo, routes, s["wd"], E, T, K, HIDDEN, *s["dq"], s["dd"],
                    workspace=s["ws"], out=(s["accum"], s["out"], s["dout"]))
        return dict(logits=s["logits"], idx=idx, weight=w, accum=s["accum"], out=s["out"], dense=s["dout"])
    if kind == "moe":
        T, E, K = s["T"], s["E"], s["K"]
        idx, w, eo, routes, *_ = bq.moe_prep(s["logits"], s["x"], s["gamma"], K, s["pes"],
                                             out=s["route"] + s["act"])
        bq.moe_phase1_quant(*s["act"], eo, routes, s["wgu"], E, T, K, INTER,
                            out=s["bucket"] + (None,))
        bq.moe_phase2(*s["bucket"], eo, routes, s["wd"], E, T, K, HIDDEN, workspace=s["ws"],
                      out=(s["accum"], s["out"]))
        return dict(idx=idx, weight=w, accum=s["accum"], out=s["out"])
    if kind == "linear":
        y, (xq, sa) = bq.norm_linear(s["x"], s["gamma"], s["w"], out=s["out"], act_out=s["act"])
        return dict(y=y, act=xq, act_scale=sa)
    if kind == "head":
        xq, sa = bq.head_prep(s["x"], s["gamma"], out=s["act"])
        o = bq.flash_sample(xq, sa, s["w"], s["wscales"], s["params"], workspace=s["ws"],
                            out=s["out"]).view(torch.int32)
        f = o.view(torch.float32)
        return dict(token=o[:, 0], logz=f[:, 1], n=o[:, 2], values=f[:, 4:260], indices=o[:, 260:516])
    codes, scales = bq.quantize_weight(s["w"], 128)
    return dict(codes=bq.retile(codes, *codes.shape), scales=scales)


def _kv_positions(case):
    w = LAYER[case["layer"]]["window"]
    return sum(min(w, b + t + 1) if w else b + t + 1 for b, n in _seqs(case) for t in range(n))


def work(case):
    kind = case["kind"]
    wb = lambda n, k: n * k + 4 * n  # noqa: E731  codes and row scales
    if kind == "attn":
        L, seqs = LAYER[case["layer"]], _seqs(case)
        T, nkv, hd = sum(n for _, n in seqs), L["nkv"], L["hd"]
        proj = (NUM_Q + nkv * (2 if L["window"] else 1)) * hd
        # each sequence's cache rows in reach are read once, new rows written once
        reach = sum(min(b, L["window"] - 1) if L["window"] else b for b, _ in seqs)
        return {"bytes": wb(proj, HIDDEN) + wb(HIDDEN, NUM_Q * hd) + 4 * T * HIDDEN + 2 * T * NUM_Q * hd +
                T * NUM_Q * hd + (reach + T) * nkv * (2 * hd + 8),
                "flops": 2 * T * HIDDEN * (proj + NUM_Q * hd) + 4 * _kv_positions(case) * NUM_Q * hd}
    if kind in ("ffn", "moe"):
        T, E, K = case["tokens"], case["experts"], case["topk"]
        touched = E * (1 - (1 - K / E) ** T)
        b = touched * (wb(2 * INTER, HIDDEN) + wb(HIDDEN, INTER)) + T * (HIDDEN * (2 + 4 + 2) + 8 * K + 4 * E)
        f = 2 * T * K * 3 * INTER * HIDDEN
        if kind == "ffn":
            b += 2 * wb(DENSE, HIDDEN) + wb(HIDDEN, DENSE) + 2 * T * HIDDEN + 2 * E * HIDDEN
            f += 2 * T * 3 * DENSE * HIDDEN + 2 * T * E * HIDDEN
        return {"bytes": b, "flops": f}
    if kind == "linear":
        T, k, n = case["tokens"], case["k"], case["n"]
        return {"bytes": wb(n, k) + 3 * T * k + 2 * k + 2 * T * n, "flops": 2 * T * n * k}
    if kind == "head":
        R, V = case["rows"], case["vocab"]
        return {"bytes": V * HIDDEN + 4 * V * (HIDDEN // 128) + R * (2 * HIDDEN + 2064),
                "flops": 2 * R * V * HIDDEN}
    n = case["rows"] * case["k"]
    return {"bytes": 3 * n + 4 * case["rows"], "flops": 9 * n}


def tolerance(case):
    """Outputs are bf16 (half a unit in the last place: 1.7e-3 in the 2-norm) or float32
    of quantized intermediates; codes and routes may move at a rounding tie."""
    if case["kind"] == "load":
        return {"rel": 1e-6, "differ": 1e-3}
    # the attention block rounds its projections to bf16 ahead of two quantizations:
    # 3.2e-3 from the same block in 64 bits; the others 1.7e-3
    return {"rel": 1.2e-2 if case["kind"] == "attn" else 7e-3, "differ": 1e-3}


# ---------------------------------------------------------------------------
# the same blocks in 64 bits, storage rounding (codes, bf16) as the path has it
# ---------------------------------------------------------------------------

def _fwht(v, block):
    sh = v.shape
    v = v.reshape(-1, block)
    s = 1
    while s < block:
        v = v.reshape(-1, block // (2 * s), 2, s)
        v = torch.stack((v[:, :, 0] + v[:, :, 1], v[:, :, 0] - v[:, :, 1]), 2).reshape(-1, block)
        s *= 2
    return (v / math.sqrt(block)).reshape(sh)


def _quant(v, floor=0.0):
    """Codes and largest magnitude over the last dimension."""
    amax = v.abs().amax(-1, keepdim=True).clamp_min(floor)
    inv = torch.where(amax > 0, 127 / amax.clamp_min(1e-300), torch.zeros_like(amax))
    return (v * inv).round().clamp(-128, 127), amax.squeeze(-1)


def _norm(x, gamma):
    x, h = x.double(), x.shape[-1]
    return x * (math.sqrt(h) / (x.square().sum(-1, keepdim=True) + h * 1e-6).sqrt()) * gamma.double()


def _round_bf(v):
    return v.float().to(torch.bfloat16).double()


def _rowlin(codes, sa, seed, tag, n, k, w=None, ws=None):
    w = _codes(seed, tag, n, k) if w is None else w
    ws = _scales(seed, tag, n) if ws is None else ws
    return codes @ w.double().T * (sa / 127)[:, None] * ws.double()


def _blocklin(v, block, fwht, w, ws):
    """Block-quant of v, then the per-block linear."""
    m, k = v.shape
    b = v.reshape(m, k // block, block)
    c, sa = _quant(_fwht(b, block) if fwht else b)
    return (c * (sa / 127)[..., None]).reshape(m, k) @ w.double().T * ws.double()


def _fast_exp(x):
    """The path's exp of the softmax: 2^(x / ln 2) through the float's bits, with its
    quadratic correction of the mantissa."""
    i = (12102203.16156148 * x.clamp_min(-87.0) + 1059208216.0).to(torch.int64)
    f = (i & 0x7FFFFF).double() / (1 << 23)
    k = i.to(torch.int32).view(torch.float32).double()
    return k * (1.6501418352127075 + f * (-0.37554836273193359 + f * 0.38696467876434326))


def _tanh(x):
    """The path's tanh through its cubic exp."""
    z = (-2 * x.abs()).clamp_min(-87.0)
    n = (z / math.log(2)).round()
    r = z - n * math.log(2)
    e = (1 + r * (0.9999 + r * (0.4985 + r * 0.1681))) * torch.exp2(n.clamp_min(-126))
    return torch.sign(x) * (1 - e) / (1 + e)


def _gelu(x):
    return 0.5 * x * (1 + _tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _attend(q, fq, kc, ks, vc, vs, lo, hi, splits, direct):
    """One sequence's tokens: q [n, heads, hd] codes of one kv head, kc / vc [P, hd]
    codes by position, ranges [lo, hi).  The softmax runs over tiles of 16 positions
    from each split's start, its weights corrected tile by tile, and the splits merge."""
    n, h, hd = q.shape
    P = kc.shape[0]
    sc = (q.reshape(n * h, hd) @ kc.T).reshape(n, h, P) * fq[..., None] * ks / 127 ** 2
    L = hi - lo
    S = torch.minimum(torch.full_like(L, splits), ((L + 31) // 32).clamp_min(1))
    per = (L + S - 1) // S
    sp = torch.arange(int(S.max()), device=DEV)
    start = torch.minimum(sp * per[:, None], L[:, None])
    end = torch.minimum(start + per[:, None], L[:, None])
    end = torch.where(sp < S[:, None], end, start)
    m = torch.full((n, h, len(sp)), -1e30, dtype=torch.float64, device=DEV)
    l = torch.zeros_like(m)
    tiles = []
    for t in range(0, int(per.max()), 16):
        at = start[..., None] + t + torch.arange(16, device=DEV)
        on = (at < end[..., None])[:, None]
        at = (lo[:, None, None] + at).clamp_max(P - 1)[:, None].expand(n, h, len(sp), 16).reshape(n, h, -1)
        s = torch.where(on, sc.gather(2, at).reshape(n, h, len(sp), 16), torch.full((), -1e30, dtype=torch.float64, device=DEV))
        new = torch.maximum(m, s.amax(-1))
        live = on.any(-1)
        corr = torch.where(live, _fast_exp(m - new), torch.ones_like(m))
        w = torch.where(on, _fast_exp(s - new[..., None]), torch.zeros_like(s))
        l = l * corr + w.sum(-1)
        m = new
        tiles.append((at, w, corr))
    c = torch.where(l > 0, _fast_exp(m - m.amax(-1, keepdim=True)), torch.zeros_like(l))
    if direct:
        c = torch.where((S == 1)[:, None, None] & (l > 0), torch.ones_like(c), c)
    full = torch.zeros(n, h, P, dtype=torch.float64, device=DEV)
    f = c / (l * c).sum(-1, keepdim=True)
    for at, w, corr in reversed(tiles):
        full.scatter_add_(2, at, (w * f[..., None]).reshape(n, h, -1))
        f = f * corr
    return (full * (vs / 127)).reshape(n * h, P) @ vc


def _exact_attn(case, seed):
    s = _attn_inputs(case, seed)
    T, nkv, hd, g = s["T"], s["nkv"], s["hd"], NUM_Q // s["nkv"]
    xq, sa = _quant(_fwht(_norm(s["x"], s["gamma"]), 128))
    heads = {}
    for tag, nh in (("wq", NUM_Q), ("wk", nkv)) + ((("wv", nkv),) if s["window"] else ()):
        heads[tag] = _round_bf(_rowlin(xq, sa, seed, tag, nh * hd, HIDDEN)).reshape(T, nh, hd)
    pos = torch.cat([torch.arange(b, b + n, device=DEV) for b, n in s["seqs"]])
    cos, sin = (s[k].double()[pos][:, None] for k in ("cos", "sin"))

    def prep(x, gain):
        one = torch.ones(hd, device=DEV)
        v = _norm(x, one if gain is None else gain)
        if gain is not None:
            r, h = s["rope"], hd // 2
            a, b = v[..., :r].clone(), v[..., h:h + r].clone()
            v[..., :r], v[..., h:h + r] = a * cos - b * sin, b * cos + a * sin
        return _quant(_fwht(v, hd), 1e-10)
    qc, fq = prep(heads["wq"], s["qn"])
    kcn, ksn = prep(heads["wk"], s["kn"])
    vcn, vsn = prep(heads["wv" if s["window"] else "wk"], None)
    splits = max(1, min(-(-2048 // (T * nkv)), -(-s["max_kv"] // 32)))
    o, t0, row0 = torch.empty(T, NUM_Q, hd, dtype=torch.float64, device=DEV), 0, 0
    rows = s["rows"].long()
    news = []
    for b, n in s["seqs"]:
        npg = 2 if s["window"] else (b + n + PAGE - 1) // PAGE
        p = torch.arange(b + n, device=DEV)
        slot = rows[row0 + ((p // PAGE) % npg)] + p % PAGE
        new = slot[b:]
        news.append(new)
        tok = slice(t0, t0 + n)
        kc, vc = s["kc"].reshape(-1, nkv, hd), s["vc"].reshape(-1, nkv, hd)
        kc[new], vc[new] = kcn[tok].to(torch.int8), vcn[tok].to(torch.int8)
        s["ks"][new], s["vs"][new] = ksn[tok].float(), vsn[tok].float()
        hi = p[b:] + 1
        lo = (hi - s["window"]).clamp_min(0) if s["window"] else torch.zeros_like(hi)
        for h in range(nkv):
            o[tok, h * g:(h + 1) * g] = _attend(
                qc[tok, h * g:(h + 1) * g], fq[tok, h * g:(h + 1) * g], kc[slot, h].double(),
                s["ks"][slot, h].double(), vc[slot, h].double(), s["vs"][slot, h].double(), lo, hi,
                splits, s["window"] > 0).reshape(n, g, hd)
        t0, row0 = t0 + n, row0 + npg
    o = _round_bf(o.reshape(T, -1))
    y = _blocklin(o, hd, False, _codes(seed, "wo", HIDDEN, NUM_Q * hd), _scales(seed, "wo", HIDDEN))
    return dict(y=y, o=o, q=None, k_cache=None, k_scale=s["ks"].double(), v_cache=None,
                v_scale=s["vs"].double())


def _exact_ffn(case, seed):
    T, E, K = case["tokens"], case["experts"], case["topk"]
    x = _bf(_normal(seed, "x", T, HIDDEN))
    gain = lambda tag: _bf(_normal(seed, tag, HIDDEN, mean=1, std=0.1))  # noqa: E731
    pes = _bf(_normal(seed, "pes", E, mean=1, std=0.1)).double()
    out = {}
    if case["kind"] == "ffn":
        proj = _bf(_normal(seed, "proj", E, HIDDEN, std=0.02)).double()
        logits = _norm(x, gain("rscale")) @ proj.T
        out["logits"] = logits
    else:
        logits = _normal(seed, "logits", T, E).double()
    top, idx = logits.topk(K, -1)
    w = _fast_exp(top - top[:, :1])
    w = w / w.sum(-1, keepdim=True) * pes[idx]
    xq, sa = _quant(_fwht(_norm(x, gain("gamma")), 128))
    wgu, sgu = _codes(seed, "wgu", E * 2 * INTER, HIDDEN), _scales(seed, "wgu", E * 2 * INTER)
    wd, sd = _codes(seed, "wd", E * HIDDEN, INTER), _scales(seed, "wd", E * HIDDEN)
    accum = torch.zeros(T, HIDDEN, dtype=torch.float64, device=DEV)
    for e in range(E):
        t, k = (idx == e).nonzero(as_tuple=True)
        if not len(t):
            continue
        rows = slice(e * 2 * INTER, (e + 1) * 2 * INTER)
        gu = _rowlin(xq[t], sa[t], 0, "", 0, 0, wgu[rows], sgu[rows])
        b = _round_bf(_gelu(gu[:, :INTER]) * gu[:, INTER:])
        rows = slice(e * HIDDEN, (e + 1) * HIDDEN)
        accum.index_add_(0, t, _blocklin(b, 64, True, wd[rows], sd[rows]) * w[t, k][:, None])
    out.update(idx=None, weight=w, accum=accum, out=accum)
    if case["kind"] == "ffn":
        dq, dsa = _quant(_fwht(_norm(x, gain("dgamma")), 128))
        gate, up = (_round_bf(_rowlin(dq, dsa, seed, t, DENSE, HIDDEN)) for t in ("dg", "du"))
        out["dense"] = _blocklin(_round_bf(_gelu(gate) * up), 64, True, _codes(seed, "dd", HIDDEN, DENSE),
                                 _scales(seed, "dd", HIDDEN))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn":
        return _exact_attn(case, seed)
    if kind in ("ffn", "moe"):
        return _exact_ffn(case, seed)
    if kind == "linear":
        T, k, n = case["tokens"], case["k"], case["n"]
        v = _norm(_bf(_normal(seed, "x", T, k)), _bf(_normal(seed, "gamma", k, mean=1, std=0.1)))
        xq, sa = _quant(_fwht(v, 128))
        return dict(y=_rowlin(xq, sa, seed, "w", n, k), act=None, act_scale=sa)
    if kind == "head":
        R, V, nb = case["rows"], case["vocab"], HIDDEN // 128
        v = _norm(_bf(_normal(seed, "x", R, HIDDEN)), _bf(_normal(seed, "gamma", HIDDEN, mean=1, std=0.1)))
        c, sa = _quant(_fwht(v, 128).reshape(R, nb, 128))
        c = (c * (sa / 127)[..., None]).reshape(R, HIDDEN)
        w, ws = _codes(seed, "w", V, HIDDEN), _scales(seed, "blocks", V, nb)
        y = torch.empty(R, V, dtype=torch.float64, device=DEV)
        for r in range(0, V, 8192):
            wr = w[r:r + 8192].double().reshape(-1, nb, 128) * ws[r:r + 8192].double()[..., None]
            y[:, r:r + 8192] = c @ wr.reshape(-1, HIDDEN).T
        y = _round_bf(_tanh(y / 30) * 30)
        temp = torch.from_numpy(_params(R, seed)["temperature"].astype(np.float64)).to(DEV)
        return dict(token=None, logz=torch.logsumexp(y / temp[:, None], -1), n=None,
                    values=y.topk(256, -1).values, indices=None)
    v = _fwht(_bf(_normal(seed, "w", case["rows"], case["k"], std=0.02)).double(), 128)
    return dict(codes=None, scales=v.abs().amax(-1) / 127)
