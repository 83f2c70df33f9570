"""GPU parity of the int8-KV attention (libbq.so through its C ABI) against
the CPU oracle: bq_attn_prep (butterquant_kernels/attention.mojo:474-534,
butterquant/head_prep.mojo:9-92) and bq_sliding_attention /
bq_full_attention (attention.mojo:32-471, kernels/logsum_merge.mojo:29-122).

Bar: bit-exact.  Codes, qi_bias, f_q and the whole K/V caches after the prep;
the bf16 attention output for the same split plan (s_max), which fixes the
f32 merge order on both sides.
"""
import numpy as np
import pytest

from attn_cases import make_case, oracle_attention
from test_attn_oracle import rope_tables
from test_gpu_parity import dev, host

pytestmark = pytest.mark.gpu


def gpu_attention(gpu, c, s_max):
    import torch
    runs = dev(np.ascontiguousarray(c.runs).view(np.int32).reshape(-1, 4))
    out, used = gpu.attention(dev(c.q_i8), dev(c.qi_bias), dev(c.f_q), dev(c.k_cache),
                              dev(c.k_scale), dev(c.v_cache), dev(c.v_scale), runs,
                              dev(c.base_rows), c.num_q, c.num_kv, c.head_dim, c.window,
                              c.page_shift, c.row_mask, c.page_mask, s_max=s_max)
    torch.cuda.synchronize()
    return host(out)


def check(gpu, O, c, s_max):
    print(f"attention T={c.T} nq={c.num_q} nkv={c.num_kv} hd={c.head_dim} window={c.window} "
          f"s_max={s_max}", flush=True)
    got = gpu_attention(gpu, c, s_max)
    ref = oracle_attention(O, c, s_max=s_max)
    np.testing.assert_array_equal(got, ref)
    return got


SHAPES = {
    # the sliding layer at decode: window 1024, head_dim 256, GQA 2, ring of two
    # 1024-row pages per sequence
    "sliding_decode_1": dict(num_q=16, num_kv=8, head_dim=256, page_len=1024, window=1024,
                             seqs=[(3000, 1)]),
    "sliding_decode_16": dict(num_q=16, num_kv=8, head_dim=256, page_len=1024, window=1024,
                              seqs=[(int(p), 1) for p in
                                    np.random.default_rng(0).integers(0, 4000, 16)]),
    "sliding_prefill": dict(num_q=16, num_kv=8, head_dim=256, page_len=1024, window=1024,
                            seqs=[(900, 48), (0, 20)]),
    # the full layer: head_dim 512, GQA 8, unbounded page table
    "full_decode_2": dict(num_q=16, num_kv=2, head_dim=512, page_len=256, window=0,
                          seqs=[(2999, 1), (700, 1)]),
    "full_prefill": dict(num_q=16, num_kv=2, head_dim=512, page_len=256, window=0,
                         seqs=[(0, 40), (300, 9)]),
}


@pytest.mark.parametrize("name", sorted(SHAPES))
@pytest.mark.parametrize("plan", ["auto", 1])
def test_attention_model_shapes(gpu, O, name, plan):
    c = make_case(O, 21, **SHAPES[name])
    w = SHAPES[name].get("window", 0)
    s_max = gpu.attention_splits(c.T, c.num_kv, w if w else int(c.positions.max()) + 1) \
        if plan == "auto" else plan
    check(gpu, O, c, s_max)


@pytest.mark.parametrize("gqa", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("hd", [64, 128, 256, 512])
def test_attention_gqa_head_dims(gpu, O, gqa, hd):
    num_kv = 2 if gqa < 16 else 1
    c = make_case(O, gqa * 7 + hd, num_q=gqa * num_kv, num_kv=num_kv, head_dim=hd, page_len=32,
                  window=0 if hd in (64, 512) else 50, seqs=[(37, 3), (5, 1), (130, 2)])
    check(gpu, O, c, 3)


def test_attention_many_splits(gpu, O):
    # s_max above ceil(L/32)/2: some tokens get up to 64 splits, the merge runs
    # over several batches of 16, and short tokens leave splits unused
    c = make_case(O, 8, num_q=4, num_kv=2, head_dim=128, page_len=64, window=0,
                  seqs=[(2100, 1), (10, 1), (64, 1)])
    check(gpu, O, c, 64)


def test_attention_splits_beyond_one_stage(gpu, O):
    # 282 splits for the long token: the merge takes them 64 corrections and 32
    # rows at a time, the last batch of each short
    c = make_case(O, 12, num_q=2, num_kv=1, head_dim=64, page_len=64, window=0,
                  seqs=[(9000, 1), (100, 1)])
    check(gpu, O, c, 300)


@pytest.mark.parametrize("gqa,hd", [(1, 64), (2, 128), (2, 256), (4, 128), (8, 64), (8, 256)])
@pytest.mark.parametrize("window,seqs", [
    (40, [(50, 70)]),             # every token past the window start: shifted tile grids
    (40, [(5, 70), (200, 3)]),    # a run straddling pos = window - 1, then a short run
    (0, [(0, 130), (37, 20)]),    # full attention, two runs
])
def test_attention_single_split_groups(gpu, O, gqa, hd, window, seqs):
    # one split per token (s_max = 1): tokens t, t + 16, ... of a run share a
    # group; those whose tile grids coincide are one set of its tiles
    c = make_case(O, gqa * 3 + hd + window, num_q=2 * gqa, num_kv=2, head_dim=hd, page_len=64,
                  window=window, ring_pages=4, seqs=seqs)
    check(gpu, O, c, 1)


def prep_case(O, seed, hd, rope_half, ps, nq, nkv, seqs, page, degree=1, rank=0,
              k_eq_v=False):
    rng = np.random.default_rng(seed)
    T = sum(n for _, n in seqs)
    bf = lambda *shape: O.f32_to_bf16(rng.standard_normal(shape).astype(np.float32) * 2)
    q, k = bf(T, nq * hd), bf(T, nkv * hd)
    v = k if k_eq_v else bf(T, nkv * hd)
    qn = O.f32_to_bf16(rng.uniform(0.5, 1.5, hd).astype(np.float32))
    kn = O.f32_to_bf16(rng.uniform(0.5, 1.5, hd).astype(np.float32))
    maxpos = max(b + n for b, n in seqs)
    cos, sin = rope_tables(maxpos + 1, rope_half)
    runs, rows, buf, off = [], [], 0, 0
    npages = 0
    for b, n in seqs:
        need = ((b + n) // degree) // page + 1
        runs.append((buf, b, off, need))
        rows.extend(range(npages, npages + need))
        npages += need
        buf += n
        off += need
    perm = rng.permutation(npages + 2)
    rows = (perm[np.array(rows)] * page).astype(np.int32)
    slots = (npages + 2) * page
    caches = dict(kc=np.zeros((slots, nkv * hd), np.int8), ks=np.zeros((slots, nkv), np.float32),
                  vc=np.zeros((slots, nkv * hd), np.int8), vs=np.zeros((slots, nkv), np.float32))
    return dict(q=q, k=k, v=v, qn=qn, kn=kn, cos=cos, sin=sin, runs=O.kv_runs(runs), rows=rows,
                shift=int(np.log2(page)), page=page, degree=degree, rank=rank, **caches)


@pytest.mark.parametrize("hd,rope_half,ps,nq,nkv,degree,rank,k_eq_v", [
    (256, 128, 128, 16, 8, 1, 0, False),    # the sliding layer
    (512, 64, 256, 16, 2, 1, 0, True),      # the full layer (K = V projection)
    (512, 64, 256, 16, 2, 2, 1, True),      # cache rank 1 of 2
    (128, 64, 64, 4, 4, 1, 0, False),
    (64, 0, 0, 2, 1, 1, 0, False),          # no RoPE
])
def test_attn_prep(gpu, O, hd, rope_half, ps, nq, nkv, degree, rank, k_eq_v):
    import torch
    p = prep_case(O, hd + nq, hd, rope_half, ps, nq, nkv, [(100, 7), (3, 2), (1500, 1)], 64,
                  degree, rank, k_eq_v)
    print(f"attn_prep hd={hd} rope_half={rope_half} degree={degree}", flush=True)
    g = {n: dev(p[n]) for n in ("kc", "ks", "vc", "vs")}
    runs = dev(np.ascontiguousarray(p["runs"]).view(np.int32).reshape(-1, 4))
    qi, qb, fq = gpu.attn_prep(dev(p["q"]), dev(p["k"]), dev(p["v"]), dev(p["qn"]), dev(p["kn"]),
                               g["kc"], g["ks"], g["vc"], g["vs"], dev(p["cos"]), dev(p["sin"]),
                               runs, dev(p["rows"]), nq, nkv, hd, rope_half, ps, p["shift"],
                               p["page"] - 1, -1, cache_degree=degree, rank=rank)
    torch.cuda.synchronize()
    rqi, rqb, rfq = O.attn_prep(p["q"], p["k"], p["v"], p["qn"], p["kn"], p["kc"], p["ks"],
                                p["vc"], p["vs"], p["cos"], p["sin"], p["runs"], p["rows"], nq,
                                nkv, hd, rope_half, ps, p["shift"], p["page"] - 1, -1,
                                cache_degree=degree, rank=rank)
    np.testing.assert_array_equal(host(qi), rqi)
    np.testing.assert_array_equal(host(qb).view(np.uint32), rqb.view(np.uint32))
    np.testing.assert_array_equal(host(fq).view(np.uint32), rfq.view(np.uint32))
    for n in ("kc", "ks", "vc", "vs"):
        np.testing.assert_array_equal(host(g[n]).view(np.uint8), p[n].view(np.uint8))


def test_prep_then_attention(gpu, O):
    """The layer's two calls back to back: prep fills the cache, attention
    reads it (sliding, decode batch of 3 sequences continuing from
    prefilled caches)."""
    import torch
    hd, nq, nkv, page = 256, 16, 8, 64
    p = prep_case(O, 99, hd, 128, 128, nq, nkv, [(0, 70), (0, 33), (0, 5)], page)
    runs = dev(np.ascontiguousarray(p["runs"]).view(np.int32).reshape(-1, 4))
    g = {n: dev(p[n]) for n in ("kc", "ks", "vc", "vs")}
    qi, qb, fq = gpu.attn_prep(dev(p["q"]), dev(p["k"]), dev(p["v"]), dev(p["qn"]), dev(p["kn"]),
                               g["kc"], g["ks"], g["vc"], g["vs"], dev(p["cos"]), dev(p["sin"]),
                               runs, dev(p["rows"]), nq, nkv, hd, 128, 128, p["shift"], page - 1,
                               -1)
    out, s_max = gpu.attention(qi, qb, fq, g["kc"], g["ks"], g["vc"], g["vs"], runs,
                               dev(p["rows"]), nq, nkv, hd, 48, p["shift"], page - 1, -1)
    torch.cuda.synchronize()
    rqi, rqb, rfq = O.attn_prep(p["q"], p["k"], p["v"], p["qn"], p["kn"], p["kc"], p["ks"],
                                p["vc"], p["vs"], p["cos"], p["sin"], p["runs"], p["rows"], nq,
                                nkv, hd, 128, 128, p["shift"], page - 1, -1)
    ref = O.flash_attention(rqi, rqb, rfq, p["kc"], p["ks"], p["vc"], p["vs"], p["runs"],
                            p["rows"], nq, nkv, hd, 48, p["shift"], page - 1, -1, s_max=s_max)
    np.testing.assert_array_equal(host(out), ref)


@pytest.mark.parametrize("gqa,hd", [(1, 64), (2, 128), (2, 256), (4, 128), (8, 512), (16, 64)])
@pytest.mark.parametrize("window,seqs,s_max", [
    (0, [(0, 75)], 2),               # neighbours in small sets; a ragged last block
    (0, [(200, 40), (3, 17)], 5),    # two runs in one block, starts unequal mod 16
    (40, [(90, 49)], 2),             # every window slides: tokens 16 apart
    (40, [(20, 37), (0, 64)], 3),    # windows start to slide inside a run; a run that begins at 0
    (33, [(31, 33)], 1),             # lengths of one position past two tiles
])
def test_attention_row_groups_split(gpu, O, gqa, hd, window, seqs, s_max):
    # chunks of many tokens per run: 16 / gqa tokens share a workgroup, those
    # with equal tile grids a set; more splits than some tokens have positions for
    c = make_case(O, gqa * 5 + hd + window, num_q=gqa, num_kv=1, head_dim=hd, page_len=32,
                  window=window, ring_pages=4, seqs=seqs)
    check(gpu, O, c, s_max)


def test_attention_row_groups_extremes(gpu, O):
    # zero scales, infinite scores and scores far below the running maximum
    c = make_case(O, 77, num_q=4, num_kv=2, head_dim=128, page_len=64, window=48, ring_pages=4,
                  seqs=[(70, 66), (0, 35)])
    c.k_scale[::7] = 0.0
    c.k_scale[3::11] *= 1e4
    c.v_scale[::5] = 1e-38
    c.f_q[::9] *= 1e30
    for s_max in (1, 2):
        check(gpu, O, c, s_max)


@pytest.mark.parametrize("hd,rope_half,nq,nkv,degree,rank,ntok", [
    (256, 128, 16, 8, 1, 0, 64),    # four waves of four heads, twice a token; the fewest tokens
    (512, 64, 16, 2, 2, 1, 116),    # a last wave of a token alone; cache rank 1 of 2
    (128, 64, 13, 3, 1, 0, 131),    # heads past the token's last
    (256, 64, 6, 5, 3, 0, 140),     # waves that mix q, k and v heads
    (256, 0, 16, 8, 1, 0, 64),      # no RoPE: one head per wave
])
def test_attn_prep_many_tokens(gpu, O, hd, rope_half, nq, nkv, degree, rank, ntok):
    # enough (token, head) items for four heads per wave
    import torch
    p = prep_case(O, hd + nq + 1, hd, rope_half, hd // 2, nq, nkv, [(100, ntok - 21), (3, 21)], 64,
                  degree, rank)
    p["q"][5, :hd] = 0  # a head of zeros: the smallest scale
    g = {n: dev(p[n]) for n in ("kc", "ks", "vc", "vs")}
    runs = dev(np.ascontiguousarray(p["runs"]).view(np.int32).reshape(-1, 4))
    args = (nq, nkv, hd, rope_half, hd // 2, p["shift"], p["page"] - 1, -1)
    got = gpu.attn_prep(dev(p["q"]), dev(p["k"]), dev(p["v"]), dev(p["qn"]), dev(p["kn"]), g["kc"],
                        g["ks"], g["vc"], g["vs"], dev(p["cos"]), dev(p["sin"]), runs,
                        dev(p["rows"]), *args, cache_degree=degree, rank=rank)
    torch.cuda.synchronize()
    ref = O.attn_prep(p["q"], p["k"], p["v"], p["qn"], p["kn"], p["kc"], p["ks"], p["vc"], p["vs"],
                      p["cos"], p["sin"], p["runs"], p["rows"], *args, cache_degree=degree, rank=rank)
    for x, y in zip(got, ref):
        np.testing.assert_array_equal(host(x).view(np.uint8), y.view(np.uint8))
    for n in ("kc", "ks", "vc", "vs"):
        np.testing.assert_array_equal(host(g[n]).view(np.uint8), p[n].view(np.uint8))


@pytest.mark.parametrize("hd", [64, 128, 512])
@pytest.mark.parametrize("s_max", [2, 3, 4, 5, 8, 9, 16, 17])
def test_attention_merge_instances(gpu, O, hd, s_max):
    # the fewest and the most splits of each merge instance, and tokens with
    # fewer splits than the plan
    c = make_case(O, hd + s_max, num_q=4, num_kv=2, head_dim=hd, page_len=64, window=0,
                  seqs=[(32 * s_max, 1), (40, 1), (0, 1)])
    check(gpu, O, c, s_max)


@pytest.mark.parametrize("gqa,s_max,window,seqs", [
    # blocks of 128 tokens (two heads per kv head)
    (2, 2, 0, [(0, 150)]),            # neighbours in pairs, a last block of 22
    (2, 2, 0, [(101, 130)]),          # ... counted round the block from an odd position
    (2, 4, 0, [(243, 77)]),           # fours, one short block
    (2, 3, 0, [(200, 140)]),          # three splits do not divide the group: a wave per token
    (2, 2, 0, [(0, 70), (5, 80)]),    # a block of two runs: a wave per token
    (2, 8, 0, [(400, 30)]),           # neighbours in launches of fewer than 16 groups
    (2, 9, 0, [(500, 60)]),
    (2, 2, 64, [(0, 300)]),           # windows slide in the later blocks only
    (2, 3, 50, [(49, 49)]),           # all slide: 49 tokens in groups,
    (2, 3, 50, [(49, 47)]),           # 47 a wave each
    (2, 2, 40, [(100, 70), (60, 90)]),
    (2, 2, 40, [(100, 70), (0, 90)]),
    # blocks of 256 tokens (a head per kv head)
    (1, 2, 0, [(30, 300)]),
    (1, 4, 0, [(333, 90)]),
    (1, 8, 0, [(700, 60)]),
    (1, 5, 0, [(0, 71)]),
    (1, 3, 64, [(0, 280)]),
])
def test_attention_row_group_forms(gpu, O, gqa, s_max, window, seqs):
    # every form of a split plan's groups, over several blocks and kv heads
    c = make_case(O, gqa + 10 * s_max + window, num_q=2 * gqa, num_kv=2, head_dim=64, page_len=64,
                  window=window, ring_pages=4, seqs=seqs)
    check(gpu, O, c, s_max)


@pytest.mark.parametrize("s_max", [1, 2])
@pytest.mark.parametrize("gqa", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("hd", [64, 128, 256, 512])
def test_attention_row_group_instances(gpu, O, hd, gqa, s_max):
    # a chunk in every instance: groups in its first run, some in the second
    c = make_case(O, hd + gqa + s_max, num_q=gqa, num_kv=1, head_dim=hd, page_len=64,
                  window=0 if gqa & 5 else 90, ring_pages=4, seqs=[(101, 131), (3, 20)])
    check(gpu, O, c, s_max)


@pytest.mark.parametrize("gqa,hd", [(1, 64), (2, 256), (4, 128), (8, 256), (8, 512), (16, 64)])
@pytest.mark.parametrize("window", [0, 40])
def test_attention_one_split_decode(gpu, O, gqa, hd, window):
    # one-split plans of many sequences of one token, and of chunks beside them
    c = make_case(O, gqa + hd + window, num_q=2 * gqa, num_kv=2, head_dim=hd, page_len=64,
                  window=window, ring_pages=4, seqs=[(37 * i % 150, 1 + 2 * (i % 9 == 0)) for i in range(40)])
    check(gpu, O, c, 1)


def test_attention_more_groups_than_a_launch(gpu, O):
    # 2^24 row groups of one token: a launch takes fewer, so it is a wave per
    # token; the first and the last tokens as in calls of their own
    import torch
    hd, nq, nkv, page, T = 64, 256, 16, 1024, 1 << 20
    d = "cuda"
    g = torch.Generator(device=d).manual_seed(5)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device=d, generator=g)  # noqa: E731
    q, kc, vc = i8(T, nq * hd), i8(2 * page, nkv * hd), i8(2 * page, nkv * hd)
    ks, vs = torch.rand(2 * page, nkv, device=d) + 1, torch.rand(2 * page, nkv, device=d) + 1
    qb = torch.zeros(T, nq, device=d)
    fq = torch.full((T, nq), 0.01, device=d)
    rows = torch.tensor([0, page], dtype=torch.int32, device=d)

    def call(t0, n):
        runs = torch.tensor([[0, t0, 0, 2]], dtype=torch.int32, device=d)
        s = slice(t0, t0 + n)
        return gpu.attention(q[s], qb[s], fq[s], kc, ks, vc, vs, runs, rows, nq, nkv, hd, 3, 10,
                             page - 1, 1, s_max=1)[0]

    print(f"attention T={T} nq={nq} nkv={nkv} hd={hd}", flush=True)
    out = call(0, T)
    torch.cuda.synchronize()
    same = [torch.equal(out[t0:t0 + 100], call(t0, 100)) for t0 in (0, T // 2 - 7, T - 100)]
    del q, qb, fq, out
    torch.cuda.empty_cache()  # (120 GB, most of it workspace)
    assert same == [True, True, True]
