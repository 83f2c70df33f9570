// int8-KV attention on gfx950: the attention prep (per-head RMS norm, RoPE,
// FWHT, absmax int8 with the code sum) that fills the paged int8 KV cache,
// and flash attention over that cache.
//
// Reference: butterquant/head_prep.mojo:9-92 (per-head prep),
// butterquant_kernels/attention.mojo:32-80 (bq_process_kv_tile), :83-146
// (decode kernel), :149-247 (sliding prefill), :250-327 (full prefill),
// :474-534 (BqAttnPrepKernel), kernels/attention_ops.mojo:45-51 (PagedKV),
// :166-182 (online_softmax_tile), kernels/logsum_merge.mojo:29-122 (merge).
//
// Layout.  KV cache rows are slots: k_cache[slot][kv_head][head_dim] int8 with
// k_scale[slot][kv_head] f32 (amax), the same for V.  A token's position p
// maps to slot base_rows[run.rows_off + ((p >> shift) & page_mask)] +
// (p & row_mask).  Q codes are [token][q_head][head_dim] int8 with
// qi_bias = 128 * sum(codes) and f_q = amax per (token, q_head).
//
// Flash attention.  A split is a contiguous range of a token's KV positions
// (worker_range of the range into S = min(s_max, ceil(L / kAttnMinSplit))
// parts), walked in tiles of 16 positions exactly as the reference does: the
// scores of a tile come from head_dim/64 int8 MFMAs (A = 16 rows of query
// heads, B = 16 K rows); per head the tile max, corr and weights use the
// reference's fast exp and its 16-lane tree sum; then acc *= corr and acc +=
// (w * vs / 127) * v position by position.  Two kernels:
//   k_flash_attn       decode: one wave per (token, kv head, split)
//   k_flash_attn_rows  prefill chunks: 16/G tokens share every K/V tile
// A token whose range is one split of a sliding layer is finalized there
// (acc * (1/l), the sliding prefill kernel), and so is every token of a
// one-split plan (full layers: the merge of one split); every other token's
// splits are written as (m, l, acc) partials and merged by k_attn_merge in
// split order with the reference's merge (corrections masked by l > 0, a
// 16-lane tree per batch of 16 splits, the first contributing split
// multiplied, the rest fma-accumulated).
#include <algorithm>

#include "bq_kernels.hpp"
#include "bq_device.hpp"

namespace bq {

namespace {

// The run holding buffer row tok: the reference advances r while
// tok >= runs[r + 1].buf_start (attention.mojo:489-492), i.e. r + 1 is the
// first j >= 1 with tok < runs[j].buf_start, else num_runs - 1.
__device__ inline int run_of(const KvRun* __restrict__ runs, int n, int tok) {
  const int lane = lane_id();
  for (int base = 1; base < n; base += kWave) {
    const int j = base + lane;
    const bool stop = j < n && tok < runs[j].buf_start;
    const unsigned long long m = __ballot(stop);
    if (m) return base + (__ffsll((long long)m) - 1) - 1;
  }
  return n - 1;
}

__device__ inline int64_t paged_slot(const int32_t* __restrict__ rows, int shift, int row_mask,
                                     int page_mask, int64_t p) {
  return (int64_t)rows[(p >> shift) & page_mask] + (p & row_mask);
}

// sum over the 16 lanes of each aligned 16-lane group in the order of a
// SIMD[f32, 16].reduce_add (halving tree: j + 8, j + 4, j + 2, j + 1); the
// result is broadcast to the group.  Lane j of each row adds lane j + H of
// the same row by a DPP row shift (the lanes whose partner falls outside the
// row compute values no one reads), so lane 0 of each row ends with the
// tree's sum; readlane brings the four row sums back.
__device__ inline float tree16(float v) {
  v = v + row_shl<8>(v);
  v = v + row_shl<4>(v);
  v = v + row_shl<2>(v);
  v = v + row_shl<1>(v);
  const int x = __float_as_int(v);
  const int s0 = __builtin_amdgcn_readlane(x, 0), s1 = __builtin_amdgcn_readlane(x, 16);
  const int s2 = __builtin_amdgcn_readlane(x, 32), s3 = __builtin_amdgcn_readlane(x, 48);
  const int row = lane_id() >> 4;
  return __int_as_float(row == 0 ? s0 : row == 1 ? s1 : row == 2 ? s2 : s3);
}

__device__ inline float max87(float x) { return x > -87.0f ? x : -87.0f; }

__device__ inline float readlane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// whether k_flash_attn_rows has blocks that it takes a wave per token (LONE)
__host__ __device__ constexpr bool attn_rows_lone(int G, int s_max) { return G <= 2 && s_max > 1; }
// and how long a split from position 0 has to be, at the end of a block, for
// its groups to beat that (200 tokens from position 0, two splits: 21 against
// 27 us; 70 tokens, four splits of up to 18: 14.7 / 14.2)
constexpr int kRowsSplitLen = 48;

// token metadata shared by the attention and merge kernels
struct TokRange {
  const int32_t* rows;
  int64_t lo;
  int L;
};

__device__ inline TokRange token_range(const AttnArgs& a, int tok) {
  const int r = run_of(a.runs, a.num_runs, tok);
  const KvRun run = a.runs[r];
  const int64_t pos = (int64_t)run.base_pos + (tok - run.buf_start);
  TokRange t;
  t.rows = a.base_rows + run.rows_off;
  if (a.window > 0) {  // attention.mojo:196-199: [max(0, pos - window + 1), pos]
    t.lo = pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
    t.L = (int)(pos + 1 - t.lo);
  } else {             // attention_ops.mojo:146-152 at one rank: rows [0, pos]
    t.lo = 0;
    t.L = pos < 0 ? 0 : (int)(pos + 1);
  }
  return t;
}

__device__ inline int num_splits(int L, int s_max) {
  if (L <= 0) return 1;
  const int s = (L + kAttnMinSplit - 1) / kAttnMinSplit;
  return s < s_max ? s : s_max;
}

}  // namespace

// ---------------------------------------------------------------------------
// attention prep: one wave per (token, head) over q heads, then k heads, then
// v heads.  Element e of the head is value r = e / 64 of lane e % 64.
// ---------------------------------------------------------------------------
template <int R>
__global__ __launch_bounds__(256) void k_attn_prep(PrepArgs a) {
  constexpr int HD = R * kWave;
  const int wave = threadIdx.x >> 6, lane = lane_id();
  const int nh = a.num_q + 2 * a.num_kv;
  const int item = blockIdx.x * 4 + wave;
  if (item >= a.T * nh) return;
  const int tok = item / nh, j = item % nh;
  const int r = run_of(a.runs, a.num_runs, tok);
  const KvRun run = a.runs[r];
  const int64_t pos = (int64_t)run.base_pos + (tok - run.buf_start);
  const bool is_q = j < a.num_q, is_v = j >= a.num_q + a.num_kv;
  const int h = is_q ? j : is_v ? j - a.num_q - a.num_kv : j - a.num_q;
  // attention.mojo:515: K/V rows only for positions this cache rank owns
  if (!is_q && pos % a.cache_degree != a.rank) return;
  const int64_t kvs = (int64_t)a.num_kv * HD;
  const uint16_t* src = is_q ? a.q_src + (int64_t)tok * a.num_q * HD + (int64_t)h * HD
                      : (is_v ? a.v_src : a.k_src) + (int64_t)tok * kvs + (int64_t)h * HD;
  float v[R];
#pragma unroll
  for (int i = 0; i < R; ++i) v[i] = bf16_to_f32(src[i * kWave + lane]);

  // head_inv_rms (head_prep.mojo:9-16): chain k of 16 takes x[16i + k] in i
  // order (product first, then fma), then the 16-lane tree.  x[16i + k] is
  // value i / 4 of lane 16 * (i % 4) + k: the row moves of row_to_row0 bring
  // it to lane k of row 0, which runs the chains (the other rows' sums are
  // not used), and lane 0 ends the tree.
  float ssq = v[0] * v[0];
#pragma unroll
  for (int i4 = 0; i4 < R; ++i4) {
    if (i4 > 0) ssq = fmaf(v[i4], v[i4], ssq);
    const float x1 = row_to_row0<1>(v[i4]), x2 = row_to_row0<2>(v[i4]);
    const float x3 = row_to_row0<3>(v[i4]);
    ssq = fmaf(x1, x1, ssq);
    ssq = fmaf(x2, x2, ssq);
    ssq = fmaf(x3, x3, ssq);
  }
  ssq = ssq + row_shl<8>(ssq);
  ssq = ssq + row_shl<4>(ssq);
  ssq = ssq + row_shl<2>(ssq);
  ssq = ssq + row_shl<1>(ssq);
  ssq = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ssq), 0));
  const float inv = a.sqrt_n / __builtin_sqrtf(ssq + a.n_eps);

  const uint16_t* gamma = is_q ? a.q_norm : a.k_norm;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    v[i] = v[i] * inv;
    if (!is_v) v[i] = v[i] * bf16_to_f32(gamma[i * kWave + lane]);
  }
  if (!is_v) {
    // RoPE on (e, pair_stride + e) for e < rope_half (head_prep.mojo:58-65);
    // rope_half and pair_stride are multiples of 64, so both elements of a
    // pair are values of the same lane
    const int ps = a.pair_stride / kWave, rh = a.rope_half / kWave;
    const float* cs = a.cos_table + pos * a.rope_half;
    const float* sn = a.sin_table + pos * a.rope_half;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i >= rh) continue;
      const float c = cs[i * kWave + lane], s = sn[i * kWave + lane];
#pragma unroll
      for (int i2 = 0; i2 < R; ++i2) {
        if (i2 != i + ps) continue;
        const float lo = v[i], hi = v[i2];
        v[i] = lo * c - hi * s;
        v[i2] = hi * c + lo * s;
      }
    }
  }
  fwht_wave<R>(v, HD);
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    v[i] = v[i] * a.fwht_scale;
    m = fmaxf(m, fabsf(v[i]));
  }
  float amax = wave_max(m);
  if (amax < 1e-10f) amax = 1e-10f;
  const float qinv = 127.0f / amax;
  int8_t* dst;
  if (is_q) {
    dst = a.q_i8 + (int64_t)tok * a.num_q * HD + (int64_t)h * HD;
  } else {
    const int64_t slot = paged_slot(a.base_rows + run.rows_off, a.page_shift, a.row_mask,
                                    a.page_mask, pos / a.cache_degree);
    dst = (is_v ? a.v_cache : a.k_cache) + slot * kvs + (int64_t)h * HD;
    if (lane == 0) (is_v ? a.v_scale : a.k_scale)[slot * a.num_kv + h] = amax;
  }
  int qs = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int8_t c = quantize_i8(v[i], qinv);
    dst[i * kWave + lane] = c;
    qs += c;
  }
  if (is_q) {
    qs = __builtin_amdgcn_readlane(wave_incl_scan(qs), 63);  // integer sum: exact
    if (lane == 0) {
      a.qi_bias[(int64_t)tok * a.num_q + h] = (float)qs * 128.0f;
      a.f_q[(int64_t)tok * a.num_q + h] = amax;
    }
  }
}

// ---------------------------------------------------------------------------
// Attention prep of many tokens: four heads of one token per wave, eight
// consecutive values per lane (head_dim / 8 lanes a head, so 512 / head_dim
// heads per round).  k_attn_prep is bound by vector-ALU issue and by its one-
// and two-byte accesses; here rows are 16-byte loads and 8-byte stores, the
// FWHT's strides 1, 2, 4 stay inside the lane, and the four heads' sums of
// squares (lane k + 16 h: chain k of head h, from LDS), square roots and
// divisions share their instructions.  Takes pair_stride == head_dim / 2, 16-
// byte aligned sources, gains and tables and 8-byte aligned codes.  The same
// values in the same order as k_attn_prep, to the bit: in the cross-lane
// stages within a row the upper lane of a pair holds -(a - b), and the sign
// (the parity of its index bits) is folded into the final scale, as in
// nq_v8_transform.
// ---------------------------------------------------------------------------
template <int HD>
__global__ __launch_bounds__(256) void k_attn_prep_v8(PrepArgs a) {
  constexpr int LPH = HD / 8, HPR = kWave / LPH, RND = 4 / HPR;  // lanes a head; heads a round; rounds
  static_assert(HPR >= 1 && RND >= 1, "128 <= head_dim <= 512");
  // (16 values of padding: the four heads' chains read different banks)
  __shared__ __attribute__((aligned(16))) uint16_t s_x[4][4][HD + 16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
  const int nh = a.num_q + 2 * a.num_kv, hg = (nh + 3) / 4;  // a token's waves
  const int item = blockIdx.x * 4 + wave, tok = item / hg, j0 = (item % hg) * 4;
  if (tok >= a.T) return;
  const int r = run_of(a.runs, a.num_runs, tok);
  const KvRun run = a.runs[r];
  const int64_t pos = (int64_t)run.base_pos + (tok - run.buf_start);
  const int64_t kvs = (int64_t)a.num_kv * HD;
  const int sub = lane / LPH;  // head within the round
  const int run8 = dpp_run(lane % LPH), e0 = run8 * 8;  // this lane's values of it
  v4i raw[RND];
#pragma unroll
  for (int q = 0; q < RND; ++q) {
    const int j = min(j0 + q * HPR + sub, nh - 1);  // (heads past the last: read, never stored)
    const uint16_t* src = j < a.num_q ? a.q_src + (int64_t)tok * a.num_q * HD + j * HD
                          : j < a.num_q + a.num_kv
                              ? a.k_src + tok * kvs + (j - a.num_q) * HD
                              : a.v_src + tok * kvs + (j - a.num_q - a.num_kv) * HD;
    raw[q] = *reinterpret_cast<const v4i*>(src + e0);
    *reinterpret_cast<v4i*>(&s_x[wave][q * HPR + sub][e0]) = raw[q];
  }
  // The position's rotation.  A pair's halves are LPH / 2 lanes apart (a row or
  // more), and go through exchanged pairs of values (row_exchange): value pair
  // i, i + 1 leaves value i + up here, so this lane needs every other entry.
  const int up = (lane / (LPH / 2)) & 1;
  const int el = (run8 % (LPH / 2)) * 8;
  const bool rot = el < a.rope_half;
  float cs[4], sn[4];
  if constexpr (LPH >= 32) {
    const int64_t o = pos * a.rope_half + (rot ? el : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cs[i] = a.cos_table[o + 2 * i + up];
      sn[i] = a.sin_table[o + 2 * i + up];
    }
  }
  // head_inv_rms: chain lane & 15 of head j0 + lane / 16, then the 16-lane tree
  float ssq;
  {
    const uint16_t* x = &s_x[wave][lane >> 4][lane & 15];
    const float x0 = bf16_to_f32(x[0]);
    ssq = x0 * x0;
#pragma unroll
    for (int i = 1; i < HD / 16; ++i) {
      const float xi = bf16_to_f32(x[16 * i]);
      ssq = fmaf(xi, xi, ssq);
    }
    ssq = row_tree16(ssq);
  }
  const float inv4 = a.sqrt_n / __builtin_sqrtf(ssq + a.n_eps);  // lane 16 h: head h's
  const float scale = (__builtin_popcount(run8 & 15) & 1) ? -a.fwht_scale : a.fwht_scale;
  const float s1 = run8 & 1 ? -1.0f : 1.0f, s2 = run8 & 2 ? -1.0f : 1.0f;
  const float s4 = run8 & 4 ? -1.0f : 1.0f, s8 = run8 & 8 ? -1.0f : 1.0f;
  // attention.mojo:515: K/V rows (and pages) only for positions this cache rank owns
  const bool owned = pos % a.cache_degree == a.rank;
  const int64_t slot = owned ? paged_slot(a.base_rows + run.rows_off, a.page_shift, a.row_mask,
                                          a.page_mask, pos / a.cache_degree) : 0;
#pragma unroll
  for (int q = 0; q < RND; ++q) {
    const int j = j0 + q * HPR + sub;
    const bool is_q = j < a.num_q, is_v = j >= a.num_q + a.num_kv;
    const float inv = __shfl(inv4, 16 * (q * HPR + sub), kWave);
    float v[8], g[8];
    bf16x8_to_f32(raw[q], v);
    v4i gr = *reinterpret_cast<const v4i*>((is_q ? a.q_norm : a.k_norm) + e0);
    if (is_v) gr = v4i{0x3F803F80, 0x3F803F80, 0x3F803F80, 0x3F803F80};  // no gain: times 1
    bf16x8_to_f32(gr, g);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = v[i] * inv * g[i];
    if constexpr (LPH >= 32) {
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        float lo, hi;
        row_exchange<LPH / 2>(v[i], v[i + 1], lo, hi);
        const float c = cs[i / 2], s = sn[i / 2];
        const float nl = lo * c - hi * s, nu = hi * c + lo * s;
        row_exchange<LPH / 2>(rot && !is_v ? nl : lo, rot && !is_v ? nu : hi, v[i], v[i + 1]);
      }
    } else {
      const int64_t o = pos * a.rope_half + (rot ? el : 0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float c = a.cos_table[o + i], s = up ? a.sin_table[o + i] : -a.sin_table[o + i];
        const float n = v[i] * c + xlane_partner<LPH / 2>(v[i]) * s;
        v[i] = rot && !is_v ? n : v[i];
      }
    }
#pragma unroll
    for (int st = 1; st < 8; st <<= 1)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i & st) continue;
        const float x = v[i], y = v[i + st];
        v[i] = x + y;
        v[i + st] = x - y;
      }
    dpp_bfly8<1>(v, s1);
    dpp_bfly8<2>(v, s2);
    dpp_bfly8<4>(v, s4);
    dpp_bfly8<8>(v, s8);
    if constexpr (LPH >= 32) row_bfly8<16>(v);
    if constexpr (LPH >= 64) row_bfly8<32>(v);
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = v[i] * scale;
      amax = fmaxf(amax, fabsf(v[i]));
    }
    for_each_xlane_stride(LPH, [&](auto st) {
      amax = fmaxf(amax, xlane_partner<decltype(st)::value>(amax));
    });
    if (amax < 1e-10f) amax = 1e-10f;
    uint32_t w[2];
    codes8_bounded(v, 127.0f / amax, w);  // (amax >= 1e-10: a finite factor)
    int qs = __builtin_amdgcn_sdot4((int)w[1], 0x01010101,
                                    __builtin_amdgcn_sdot4((int)w[0], 0x01010101, 0, false), false);
    for_each_xlane_stride(LPH, [&](auto st) {  // the head's code sum
      qs += __float_as_int(xlane_partner<decltype(st)::value>(__int_as_float(qs)));
    });
    if (j >= nh || (!is_q && !owned)) continue;
    const int h = is_q ? j : is_v ? j - a.num_q - a.num_kv : j - a.num_q;
    int8_t* dst = is_q ? a.q_i8 + ((int64_t)tok * a.num_q + h) * HD
                       : (is_v ? a.v_cache : a.k_cache) + slot * kvs + (int64_t)h * HD;
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    *reinterpret_cast<u2*>(dst + e0) = u2{w[0], w[1]};
    if (e0 == 0) {
      if (is_q) {
        a.qi_bias[(int64_t)tok * a.num_q + h] = (float)qs * 128.0f;
        a.f_q[(int64_t)tok * a.num_q + h] = amax;
      } else {
        (is_v ? a.v_scale : a.k_scale)[slot * a.num_kv + h] = amax;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// flash attention: one wave per (token, kv head, split); G query heads share
// the kv head (G <= 16).  wsh: the wave's LDS for 16 x G weights [p][head].
// ---------------------------------------------------------------------------
template <int HD, int G>
__device__ __forceinline__ void flash_attn_wave(const AttnArgs& a, int tok, int kvh, int s,
                                                float* wsh) {
  constexpr int C = HD / 64;  // 64-byte K chunks per row = V bytes per lane
  const int lane = lane_id();
  const TokRange tr = token_range(a, tok);
  const int S = num_splits(tr.L, a.s_max);
  if (s >= S) return;
  int start, end;
  {
    const int per = (tr.L + S - 1) / S;
    start = s * per;
    end = start + per < tr.L ? start + per : tr.L;
    if (start >= tr.L) start = end = tr.L;
  }
  const int64_t kvs = (int64_t)a.num_kv * HD;
  const int p16 = lane & 15, grp = lane >> 4;
  const int qh0 = kvh * G;  // first query head of this kv head

  // A operand: lane (h + 16 g) holds head h's bytes [c*64 + g*16, +16)
  v4i qa[C];
  const v4i zero4 = {0, 0, 0, 0};
  {
    const int hq = lane & 15;
    const int8_t* qrow = a.q_i8 + ((int64_t)tok * a.num_q + qh0 + hq) * HD + grp * 16;
#pragma unroll
    for (int c = 0; c < C; ++c) qa[c] = hq < G ? ld16(qrow + c * 64) : zero4;
  }
  // score layout: lane (p + 16 g), value i <-> head 4 g + i, position p.
  // The u8-shifted dot of the reference is dot + 128 * sum(q).
  float qb[4], fq[4];
  int qsum128[4];
  {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int h = 4 * grp + i;
      qb[i] = 0.0f; fq[i] = 0.0f; qsum128[i] = 0;
      if (h < G) {
        qb[i] = a.qi_bias[(int64_t)tok * a.num_q + qh0 + h];
        fq[i] = a.f_q[(int64_t)tok * a.num_q + qh0 + h];
      }
    }
    // sum of the query codes of head hq, lane-parallel over the 16-byte pieces
    int part = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int w4[4] = {qa[c].x, qa[c].y, qa[c].z, qa[c].w};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part += (int)(int8_t)w4[q] + (int)(int8_t)(w4[q] >> 8) + (int)(int8_t)(w4[q] >> 16) +
                (w4[q] >> 24);
    }
    part += __shfl_xor(part, 16, kWave);
    part += __shfl_xor(part, 32, kWave);  // lane hq (and hq + 16 g): sum of head hq
#pragma unroll
    for (int i = 0; i < 4; ++i) qsum128[i] = 128 * __shfl(part, 4 * grp + i, kWave);
  }

  const float inv127 = 1.0f / 127.0f;
  const float inv127sq = inv127 * inv127;
  float m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) { m[i] = -1e30f; l[i] = 0.0f; }
  // acc[h / 4][c][h % 4]: head h, column lane * C + c
  constexpr int HB = (G + 3) / 4;
  v4f acc[HB][C];
#pragma unroll
  for (int b = 0; b < HB; ++b)
#pragma unroll
    for (int c = 0; c < C; ++c) acc[b][c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

  const int8_t* kbase = a.k_cache + (int64_t)kvh * HD;
  const int8_t* vbase = a.v_cache + (int64_t)kvh * HD + lane * C;
  // Slots of 64 consecutive positions [sb, sb + 64) of the split, one per
  // lane (lanes past the end repeat the last position); slots fit in 32 bits.
  auto slot_batch = [&](int sb) -> int {
    const int pj = sb + lane < end ? sb + lane : end - 1;
    return (int)paged_slot(tr.rows, a.page_shift, a.row_mask, a.page_mask, tr.lo + pj);
  };
  // One tile's operands: lane (p + 16 g) holds K row p's bytes [c*64 + g*16,
  // +16) for every chunk c, its ks and vs; every lane holds its C bytes of
  // each V row.  Idle positions repeat the tile's first row.  (Requesting the
  // next tile's registers as this tile frees them measured slower: the waves of
  // a SIMD already cover each other's loads.  Sliding, head 256, two heads per
  // kv head, caches not in L2: 16 x 1000 positions 24.5 us against 23.4, 32
  // 36.0 / 34.1, one sequence 12.3 / 12.0; head 512, eight heads, the registers
  // it takes: a decode block 91 -> 111.)
  v4i kb[C];
  uint32_t vraw[16][(C + 3) / 4];
  float ks, vs;
  auto load_k = [&](int slots, int off, int tl) {
    const int my = __shfl(slots, off + (p16 < tl ? p16 : 0), kWave);
    const int8_t* krow = kbase + (int64_t)my * kvs + grp * 16;
#pragma unroll
    for (int c = 0; c < C; ++c) kb[c] = ld16(krow + c * 64);
    ks = a.k_scale[(int64_t)my * a.num_kv + kvh];
    vs = a.v_scale[(int64_t)my * a.num_kv + kvh];
  };
  auto load_v = [&](int p, int slots, int off, int tl) {
    const int sp = __builtin_amdgcn_readlane(slots, off + (p < tl ? p : 0));
    const int8_t* vr = vbase + (int64_t)sp * kvs;
    if constexpr (C >= 8) {
      const uint2 w = *reinterpret_cast<const uint2*>(vr);
      vraw[p][0] = w.x; vraw[p][1] = w.y;
    } else if constexpr (C == 4) {
      vraw[p][0] = *reinterpret_cast<const uint32_t*>(vr);
    } else if constexpr (C == 2) {
      vraw[p][0] = *reinterpret_cast<const uint16_t*>(vr);
    } else {
      vraw[p][0] = (uint8_t)*vr;
    }
  };

  // The batch after is requested ahead, behind a tile's loads: a branch in
  // front of them holds them back (128 sequences of 1500 positions, sliding:
  // 124 us against 108).  Head 512 with a query head of its own per kv head is
  // bound by HBM and takes its batches when due: a fourth wave per SIMD fits
  // its registers then (8 sequences of 3000 positions, 16 heads: 77 us, 81 ahead).
  constexpr bool NEXT = HD / G < 512;
  int off = 0, slots = 0, slots_n = 0;  // the next tile: its batch, and the batch after
  if (start < end) {
    slots = slot_batch(start);
    if constexpr (NEXT) slots_n = slot_batch(start + 64);
  }
  for (int p0 = start; p0 < end; p0 += 16) {
    const int tl = end - p0 < 16 ? end - p0 : 16;
    if (!NEXT && off == 64) {
      off = 0;
      slots = slot_batch(p0);
    }
    load_k(slots, off, tl);
#pragma unroll
    for (int p = 0; p < 16; ++p) load_v(p, slots, off, tl);
    off += 16;
    if (NEXT && off == 64) {
      off = 0;
      slots = slots_n;
      slots_n = slot_batch(p0 + 80);
    }
    v4i d = zero4;
#pragma unroll
    for (int c = 0; c < C; ++c) d = mfma16x16x64(qa[c], kb[c], d);
    const int dv[4] = {d.x, d.y, d.z, d.w};
    // per head of this lane's group (heads 4 g + i, only i < G exist)
    constexpr int NI = G < 4 ? G : 4;
    float sc[4], corr[4];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float sco = -1e30f;
      if (4 * grp + i < G && p16 < tl)
        sco = (((float)(dv[i] + qsum128[i]) - qb[i]) * fq[i]) * ks * inv127sq;
      const float tmax = group_max(sco, 16);
      const float m_new = tmax > m[i] ? tmax : m[i];
      corr[i] = fast_exp_softmax_biased(max87(m[i] - m_new));
      const float w = fast_exp_softmax_biased(max87(sco - m_new));
      l[i] = l[i] * corr[i] + tree16(w);
      m[i] = m_new;
      sc[i] = p16 < tl ? w * vs * inv127 : 0.0f;
    }
#pragma unroll
    for (int h = 0; h < G; ++h) {
      const float ch = readlane_f(corr[h % 4], 16 * (h / 4));
#pragma unroll
      for (int c = 0; c < C; ++c) acc[h / 4][c][h % 4] = acc[h / 4][c][h % 4] * ch;
    }
    // positions past the tile's end carry weight 0: acc + v*0 leaves acc
    // unchanged bit for bit (acc is never -0: it starts at +0 and only an
    // exact -0 product added to -0 gives -0), so the loop needs no branch.
    // The weights go through LDS, from G = 4 as [p][head % 4][head / 4]: lane
    // L reads those of heads L % 4, + 4, ..., the rows of the f32 MFMA that
    // takes four heads' fmaf at once; else as [p][head], read broadcast.  What
    // the MFMA gives is fewer instructions in a wave's chain.  Head 512, eight
    // heads, attention and merge: one sequence of 100 positions 15.8 us with
    // v_fma, 14.7 so; 4 x 3000 29.1 / 27.9; 16 x 4096 55.0 / 53.9, where the
    // SIMDs are full (the attention alone 36.4 / 37.5).  Sixteen heads, 8 x
    // 3000: head 512 22.6 / 20.4 for the attention, head 64 10.0 / 9.1.
    if constexpr (G >= 4) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (4 * grp + i < G) wsh[p16 * G + i * HB + grp] = sc[i];
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (grp == 0) wsh[p16 * G + i] = sc[i];
    }
#pragma unroll
    for (int p = 0; p < 16; ++p) {
      float vf[C];
#pragma unroll
      for (int c = 0; c < C; ++c) vf[c] = (float)(int8_t)(vraw[p][c / 4] >> (8 * (c % 4)));
      if constexpr (G >= 4) {
        float w[HB];
#pragma unroll
        for (int b = 0; b < HB; ++b) w[b] = wsh[p * G + (lane & 3) * HB + b];
#pragma unroll
        for (int b = 0; b < HB; ++b)
#pragma unroll
          for (int c = 0; c < C; ++c) acc[b][c] = mfma4x64x1f(w[b], vf[c], acc[b][c]);
      } else {
#pragma unroll
        for (int h = 0; h < G; ++h) {
          const float w = wsh[p * G + h];
#pragma unroll
          for (int c = 0; c < C; ++c) acc[0][c][h] = fmaf(vf[c], w, acc[0][c][h]);
        }
      }
    }
  }

  // finished here: a sliding token with one split (acc * (1/l)), and every
  // token when the plan has one split (full layers: the merge of one split,
  // (acc * c) * (1/(l * c)) with c = fast_exp(0))
  const bool direct = S == 1 && (a.window > 0 || a.s_max == 1);
#pragma unroll
  for (int h = 0; h < G; ++h) {
    const float mh = readlane_f(m[h % 4], 16 * (h / 4));
    const float lh = readlane_f(l[h % 4], 16 * (h / 4));
    const int64_t qrow = (int64_t)tok * a.num_q + qh0 + h;
    if (direct) {
      uint16_t o[C];
      if (a.window > 0) {
        const float inv_l = lh > 0.0f ? 1.0f / lh : 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c)
          o[c] = lh > 0.0f ? f32_to_bf16(acc[h / 4][c][h % 4] * inv_l) : 0;
      } else {
        const float cm = lh > 0.0f ? fast_exp_softmax_biased(0.0f) : 0.0f;
        const float gl = 0.0f + lh * cm;
        const float inv_l = gl > 0.0f ? 1.0f / gl : 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c)
          o[c] = gl > 0.0f ? f32_to_bf16((acc[h / 4][c][h % 4] * cm) * inv_l) : 0;
      }
      uint16_t* dst = a.out + qrow * HD + lane * C;
#pragma unroll
      for (int c = 0; c < C; ++c) dst[c] = o[c];
    } else {
      float* pa = a.ws_acc + (qrow * a.s_max + s) * HD + lane * C;
#pragma unroll
      for (int c = 0; c < C; ++c) pa[c] = acc[h / 4][c][h % 4];
      if (lane == 0) {
        a.ws_ml[(qrow * a.s_max + s) * 2 + 0] = mh;
        a.ws_ml[(qrow * a.s_max + s) * 2 + 1] = lh;
      }
    }
  }
}

// Two waves per SIMD keep the accumulators out of the AGPRs (head 512, eight
// heads: 16 sequences of 4096 positions 61.6 -> 53.4 us); head 512 with sixteen
// does not fit the registers of two (36 spilled: 38.9 us against 33.5 with one).
template <int HD, int G>
__global__ __launch_bounds__(256, HD * G >= 8192 ? 1 : 2) void k_flash_attn(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) float s_w[4][16 * G];
  const int wave = threadIdx.x >> 6;
  const int per_tok = a.num_kv * a.s_max;
  const int item = blockIdx.x * 4 + wave;
  if (item >= a.T * per_tok) return;
  // later buffer rows first: in a prefill chunk they have the longest KV
  // ranges, so the long waves start early and the short ones fill the tail
  const int tok = a.T - 1 - item / per_tok, rem = item % per_tok;
  flash_attn_wave<HD, G>(a, tok, rem / a.s_max, rem % a.s_max, s_w[wave]);
}

// ---------------------------------------------------------------------------
// Row-group attention: one workgroup of four waves per (16 / G query tokens,
// kv head, split).  The group's 16 (token, head) rows are the rows of every
// MFMA, and each step of the workgroup takes four of the reference's
// 16-position tiles.
//   A  wave w scores tile w (int8 MFMA, K rows from memory), and its tile
//      maxima go to LDS; after a barrier every row's running maximum, the
//      tile's correction, weights and 16-lane weight sum follow, and go to LDS.
//   B  after a second barrier every wave applies the four tiles, in order, to
//      its quarter of the head's columns: acc *= corr, then acc += w * v by
//      f32 MFMA, whose products are exactly the reference's fmaf chain over
//      the positions (mfma16x16x4f).
// Rows keep their own m, l and acc and the reference's tile recursion, which
// needs tiles counted from the row's own first position: tokens of one run
// whose ranges start equal mod 16 are one set, on one tile grid; the tiles of
// a group's sets follow each other.  A row outside a tile has corr 1 and
// weights 0, which leave its acc (never -0) bit for bit.
// It is bound by instruction issue: the f32 MFMA runs on the vector ALU's own
// multipliers (33 cycles for 1024 fmaf per SIMD, and none of another wave's
// vector work beside it), so a step of head 256 costs 64 of them plus about
// 400 vector instructions per wave.  The block of 2048 tokens from position 0
// (sliding, head 256): 598 -> 412 us, attention alone 403 -> 222 us against a
// wave per 8 tokens on v_fma; 700 + 411 tokens (full, head 512): 699 -> 396 us.
// LONE: the instance of split plans with one or two heads per kv head, whose
// sets need several tokens to fill a group's rows: a workgroup with few takes
// four tokens, a wave each, as k_flash_attn does.  A group walks its tiles in
// the time of about three such waves, so it pays from three tokens per set.
template <int HD, int G, bool LONE>
__global__ __launch_bounds__(256, HD >= 512 ? 2 : 3) void k_flash_attn_rows(AttnArgs a, int nblk) {
  constexpr int C = HD / 64;    // 64-byte K chunks per row; column tiles per wave
  constexpr int TPW = 16 / G;   // tokens per group
  constexpr int NL = G >= 4 ? 1 : 4 / G;  // tokens among a lane's four rows
  constexpr int NT = 16 * TPW;  // tokens per block
  // a step's weights [position][row]; corrections, weight sums (row 4: a spare)
  // and maxima [tile][row]
  __shared__ __attribute__((aligned(16))) float s_w[64 * 16];
  __shared__ __attribute__((aligned(16))) float s_corr[4][16], s_sum[5][16], s_tm[4][16];
  __shared__ __attribute__((aligned(16))) float s_mn[4][16];  // per wave: its tile's new maxima
  __shared__ __attribute__((aligned(16))) int8_t s_q[C][1024];  // the A operands, by lane
  __shared__ __attribute__((aligned(16))) float s_qb[16], s_fq[16];  // per row
  __shared__ __attribute__((aligned(16))) int s_qs[16];
  __shared__ uint64_t s_row[4][64];  // per wave: the step's cache row offsets
  __shared__ int s_set[TPW][4];      // sets: first position, end, page table offset, first tile
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
  const int p16 = lane & 15, grp = lane >> 4;
  // kv head fastest (workgroups go round the XCDs, so an XCD's L2 sees few kv
  // heads), then split, then the block's groups; later tokens first: in a
  // prefill chunk they have the longest ranges, and the short ones fill the tail
  int item = blockIdx.x;
  const int kvh = item % a.num_kv;
  item /= a.num_kv;
  const int s = item % a.s_max;
  item /= a.s_max;
  // (the parts come last: where one alone has work, workgroups without any
  // between it would leave some shader engines idle)
  const int part = item / (nblk * 16);
  item -= part * nblk * 16;
  // (every other block's groups in reverse: a CU takes every 32nd workgroup of
  // its XCD, which would be the longest ranges of each block for some CUs and
  // the shortest for others)
  const int cls = (item / 16) & 1 ? 15 - item % 16 : item % 16;
  const int t0 = (nblk - 1 - item / 16) * NT, t1 = min(t0 + NT, a.T);
  const int run0 = run_of(a.runs, a.num_runs, t0);
  auto run_from = [&](int tok) {  // run_of(tok), tok >= t0
    int r = run0;
    while (r + 1 < a.num_runs && tok >= a.runs[r + 1].buf_start) ++r;
    return r;
  };
  // whether f(position) holds for a token of the block
  auto any_pos = [&](auto f) {
    bool x = false;
#pragma unroll
    for (int q = 0; q < NT; q += kWave) {
      const int tok = t0 + q + lane;
      if (tok < t1) {
        const KvRun run = a.runs[run_from(tok)];
        x |= f(run.base_pos + (tok - run.buf_start));
      }
    }
    return __ballot(x) != 0;
  };
  // the first token's position and, in a block of one run, the last one's
  const bool one = run0 + 1 >= a.num_runs || a.runs[run0 + 1].buf_start >= t1;
  const int pos0 = a.runs[run0].base_pos + (t0 - a.runs[run0].buf_start), pos1 = pos0 + (t1 - 1 - t0);
  // Groups take neighbours where every range starts at position 0 (no tile of
  // one is past the other), and tokens 16 apart where windows slide (equal
  // starts mod 16).
  int tok0 = t0 + cls * TPW, step = 1;
  // LONE, from position 0: split s starts at s * ceil(L / S), so with fewer
  // splits than the group has tokens those that start together are S neighbours
  // (from a position that S divides), and equal mod 16 those 16 S, 32 S, ...
  // on.  sn > 0: the group is these, sn = S, counted round the block; S divides
  // the group, so the block's end fits its beginning.
  int sn = 0, turn = 0;
  if constexpr (LONE) {
    // three tokens per group of those 16 (S) apart, or fewer at the end of a
    // long chunk, whose other blocks fill the chip; the launch has the groups then
    const bool spread = t1 - t0 >= 48 || nblk > 1;
    bool lone = true;
    if (a.window > 0 && pos0 >= a.window - 1) {  // every window of the block slides
      lone = !(spread &&
               (one || !any_pos([&](int pos) { return pos < a.window - 1; })));
      tok0 = t0 + cls;
      step = 16;
    } else if (one && (a.window <= 0 || pos1 < a.window) && pos1 + 1 >= a.s_max * kRowsSplitLen &&
               (a.s_max >= TPW || (TPW % a.s_max == 0 && spread))) {
      lone = false;
      if (a.s_max < TPW) {
        sn = a.s_max;
        turn = pos0 % sn;
      }
    }
    if (lone) {
      // the block's tokens from the last, over its workgroups of all parts
      const int wgs = nblk > 1 ? NT / 4 : (a.T + 3) / 4;
      const int tok = t0 + 4 * (wgs - 1 - (part * 16 + item % 16)) + wave;
      if (part * 16 + item % 16 < wgs && tok < a.T)
        flash_attn_wave<HD, G>(a, tok, kvh, s, s_w + wave * 16 * G);
      return;
    }
    if (part > 0) return;
  } else if (a.window > 0 && (one ? pos1 >= a.window : any_pos([&](int pos) { return pos >= a.window; }))) {
    tok0 = t0 + cls;
    step = 16;
  }
  // token k of the group (none from a.T on)
  auto token = [&](int k) {
    if (!LONE || sn == 0) return tok0 + step * k;
    return t0 + ((k % sn + sn * cls + 16 * sn * (k / sn) - turn) & (NT - 1));
  };
  if (sn == 0 && tok0 >= a.T) return;
  const int64_t kvs = (int64_t)a.num_kv * HD;

  // token lane % TPW of the group: its positions [t_beg, t_end) of this split,
  // its number of splits (0: no token), its set
  int t_beg = 0, t_end = 0, t_S, t_set = -1, nsets = 0, tiles = 0;
  {
    const int tok = token(lane % TPW);
    const int r = run_from(min(tok, a.T - 1));
    const KvRun run = a.runs[r];
    const int pos = run.base_pos + (tok - run.buf_start);
    const int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
    const int L = pos + 1 - lo;  // <= 0: no positions
    t_S = num_splits(L, a.s_max);
    const int per = (L + t_S - 1) / t_S;
    if (tok < a.T && s < t_S && s * per < L) {
      t_beg = lo + s * per;
      t_end = lo + (s * per + per < L ? s * per + per : L);
    }
    if (tok >= a.T) t_S = 0;
    if (!__ballot(s < t_S)) return;  // no token has this split
    unsigned todo = (unsigned)__ballot(lane < TPW && t_end > t_beg);
    for (; todo; ++nsets) {  // uniform; every wave makes the same table
      const int f = __ffs((int)todo) - 1;
      const bool in = ((todo >> (lane % TPW)) & 1u) && r == __builtin_amdgcn_readlane(r, f) &&
                      ((t_beg - __builtin_amdgcn_readlane(t_beg, f)) & 15) == 0;
      if (in) t_set = nsets;
      todo &= ~(unsigned)__ballot(lane < TPW && in);
      int pbeg = in ? t_beg : 0x7FFFFFFF, pend = in ? t_end : 0;
#pragma unroll
      for (int o = 1; o < TPW; o <<= 1) {
        pbeg = min(pbeg, __shfl_xor(pbeg, o, kWave));
        pend = max(pend, __shfl_xor(pend, o, kWave));
      }
      if (lane == 0) {
        s_set[nsets][0] = pbeg;
        s_set[nsets][1] = pend;
        s_set[nsets][2] = __builtin_amdgcn_readlane(run.rows_off, f);
        s_set[nsets][3] = tiles;
      }
      tiles += (__builtin_amdgcn_readfirstlane(pend) - __builtin_amdgcn_readfirstlane(pbeg) + 15) >> 4;
    }
  }

  // A operand: row r = k * G + h (token k, head h); lane (r + 16 g) holds row
  // r's bytes [c*64 + g*16, +16).  Scores: lane (p + 16 g), value i <-> row
  // 4 g + i, position p.
  const v4i zero4 = {0, 0, 0, 0};
  {
    const int tok = min(token(p16 / G), a.T - 1);  // (rows without a token: never used)
    const int64_t qrow = (int64_t)tok * a.num_q + kvh * G + p16 % G;
    int part = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const v4i q = ld16(a.q_i8 + qrow * HD + c * 64 + grp * 16);
      const int w4[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        part += (int)(int8_t)w4[j] + (int)(int8_t)(w4[j] >> 8) + (int)(int8_t)(w4[j] >> 16) +
                (w4[j] >> 24);
      if (c % 4 == wave) *reinterpret_cast<v4i*>(&s_q[c][lane * 16]) = q;
    }
    part += __shfl_xor(part, 16, kWave);
    part += __shfl_xor(part, 32, kWave);  // lane r (and r + 16 g): sum of row r's codes
    if (wave == 0 && lane < 16) {
      s_qs[lane] = 128 * part;  // the u8-shifted dot of the reference is dot + 128 * sum(q)
      s_qb[lane] = a.qi_bias[qrow];
      s_fq[lane] = a.f_q[qrow];
    }
  }
  lds_barrier();

  // positions of this lane's rows 4 grp + i, and of row p16, and their sets
  int lo[NL], hi[NL], rs[NL];
#pragma unroll
  for (int t = 0; t < NL; ++t) {
    const int k = 4 * grp / G + t;
    lo[t] = __shfl(t_beg, k, kWave);
    hi[t] = __shfl(t_end, k, kWave);
    rs[t] = __shfl(t_set, k, kWave);
  }
  const int lo_r = __shfl(t_beg, p16 / G, kWave), hi_r = __shfl(t_end, p16 / G, kWave);
  const int rs_r = __shfl(t_set, p16 / G, kWave);

  const float inv127 = 1.0f / 127.0f;
  const float inv127sq = inv127 * inv127;
  float m = -1e30f, l = 0.0f;  // row p16's running maximum and sum
  v4f acc[C];                  // columns (wave * 16 + p16) * C + ct, rows 4 grp + i
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  const int8_t* kbase = a.k_cache + (int64_t)kvh * HD + grp * 16;
  const int8_t* vbase = a.v_cache + (int64_t)kvh * HD + (wave * 16 + p16) * C;

  // Tile n0 + grp of the list: its set (-1 past the last tile), its first
  // position and the slot of its position p16 (those past the set's end, or
  // the list's, repeat a position: their weights are 0).
  int n_set = 0, n_pos = 0, slot = 0;
  auto next_tiles = [&](int n0) {
    const int n = min(n0 + grp, tiles - 1);
    int c = n_set < 0 ? nsets - 1 : n_set;
    while (c + 1 < nsets && n >= s_set[c + 1][3]) ++c;
    const int beg = s_set[c][0] + 16 * (n - s_set[c][3]);
    const int p = min(beg + p16, s_set[c][1] - 1);
    slot = (int)paged_slot(a.base_rows + s_set[c][2], a.page_shift, a.row_mask, a.page_mask, p);
    n_set = n0 + grp < tiles ? c : -1;
    n_pos = beg;
  };
  v4i kb[C];
  float ks, vs;
  auto load_k = [&]() {  // K rows of tile `wave`; all rows' byte offsets through LDS
    // (a wave's own LDS accesses are in order: no barrier)
    s_row[wave][lane] = (uint64_t)(uint32_t)slot * (uint32_t)kvs;
    const int64_t my = __shfl(slot, 16 * wave + p16, kWave);
    const int8_t* kr = kbase + s_row[wave][16 * wave + p16];
#pragma unroll
    for (int c = 0; c < C; ++c) kb[c] = ld16(kr + c * 64);
    ks = a.k_scale[my * a.num_kv + kvh];
    vs = a.v_scale[my * a.num_kv + kvh];
  };
  if (tiles > 0) {
    next_tiles(0);
    load_k();
  }
  for (int n0 = 0; n0 < tiles; n0 += 4) {
    const int set = n_set, pos = n_pos;  // of tile n0 + grp
    // this step's V: lane (j + 16 k) holds C bytes of position 4 u + k
    uint32_t vraw[16][(C + 3) / 4];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int8_t* vr = vbase + s_row[wave][4 * u + grp];
      if constexpr (C == 8) {
        const uint2 w = *reinterpret_cast<const uint2*>(vr);
        vraw[u][0] = w.x; vraw[u][1] = w.y;
      } else if constexpr (C == 4) {
        vraw[u][0] = *reinterpret_cast<const uint32_t*>(vr);
      } else if constexpr (C == 2) {
        vraw[u][0] = *reinterpret_cast<const uint16_t*>(vr);
      } else {
        vraw[u][0] = (uint8_t)*vr;
      }
    }
    next_tiles(n0 + 4);
    // ---- A: scores of tile `wave` -------------------------------------------
    const int w_set = __builtin_amdgcn_readlane(set, 16 * wave);
    const int w_pos = __builtin_amdgcn_readlane(pos, 16 * wave);
    v4i d = zero4;
#pragma unroll
    for (int c = 0; c < C; ++c)
      d = mfma16x16x64(*reinterpret_cast<const v4i*>(&s_q[c][lane * 16]), kb[c], d);
    const v4i qs4 = *reinterpret_cast<const v4i*>(&s_qs[4 * grp]);
    const v4f qb4 = *reinterpret_cast<const v4f*>(&s_qb[4 * grp]);
    const v4f fq4 = *reinterpret_cast<const v4f*>(&s_fq[4 * grp]);
    float sco[4], tm[4];
    bool on[4], ok[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = NL == 1 ? 0 : i / (4 / NL);
      const bool in = rs[t] == w_set && w_pos >= lo[t];
      on[i] = in && w_pos < hi[t];
      ok[i] = in && w_pos + p16 < hi[t];
      sco[i] = (((float)(d[i] + qs4[i]) - qb4[i]) * fq4[i]) * ks * inv127sq;
      sco[i] = ok[i] ? sco[i] : -1e30f;
      tm[i] = sco[i];
    }
    row_max16_x4(tm);
    const float vs_t = vs;
    *reinterpret_cast<float4*>(&s_tm[wave][4 * grp]) = float4{tm[0], tm[1], tm[2], tm[3]};
    lds_barrier();
    // row p16, tile grp: the running maximum before and after the tile, and
    // the correction (every wave the same; 1 where the row is outside the tile)
    {
      const float x0 = s_tm[0][p16], x1 = s_tm[1][p16], x2 = s_tm[2][p16], x3 = s_tm[3][p16];
      const float a0 = max_num(m, x0), a1 = max_num(a0, x1), a2 = max_num(a1, x2);
      const float a3 = max_num(a2, x3);
      const float before = grp < 2 ? (grp == 0 ? m : a0) : (grp == 2 ? a1 : a2);
      const float after = grp < 2 ? (grp == 0 ? a0 : a1) : (grp == 2 ? a2 : a3);
      const float cr = fast_exp_softmax_le0(max_num(before - after, -87.0f));
      s_corr[grp][p16] = rs_r == set && pos >= lo_r && pos < hi_r ? cr : 1.0f;
      if (grp == wave) s_mn[wave][p16] = after;
      m = a3;
    }
    const v4f mn = *reinterpret_cast<const v4f*>(&s_mn[wave][4 * grp]);
    float wt[4], sum[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float w = fast_exp_softmax_le0(max_num(sco[i] - mn[i], -87.0f));
      const float t = row_tree16(w);  // in lane 0 of the row
      sum[i] = on[i] ? t : 0.0f;
      wt[i] = ok[i] ? w * vs_t * inv127 : 0.0f;
    }
    *reinterpret_cast<float4*>(&s_w[(16 * wave + p16) * 16 + 4 * grp]) =
        float4{wt[0], wt[1], wt[2], wt[3]};
    // (lanes without a sum write to the spare row: no branch)
    *reinterpret_cast<float4*>(&s_sum[p16 == 0 ? wave : 4][4 * grp]) =
        float4{sum[0], sum[1], sum[2], sum[3]};
    load_k();
    lds_barrier();
    // ---- B: the tiles' updates of this wave's columns -----------------------
    auto update = [&](int t) {
      const v4f cv = *reinterpret_cast<const v4f*>(&s_corr[t][4 * grp]);
      l = l * s_corr[t][p16] + s_sum[t][p16];
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][i] = acc[c][i] * cv[i];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int u = 4 * t + q;
        const float w = s_w[(4 * u + grp) * 16 + p16];
#pragma unroll
        for (int c = 0; c < C; ++c)
          acc[c] = mfma16x16x4f(w, (float)(int8_t)(vraw[u][c / 4] >> (8 * (c % 4))), acc[c]);
      }
    };
    if (n0 + 4 <= tiles) {
#pragma unroll
      for (int t = 0; t < 4; ++t) update(t);
    } else {  // a short last step
      update(0);
      if (n0 + 1 < tiles) update(1);
      if (n0 + 2 < tiles) update(2);
    }
  }

  // finished here: a sliding token with one split (acc * (1/l)), and every
  // token when the plan has one split (full layers: the merge of one split,
  // (acc * c) * (1/(l * c)) with c = fast_exp(0)); other splits are partials
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * grp + i, k = r / G, tok = token(k);
    const float lr = __shfl(l, r, kWave), mr = __shfl(m, r, kWave);
    const int S = __shfl(t_S, k, kWave);
    if (s >= S) continue;  // no such token, or no such split of it
    const int64_t qrow = (int64_t)tok * a.num_q + kvh * G + r % G;
    const int col = (wave * 16 + p16) * C;
    if (S == 1 && (a.window > 0 || a.s_max == 1)) {
      const float cm = a.window > 0 ? 1.0f : lr > 0.0f ? fast_exp_softmax_biased(0.0f) : 0.0f;
      const float gl = a.window > 0 ? lr : 0.0f + lr * cm;
      const float inv_l = gl > 0.0f ? 1.0f / gl : 0.0f;
      uint16_t* dst = a.out + qrow * HD + col;
#pragma unroll
      for (int c = 0; c < C; ++c) dst[c] = gl > 0.0f ? f32_to_bf16((acc[c][i] * cm) * inv_l) : 0;
    } else {
      float* pa = a.ws_acc + (qrow * a.s_max + s) * HD + col;
#pragma unroll
      for (int c = 0; c < C; ++c) pa[c] = acc[c][i];
      if (wave == 0 && p16 == 0) {
        a.ws_ml[(qrow * a.s_max + s) * 2 + 0] = mr;
        a.ws_ml[(qrow * a.s_max + s) * 2 + 1] = lr;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// merge of the split partials: one wave per (token, query head, 64 * CL
// columns), CL columns per lane.  It is latency: a wave's rows (NB splits) are
// all requested before the corrections are computed from the (m, l), and the
// chain over the splits in order then runs from registers.
// ---------------------------------------------------------------------------
template <int HD, int NB, int CL>
__global__ __launch_bounds__(256) void k_attn_merge(AttnArgs a) {
  constexpr int NW = HD / (64 * CL);
  const int wave = threadIdx.x >> 6, lane = lane_id();
  const int witem = blockIdx.x * 4 + wave;
  if (witem >= a.T * a.num_q * NW) return;
  const int item = witem / NW, col = ((witem % NW) * 64 + lane) * CL;
  const int tok = item / a.num_q;
  const TokRange tr = token_range(a, tok);
  const int S = num_splits(tr.L, a.s_max);
  if (a.window > 0 && S == 1) return;  // finalized by the attention wave
  const int64_t base = (int64_t)item * a.s_max;
  const float* ml = a.ws_ml + base * 2;
  const float* src = a.ws_acc + base * HD + col;
  float rows[NB][CL];
  auto load_rows = [&](int s0) {  // splits past S repeat the last (never used)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < CL; ++j) rows[b][j] = src[(int64_t)min(s0 + b, S - 1) * HD + j];
  };
  float gm = -1e30f;
  for (int s0 = 0; s0 < S; s0 += kWave) {
    const float v = s0 + lane < S ? ml[(s0 + lane) * 2] : -1e30f;
    gm = fmaxf(gm, wave_max(v));
  }
  load_rows(0);
  float gl = 0.0f, out[CL];
#pragma unroll
  for (int j = 0; j < CL; ++j) out[j] = 0.0f;
  bool first = true;
  for (int s0 = 0; s0 < S; s0 += kWave) {
    // the corrections of 64 splits, lane-parallel; masked by l > 0
    const int sidx = s0 + lane;
    float d = -1e30f, ls = 0.0f;
    if (sidx < S) { d = ml[sidx * 2] - gm; ls = ml[sidx * 2 + 1]; }
    float c = fast_exp_softmax_biased(max87(d));
    if (!(ls > 0.0f)) c = 0.0f;
    // global l: batches of 16 splits, each a 16-lane tree of l * c
    const float bsum = tree16(ls * c);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (s0 + 16 * q < S) gl = gl + readlane_f(bsum, 16 * q);
    // acc: splits in order; those with a correction of 0 are left out, and the
    // first of the others is multiplied
    const unsigned long long live = __ballot(c > 0.0f);
#pragma unroll
    for (int h = 0; h < kWave; h += NB) {
      if (s0 + h >= S) break;
      if (s0 + h > 0) load_rows(s0 + h);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        if (!((live >> (h + b)) & 1ull)) continue;  // uniform
        const float cb = readlane_f(c, h + b);
#pragma unroll
        for (int j = 0; j < CL; ++j) out[j] = first ? rows[b][j] * cb : fmaf(rows[b][j], cb, out[j]);
        first = false;
      }
    }
  }
  uint16_t* dst = a.out + (int64_t)item * HD + col;
#pragma unroll
  for (int j = 0; j < CL; ++j) dst[j] = gl > 0.0f ? f32_to_bf16(out[j] * (1.0f / gl)) : (uint16_t)0;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// (token, head) items from which the prep takes four heads per wave: 3200 items
// (100 tokens, 32 heads of 256) 1.3 us faster than a wave per head, 65536 items
// 48.4 -> 23.4 us; below 2048 a wave per item still leaves CUs to spare
constexpr int kPrepV8Items = 2048;

hipError_t launch_attn_prep(const PrepArgs& args, int head_dim, hipStream_t st) {
  PrepArgs a = args;
  a.fwht_scale = fwht_scale_host(head_dim);
  const int items = a.T * (a.num_q + 2 * a.num_kv);
  if (items <= 0) return hipSuccess;
  const dim3 g((items + 3) / 4), b(256);
  auto aligned = [](const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; };
  if (head_dim >= 128 && items >= kPrepV8Items && a.pair_stride == head_dim / 2 &&
      a.rope_half > 0 && aligned(a.q_src, 16) && aligned(a.k_src, 16) &&
      aligned(a.v_src, 16) && aligned(a.q_norm, 16) && aligned(a.k_norm, 16) &&
      aligned(a.cos_table, 16) && aligned(a.sin_table, 16) && aligned(a.q_i8, 8) &&
      aligned(a.k_cache, 8) && aligned(a.v_cache, 8)) {
    const dim3 gv((a.T * ((a.num_q + 2 * a.num_kv + 3) / 4) + 3) / 4);
    switch (head_dim) {
      case 128: hipLaunchKernelGGL(k_attn_prep_v8<128>, gv, b, 0, st, a); break;
      case 256: hipLaunchKernelGGL(k_attn_prep_v8<256>, gv, b, 0, st, a); break;
      case 512: hipLaunchKernelGGL(k_attn_prep_v8<512>, gv, b, 0, st, a); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  switch (head_dim) {
    case 64: hipLaunchKernelGGL(k_attn_prep<1>, g, b, 0, st, a); break;
    case 128: hipLaunchKernelGGL(k_attn_prep<2>, g, b, 0, st, a); break;
    case 256: hipLaunchKernelGGL(k_attn_prep<4>, g, b, 0, st, a); break;
    case 512: hipLaunchKernelGGL(k_attn_prep<8>, g, b, 0, st, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int HD>
static hipError_t launch_attn_hd(const AttnArgs& a, int gqa, hipStream_t st) {
  const dim3 b(256);
  // Row groups need neighbours in a run to share tiles with: two groups' tokens
  // per run, and 20 with four heads or fewer, whose sliding windows share tiles
  // 16 tokens apart (200 tokens of one run at position 2000, sliding, both
  // kernels: a wave per token 130 us, groups 54; 16 tokens of four heads 14.6 /
  // 23).  A decode step's tokens share nothing and take a wave each (one split,
  // two heads of 256, 512 sequences of 1000 positions 325 us, in groups 496;
  // eight of 512, 256 sequences of 1500 545 / 700).  One-split plans of 16
  // heads, which fill a group's rows by themselves, and of eight up to head 256
  // stay in groups, whose four waves walk a range in a quarter of the steps (16
  // heads of 256, 600 sequences of 1500 346 / 176; eight of 128, 512 sequences
  // 221 / 165).
  const int tpw = 16 / gqa, nblk = (a.T + 16 * tpw - 1) / (16 * tpw);
  const int chunk = gqa >= 8 ? 2 * tpw : std::max(2 * tpw, 20);
  // LONE: workgroups for four tokens each, and for a block's 16 groups where it
  // can have them
  const bool lone = attn_rows_lone(gqa, a.s_max);
  const int need = (a.T + 3) / 4, groups = a.T < 48 ? need : std::max(16, need);
  const int per = !lone ? nblk * 16 : nblk > 1 ? nblk * 4 * tpw : groups;
  // (a launch has fewer than 2^24 workgroups of 256: past that a wave per token,
  // of which a workgroup has four)
  const bool fits = (int64_t)per * a.num_kv * a.s_max < (1 << 24);
  if (fits && (a.T >= chunk * a.num_runs ||
               (a.s_max == 1 && (gqa == 16 || (gqa == 8 && HD <= 256))))) {
    const dim3 g(per * a.num_kv * a.s_max);
    switch (gqa) {
      case 1:
        if (lone) hipLaunchKernelGGL((k_flash_attn_rows<HD, 1, true>), g, b, 0, st, a, nblk);
        else hipLaunchKernelGGL((k_flash_attn_rows<HD, 1, false>), g, b, 0, st, a, nblk);
        break;
      case 2:
        if (lone) hipLaunchKernelGGL((k_flash_attn_rows<HD, 2, true>), g, b, 0, st, a, nblk);
        else hipLaunchKernelGGL((k_flash_attn_rows<HD, 2, false>), g, b, 0, st, a, nblk);
        break;
      case 4: hipLaunchKernelGGL((k_flash_attn_rows<HD, 4, false>), g, b, 0, st, a, nblk); break;
      case 8: hipLaunchKernelGGL((k_flash_attn_rows<HD, 8, false>), g, b, 0, st, a, nblk); break;
      case 16: hipLaunchKernelGGL((k_flash_attn_rows<HD, 16, false>), g, b, 0, st, a, nblk); break;
      default: return hipErrorInvalidValue;
    }
  } else {
    const int items = a.T * a.num_kv * a.s_max;
    const dim3 g((items + 3) / 4);
    switch (gqa) {
      case 1: hipLaunchKernelGGL((k_flash_attn<HD, 1>), g, b, 0, st, a); break;
      case 2: hipLaunchKernelGGL((k_flash_attn<HD, 2>), g, b, 0, st, a); break;
      case 4: hipLaunchKernelGGL((k_flash_attn<HD, 4>), g, b, 0, st, a); break;
      case 8: hipLaunchKernelGGL((k_flash_attn<HD, 8>), g, b, 0, st, a); break;
      case 16: hipLaunchKernelGGL((k_flash_attn<HD, 16>), g, b, 0, st, a); break;
      default: return hipErrorInvalidValue;
    }
  }
  if (a.s_max == 1) return hipGetLastError();  // every token finished in the wave
  // up to 16 splits: two columns per lane and as many rows in flight as the
  // plan can have (16 sequences of 1024 positions, sliding, 16 splits: the two
  // attention kernels 24.4 us, with 32 rows 25.0); more splits (few tokens):
  // one column, 32 rows (64 splits, 16 tokens, head 512, partials not in L2:
  // 9.8 us; with the rows staged in LDS for one wave's chain 16.6)
  constexpr int CL = HD >= 128 ? 2 : 1;
  const int waves = a.T * a.num_q * (HD / 64);
  const dim3 g2((waves / CL + 3) / 4), g1((waves + 3) / 4);
  if (a.s_max <= 2) hipLaunchKernelGGL((k_attn_merge<HD, 2, CL>), g2, b, 0, st, a);
  else if (a.s_max <= 4) hipLaunchKernelGGL((k_attn_merge<HD, 4, CL>), g2, b, 0, st, a);
  else if (a.s_max <= 8) hipLaunchKernelGGL((k_attn_merge<HD, 8, CL>), g2, b, 0, st, a);
  else if (a.s_max <= 16) hipLaunchKernelGGL((k_attn_merge<HD, 16, CL>), g2, b, 0, st, a);
  else hipLaunchKernelGGL((k_attn_merge<HD, 32, 1>), g1, b, 0, st, a);
  return hipGetLastError();
}

hipError_t launch_flash_attn(const AttnArgs& a, int head_dim, hipStream_t st) {
  if (a.T <= 0) return hipSuccess;
  const int gqa = a.num_q / a.num_kv;
  switch (head_dim) {
    case 64: return launch_attn_hd<64>(a, gqa, st);
    case 128: return launch_attn_hd<128>(a, gqa, st);
    case 256: return launch_attn_hd<256>(a, gqa, st);
    case 512: return launch_attn_hd<512>(a, gqa, st);
    default: return hipErrorInvalidValue;
  }
}

int attn_splits(int seq_len, int num_kv, int max_kv_len) {
  // enough splits for ~2048 waves (BQ_ATTN_WAVES), each at least
  // kAttnMinSplit positions
  if (seq_len <= 0 || num_kv <= 0) return 1;
  const int64_t items = (int64_t)seq_len * num_kv;
  const int64_t target = tune().attn_waves ? tune().attn_waves : 2048;
  int s = (int)((target + items - 1) / items);
  const int cap = max_kv_len > 0 ? (max_kv_len + kAttnMinSplit - 1) / kAttnMinSplit : 1;
  if (s > cap) s = cap;
  return s < 1 ? 1 : s;
}

}  // namespace bq
