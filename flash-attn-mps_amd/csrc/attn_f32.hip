// Attention in single precision on the matrix cores: fp32 queries, keys and
// values, one kernel for prefill and for decode (counterpart of the
// reference's fp32 use of its fast and decode kernels,
// flash_attn_mps/_attention.py:134-158, with the features of its tiled one,
// kernels/attention.metal:29-51).
//
// What bounds it: v_mfma_f32_32x32x2_f32 does 64 FLOP per SIMD and clock
// (157 TFLOP/s), 1/16 of the bf16 rate, so a 32-key x 32-column stage at d128
// is 128 MFMAs = 8192 cycles against ~300 VALU instructions of softmax and
// 32 KiB of K/V: prefill is MFMA-bound, and every score feature (softcap with
// tanhf, ALiBi, masks) is a run-time branch that hides behind the MFMAs.
// Decode is HBM-bound: a stage reads its 32 KiB in 8192 cycles per SIMD,
// 1024 SIMDs x 32 KiB / 3.4 us = 9.8 TB/s, above what HBM delivers.  All
// products, probabilities and sums are fp32, as in the generic kernel.
//
// * A workgroup takes 32 columns, (query head, query row) pairs of one KV
//   head: 32 rows of one head in prefill, the group's heads at one row each
//   in decode, or R rows of 32 / R heads between.  Its four waves take the
//   32-key stages j = w, w + 4, ... (by absolute key, so a row's order of
//   summation does not depend on the rest of the batch) and combine (m, l, O)
//   through LDS at the end.  Splitting the keys over the waves, rather than
//   giving each wave its own rows, quarters the longest chain of a causal
//   block and lets a grid of 32-row blocks fill the 1024 SIMDs.
// * S^T = K Q^T: lane (key l32, half hh) loads its key row 16 bytes at a
//   time straight from global memory (dims 8 t + 4 hh .. +4 feed four MFMAs;
//   the contraction order is free), Q^T comes from LDS in operand order.
//   S^T's accumulator i then holds key 8 (i / 4) + 4 hh + i % 4 of the lane's
//   column, which is the B operand of O^T += V^T P^T as it stands when V's
//   lanes load that key's row: no shuffle, no LDS trip, no rounding of P.
//   V lane m holds dims 4 m .. 4 m + 3 (one 16-byte load feeds four MFMAs,
//   each of its own 32-dim block {4 m + n}).
// * K and V move in quarters (of the row's dims; of the stage's keys), each
//   loaded one quarter ahead of its MFMAs (1024 cycles at d128, three times
//   that with three waves on the SIMD).  K and V then share 32 registers and
//   three workgroups fit a CU at d128, four at d64.  Same process against
//   halves (64 registers, two workgroups): 2 x 4096 tokens 16/8 heads d128
//   2338 -> 2238 us (123 TFLOP/s; a 8192^3 fp32 matrix product of the library
//   154), 2 x 1024 causal d64 68.1 -> 61.8, d128 unchanged at 111; whole tiles
//   in flight (128 registers) spilled 35.
//   K/V go through registers: at 16 bytes per clock and CU they leave the
//   load path three quarters idle, and LDS tiles would only add barriers.
//   Two accumulators for S^T instead of one chain: no change.
// * A product with weight 0 still meets its V, so a NaN or an infinity in V
//   reaches every row of the block.  The outputs show it: a block with one
//   that is not finite runs its rows again one by one (f32_row), over the keys
//   each sees, at the generic kernel's speed.  The check costs the others one
//   barrier (2 x 1024 causal 16/8 d128 114 us with and without).
// * Measured (generic kernel before): 2 x 1024 tokens causal, 16/8 heads,
//   d128 4971 -> 111 us (77 TFLOP/s; 1024 workgroups for 256 CUs); decode of
//   4 requests x 2048 keys 252 + 14 (merge) -> 22 + 4 us.
#include "attn_common.h"

#include <climits>
#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int F32_COLS = 32, F32_STAGE = 32, F32_WAVES = 4;
constexpr int F32_ROUND = F32_STAGE * F32_WAVES;   // keys per pass of the four waves

struct F32Shape {
  int log2_rows;    // a column block holds 2^log2_rows query rows of each of `heads` heads
  int heads;        // query heads per workgroup
  int tiles;        // workgroups per KV head: ceil(group / heads)
  int n_qblocks;
  int log2_page;    // >= 0: page size 2^log2_page; -1: any other page size; packed K/V unused
  int vec_out;      // fp32 output rows take 16-byte stores
};

// 32-dim blocks of O^T (one, two, four or eight).
template <int DV> constexpr int f32_blocks() { return DV <= 32 ? 1 : DV <= 64 ? 2 : DV <= 128 ? 4 : 8; }
template <int DQ, int DV> constexpr size_t f32_lds_bytes() {
  const size_t q = (size_t)(DQ / 8) * 64 * 16;
  const size_t combine = (size_t)F32_COLS * (2 * (32 * f32_blocks<DV>() + 4) + 2 * F32_WAVES) * 4;
  return q > combine ? q : combine;
}

FA_DEV float f32_sum_hh(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
FA_DEV float f32_max_hh(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
FA_DEV uint64_t shfl_u64(uint64_t x, int src) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)(uint32_t)x);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)(uint32_t)(x >> 32));
  return (uint64_t)hi << 32 | lo;
}

// One row (query row tq at position qa, head h, of KV head kh) over its keys of
// [t0, t1), one key per lane and only the values of keys with weight, as the
// generic kernel does: for blocks whose products met a value that is not
// finite (0 * inf in the rows that do not see it).
template <int DQ, int DV>
FA_DEV void f32_row(const fa_attn_args& a, int64_t b, const RequestInfo& r, int kh, int64_t h, int64_t tq, int qa, int split,
                    int lo, int hi, int lo2, int hi2, int t0, int t1, float scale, float slope, int lane) {
  const float* const q = (const float*)a.q + tq * a.q_stride[0] + h * a.q_stride[1];
  float m = a.sinks && split == 0 ? a.sinks[h * a.sink_stride] : -INFINITY, l = m > -INFINITY ? 1.0f : 0.0f;
  constexpr int ACC = (DV + 63) / 64;
  float acc[ACC];
#pragma unroll
  for (int i = 0; i < ACC; ++i) acc[i] = 0.0f;
  for (; t0 < t1; t0 += 64) {
    const int t = t0 + lane;
    const bool valid = t < t1 && ((t >= lo && t < hi) || (t >= lo2 && t < hi2));
    float s = -INFINITY;
    if (valid) {
      const float* const k = (const float*)a.k + kv_offset(a, a.k_stride, b, r, t, kh);
      float dot = 0.0f;
      for (int d = 0; d < DQ; d += 4) {
        const f32x4 x = *(const f32x4*)(q + d), y = *(const f32x4*)(k + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) dot = fmaf(x[e], y[e], dot);
      }
      s = dot * scale;
      if (a.softcap > 0.0f) s = a.softcap * tanhf(s / a.softcap);
      s -= slope * (float)abs(qa - t);
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float ref = m_new == -INFINITY ? 0.0f : m_new;
    const float factor = expf(m - ref), p = valid ? expf(s - ref) : 0.0f;
    l = l * factor + wave_sum(p);
#pragma unroll
    for (int i = 0; i < ACC; ++i) acc[i] *= factor;
    const int n = min(64, t1 - t0);
    for (int j = 0; j < n; ++j) {
      const float pj = readlane_f(p, j);
      if (pj == 0.0f) continue;
      const float* const v = (const float*)a.v + kv_offset(a, a.v_stride, b, r, t0 + j, kh);
#pragma unroll
      for (int i = 0; i < ACC; ++i)
        if (lane + 64 * i < DV) acc[i] = fmaf(pj, v[lane + 64 * i], acc[i]);
    }
    m = m_new;
  }
  const float norm = l > 0.0f ? descale_of(a.v_descale, a.v_descale_stride, b, kh) / l : 0.0f;
  const int S = a.num_splits;
  // A NaN sum is no split without keys: its LSE is NaN for the merge.
  const float lse = l > 0.0f || (S > 1 && l != 0.0f) ? m + logf(l) : -INFINITY;
#pragma unroll
  for (int i = 0; i < ACC; ++i) {
    const int d = lane + 64 * i;
    if (d >= DV) continue;
    if (S > 1) a.partial_out[((split * a.total_q + tq) * a.heads_q + h) * DV + d] = acc[i] * norm;
    else store_any(a.out, tq * a.out_stride[0] + h * a.out_stride[1] + d * a.out_stride[2], a.out_dtype, acc[i] * norm);
  }
  if (lane != 0) return;
  if (S > 1) a.partial_lse[((int64_t)split * a.heads_q + h) * a.total_q + tq] = lse;
  else a.lse[h * a.lse_stride[0] + tq * a.lse_stride[1]] = lse;
}

// DQ, DV: the tensors' head dims (multiples of 8).  V columns past DV inside
// the 32-dim blocks re-read real columns and are not stored.  MASKS: the vLLM
// mask kinds (a.mask_kind 1 or 2), in variants of their own: their second key
// range and the gaps it leaves would cost the others 4-24 spilled registers.
template <int DQ, int DV, int MINB, bool MASKS>
__global__ __launch_bounds__(64 * F32_WAVES, MINB) void attn_f32_kernel(const fa_attn_args a, const F32Shape shp) {
  static_assert(DQ % 8 == 0 && DV % 8 == 0 && DQ <= 256 && DV <= 256, "head dims");
  constexpr int KT = DQ / 8;                       // 16-byte key pieces per lane
  constexpr int NB = f32_blocks<DV>();
  constexpr int VW = NB < 4 ? NB : 4;              // dims per lane and V load (one per block)
  constexpr int VL = NB / VW;                      // V loads per key: 32 VW dims each
  typedef __attribute__((ext_vector_type(VW))) float vpiece;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Work order: KV heads fastest (a KV head of a multiple of 8 stays on one
  // XCD, whose L2 then serves all its query blocks), then head tiles,
  // requests and splits; query blocks last to first, since causal ones are
  // the longest.
  const int S = a.num_splits, hk = (int)a.heads_k, group = (int)(a.heads_q / a.heads_k);
  uint32_t id = blockIdx.x;   // 32-bit: a 64-bit division costs ~100 instructions
  const int kh = (int)(id % (uint32_t)hk);
  id /= (uint32_t)hk;
  const int tile = (int)(id % (uint32_t)shp.tiles);
  id /= (uint32_t)shp.tiles;
  const int64_t b = id % (uint32_t)a.batch;
  id /= (uint32_t)a.batch;
  const int split = (int)(id % (uint32_t)S);
  const int qb = shp.n_qblocks - 1 - (int)(id / (uint32_t)S);
  const RequestInfo r = load_request(a, b);
  const int rl = shp.log2_rows, R = 1 << rl, q0 = qb << rl;
  if (q0 >= r.q_len) return;
  const int t0 = tile * shp.heads, nheads = min(shp.heads, group - t0);
  const int h0 = kh * group + t0;

  // This lane's column: head h0 + chead, query row q0 + crow, and the keys it
  // sees, [lo, hi) and, with mask kinds, [lo2, hi2) too.
  const int chead = l32 >> rl, crow = l32 & (R - 1);
  const bool col_ok = chead < nheads && q0 + crow < r.q_len;
  const int qa = q0 + crow + r.k_len - r.q_len;
  const int64_t tq = (int64_t)r.q_begin + q0 + (col_ok ? crow : 0);
  const int hq = h0 + (col_ok ? chead : 0);
  int lo = INT_MAX, hi = 0, lo2 = INT_MAX, hi2 = 0;
  if (col_ok) {
    lo = 0, hi = r.k_len;
    auto from_window = [&](int w) { return max(qa - min(w, 1 << 30) + 1, 0); };   // keys of the last w positions
    if (!MASKS) {
      if (r.causal) hi = min(hi, qa + 1);
      if (a.window_right >= 0) hi = min(hi, qa + a.window_right + 1);
      if (a.window_left >= 0) lo = max(qa - a.window_left, 0);
    } else if (a.mask_kind == 1) {   // the causal window, and the row's range
      const int first = a.mask_window >= 0 ? from_window(a.mask_window) : 0;
      const int from = a.mask_ranges[tq * a.ranges_stride[0]];
      const int to = a.mask_ranges[tq * a.ranges_stride[0] + a.ranges_stride[1]];
      lo = first, hi = min(hi, qa + 1);
      if (from >= 0) lo2 = a.mask_clamp ? max(from, first) : from, hi2 = min(to, r.k_len - 1) + 1;
    } else {                         // the prefix, and the causal window
      lo2 = from_window(a.mask_window_len[0]), hi2 = min(hi, qa + 1);
      hi = min(hi2, a.mask_prefix[b * a.prefix_stride]);
    }
    if (hi <= lo) lo = INT_MAX, hi = 0;   // a range without keys bounds nothing
    if (hi2 <= lo2) lo2 = INT_MAX, hi2 = 0;
  }
  // Keys of the workgroup, [kbeg, kend), and those every column sees.
  const int kbeg = __builtin_amdgcn_readfirstlane(wave_min_i(min(lo, lo2)));
  const int kend = __builtin_amdgcn_readfirstlane(wave_max_i(max(hi, hi2)));
  const bool bounds = col_ok && hi > lo;
  const int full_lo = __builtin_amdgcn_readfirstlane(wave_max_i(bounds ? lo : INT_MIN));
  const int full_hi = __builtin_amdgcn_readfirstlane(wave_min_i(bounds ? hi : INT_MAX));
  // A column without keys among columns that have some: masked everywhere.
  const bool any_empty = __any(col_ok && !bounds) || MASKS;
  // This split's rounds of 128 keys.
  const int rnd0 = kbeg < kend ? kbeg / F32_ROUND : 0;
  const int nrnd = kbeg < kend ? (kend + F32_ROUND - 1) / F32_ROUND - rnd0 : 0;
  const int rb = rnd0 + (int)((int64_t)nrnd * split / S), re = rnd0 + (int)((int64_t)nrnd * (split + 1) / S);

  const float scale = a.softmax_scale * descale_of(a.q_descale, a.q_descale_stride, b, kh) *
                      descale_of(a.k_descale, a.k_descale_stride, b, kh);
  const float slope = a.alibi ? a.alibi[b * a.alibi_stride[0] + (int64_t)hq * a.alibi_stride[1]] : 0.0f;
  const bool plain = a.softcap <= 0.0f && !a.alibi;
  const float c_scale = scale * LOG2E;   // raw dot -> log2 units
  const float cap = a.softcap, cap_in = cap > 0.0f ? scale / cap : 0.0f;

  // A sink logit seeds the state of one wave of split 0 (max = sink, sum = 1).
  const float sink = (a.sinks && split == 0 && wave == 0 && col_ok) ? a.sinks[(int64_t)hq * a.sink_stride] * LOG2E : -INFINITY;
  float m_run = sink, l_run = sink > -INFINITY && hh == 0 ? 1.0f : 0.0f;
  f32x16 o[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] = 0.0f;

  const float* const khead = (const float*)a.k + (int64_t)kh * a.k_stride[2];
  const float* const vhead = (const float*)a.v + (int64_t)kh * a.v_stride[2];
  const int P = (int)a.page_size, lp = shp.log2_page;
  const int32_t* const trow = P ? a.block_table + b * a.bt_stride[0] : nullptr;
  // Mask kinds: the keys of the stage at k0 that some column sees, as bits
  // (without them, the stage's keys between kbeg and kend).
  auto seen_of = [&](int k0) -> uint32_t {
    auto ones = [](int n) { return n >= 32 ? ~0u : (1u << max(n, 0)) - 1u; };
    uint32_t mine = hi > lo ? ones(hi - k0) & ~ones(lo - k0) : 0u;
    if (hi2 > lo2) mine |= ones(hi2 - k0) & ~ones(lo2 - k0);
#pragma unroll
    for (int m = 16; m >= 1; m >>= 1) mine |= (uint32_t)__shfl_xor((int)mine, m);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)mine);
  };
  // This wave's first round from `rnd` on with such a key, and its keys.
  auto next_round = [&](int rnd, uint32_t& seen) {
    if constexpr (MASKS) {
      seen = 0u;
      for (; rnd < re; ++rnd)
        if ((seen = seen_of(F32_ROUND * rnd + F32_STAGE * wave))) break;
    }
    return rnd;
  };
  // Row offsets (elements) of key k0 + l32 in K and V.  Keys that no column
  // sees take a row that one does: their table entries and rows, which may
  // hold anything, are never read.
  auto rows_of = [&](int k0, uint32_t seen, uint64_t& kr, uint64_t& vr) {
    const int key = !MASKS ? min(max(k0 + l32, kbeg), kend - 1) : (seen >> l32) & 1 ? k0 + l32 : kbeg;
    const int64_t pos = (int64_t)r.k_base + r.left + key;
    if (P) {
      const int page = lp >= 0 ? (int)pos >> lp : (int)pos / P;
      const int64_t blk = trow[(int64_t)page * a.bt_stride[1]];
      const int64_t slot = (int)pos - page * P;
      kr = (uint64_t)(blk * a.k_stride[0] + slot * a.k_stride[1]);
      vr = (uint64_t)(blk * a.v_stride[0] + slot * a.v_stride[1]);
    } else {
      kr = (uint64_t)(pos * a.k_stride[1]);
      vr = (uint64_t)(pos * a.v_stride[1]);
    }
  };
  // Quarters: key pieces [KT q / 4, KT (q + 1) / 4) and the stage's V rows
  // 8 q + 4 hh .. +4; buffers 0 and 1 take turns.
  constexpr int KQ = (KT + 3) / 4;
  f32x4 kq[2][KQ];
  vpiece vq[2][4][VL];
  auto load_k = [&](uint64_t kr, auto q) {
    constexpr int Q = decltype(q)::value, T0 = KT * Q / 4, T1 = KT * (Q + 1) / 4;
    const float* p = khead + kr + 4 * hh;
#pragma unroll
    for (int t = T0; t < T1; ++t) kq[Q & 1][t - T0] = *(const f32x4*)(p + 8 * t);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Element 4 m + n of the row feeds block n (VW = 4; likewise 2 m + n, m);
  // lanes past the row's end re-read its last piece.
  int vcol[VL];
#pragma unroll
  for (int u = 0; u < VL; ++u) vcol[u] = min(32 * VW * u + VW * l32, DV - VW);
  auto load_v = [&](uint64_t vr, auto q) {
    constexpr int Q = decltype(q)::value;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* p = vhead + shfl_u64(vr, 8 * Q + 4 * hh + i);
#pragma unroll
      for (int u = 0; u < VL; ++u) vq[Q & 1][i][u] = *(const vpiece*)(p + vcol[u]);
      if (i % 2) __builtin_amdgcn_sched_barrier(0);
    }
  };
  const std::integral_constant<int, 0> q0c;
  const std::integral_constant<int, 1> q1c;
  const std::integral_constant<int, 2> q2c;
  const std::integral_constant<int, 3> q3c;

  // The first keys, then the queries: both round trips to memory run together.
  uint64_t kr = 0, vr = 0, kn, vn;
  int rnd = rb;
  uint32_t seen = 0;
  if (rb < re) {
    rnd = next_round(rb, seen);
    rows_of(F32_ROUND * rnd + F32_STAGE * wave, seen, kr, vr);
    load_k(kr, q0c);
  }
  // Q^T operands in LDS: piece t of lane (column l32, half hh) is dims
  // 8 t + 4 hh .. +4 of the column's query (zeros for columns without one).
  f32x4* const qs = (f32x4*)smem;
  {
    const float* qp = (const float*)a.q + tq * a.q_stride[0] + (int64_t)hq * a.q_stride[1] + 4 * hh;
    constexpr int TW = (KT + F32_WAVES - 1) / F32_WAVES;
    f32x4 x[TW];
#pragma unroll
    for (int i = 0; i < TW; ++i) x[i] = *(const f32x4*)(qp + 8 * min(wave + F32_WAVES * i, KT - 1));
#pragma unroll
    for (int i = 0; i < TW; ++i)
      if (wave + F32_WAVES * i < KT) qs[(wave + F32_WAVES * i) * 64 + lane] = col_ok ? x[i] : f32x4{0, 0, 0, 0};
  }
  __syncthreads();
  if (rb < re) {
    int next;
    for (; rnd < re; rnd = next) {
      const int k0 = F32_ROUND * rnd + F32_STAGE * wave;
      uint32_t seen_next = 0u;   // the next stage's rows (past the last one: a valid row, unused)
      next = next_round(rnd + 1, seen_next);
      rows_of(F32_ROUND * next + F32_STAGE * wave, seen_next, kn, vn);
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f;
      auto qk = [&](auto q) {
        constexpr int Q = decltype(q)::value, T0 = KT * Q / 4, T1 = KT * (Q + 1) / 4;
#pragma unroll
        for (int t = T0; t < T1; ++t) {
          const f32x4 x = qs[t * 64 + lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kq[Q & 1][t - T0][e], x[e], s, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      load_k(kr, q1c);
      qk(q0c);
      load_k(kr, q2c);
      qk(q1c);
      load_k(kr, q3c);
      qk(q2c);
      load_v(vr, q0c);
      qk(q3c);
      // s[i] = score of key k0 + 8 (i / 4) + 4 hh + i % 4.
      const int key0 = k0 + 4 * hh;
      if (plain) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] *= c_scale;
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          float x = s[i] * scale;
          if (cap > 0.0f) x = cap * tanhf(s[i] * cap_in);
          x -= slope * (float)abs(qa - (key0 + 8 * (i >> 2) + (i & 3)));
          s[i] = x * LOG2E;
        }
      }
      const bool edge = k0 < kbeg || k0 + F32_STAGE > kend;
      if (k0 < full_lo || k0 + F32_STAGE > full_hi || any_empty) {
        // Bounds relative to the stage cost the fewest registers to 64 dims,
        // absolute keys beyond (16 x 8192 keys, 16/8 heads d64 120.5 / 132.5
        // us; 32/8 d128 204.8 / 201.9; 2 x 1024 causal 16/8 d128 115.4 / 113.2).
        const int from = NB < 4 ? key0 : 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = key0 - from + 8 * (i >> 2) + (i & 3);
          const bool see = (key >= lo - from && key < hi - from) || (MASKS && key >= lo2 - from && key < hi2 - from);
          s[i] = see ? s[i] : -INFINITY;
        }
      }
      float mx = s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
      const float m_new = fmaxf(m_run, f32_max_hh(mx));
      const float mref = m_new == -INFINITY ? 0.0f : m_new;
      if (__any(m_new != m_run)) {
        const float f = fast_exp2(m_run - mref);   // 1 where the maximum stays
        l_run *= f;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[n][i] *= f;
      }
      m_run = m_new;
      float psum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[i] = fast_exp2(s[i] - mref);
        psum += s[i];
      }
      l_run += psum;
      auto pv = [&](auto q) {
        constexpr int Q = decltype(q)::value;
        if (MASKS ? seen != ~0u : edge) {   // rows that are not the stage's own: no value of theirs may reach O
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = key0 + 8 * Q + i;
            const bool own = MASKS ? (seen >> (key - k0)) & 1 : key >= kbeg && key < kend;
#pragma unroll
            for (int u = 0; u < VL; ++u)
#pragma unroll
              for (int n = 0; n < VW; ++n) vq[Q & 1][i][u][n] = own ? vq[Q & 1][i][u][n] : 0.0f;
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int u = 0; u < VL; ++u)
#pragma unroll
            for (int n = 0; n < VW; ++n)
              o[u * VW + n] =
                  __builtin_amdgcn_mfma_f32_32x32x2f32(vq[Q & 1][i][u][n], s[4 * Q + i], o[u * VW + n], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      };
      __builtin_amdgcn_sched_barrier(0);
      load_v(vr, q1c);
      pv(q0c);
      load_v(vr, q2c);
      pv(q1c);
      load_v(vr, q3c);
      pv(q2c);
      kr = kn, vr = vn;
      load_k(kr, q0c);
      pv(q3c);
      seen = seen_next;
    }
  }

  // Combine the four waves: per column the common max and the sum of the
  // scaled (l, O^T), O^T pairwise through LDS (waves 2, 3 onto 0, 1, then 1
  // onto 0), which takes half the room of four at once.
  const float lt = f32_sum_hh(l_run);
  __syncthreads();   // every wave is done with the queries
  float* const cm = (float*)smem;              // [4][32]
  float* const cl = cm + F32_WAVES * F32_COLS; // [4][32]
  constexpr int ROW = 32 * NB + 4;             // padded: one instruction's stores fall on distinct bank groups
  float* const co = cl + F32_WAVES * F32_COLS; // [2][32][ROW]
  if (hh == 0) {
    cm[wave * F32_COLS + l32] = m_run;
    cl[wave * F32_COLS + l32] = lt;
  }
  __syncthreads();
  float M = cm[l32], L = 0.0f;
#pragma unroll
  for (int w = 1; w < F32_WAVES; ++w) M = fmaxf(M, cm[w * F32_COLS + l32]);
  const float ref = M == -INFINITY ? 0.0f : M;
#pragma unroll
  for (int w = 0; w < F32_WAVES; ++w) L += cl[w * F32_COLS + l32] * fast_exp2(cm[w * F32_COLS + l32] - ref);
  const float norm = L > 0.0f ? descale_of(a.v_descale, a.v_descale_stride, b, kh) / L : 0.0f;
  const float fw = fast_exp2(m_run - ref) * norm;
  // o[u VW + n][i]: column l32, dim 32 VW u + VW (8 (i / 4) + 4 hh + i % 4) + n.
  auto piece = [&](int w, int u, int i) -> vpiece* {
    return (vpiece*)(co + (w * F32_COLS + l32) * ROW + 32 * VW * u + VW * (8 * (i >> 2) + 4 * hh + (i & 3)));
  };
  auto put = [&](int w) {
#pragma unroll
    for (int u = 0; u < VL; ++u)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        vpiece x;
#pragma unroll
        for (int n = 0; n < VW; ++n) x[n] = o[u * VW + n][i];
        *piece(w, u, i) = x;
      }
  };
  auto add = [&](int w) {
#pragma unroll
    for (int u = 0; u < VL; ++u)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const vpiece x = *piece(w, u, i);
#pragma unroll
        for (int n = 0; n < VW; ++n) o[u * VW + n][i] += x[n];
      }
  };
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[n][i] *= fw;
  if (wave >= 2) put(wave - 2);
  __syncthreads();
  if (wave < 2) add(wave);
  if (wave == 1) put(1);
  if (wave == 0) put(0);
  __syncthreads();
  // O of this thread's output pieces.  One that is not finite comes from a
  // value of the block's rows that is not (every column's sum then holds it,
  // those that give it weight 0 as NaN) or from the row's own scores.
  constexpr int D4 = DV / 4, PIECES = (F32_COLS * D4 + 64 * F32_WAVES - 1) / (64 * F32_WAVES);
  f32x4 O[PIECES];
  float probe = 0.0f;
  auto column_row = [&](int c, int& head) {   // column c's query row, -1 without one
    head = h0 + (c >> rl);
    const int row = q0 + (c & (R - 1));
    return (c >> rl) < nheads && row < r.q_len ? row : -1;
  };
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int idx = tid + 64 * F32_WAVES * i, c = idx / D4, d = 4 * (idx - c * D4);
    int h;
    if (idx >= F32_COLS * D4 || column_row(c, h) < 0) continue;
    O[i] = *(const f32x4*)(co + c * ROW + d) + *(const f32x4*)(co + (F32_COLS + c) * ROW + d);
#pragma unroll
    for (int e = 0; e < 4; ++e) probe = fmaf(O[i][e], 0.0f, probe);
  }
  int* const flags = (int*)cm;   // every wave has read the maxima
  if (lane == 0) flags[wave] = 0;
  if (__any(probe != 0.0f) && lane == 0) flags[wave] = 1;
  __syncthreads();
  if (__builtin_expect(flags[0] | flags[1] | flags[2] | flags[3], 0)) {
    for (int c = wave; c < F32_COLS; c += F32_WAVES) {
      int h;
      const int row = column_row(c, h);
      if (row < 0) continue;
      const float slope_c = a.alibi ? a.alibi[b * a.alibi_stride[0] + (int64_t)h * a.alibi_stride[1]] : 0.0f;
      f32_row<DQ, DV>(a, b, r, kh, h, (int64_t)r.q_begin + row, row + r.k_len - r.q_len, split,
                      __builtin_amdgcn_readlane(lo, c), __builtin_amdgcn_readlane(hi, c),
                      __builtin_amdgcn_readlane(lo2, c), __builtin_amdgcn_readlane(hi2, c),
                      max(kbeg, F32_ROUND * rb), min(kend, F32_ROUND * re), scale, slope_c, lane);
    }
    return;
  }
  const float lse = L > 0.0f ? M * LN2 + logf(L) : -INFINITY;
  if (wave == 0 && hh == 0 && col_ok) {
    if (S > 1) a.partial_lse[((int64_t)split * a.heads_q + hq) * a.total_q + tq] = lse;
    else a.lse[hq * a.lse_stride[0] + tq * a.lse_stride[1]] = lse;
  }
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int idx = tid + 64 * F32_WAVES * i, c = idx / D4, d = 4 * (idx - c * D4);
    int head;
    const int row = idx < F32_COLS * D4 ? column_row(c, head) : -1;
    if (row < 0) continue;
    const int64_t t = (int64_t)r.q_begin + row, h = head;
    if (S > 1) {   // partials [S][T][Hq][Dv], LSEs [S][Hq][T], as the generic kernel's
      *(f32x4*)(a.partial_out + ((split * a.total_q + t) * a.heads_q + h) * DV + d) = O[i];
    } else {
      const int64_t off = t * a.out_stride[0] + h * a.out_stride[1] + (int64_t)d * a.out_stride[2];
      if (shp.vec_out) {
        *(f32x4*)((float*)a.out + off) = O[i];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) store_any(a.out, off + e * a.out_stride[2], a.out_dtype, O[i][e]);
      }
    }
  }
}

using F32Kernel = void (*)(fa_attn_args, F32Shape);
struct F32Choice {
  F32Kernel kern;
  size_t lds;
};

// Workgroups per CU (waves per SIMD): 168 registers at three (d128 spills
// 13), 128 at four; d256 holds 128 for O^T alone and runs one.
template <int DQ, int DV, int MINB> F32Choice f32_choice(bool masks) {
  return F32Choice{masks ? attn_f32_kernel<DQ, DV, MINB, true> : attn_f32_kernel<DQ, DV, MINB, false>,
                   f32_lds_bytes<DQ, DV>()};
}

F32Choice pick_f32(int64_t dq, int64_t dv, bool masks) {
  if (dq == 192 && dv == 128) return f32_choice<192, 128, 2>(masks);
  if (dq != dv) return F32Choice{nullptr, 0};
  switch (dq) {
    case 32: return f32_choice<32, 32, 4>(masks);
    case 64: return f32_choice<64, 64, 4>(masks);
    case 72: return f32_choice<72, 72, 3>(masks);
    case 80: return f32_choice<80, 80, 3>(masks);
    case 96: return f32_choice<96, 96, 3>(masks);
    case 128: return f32_choice<128, 128, 3>(masks);
    case 256: return f32_choice<256, 256, 1>(masks);
    default: return F32Choice{nullptr, 0};
  }
}

// Every 16-byte piece of a Q, K or V row starts on a 16-byte boundary.
bool rows_aligned(const void* p, const int64_t* st, int n) {
  if ((uintptr_t)p & 15) return false;
  for (int i = 0; i < n; ++i)
    if (st[i] % 4) return false;
  return st[n] == 1;
}

}  // namespace

bool fa_f32_supported(const fa_attn_args& a) {
  if (a.q_dtype != FA_F32 || a.k_dtype != FA_F32 || a.v_dtype != FA_F32) return false;
  if (a.heads_k < 1 || a.heads_q % a.heads_k) return false;
  if (!pick_f32(a.head_dim_qk, a.head_dim_v, a.mask_kind != 0).kern) return false;
  if (a.num_splits > 1 && ((uintptr_t)a.partial_out & 15)) return false;   // 16-byte partial stores
  return rows_aligned(a.q, a.q_stride, 2) && rows_aligned(a.k, a.k_stride, 3) && rows_aligned(a.v, a.v_stride, 3);
}

int fa_f32_launch(const fa_attn_args& a, void* stream) {
  const F32Choice ch = pick_f32(a.head_dim_qk, a.head_dim_v, a.mask_kind != 0);
  const int64_t group = a.heads_q / a.heads_k;
  F32Shape shp;
  shp.log2_rows = 0;
  while (shp.log2_rows < 5 && (1ll << shp.log2_rows) < a.max_seqlen_q) ++shp.log2_rows;
  shp.heads = F32_COLS >> shp.log2_rows;
  if (shp.heads > group) shp.heads = (int)group;
  shp.tiles = (int)fa_ceil_div(group, shp.heads);
  const int64_t qblocks = fa_ceil_div(a.max_seqlen_q, 1ll << shp.log2_rows);
  const int64_t blocks = a.heads_k * shp.tiles * a.batch * a.num_splits * qblocks;
  FA_REQUIRE(qblocks <= 0x7fffffffll && blocks <= 0x7fffffffll, "fa_attn_fwd: grid too large");
  shp.n_qblocks = (int)qblocks;
  shp.log2_page = -1;
  if (a.page_size && (a.page_size & (a.page_size - 1)) == 0)
    for (shp.log2_page = 0; (1ll << shp.log2_page) < a.page_size; ++shp.log2_page) {}
  shp.vec_out = a.out_dtype == FA_F32 && a.out_stride[2] == 1 && a.out_stride[0] % 4 == 0 && a.out_stride[1] % 4 == 0 &&
                ((uintptr_t)a.out & 15) == 0;
  const hipError_t err = hipFuncSetAttribute((const void*)ch.kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ch.lds);
  if (err != hipSuccess) {
    fa_set_error("fa_attn_fwd: cannot reserve %zu bytes of LDS: %s", ch.lds, hipGetErrorString(err));
    return FA_ERR_LAUNCH;
  }
  hipLaunchKernelGGL(ch.kern, dim3((unsigned)blocks), dim3(64 * F32_WAVES), ch.lds, (hipStream_t)stream, a, shp);
  return fa_check_launch("fa_attn_fwd");
}
