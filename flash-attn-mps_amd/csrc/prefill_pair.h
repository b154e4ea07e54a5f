// MFMA prefill of 256-dim heads over 16-bit K/V by wave pairs.
//
// What bounds 256-dim heads: O^T of 32 rows is 128 registers and Q 64, so a
// wave that owns 32 whole rows fills the 512 registers of a SIMD by itself,
// spills 62 and more, and has no second wave to overlap its softmax with
// (one-pass 256/256 tile: 560 TFLOP/s with softcap, 346 with softcap and a
// window); as two workgroups per V half S and its softmax are computed twice
// (600 TFLOP/s without softcap).  Here two waves share 32 rows: each takes one
// 32-key half of every 64-key tile for S and the softmax and one 128-column
// half of V for O^T, and they exchange their probabilities through LDS.
// Nothing is computed twice, a wave holds 64 + 64 registers of O^T and Q, and
// two waves fit a SIMD (256 registers each, of which 13-15 still spill, 26 with
// softcap and a window that is not causal).  (Reference counterpart as prefill_kernel.h.)
//
// * A workgroup is eight waves, four row blocks of 32 (of one head, or two
//   blocks of each of two heads of a KV head).  Layouts, DMA, MFMA operand
//   order and numerics are those of prefill_kernel.h; the tile buffers take
//   2 x 32 KiB each for K and V, P 16 KiB, the maxima 1 KiB: one workgroup
//   per CU.
// * Per tile t, one barrier: K(t+1) and V(t) have landed, and the pair's column
//   maxima of S(t) are visible.  Then P(t) = exp2(S(t) - m) runs on the VALU
//   under the MFMAs of S(t+1) and of this wave's keys of O^T += V(t) P(t); a
//   flag in LDS says that the partner's P(t) is there (nearly always already),
//   and its keys' P.V runs over softcap, mask and maximum of S(t+1).  With a
//   workgroup barrier instead of the flag: 628 / 544 / 475 / 499 TFLOP/s where
//   the table below has 721 / 562 / 581 / 538.  Both waves of a pair take the
//   larger maximum, so their running maxima agree (lazily moved, as in
//   prefill_kernel.h); row sums are added at the end.
// * Measured, 16 sequences of 256..4096 tokens, 16/8 heads, bf16, TFLOP/s of
//   visible pairs, before -> here: causal 608 -> 721, softcap 556 -> 562, left
//   window of 1023 291 -> 581, softcap and window 346 -> 538, not causal 712
//   -> 828.  What bounds it now (counters): causal MFMA busy 30%, VALU 31%, 34%
//   of wave time waiting; softcap and window 24%, 37%, 31%: two waves per SIMD
//   do not cover the barrier, the softmax chain and LDS operand latency.
#ifndef FA_PREFILL_PAIR_H
#define FA_PREFILL_PAIR_H

#include "prefill_kernel.h"

namespace fa_prefill {

constexpr int PAIR_D = 256, PAIR_WAVES = 8, PAIR_ROWS = 128;
constexpr int PAIR_TILE = 4 * PF_GROUP_BYTES;                 // a K or V tile
constexpr int PAIR_P = 4 * PAIR_TILE;                         // P: 2 KiB a wave
constexpr int PAIR_MAX = PAIR_P + PAIR_WAVES * 2048;          // column maxima: 128 bytes a wave
constexpr int PAIR_FLAG = PAIR_MAX + PAIR_WAVES * 128;        // the tile whose P a wave has written, plus one
constexpr size_t PAIR_LDS = PAIR_FLAG + PAIR_WAVES * 16;

template <typename T, bool CAUSAL, bool CAP, bool WIN>
__global__ __launch_bounds__(64 * PAIR_WAVES, 1) void prefill_pair_kernel(const fa_attn_args a, const PrefillShape shp) {
  constexpr int KST = PAIR_D / 16, DB = 4;   // k-steps of S^T; 32-dim blocks of this wave's half of O^T
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const kbuf = smem;
  char* const vbuf = smem + 2 * PAIR_TILE;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave & 1, block = wave >> 1;
  // Work item: as prefill_kernel (requests longest first, an XCD's own KV heads).
  const int G = (int)(a.heads_q / a.heads_k) / shp.hp;
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  WorkItem wi;
  if (shp.compact) {
    bool found;
    if (a.batch <= 64)
      found = shp.hp == 2 ? compact_item<PAIR_ROWS / 2, 1>(a, slot, xcd, lane, G, wi)
                          : compact_item<PAIR_ROWS, 1>(a, slot, xcd, lane, G, wi);
    else
      found = shp.hp == 2 ? compact_item<PAIR_ROWS / 2, PF_COMPACT_MAX_BATCH / 64>(a, slot, xcd, lane, G, wi)
                          : compact_item<PAIR_ROWS, PF_COMPACT_MAX_BATCH / 64>(a, slot, xcd, lane, G, wi);
    if (!found) return;
  } else {
    const int per_pair = shp.n_qblocks * G;
    const int64_t pair = (int64_t)(slot / per_pair) * 8 + xcd;
    if (pair >= a.batch * a.heads_k) return;
    const int rem = slot % per_pair;
    wi.qb = shp.n_qblocks - 1 - rem / G;
    wi.g = rem % G;
    wi.b = a.batch > 1 && a.batch <= 64 ? request_by_rank(a, pair / a.heads_k, lane) : pair / a.heads_k;
    wi.kh = (int)(pair % a.heads_k);
    wi.r = load_request(a, wi.b);
    if ((a.flags & FA_FLAG_SKIP_SINGLE_QUERY) && wi.r.q_len == 1) return;   // the decode kernel owns it
  }
  const int64_t b = wi.b;
  const RequestInfo r = wi.r;
  const int bph = 4 / shp.hp, bmh = 32 * bph;   // row blocks and rows per head
  const int kh = wi.kh, h = (kh * G + wi.g) * shp.hp + block / bph;
  const int q0 = wi.qb * bmh;
  if (q0 >= r.q_len) return;
  const int off = r.k_len - r.q_len;   // row i sits at key position i + off
  const int wq0 = q0 + (block % bph) * 32;
  const int row = wq0 + l32, qa = row + off;

  // Keys (as prefill_kernel): window [qa - WL, qa + WR], causal up to qa.
  const int WL = WIN ? a.window_left : -1, WR = (WIN && !CAUSAL) ? (r.causal ? 0 : a.window_right) : -1;
  const int qa_first = q0 + off, qa_last = min(q0 + bmh, r.q_len) - 1 + off;
  int kv_end = r.k_len;
  if (CAUSAL) kv_end = min(kv_end, qa_last + 1);
  else if (WR >= 0) kv_end = min(kv_end, max(qa_last + WR + 1, 0));
  const int kv_begin = WL >= 0 ? min(max(qa_first - WL, 0), max(kv_end, 0)) : 0;
  const int n_tiles = kv_end > 0 ? (kv_end + PF_BN - 1) / PF_BN : 0, tile0 = kv_begin / PF_BN;
  // The pair's rows, the tiles that hold a key of theirs, [act_lo, act_hi),
  // and those whose keys all of them see, [hot_lo, hot_hi).
  const bool rows_ok = wq0 < r.q_len;
  const int lo_row = wq0 + off, hi_row = min(wq0 + 32, r.q_len) - 1 + off;
  const int key_hi = min(CAUSAL ? hi_row : WR >= 0 ? hi_row + WR : INT_MAX - PF_BN, r.k_len - 1);
  const int act_lo = WL >= 0 ? max(lo_row - WL, 0) / PF_BN : 0;
  const int act_hi = rows_ok && key_hi >= 0 ? min(n_tiles, key_hi / PF_BN + 1) : 0;
  const int hot_lo = WL >= 0 ? (max(hi_row - WL, 0) + PF_BN - 1) / PF_BN : 0;
  const int see = CAUSAL ? lo_row + 1 : WR >= 0 ? lo_row + WR + 1 : r.k_len;   // keys below this: every row
  const int hot_hi = min(act_hi, max(min(see, r.k_len), 0) / PF_BN);

  const float kdsc = descale_of(a.q_descale, a.q_descale_stride, b, kh) * descale_of(a.k_descale, a.k_descale_stride, b, kh);
  const float vdsc = descale_of(a.v_descale, a.v_descale_stride, b, kh);
  // A negative score scale flips Q's sign bits, so that the raw maximum is
  // the score's (prefill_kernel).
  const bool q_flip = a.softmax_scale * kdsc < 0.0f;
  const float kscale = q_flip ? -(a.softmax_scale * kdsc) : a.softmax_scale * kdsc;
  u32x4 qop[KST];
  {
    const uint16_t* qp = (const uint16_t*)a.q + ((int64_t)r.q_begin + min(row, r.q_len - 1)) * a.q_stride[0] +
                         (int64_t)h * a.q_stride[1] + 8 * hh;
#pragma unroll
    for (int kk = 0; kk < KST; ++kk) qop[kk] = *(const u32x4*)(qp + 16 * kk);
    if (q_flip) {
#pragma unroll
      for (int kk = 0; kk < KST; ++kk)
#pragma unroll
        for (int e = 0; e < 4; ++e) qop[kk][e] ^= 0x80008000u;
    }
  }
  // V rows past the request's last key must be finite (prefill_kernel).
  if ((tile0 + 1) * PF_BN > r.k_len || (tile0 + 1 < n_tiles && (tile0 + 2) * PF_BN > r.k_len)) {
    for (int i = tid; i < 2 * PAIR_TILE / 16; i += 64 * PAIR_WAVES) *(u32x4*)(vbuf + 16 * i) = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
  }

  // DMA: wave w moves K row block w (four 64-dim column groups) and, of V's
  // 16-key group w / 2, the four 32-dim blocks of half w % 2.
  const bool paged = a.page_size != 0;
  const int lp = shp.log2_page, pmask = (1 << lp) - 1;
  const int drow = 8 * (wave & 1) + (lane >> 3);
  const int kdoff = 2 * (int)(sigma(drow) * a.k_stride[1]) + (((lane & 7) ^ ((drow >> 1) & 7)) * 16);
  const int vdoff = 2 * (int)((lane >> 2) * a.v_stride[1]) + (lane & 3) * 16;
  const char* const khead = (const char*)a.k + 2 * (int64_t)kh * a.k_stride[2];
  const char* const vhead = (const char*)a.v + 2 * (int64_t)kh * a.v_stride[2] + 256 * half;
  const uint32_t krow_b = (uint32_t)(2 * a.k_stride[1]), vrow_b = (uint32_t)(2 * a.v_stride[1]);
  const uint32_t kpage_b = (uint32_t)(2 * a.k_stride[0]), vpage_b = (uint32_t)(2 * a.v_stride[0]);
  const int32_t* const trow = paged ? a.block_table + b * a.bt_stride[0] : nullptr;
  const int bt1 = (int)a.bt_stride[1];
  // The 16-key group from key0: base at its first row, bounded at the
  // request's last key (group_rsrc of prefill_kernel).
  auto group_rsrc = [&](const char* head, uint32_t row_b, uint32_t page_b, int key0, int row_bytes) {
    const int nvalid = min(max(r.k_len - key0, 0), 16);
    const char* g = head;
    if (nvalid > 0) {
      const int pos = key0 + r.left;
      if (paged) {
        const uint32_t blk = (uint32_t)load_invariant_i32(trow, (int64_t)(pos >> lp) * bt1);
        g = head + (uint64_t)blk * page_b + (uint32_t)(pos & pmask) * row_b;
      } else {
        g = head + (uint64_t)(uint32_t)(r.k_base + pos) * row_b;
      }
    }
    const int bytes = __builtin_amdgcn_readfirstlane(nvalid > 0 ? (nvalid - 1) * (int)row_b + row_bytes : 0);
    return __builtin_amdgcn_make_buffer_rsrc((void*)g, (short)0, bytes, 0x00020000);
  };
  auto dma_k = [&](int t) {
    const auto rsrc = group_rsrc(khead, krow_b, kpage_b, t * PF_BN + 16 * (wave >> 1), 2 * PAIR_D);
    dma_columns<4>(rsrc, kbuf + (t & 1) * PAIR_TILE + wave * 1024, kdoff);
  };
  auto dma_v = [&](int t) {
    const auto rsrc = group_rsrc(vhead, vrow_b, vpage_b, t * PF_BN + 16 * (wave >> 1), PAIR_D);
    dma_blocks<4>(rsrc, vbuf + (t & 1) * PAIR_TILE + half * 4 * PF_VBLOCK_BYTES + (wave >> 1) * 1024, vdoff);
  };

  // Operand reads (prefill_kernel): K rows 32 half .. +32 of the tile; V
  // blocks 4 half .. +4, first this wave's keys, then its partner's.
  int krd[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) krd[s] = half * 32 * 128 + l32 * 128 + (((2 * s + hh) ^ ((l32 >> 1) & 7)) * 16);
  const int vg16 = lane >> 4, vi = lane & 15, va = vi & 3, vt = vi >> 2;
  const int vrd = half * 4 * PF_VBLOCK_BYTES + (8 * (vg16 >> 1) + vt) * 64 + (4 * (vg16 & 1) + va) * 8;
  u32x4* const p_own = (u32x4*)(smem + PAIR_P + wave * 2048) + lane;
  const u32x4* const p_partner = (const u32x4*)(smem + PAIR_P + (wave ^ 1) * 2048) + lane;
  float* const max_own = (float*)(smem + PAIR_MAX + wave * 128) + l32;
  const float* const max_partner = (const float*)(smem + PAIR_MAX + (wave ^ 1) * 128) + l32;

  typedef __attribute__((address_space(3))) volatile int lds_flag;
  lds_flag* const flag_own = (lds_flag*)(smem + PAIR_FLAG + wave * 16);
  lds_flag* const flag_partner = (lds_flag*)(smem + PAIR_FLAG + (wave ^ 1) * 16);
  *flag_own = 0;   // before the first barrier
  // P(t) of the partner is in LDS: it wrote its flag after P (a wave's LDS
  // accesses complete in order), on its way from barrier A(t), which this
  // wave has passed too, without waiting for anything of this wave.
  auto wait_partner = [&](int t) {
    while (__builtin_amdgcn_readfirstlane(*flag_partner) < t + 1) {}
    asm volatile("" ::: "memory");
  };

  const float c_scale = kscale * LOG2E;
  const float cap_in = CAP ? 2.0f * LOG2E * kscale / a.softcap : 0.0f, cap_out = a.softcap * LOG2E;
  float m_run = a.sinks ? a.sinks[(int64_t)h * a.sink_stride] * LOG2E : -INFINITY;
  float l_run = (a.sinks && half == 0 && hh == 0) ? 1.0f : 0.0f;
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;

  // S^T of this wave's half of tile t: s[i] = score of key
  // 64 t + 32 half + 16 (i >> 3) + 8 hh + (i & 7).
  auto qk = [&](int t, f32x16& s) {
    const char* const kl = kbuf + (t & 1) * PAIR_TILE;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
    for (int kk = 0; kk < KST; ++kk) s = mfma32<T>(lds_read16(kl, krd[kk % 4] + (kk / 4) * PF_GROUP_BYTES), qop[kk], s);
  };
  // Softcap, mask and this wave's column maxima (log2 units) for its partner.
  float mx_own = -INFINITY;
  auto phase_a = [&](auto mask_tag, int t, f32x16& s) {
    if constexpr (CAP) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float e = fast_exp2(cap_in * s[i]);
        s[i] = cap_out * (1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f));
      }
    }
    if constexpr (decltype(mask_tag)::value) {
      const int t0 = t * PF_BN + 32 * half + 8 * hh;
      int lim = r.k_len - 1 - t0;
      if (CAUSAL) lim = min(lim, qa - t0);
      else if (WR >= 0) lim = min(lim, qa + WR - t0);
      const int lo = WL >= 0 ? qa - WL - t0 : INT_MIN;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (16 * (i >> 3) + (i & 7) > lim || 16 * (i >> 3) + (i & 7) < lo) s[i] = -INFINITY;
    }
    float mx = fmaxf(s[0], s[1]);
#pragma unroll
    for (int i = 2; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = max_hh(mx);
    mx_own = CAP ? mx : mx * c_scale;
    *max_own = mx_own;   // both lanes of a column write the same value
  };
  // The running maximum, which both waves of the pair move alike, and O^T's rescale.
  auto move_max = [&]() {
    const float cand = fmaxf(mx_own, *max_partner);
    const bool need = cand > m_run + PF_RESCALE;
    if (__builtin_expect(__any(need), 0)) {
      const float f = need ? fast_exp2(m_run - cand) : 1.0f;
      m_run = need ? cand : m_run;
      l_run *= f;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= f;
    }
  };
  auto phase_b = [&](int t, f32x16& s, u32x4 (&pop)[2]) {
    const float sc = CAP ? 1.0f : c_scale;
    const float mref = m_run == -INFINITY ? 0.0f : m_run;
    float psum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = fast_exp2(fmaf(s[i], sc, -mref));
      psum += s[i];
    }
    l_run += psum;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int q = 0; q < 4; ++q) pop[c][q] = pack2<T>(s[8 * c + 2 * q], s[8 * c + 2 * q + 1]);
      p_own[64 * c] = pop[c];
    }
    asm volatile("" ::: "memory");
    *flag_own = t + 1;
  };
  auto pv = [&](const char* vl, const u32x4 (&pop)[2]) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int imm = 16 * c * 64 + db * PF_VBLOCK_BYTES;
        const u32x2 lo = lds_read_tr(vl, vrd + imm), hi = lds_read_tr(vl, vrd + imm + 4 * 64);
        o[db] = mfma32<T>(u32x4{lo[0], lo[1], hi[0], hi[1]}, pop[c], o[db]);
      }
  };
  auto barrier_a = [&](int t) {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // this wave's DMAs
    __syncthreads();
    if (t + 1 < n_tiles) dma_v(t + 1);
    if (t + 2 < n_tiles) dma_k(t + 2);
  };
  auto pv_own = [&](int t, const u32x4 (&own)[2]) { pv(vbuf + (t & 1) * PAIR_TILE + half * 32 * 64, own); };
  auto pv_partner = [&](int t) {
    const u32x4 other[2] = {p_partner[0], p_partner[64]};
    pv(vbuf + (t & 1) * PAIR_TILE + (1 - half) * 32 * 64, other);
  };

  const std::integral_constant<bool, true> masked;
  const std::integral_constant<bool, false> unmasked;
  auto active = [&](int t) { return t >= act_lo && t < act_hi; };
  auto hot = [&](int t) { return t >= hot_lo && t < hot_hi; };
  if (tile0 < n_tiles) {
    dma_k(tile0);
    dma_v(tile0);
    if (tile0 + 1 < n_tiles) dma_k(tile0 + 1);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    f32x16 s;
    if (active(tile0)) {
      qk(tile0, s);
      phase_a(masked, tile0, s);
    }
    // Every path of a tile passes both barriers, so the pairs of a workgroup
    // may take different ones.
    for (int t = tile0; t < n_tiles; ++t) {
      barrier_a(t);
      u32x4 pop[2];
      if (active(t) && hot(t + 1)) {
        move_max();
        f32x16 n;
        phase_b(t, s, pop);
        qk(t + 1, n);
        pv_own(t, pop);
        // As in prefill_kernel's hot stage (+6.5% causal, +21% softcap and window).
        __builtin_amdgcn_iglp_opt(0);
        asm volatile("" : "+v"(n));   // or the compiler moves these MFMAs past the wait, away from phase B
        wait_partner(t);
        pv_partner(t);
        phase_a(unmasked, t + 1, n);
        __builtin_amdgcn_iglp_opt(0);
        s = n;
      } else {
        const bool act = active(t), next = t + 1 < n_tiles && active(t + 1);
        if (act) {
          move_max();
          phase_b(t, s, pop);
        }
        if (next) qk(t + 1, s);
        if (act) {
          pv_own(t, pop);
          wait_partner(t);
          pv_partner(t);
        }
        if (next) phase_a(masked, t + 1, s);
      }
    }
  }

  // The pair's row sums; O = O^T / l, LSE = m ln2 + ln(l).
  const float own = sum_hh(l_run);
  __syncthreads();
  *max_own = own;
  __syncthreads();
  const float lt = half == 0 ? own + *max_partner : *max_partner + own;
  if (row < r.q_len) {
    const float inv = lt > 0.0f ? vdsc / lt : 0.0f;
    const int64_t tq = (int64_t)r.q_begin + row;
    uint16_t* op = (uint16_t*)a.out + tq * a.out_stride[0] + (int64_t)h * a.out_stride[1] + 128 * half + 4 * hh;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint2 w;
        w.x = pack2<T>(o[db][4 * g] * inv, o[db][4 * g + 1] * inv);
        w.y = pack2<T>(o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv);
        *(uint2*)(op + 32 * db + 8 * g) = w;
      }
    if (hh == 0 && half == 0)
      a.lse[(int64_t)h * a.lse_stride[0] + tq * a.lse_stride[1]] = lt > 0.0f ? m_run * LN2 + logf(lt) : -INFINITY;
  }
}

// Defined in prefill_inst_pair.hip.
PrefillChoice pick_pair(bool bf16, bool causal, bool cap, bool win);

}  // namespace fa_prefill

#endif  // FA_PREFILL_PAIR_H
