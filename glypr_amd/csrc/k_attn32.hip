// k_attn32.hip — flash attention on the full-rate f16 MFMA
// (v_mfma_f32_32x32x16_f16; the 16x16x32 form of attn_partial_kernel issues at
// half the rate), for the longer sequences and batches (attn_plan.cpp).
//
// A wave owns 32 queries of one q head and all HD dims of their O^T, one wave
// per SIMD (HD 512: Q 128 + O^T 256 + two S^T tiles 32 registers of the 512);
// four waves share every 32-key K / V^T tile, which LDS DMA streams into two
// slots.  Transposed products as in attn_partial_kernel: S^T = K Q^T and
// O^T = V^T P^T, so a lane's S^T column is its query's and P^T goes from the
// accumulator into the PV product's B operand.  The S^T products of tile kb+1
// issue over the exponentials of tile kb, fragments four MFMAs ahead of use;
// one barrier per tile.
//
// What bounds it: the one wave of each SIMD.  At T = 8192, 4 heads on one kv head
// of 512, the MFMAs take 47 % of the SIMD cycles (64 of 32 clocks per tile and wave,
// at the 1.8 GHz the card holds under them), 23 % of the wave's time are waits at the
// tile's barrier and for fragments, 13 % VALU, and nothing else runs on the
// SIMD meanwhile.  LDS is not it: the fragment reads are 23 % of its cycles (a
// conflict-free ds_read_b128 takes 4 clocks, 256 B/clock per CU) without one bank
// conflict.  Same shape: 1350 + 59 us (16-query blocks, 4 partitions, combine) ->
// 553 us in one launch, 0.99 PFLOP/s of the card's 1.36 for a large f16 product; the
// whole call 1472 -> 594 us.  T = 1777, window 512, 2 x 2 heads of 256: 49.9 -> 37.3 us
// (the tile kernel 22.8, the prologue and combine launches 8.3 and 7.1).
#include "attn_common.hpp"
#include "device_common.hpp"
#include "internal.hpp"

namespace glypr {

namespace {
typedef _Float16 f16;
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int A32_K = ATTN_AK;   // keys per tile

// Rows of an S^T tile are dealt to keys with bits 2 and 3 of the row swapped:
// lane half h then holds keys 16 u + 8 h .. + 7 in accumulator registers
// 8 u .. 8 u + 7, the k-slots of the PV product's B operand.
__device__ __forceinline__ int key_of_row(int r) {
  return (r & 19) | ((r & 4) << 1) | ((r & 8) >> 1);
}

// O^T accumulators stay in AGPRs (HD 512: all 256 of a lane, while the other 256
// registers hold Q and the tile in work), which only an asm operand pins; s_nop 1 covers a vector ALU write of an operand right in
// front, and acc_settle the reads of o behind the last product.
__device__ __forceinline__ void pv_mfma(v16f& o, const v8h& a, const v8h& b) {
  asm("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(o) : "v"(a), "v"(b));
}
template <int NT>
__device__ __forceinline__ void acc_settle(v16f (&o)[NT]) {
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int t = 0; t < NT; t++) asm volatile("" : "+a"(o[t]));
}

template <int HD, int NWV, bool DIRECT>
__global__ void __launch_bounds__(NWV * 64)
    __attribute__((amdgpu_waves_per_eu(1, 1)))
attn_tile32_kernel(const f16* __restrict__ q16, const f16* __restrict__ kk,
                   const f16* __restrict__ vt, float* __restrict__ part_o,
                   float* __restrict__ part_ml, int T, int Tp, int nq, int nkv, int window,
                   int kb_per_part, int kparts, const int2* __restrict__ seg,
                   float* __restrict__ ctx, int8_t* __restrict__ cq, float* __restrict__ dc,
                   uint16_t* __restrict__ cb) {
  static_assert(HD == 256 || HD == 512, "head dims 256 and 512");
  constexpr int NS = HD / 16;            // S^T steps (16 dims each)
  constexpr int NT = HD / 32;            // O^T tiles (32 dims each)
  constexpr int TILE_H = A32_K * HD;     // halves per K (or V^T) tile
  constexpr int KU = HD / 16;            // 1 KB DMA units per K tile (= per V^T tile)
  constexpr int KLPR = HD / 8;           // 16-byte chunks per K row
  constexpr int KRPU = 64 / KLPR;        // K rows per unit
  __shared__ __attribute__((aligned(16))) f16 Ks[2][TILE_H];
  __shared__ __attribute__((aligned(16))) f16 Vs[2][TILE_H];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, lh = lane >> 5;
  // Column groups: 32 queries of one q head, head-minor; a workgroup takes NWV
  // consecutive ones of a kv group (wave w the w-th), so that its four waves
  // fill the CU's SIMDs whatever the number of q heads per kv head.
  const int G = nq / nkv;
  const int ngrp = (Tp >> 5) * G;
  const int nblk = (ngrp + NWV - 1) / NWV;
  const int items = nkv * kparts * nblk;
  const int n8 = (items + 7) / 8;
  const int W = (int)(blockIdx.x % 8) * n8 + (int)(blockIdx.x / 8);
  if (W >= items) return;   // grid padding (whole block)
  const int g = W / (kparts * nblk);
  const int kp = (W / nblk) % kparts;
  const int c0 = (W % nblk) * NWV;
  const int c1 = c0 + NWV < ngrp ? c0 + NWV : ngrp;     // past the last group
  const int cw = c0 + w < c1 ? c0 + w : c1 - 1;         // spare waves repeat it
  const int q0 = 32 * (c0 / G), q1 = 32 * ((c1 - 1) / G) + 32;   // the block's queries
  const int h = g * G + cw % G;
  const int qi = 32 * (cw / G) + l31;    // this lane's query
  // keys of this block's sequence (with a segment table a block's rows stay
  // within one sequence), then its key tiles
  int kstart = 0, kend = T;
  if (seg) {
    const int2 sg = seg[q0];
    kstart = sg.x;
    kend = sg.x + sg.y;
  }
  const bool banded = window > 0 && kend - kstart > window;
  int kb_lo = kstart / A32_K, kb_hi = (kend + A32_K - 1) / A32_K;
  if (banded) {
    const int lo_key = q0 - window, hi_key = q1 - 1 + window;
    kb_lo = (lo_key > kstart ? lo_key : kstart) / A32_K;
    kb_hi = (hi_key < kend - 1 ? hi_key : kend - 1) / A32_K + 1;
  }
  const int kb0 = kb_lo + kp * kb_per_part;
  const int kb1 = kb0 + kb_per_part < kb_hi ? kb0 + kb_per_part : kb_hi;
  const int qw = qi - l31;               // the wave's first query

  const f16* kbase = kk + (int64_t)g * Tp * HD;
  const f16* vbase = vt + (int64_t)g * HD * Tp;
  // DMA lane offsets: K unit u = rows KRPU u .. (chunk c of row r at LDS chunk
  // c ^ (key_of_row(r) & 15)); V^T unit u = dim rows 16 u .. 16 u + 15 (chunk
  // c of row r at c ^ ((r >> 2) & 3)).  LDS serves a ds_read_b128 in groups of
  // 16 lanes (0-3, 12-15, 20-27 and the other 16, then the upper half alike)
  // over 64 banks: both swizzles give a group's rows distinct banks (for these 32-row
  // fragments; (r >> 1) & 3, right for the 16-row ones, halves the V^T rate).
  const int krow = lane / KLPR;
  const int kl = krow * HD * 2 + (((lane % KLPR) ^ krow) << 4);
  const int vl = (lane >> 2) * Tp * 2 + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  auto issue_k = [&](int kb, int sl) {
    const int8_t* base = reinterpret_cast<const int8_t*>(kbase + (int64_t)kb * TILE_H);
    int kl_ = kl;   // opaque with two waves: sixteen offsets held across the loop would spill
    if constexpr (NWV == 2) asm volatile("" : "+v"(kl_));
#pragma unroll
    for (int j = 0; j < (KU + NWV - 1) / NWV; j++) {
      const int u = w + NWV * j;
      if (KU % NWV == 0 || u < KU)
        dma16(base + u * 1024, kl_ ^ ((key_of_row(u * KRPU) & 15) << 4),
              lds_u32(&Ks[sl][u * 512]));
    }
  };
  auto issue_v = [&](int kb, int sl) {
    const int8_t* base = reinterpret_cast<const int8_t*>(vbase + (int64_t)kb * A32_K);
#pragma unroll
    for (int j = 0; j < (KU + NWV - 1) / NWV; j++) {
      const int u = w + NWV * j;
      if (KU % NWV == 0 || u < KU)
        dma16(base + (int64_t)u * 32 * Tp, vl, lds_u32(&Vs[sl][u * 512]));
    }
  };

  if (kb0 < kb1) {
    issue_k(kb0, 0);
    issue_v(kb0, 0);
  }
  // Q fragments (B operand of S^T): query qi, dims 16 s + 8 lh .. + 7
  v8h qf[NS];
  {
    const f16* qp = q16 + ((int64_t)h * Tp + qi) * HD + 8 * lh;
#pragma unroll
    for (int s = 0; s < NS; s++) qf[s] = *reinterpret_cast<const v8h*>(qp + 16 * s);
  }
  const int kfo = key_of_row(l31) * HD;
  const int kx = l31 & 15;
  const int vfo = l31 * A32_K;
  const int vx = (l31 >> 2) & 3;

  // l_run + l_lo: the sum of the tiles' sums with the additions' rounding errors
  // kept apart, so a partition of any length is as exact as one of few tiles
  float m_run = -INFINITY, l_run = 0.0f, l_lo = 0.0f, thr = -INFINITY, m_use = 0.0f;
  v16f o[NT];
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[t][r] = 0.0f;

  auto scores = [&](int sl, v16f& s) {
    const f16* Kt = Ks[sl] + kfo;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll
    for (int i = 0; i < NS; i++) {
      const v8h kf = *reinterpret_cast<const v8h*>(Kt + (((2 * i + lh) ^ kx) << 3));
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[i], s, 0, 0, 0);
    }
  };

  v16f sc;
  if (kb0 < kb1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kb0 + 1 < kb1) issue_k(kb0 + 1, 1);
    scores(0, sc);
  }
  for (int kb = kb0, sl = 0; kb < kb1; kb++, sl ^= 1) {
    // mask the scores of tile kb (only where a key can be out of range or band)
    const int k0 = kb * A32_K;
    const bool edge = k0 + A32_K > kend ||
                      (banded && (k0 < qw + 31 - window || k0 + A32_K - 1 > qw + window));
    if (edge) {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int key = k0 + 16 * (r >> 3) + 8 * lh + (r & 7);
        const bool out = (key >= kend) | (banded & (abs(qi - key) > window));
        sc[r] = out ? -INFINITY : sc[r];
      }
    }
    float mloc = sc[0];
#pragma unroll
    for (int r = 1; r < 16; r++) mloc = fmaxf(mloc, sc[r]);
    if (__any(mloc > thr)) {
      const float mx = pair_max32(mloc);
      const float m_new = mx > thr ? mx : m_run;
      m_use = m_new == -INFINITY ? 0.0f : m_new;
      if (__any(m_run != -INFINITY)) {   // O and l are still zero otherwise
        const float alpha = __expf(m_run - m_use);
        l_run *= alpha;
        l_lo *= alpha;
        acc_settle(o);
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
          for (int r = 0; r < 16; r++) o[t][r] *= alpha;
          asm volatile("" : "+a"(o[t]));
        }
      }
      m_run = m_new;
      thr = m_new + ATTN_TAU;
    }
    // K of tile kb+1 and V^T of tile kb have landed, for every wave
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kb + 1 < kb1) issue_v(kb + 1, sl ^ 1);
    if (kb + 2 < kb1) issue_k(kb + 2, sl);
    v16f sn;
#pragma unroll
    for (int r = 0; r < 16; r++) sn[r] = 0.0f;
    v8h pf[2];
    const f16* Kt = Ks[sl ^ 1] + kfo;
    const f16* Vt = Vs[sl] + vfo;
    auto kfrag = [&](int i) {
      return *reinterpret_cast<const v8h*>(Kt + (((2 * i + lh) ^ kx) << 3));
    };
    auto vfrag = [&](int i) {   // tile i / 2, keys 16 (i % 2) + 8 lh ..
      return *reinterpret_cast<const v8h*>(Vt + (i >> 1) * 32 * A32_K +
                                           (((2 * (i & 1) + lh) ^ vx) << 3));
    };
    // S^T of tile kb+1 (past the last tile: stale LDS, unused) over the
    // exponentials of tile kb, then O^T += V^T P^T; fragments one chunk ahead
    constexpr int CH = 4;
    v8h fr[2][CH];
    float ps[2] = {0.0f, 0.0f};
#pragma unroll
    for (int e = 0; e < CH; e++) fr[0][e] = kfrag(e);
#pragma unroll
    for (int c = 0; c < NS / CH; c++) {
#pragma unroll
      for (int e = 0; e < CH; e++)
        fr[(c + 1) & 1][e] = c + 1 < NS / CH ? kfrag((c + 1) * CH + e) : vfrag(e);
#pragma unroll
      for (int e = 0; e < CH; e++)
        sn = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[c & 1][e], qf[c * CH + e], sn, 0, 0, 0);
      constexpr int EPC = 16 * CH / NS;   // exponentials per chunk
#pragma unroll
      for (int e = 0; e < EPC; e++) {
        const int r = c * EPC + e;
        // (the difference first: a product m * log2(e) rounded on its own would
        // shift partitions and rescales against each other by |m| 2^-24; one
        // instruction more each, T = 8192 at head_dim 512: 588 -> 593 us)
        const float pv = __expf(sc[r] - m_use);
        ps[r >> 3] += pv;
        pf[r >> 3][r & 7] = (f16)pv;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    {
      const float pt = ps[0] + ps[1], l_new = l_run + pt;
      l_lo += pt - (l_new - l_run);
      l_run = l_new;
    }
    constexpr int PB = (NS / CH) & 1;     // the buffer the first V^T chunk is in
#pragma unroll
    for (int c = 0; c < 2 * NT / CH; c++) {
      if (c + 1 < 2 * NT / CH)
#pragma unroll
        for (int e = 0; e < CH; e++) fr[(c + 1 + PB) & 1][e] = vfrag((c + 1) * CH + e);
#pragma unroll
      for (int e = 0; e < CH; e++) {
        const int i = c * CH + e;
        pv_mfma(o[i >> 1], fr[(c + PB) & 1][e], pf[i & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    sc = sn;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  l_run = pair_sum32(l_run + l_lo);
  acc_settle(o);

  if (c0 + w >= c1) return;   // a spare wave (no barrier follows)
  // O^T tile t, register r: dim 32 t + 8 (r >> 2) + 4 lh + (r & 3) of query qi
  if constexpr (DIRECT) {
    const float inv = 1.0f / l_run;
    const bool live = qi < T;
    const int width = nq * HD;
    const int64_t rowoff = (int64_t)qi * width + (int64_t)h * HD;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      asm volatile("" : "+a"(o[t]));
      float y[16];
#pragma unroll
      for (int r = 0; r < 16; r++) y[r] = o[t][r] * inv;
      if (ctx && live)
#pragma unroll
        for (int c = 0; c < 4; c++)
          *reinterpret_cast<v4f*>(ctx + rowoff + 32 * t + 8 * c + 4 * lh) =
              v4f{y[4 * c], y[4 * c + 1], y[4 * c + 2], y[4 * c + 3]};
      if (cb && live)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          uint32_t* dst = reinterpret_cast<uint32_t*>(cb + rowoff + 32 * t + 8 * c + 4 * lh);
#pragma unroll
          for (int e = 0; e < 2; e++)
            dst[e] = (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)y[4 * c + 2 * e]) |
                     ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)y[4 * c + 2 * e + 1]) << 16);
        }
      if (cq) {
        float a = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) a = fmaxf(a, fabsf(y[r]));
        const QScale qsc = q8_scale(pair_max32(a));
        if (live) {
#pragma unroll
          for (int c = 0; c < 4; c++) {
            uint32_t packed = 0;
#pragma unroll
            for (int e = 0; e < 4; e++)
              packed |= ((uint32_t)(quant_round(y[4 * c + e] * qsc.id) & 0xFF)) << (8 * e);
            *reinterpret_cast<uint32_t*>(cq + rowoff + 32 * t + 8 * c + 4 * lh) = packed;
          }
          if (lh == 0) dc[(int64_t)qi * (width / QK) + (h * HD) / QK + t] = qsc.dq;
        }
      }
    }
  } else {
  const int64_t prow = (int64_t)kp * Tp + qi;
  float* po = part_o + prow * nq * HD + (int64_t)h * HD;
#pragma unroll
  for (int t = 0; t < NT; t++) {
    asm volatile("" : "+a"(o[t]));
#pragma unroll
    for (int c = 0; c < 4; c++)
      *reinterpret_cast<v4f*>(po + 32 * t + 8 * c + 4 * lh) =
          v4f{o[t][4 * c], o[t][4 * c + 1], o[t][4 * c + 2], o[t][4 * c + 3]};
  }
  if (lh == 0) {
    part_ml[(prow * nq + h) * 2] = m_run;
    part_ml[(prow * nq + h) * 2 + 1] = l_run;
  }
  }
}

template <int HD, int NWV>
void run_tile32(const f16* q, const f16* k, const f16* v, float* part_o, float* part_ml,
                int64_t T, int64_t Tp, int64_t nq, int64_t nkv, int64_t window,
                const AttnPlan& p, const int2* seg, float* ctx, int8_t* cq, float* dc,
                uint16_t* cb, hipStream_t s) {
  const int64_t items = nkv * p.kparts * (((Tp >> 5) * (nq / nkv) + NWV - 1) / NWV);
  const unsigned grid = (unsigned)((items + 7) / 8 * 8);
  if (p.kparts == 1)
    attn_tile32_kernel<HD, NWV, true><<<grid, NWV * 64, 0, s>>>(
        q, k, v, part_o, part_ml, (int)T, (int)Tp, (int)nq, (int)nkv, (int)window, p.per, 1, seg,
        ctx, cq, dc, cb);
  else
    attn_tile32_kernel<HD, NWV, false><<<grid, NWV * 64, 0, s>>>(
        q, k, v, part_o, part_ml, (int)T, (int)Tp, (int)nq, (int)nkv, (int)window, p.per,
        p.kparts, seg, ctx, cq, dc, cb);
}
}  // namespace

hipError_t launch_attn_tile32(const uint16_t* q16, const uint16_t* k16, const uint16_t* vt16,
                              float* part_o, float* part_ml, int64_t T, int64_t Tp, int64_t nq,
                              int64_t nkv, int64_t hd, int64_t window, const AttnPlan& plan,
                              const int32_t* seg, float* ctx, int8_t* cq, float* dc, uint16_t* cb,
                              hipStream_t s) {
  const f16* q = reinterpret_cast<const f16*>(q16);
  const f16* k = reinterpret_cast<const f16*>(k16);
  const f16* v = reinterpret_cast<const f16*>(vt16);
  const int2* sg = reinterpret_cast<const int2*>(seg);
#define A32_CASE(H, N)                                                                         \
  if (hd == H && plan.waves == N) {                                                            \
    run_tile32<H, N>(q, k, v, part_o, part_ml, T, Tp, nq, nkv, window, plan, sg, ctx, cq, dc,  \
                     cb, s);                                                                   \
    return hipGetLastError();                                                                  \
  }
  A32_CASE(512, 2)
  A32_CASE(512, 3)
  A32_CASE(512, 4)
  A32_CASE(256, 2)
  A32_CASE(256, 3)
  A32_CASE(256, 4)
#undef A32_CASE
  return hipErrorInvalidValue;
}

}  // namespace glypr
