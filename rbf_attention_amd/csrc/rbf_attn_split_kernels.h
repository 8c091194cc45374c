// Split kernels for problems with few 32-token blocks (16-bit elements, D <= 128).
//
// The streaming kernels give each 32-query (or key) block one wave.  With fewer
// blocks than the GPU has room for waves, the launch lasts as long as the
// longest causal chain: one wave alone on its SIMD takes ~1000 cycles per
// 32 x 32 block at D = 64 (LDS reads, dependent MFMAs, exponentials, MFMAs; 256
// of them MFMA cycles), with nothing to overlap them.  Here KSP waves share a
// block: of every tile of 32 * KSP streamed tokens each takes one 32-token
// block, and their partial accumulators are added through LDS at the end
// (split_sum).  The chain is KSP times shorter and the SIMDs hold more waves,
// whose latencies overlap.
//
// What a tile costs beside its blocks is kept to one barrier: tiles are staged
// by LDS-DMA in whole rows (SLayout, DmaRows) into two buffers, tile t + 1 in
// flight while tile t is computed, and the per-row terms (-0.5||k||^2, -L/c,
// -Delta) enter through one more MFMA per product instead of an LDS array that
// has to be formed and read back: the wave splits its row's term into three
// bf16 values that add up to it exactly (row_term) and multiplies them by
// ones.  (That costs ~25 VALU instructions per block, which a GPU full of waves
// does not have to spare: with KSP = 1 and two blocks per tile the B16 H8 N2052
// D64 forward took 116 us against the streaming kernel's 107.)
#pragma once

#include "rbf_attn_kernels.h"

namespace rbf {

// ---------------------------------------------------------------------------
// Swizzled row-major tile (16-bit elements).  Row r holds its DP/8 16-byte
// chunks without padding, chunk c at slot c ^ swz(r).  Whole rows are
// contiguous, so a DMA instruction (1 KB of LDS, 16 consecutive bytes per lane)
// fetches 512 / DP whole rows of global memory: streaming 64-row K and V tiles
// from L2 with nothing else in the loop (32 heads of 1024 rows, 768
// work-groups) ran at 25.7 TB/s, against 8.9 TB/s for 64-row gathers of one
// 16-byte chunk (64 cache lines per instruction).  The XOR spreads the kernels'
// reads over all 64 LDS banks:
//   * row reads (16 lanes, one chunk of 16 consecutive rows): rows that share
//     a 256-byte bank position modulo the XOR (all 16 at DP = 128, the 8 of one
//     parity at DP = 64, the 4 of one r % 4 at DP = 32) have distinct swz;
//   * transposing reads (32 lanes, chunks 4m .. 4m + 3 of rows 4i .. 4i + 3):
//     the four rows differ in address bits 6-7 (slot bits 2-3, or the row's low
//     bits where rows are shorter than 256 bytes).
// swz depends on the row's low four bits only, so a block of 32 rows is an
// additive offset.
// ---------------------------------------------------------------------------
template <int DP>
struct SLayout {
  static_assert(DP == 32 || DP == 64 || DP == 128, "swizzle written for 64-, 128- and 256-byte rows");
  __device__ static inline int swz(int r) {
    if constexpr (DP == 32) return (r >> 2) & 3;
    else if constexpr (DP == 64) return ((r & 2) << 1) | ((r >> 2) & 3);
    else return ((r & 3) << 2) | ((r >> 2) & 3);
  }
  // element offset of the 8-feature chunk that starts at col
  __device__ static inline int off(int row, int col) { return row * DP + (((col >> 3) ^ swz(row)) << 3); }

  // Transposing read: 8 tokens (in the P / dS contraction order tbase + 8(s/4)
  // + 4h + s%4) of feature fbase + n, as ld_tr8.
  template <typename T>
  __device__ static inline typename Elem<T>::frag tr(const T* tile, int tbase, int fbase, int lane) {
    static_assert(sizeof(T) == 2, "transposing LDS reads are for 16-bit elements");
    typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
    const int g = lane & 15;
    const int row = tbase + 4 * (lane >> 5) + (g >> 2);
    const int col = fbase + 16 * ((lane >> 4) & 1) + 4 * (g & 3);
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off(row, col) + (col & 7)));
    const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + off(row + 8, col) + (col & 7)));
    typedef short s16x8_t __attribute__((ext_vector_type(8)));
    const s16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(typename Elem<T>::frag, v);
  }
};

// The LDS-DMA of two (ROWS x DP) SLayout tiles -- tokens tok0 .. tok0 + ROWS - 1
// of slices A and B, each (N, D) with row stride sa / sb -- by W waves: 1 KB
// (512 / DP whole rows) per instruction, dealt round-robin to the waves.  A
// wave's lane offsets (relative to the tile's first row) are fixed, so a tile
// costs one add per instruction.  Tokens outside [0, N) and features >= D read
// zeros: lanes of such features start at offset 2^31, past every buffer range
// and, with a tile's row offset added, below 2^32 (the host keeps
// (N + ROWS) * stride * sizeof(T) within 2^31, split_rows_ok).
template <typename T, int ROWS, int DP, int W>
struct DmaRows {
  static_assert(sizeof(T) == 2 && ROWS % 16 == 0, "DMA tiles: 16-bit, whole swizzle periods");
  static constexpr int CPR = DP / 8, RPI = 64 / CPR, PER = ROWS / RPI, NIW = 2 * PER / W;
  static_assert(PER % W == 0, "every wave issues the same instructions of both tiles");
  i32x4_t ra, rb;
  uint32_t voff[NIW];  // lane byte offset of instruction j, tile row 0 at offset 0
  int rowa, rowb;      // row strides in bytes
  int wave;

  __device__ inline void init(const T* A, int64_t sa, const T* B, int64_t sb, int N, int D, int wave_, int lane) {
    wave = wave_;
    rowa = (int)(sa * (int64_t)sizeof(T));
    rowb = (int)(sb * (int64_t)sizeof(T));
    ra = buffer_rsrc(A, (uint32_t)N * (uint32_t)rowa);
    rb = buffer_rsrc(B, (uint32_t)N * (uint32_t)rowb);
#pragma unroll
    for (int j = 0; j < NIW; ++j) {
      const int r = (wave + j * W) % PER * RPI + lane / CPR;
      const int ch = (lane % CPR) ^ SLayout<DP>::swz(r);
      voff[j] = 8 * ch < D ? (uint32_t)(r * (j < NIW / 2 ? rowa : rowb) + 16 * ch) : 0x80000000u;
    }
  }

  __device__ inline void issue(int tok0, T* tA, T* tB) const {
    const uint32_t la = lds_addr(tA), lb = lds_addr(tB);
#pragma unroll
    for (int j = 0; j < NIW; ++j) {
      const uint32_t at = 1024u * (uint32_t)((wave + j * W) % PER);
      if (j < NIW / 2) dma16(voff[j] + (uint32_t)(tok0 * rowa), ra, la + at);
      else dma16(voff[j] + (uint32_t)(tok0 * rowb), rb, lb + at);
    }
  }
};

// s + x[row] for every element of the 32x32 accumulator s, where lane (n, h)
// gives the x of row n: x = x0 + x1 + x2 with bf16 x0, x1, x2 (24 significant
// bits cut into three of 8, each exact; infinities and NaN stay what they are),
// multiplied by ones as three contraction indices of one MFMA.
__device__ __forceinline__ f32x16_t row_term(float x, int h, f32x16_t s) {
  const bool fin = (__float_as_uint(x) & 0x7fffffffu) < 0x7f800000u;
  const uint32_t b0 = __float_as_uint(x) & 0xffff0000u;
  const float r0 = fin ? x - __uint_as_float(b0) : 0.f;
  const uint32_t b1 = __float_as_uint(r0) & 0xffff0000u;
  const float r1 = r0 - __uint_as_float(b1);
  u32x4_t a = {(b0 >> 16) | b1, __float_as_uint(r1) >> 16, 0u, 0u};
  if (h) a = u32x4_t{0u, 0u, 0u, 0u};
  const u32x4_t one = {0x3f803f80u, 0x00003f80u, 0u, 0u};
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, one), s, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// split_sum adds acc[0 .. NA) and x[0 .. NX) over the KSP consecutive waves
// that share a block; wave ki = 0 of them receives the sums (the others' values
// are then meaningless).  Pairwise in a fixed order: the upper half of the
// remaining waves stores, the lower half adds.  buf: LDS no longer in use (the
// function starts with a barrier), W / 2 slots of NA * 4 KB.  Every wave of the
// work-group calls it.
// ---------------------------------------------------------------------------
template <int W, int KSP, int NA, int NX>
__device__ __forceinline__ void split_sum(f32x16_t* acc, float* x, f32x4_t* buf, float (*sx)[NX][64], int wave, int lane) {
  static_assert(KSP == 2 || KSP == 4 || KSP == 8, "split over 2, 4 or 8 waves");
  const int q = wave / KSP, ki = wave % KSP;
#pragma unroll
  for (int half = KSP / 2; half >= 1; half /= 2) {
    lds_barrier();
    if (ki >= half && ki < 2 * half) {
      const int slot = q * half + (ki - half);
      f32x4_t* o = buf + slot * NA * 256 + lane;
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          o[(4 * a + g) * 64] = f32x4_t{acc[a][4 * g], acc[a][4 * g + 1], acc[a][4 * g + 2], acc[a][4 * g + 3]};
#pragma unroll
      for (int e = 0; e < NX; ++e) sx[slot][e][lane] = x[e];
    }
    lds_barrier();
    if (ki < half) {
      const int slot = q * half + ki;
      const f32x4_t* o = buf + slot * NA * 256 + lane;
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4_t v = o[(4 * a + g) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[a][4 * g + e] += v[e];
        }
#pragma unroll
      for (int e = 0; e < NX; ++e) x[e] += sx[slot][e][lane];
    }
  }
}

// Work-group -> (head, group rank), as decode_wg where B*H is a multiple of 8.
// Otherwise rank-major: the heaviest groups of all heads start first.
__device__ inline void split_wg(int ngrp, int hchunk, int& bh, int& rank) {
  const int BH = gridDim.x / ngrp;
  if ((BH & 7) == 0) {
    decode_wg(ngrp, hchunk, bh, rank);
  } else {
    rank = blockIdx.x / BH;
    bh = blockIdx.x - rank * BH;
  }
}

// The two-buffer pipeline: issue(t, b) requests tile t into buffer b = t mod 2,
// compute(t, b) runs it; the caller has requested tile 0.  One barrier per
// tile: after it tile t has landed for every wave and every wave has finished
// reading tile t - 1, whose buffer tile t + 1 then takes.
template <typename Issue, typename Compute>
__device__ __forceinline__ void split_pipeline(int nt, Issue&& issue, Compute&& compute) {
  for (int t = 0; t < nt; ++t) {
    wait_vmem();
    lds_barrier();
    if (t + 1 < nt) issue(t + 1, (t + 1) & 1);
    compute(t, t & 1);
  }
}

// ---------------------------------------------------------------------------
// Forward.  W / KSP query blocks per work-group; per 32-key block as
// rbf_fwd_group (static softmax bound with a rerun, online max for fp16).
// ---------------------------------------------------------------------------
template <typename T, int DP, int W, int KSP, bool SOFTMAX>
__global__ __launch_bounds__(64 * W) void rbf_fwd_split_kernel(const Params p) {
  typedef Elem<T> E;
  typedef typename E::frag frag;
  typedef SLayout<DP> L;
  constexpr int KS = DP / 16, ND = DP / 32, GB = W / KSP, ROWS = 32 * KSP;
  __shared__ __attribute__((aligned(1024))) T sT[2][2][ROWS * DP];
  __shared__ float sM[2][W][32];  // the waves' row maxima of a tile, by the tile's parity
  __shared__ float sX[W / 2][2][64];
  static_assert(W / 2 * ND * 4096 <= (int)sizeof(sT), "the partials fit the tiles");

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ki = wave % KSP;  // this wave's block of every tile
  const int N = p.N, D = p.D, org = p.org, nblk = p.nblk;
  const bool causal = p.causal != 0;
  const int npre = p.num_prefix;
  const float c = p.c;
  const int ngrp = (nblk + GB - 1) / GB;
  int bh, rank;
  split_wg(ngrp, p.hchunk, bh, rank);
  const int grp = causal ? ngrp - 1 - rank : rank;
  const int b = bh / p.H, hh = bh - b * p.H;
  const T* Q = reinterpret_cast<const T*>(p.q) + b * p.sq[0] + hh * p.sq[1];
  const T* K = reinterpret_cast<const T*>(p.k) + b * p.sk[0] + hh * p.sk[1];
  const T* V = reinterpret_cast<const T*>(p.v) + b * p.sv[0] + hh * p.sv[1];
  T* O = reinterpret_cast<T*>(const_cast<void*>(p.o)) + b * p.so[0] + hh * p.so[1];

  const int blk0 = nblk - (ngrp - grp) * GB;
  const int qblk = blk0 + wave / KSP;
  const bool wave_on = qblk >= 0;
  const int q0 = org + 32 * qblk, qtok = q0 + n;
  const bool qvalid = wave_on && qtok >= 0;
  const int jmax = last_key(qtok, N, causal, npre);
  const int hi = min(causal ? max(org + 32 * (blk0 + GB), npre) : N, N);  // keys any query of the group sees
  const int nkt = ((hi - 1 - org) >> 5) / KSP + 1;

  DmaRows<T, ROWS, DP, W> dma;
  dma.init(K, p.sk[2], V, p.sv[2], N, D, wave, lane);
  auto issue = [&](int kt, int buf) { dma.issue(org + kt * ROWS, sT[buf][0], sT[buf][1]); };
  issue(0, 0);

  frag qf[KS];
  float qn2 = 0.f;  // c * 0.5 ||q||^2
#pragma unroll
  for (int t = 0; t < KS; ++t)
    qf[t] = (qvalid && 16 * t + 8 * h < D) ? ld8<T>(Q + (int64_t)qtok * p.sq[2] + 16 * t + 8 * h) : zero_frag<T>();
#pragma unroll
  for (int t = 0; t < KS; ++t) qn2 += sumsq8<T>(qf[t]);
  qn2 = c * 0.5f * xhalf_sum(qn2);
  const frag ones = ones_frag<T>();

  constexpr bool STATIC = SOFTMAX && !std::is_same<T, _Float16>::value;
  f32x16_t oacc[ND];
  float x[2];  // sums of the rounded P (normalises O) and of the unrounded P (gives L)
  float m_run;
  auto run = [&](auto safe_tag) {
    constexpr bool SAFE = decltype(safe_tag)::value;
    // fp16, whose every pass is this one: one offset for the block's waves (bf16
    // comes here only in the rerun; sharing there too would cost its static pass
    // 2 %, B1 H16 N1333 D128 28.25 -> 28.93 us, by the compiler's register use)
    constexpr bool SHARED = SOFTMAX && SAFE && !STATIC;
#pragma unroll
    for (int d = 0; d < ND; ++d) oacc[d] = zero16();
    x[0] = x[1] = 0.f;
    m_run = !SOFTMAX ? qn2 : (SAFE ? -__builtin_inff() : qn2 - kBoundMargin);
    // SHARED: the offset after all blocks so far, the same in the block's KSP waves.
    // take() moves it over the first `upto` blocks of a tile, in key order and by the
    // streaming kernel's rule, by the maxima that the waves left in sM (a second time
    // over the same blocks changes nothing).
    float m_all = m_run;
    auto maxima = [&](int par, float (&me)[KSP]) {
#pragma unroll
      for (int e = 0; e < KSP; ++e) me[e] = sM[par][wave - ki + e][n];
    };
    auto take = [&](const float (&me)[KSP], int upto) {
#pragma unroll
      for (int e = 0; e < KSP; ++e)
        if (e < upto && __any(me[e] > m_all + kTau)) m_all = fmaxf(m_all, me[e]);
    };
    split_pipeline(nkt, issue, [&](int kt, int buf) {
      const int k0 = org + 32 * (kt * KSP + ki);
      const bool on = wave_on && k0 < N && blk_any(q0, k0, causal, npre);
      float me[KSP];
      if constexpr (SHARED) maxima((kt - 1) & 1, me);
      if (!SHARED && !on) return;
      const T* kt_ = sT[buf][0] + 32 * ki * DP;
      const T* vt_ = sT[buf][1] + 32 * ki * DP;
      frag kA[KS];
#pragma unroll
      for (int t = 0; t < KS; ++t) kA[t] = ld8<T>(kt_ + L::off(n, 16 * t + 8 * h));
      f32x16_t s = zero16();
      float kn = 0.f;
#pragma unroll
      for (int t = 0; t < KS; ++t) {
        s = E::mma(kA[t], qf[t], s);
        kn += sumsq8<T>(kA[t]);
      }
      kn = xhalf_sum(kn);
      s = row_term((k0 + n >= 0 && k0 + n < N) ? -0.5f * kn : -__builtin_inff(), h, s);
      frag vA[ND][2];
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int t = 0; t < 2; ++t) vA[d][t] = L::template tr<T>(vt_, 16 * t, 32 * d, lane);
      if (!blk_nomask(q0, k0, causal, npre)) mask_key_rows(s, k0, h, jmax);
      if constexpr (SOFTMAX && SAFE && !SHARED) {
        const float mt = xhalf_max(tree_max16(s)) * c;
        if (__any(mt > m_run + kTau)) {
          const float mnew = fmaxf(m_run, mt);
          const float alpha = (mnew == -__builtin_inff()) ? 1.f : fast_exp2(m_run - mnew);
#pragma unroll
          for (int d = 0; d < ND; ++d) oacc[d] *= alpha;
          x[0] *= alpha;
          x[1] *= alpha;
          m_run = mnew;
        }
      }
      if constexpr (SHARED) {
        // So that P is rounded to T at the same scale as in the streaming kernel, its
        // offset is that kernel's: of all blocks up to this one.  In the first tile,
        // where they all raise it, the waves wait for one another's maxima; later an
        // earlier block of the same tile that raises it (by more than kTau) is
        // seen one tile late.  Outputs of the two kernels at B4 H8 N1024 D64: 2.6e-4
        // apart (as much as fp16's own error) where a wave went by its own blocks
        // alone, 0.2e-4 this way.  Times (us; own blocks alone / this / a barrier in
        // every tile / the streaming kernel): B4 H8 N1024 D64 17.8 / 19.5 / 19.5 / 22.3,
        // B1 H4 N8000 D64 98 / 107 / 113 / 140, B1 H4 N4000 D128 56 / 60 / 64 / 125.
        const float mt = on ? xhalf_max(tree_max16(s)) * c : -__builtin_inff();
        if (h == 0) sM[kt & 1][wave][n] = mt;
        float mnew = m_run;
        bool moved = true;
        if (kt == 0) {
          lds_barrier();
          maxima(0, me);
          take(me, ki + 1);
          mnew = m_all;
        } else {
          float most = mt;
#pragma unroll
          for (int e = 0; e < KSP; ++e) most = fmaxf(most, me[e]);
          moved = __any(most > m_all + kTau);
          if (moved) {
            take(me, KSP);
            mnew = __any(mt > m_all + kTau) ? fmaxf(m_all, mt) : m_all;
          }
        }
        if (!on) return;
        if (moved) {
          const float alpha = (mnew == -__builtin_inff()) ? 1.f : fast_exp2(m_run - mnew);
#pragma unroll
          for (int d = 0; d < ND; ++d) oacc[d] *= alpha;
          x[0] *= alpha;
          x[1] *= alpha;
          m_run = mnew;
        }
      }
      const float moff = (SAFE && m_run == -__builtin_inff()) ? 0.f : m_run;
      frag pf[2];
      float pe[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        pe[i] = fast_exp2(fmaf(s[i], c, -moff));
        pf[i >> 3][i & 7] = (T)pe[i];
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int d = 0; d < ND; ++d) oacc[d] = E::mma(vA[d][t], pf[t], oacc[d]);
      if constexpr (SOFTMAX) {
        x[1] += tree_sum16(pe);
        x[0] += dot8<T>(pf[0], ones) + dot8<T>(pf[1], ones);
      }
    });
    if constexpr (SOFTMAX && SAFE) {
      // bring the wave's partials from its last offset to the block's
      if constexpr (SHARED) {
        lds_barrier();
        float me[KSP];
        maxima((nkt - 1) & 1, me);
        take(me, KSP);
      } else {
        if (h == 0) sM[0][wave][n] = m_run;
        __syncthreads();
        m_all = m_run;
#pragma unroll
        for (int e = 0; e < KSP; ++e) m_all = fmaxf(m_all, sM[0][wave - ki + e][n]);
      }
      const float w = (m_run == -__builtin_inff()) ? 0.f : fast_exp2(m_run - m_all);
#pragma unroll
      for (int d = 0; d < ND; ++d) oacc[d] *= w;
      x[0] *= w;
      x[1] *= w;
      m_run = m_all;
    }
    split_sum<W, KSP, ND, 2>(oacc, x, reinterpret_cast<f32x4_t*>(&sT[0][0][0]), sX, wave, lane);
  };

  if constexpr (SOFTMAX && !STATIC) run(std::true_type{});
  else run(std::false_type{});
  if constexpr (STATIC) {
    const float l = xhalf_sum(x[1]);
    const bool bad = qvalid && ki == 0 && !(l >= kSumLow && l <= kSumHigh);
    if (__syncthreads_or(bad)) {
      __syncthreads();
      issue(0, 0);
      run(std::true_type{});
    }
  }

  if (!wave_on || ki != 0) return;
  const float inv = SOFTMAX ? 1.f / xhalf_sum(x[0]) : 1.f;
  const float lsum = SOFTMAX ? xhalf_sum(x[1]) : 1.f;
  if (qtok < 0) return;
  T* orow = O + (int64_t)qtok * p.so[2];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * d + 8 * g + 4 * h;
      if (dd < D) {
        float v4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v4[e] = oacc[d][4 * g + e] * inv;
        st4f<T>(orow + dd, v4);
      }
    }
  if (SOFTMAX && h == 0) p.lse[(int64_t)bh * N + qtok] = m_run + __log2f(lsum);
}

// ---------------------------------------------------------------------------
// dQ (and Delta, or the non-softmax norm offsets), as rbf_bwd_dq_group.
// ---------------------------------------------------------------------------
template <typename T, int DP, int W, int KSP, bool SOFTMAX>
__global__ __launch_bounds__(64 * W) void rbf_bwd_dq_split_kernel(const Params p) {
  typedef Elem<T> E;
  typedef typename E::frag frag;
  typedef SLayout<DP> L;
  constexpr int KS = DP / 16, ND = DP / 32, GB = W / KSP, ROWS = 32 * KSP;
  __shared__ __attribute__((aligned(1024))) T sT[2][2][ROWS * DP];
  __shared__ float sX[W / 2][1][64];
  static_assert(W / 2 * ND * 4096 <= (int)sizeof(sT), "the partials fit the tiles");

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ki = wave % KSP;
  const int N = p.N, D = p.D, org = p.org, nblk = p.nblk;
  const bool causal = p.causal != 0;
  const int npre = p.num_prefix;
  const float c = p.c;
  const int ngrp = (nblk + GB - 1) / GB;
  int bh, rank;
  split_wg(ngrp, p.hchunk, bh, rank);
  const int grp = causal ? ngrp - 1 - rank : rank;
  const int b = bh / p.H, hh = bh - b * p.H;
  const T* Q = reinterpret_cast<const T*>(p.q) + b * p.sq[0] + hh * p.sq[1];
  const T* K = reinterpret_cast<const T*>(p.k) + b * p.sk[0] + hh * p.sk[1];
  const T* V = reinterpret_cast<const T*>(p.v) + b * p.sv[0] + hh * p.sv[1];
  const T* Og = reinterpret_cast<const T*>(p.o) + b * p.so[0] + hh * p.so[1];
  const T* dO = reinterpret_cast<const T*>(p.dout) + b * p.sdo[0] + hh * p.sdo[1];
  T* dQ = reinterpret_cast<T*>(p.dq) + b * p.sdq[0] + hh * p.sdq[1];

  const int blk0 = nblk - (ngrp - grp) * GB;
  const int qblk = blk0 + wave / KSP;
  const bool wave_on = qblk >= 0;
  const int q0 = org + 32 * qblk, qtok = q0 + n;
  const bool qvalid = wave_on && qtok >= 0;
  const int jmax = last_key(qtok, N, causal, npre);
  const int hi = min(causal ? max(org + 32 * (blk0 + GB), npre) : N, N);
  const int nkt = ((hi - 1 - org) >> 5) / KSP + 1;

  DmaRows<T, ROWS, DP, W> dma;
  dma.init(K, p.sk[2], V, p.sv[2], N, D, wave, lane);
  auto issue = [&](int kt, int buf) { dma.issue(org + kt * ROWS, sT[buf][0], sT[buf][1]); };
  issue(0, 0);

  frag qf[KS], df[KS];
#pragma unroll
  for (int t = 0; t < KS; ++t) {
    const bool ok = qvalid && 16 * t + 8 * h < D;
    qf[t] = ok ? ld8<T>(Q + (int64_t)qtok * p.sq[2] + 16 * t + 8 * h) : zero_frag<T>();
    df[t] = ok ? ld8<T>(dO + (int64_t)qtok * p.sdo[2] + 16 * t + 8 * h) : zero_frag<T>();
  }
  float off, dlt = 0.f;
  if constexpr (SOFTMAX) {
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      const bool ok = qvalid && 16 * t + 8 * h < D;
      const frag of = ok ? ld8<T>(Og + (int64_t)qtok * p.so[2] + 16 * t + 8 * h) : zero_frag<T>();
      s += dot8<T>(of, df[t]);
    }
    dlt = xhalf_sum(s);
    off = qvalid ? p.lse[(int64_t)bh * N + qtok] : 0.f;
    if (qvalid && h == 0 && ki == 0) p.delta[(int64_t)bh * N + qtok] = dlt;
  } else {
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < KS; ++t) s += sumsq8<T>(qf[t]);
    off = c * 0.5f * xhalf_sum(s);
    if (qvalid && h == 0 && ki == 0) p.lse[(int64_t)bh * N + qtok] = off;
  }

  f32x16_t dqacc[ND];
  float rsum = 0.f;
#pragma unroll
  for (int d = 0; d < ND; ++d) dqacc[d] = zero16();
  split_pipeline(nkt, issue, [&](int kt, int buf) {
    const int k0 = org + 32 * (kt * KSP + ki);
    if (!wave_on || k0 >= N || !blk_any(q0, k0, causal, npre)) return;
    const T* kt_ = sT[buf][0] + 32 * ki * DP;
    const T* vt_ = sT[buf][1] + 32 * ki * DP;
    f32x16_t s = zero16(), dp = SOFTMAX ? splat16(-dlt) : zero16();
    float kn = 0.f;
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      const frag kA = ld8<T>(kt_ + L::off(n, 16 * t + 8 * h));
      const frag vA = ld8<T>(vt_ + L::off(n, 16 * t + 8 * h));
      s = E::mma(kA, qf[t], s);
      dp = E::mma(vA, df[t], dp);
      kn += sumsq8<T>(kA);
    }
    kn = xhalf_sum(kn);
    s = row_term((k0 + n >= 0 && k0 + n < N) ? -0.5f * kn : -__builtin_inff(), h, s);
    if (!blk_nomask(q0, k0, causal, npre)) mask_key_rows(s, k0, h, jmax);
    float ds[16];
    frag sf[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      ds[i] = fast_exp2(fmaf(s[i], c, -off)) * dp[i];
      sf[i >> 3][i & 7] = (T)ds[i];
    }
    if constexpr (!SOFTMAX) rsum += tree_sum16(ds);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int d = 0; d < ND; ++d) dqacc[d] = E::mma(L::template tr<T>(kt_, 16 * t, 32 * d, lane), sf[t], dqacc[d]);
  });
  split_sum<W, KSP, ND, 1>(dqacc, &rsum, reinterpret_cast<f32x4_t*>(&sT[0][0][0]), sX, wave, lane);

  if (!wave_on || ki != 0) return;
  const float g2 = 2.f * p.gamma;
  float rs = 0.f;
  if constexpr (!SOFTMAX) rs = xhalf_sum(rsum);
  if (qtok < 0) return;
  T* drow = dQ + (int64_t)qtok * p.sdq[2];
  const T* qrow = Q + (int64_t)qtok * p.sq[2];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * d + 8 * g + 4 * h;
      if (dd < D) {
        float v4[4];
        if constexpr (SOFTMAX) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v4[e] = g2 * dqacc[d][4 * g + e];
        } else {
          float q4[4];
          ld4f<T>(qrow + dd, q4);
#pragma unroll
          for (int e = 0; e < 4; ++e) v4[e] = g2 * (dqacc[d][4 * g + e] - rs * q4[e]);
        }
        st4f<T>(drow + dd, v4);
      }
    }
}

// ---------------------------------------------------------------------------
// dK and dV, as rbf_bwd_dkdv_group: W / KSP key blocks per work-group, tiles of
// 32 * KSP queries (Q, dO and the raw L, Delta rows).
// ---------------------------------------------------------------------------
template <typename T, int DP, int W, int KSP, bool SOFTMAX>
__global__ __launch_bounds__(64 * W) void rbf_bwd_dkdv_split_kernel(const Params p) {
  typedef Elem<T> E;
  typedef typename E::frag frag;
  typedef SLayout<DP> L;
  constexpr int KS = DP / 16, ND = DP / 32, GB = W / KSP, ROWS = 32 * KSP;
  __shared__ __attribute__((aligned(1024))) T sT[2][2][ROWS * DP];
  __shared__ __attribute__((aligned(16))) float sRaw[2][2][ROWS];  // L, Delta as loaded
  __shared__ float sX[W / 2][1][64];
  static_assert(W / 2 * 2 * ND * 4096 <= (int)sizeof(sT), "the partials fit the tiles");
  static_assert(ROWS % 64 == 0, "L and Delta by 64-lane DMA");

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ki = wave % KSP;  // this wave's query block of every tile
  const int N = p.N, D = p.D, org = p.org, nblk = p.nblk;
  const bool causal = p.causal != 0;
  const int npre = p.num_prefix;
  const float c = p.c;
  const float inv_c = 1.f / c;
  const int ngrp = (nblk + GB - 1) / GB;
  int bh, grp;
  split_wg(ngrp, p.hchunk, bh, grp);
  const int b = bh / p.H, hh = bh - b * p.H;
  const T* Q = reinterpret_cast<const T*>(p.q) + b * p.sq[0] + hh * p.sq[1];
  const T* K = reinterpret_cast<const T*>(p.k) + b * p.sk[0] + hh * p.sk[1];
  const T* V = reinterpret_cast<const T*>(p.v) + b * p.sv[0] + hh * p.sv[1];
  const T* dO = reinterpret_cast<const T*>(p.dout) + b * p.sdo[0] + hh * p.sdo[1];
  T* dK = reinterpret_cast<T*>(p.dk) + b * p.sdk[0] + hh * p.sdk[1];
  T* dV = reinterpret_cast<T*>(p.dv) + b * p.sdv[0] + hh * p.sdv[1];
  const float* offg = p.lse + (int64_t)bh * N;
  const float* delg = SOFTMAX ? p.delta + (int64_t)bh * N : offg;

  const int blk0 = grp * GB;
  const int kblk = blk0 + wave / KSP;
  const bool wave_on = kblk < nblk;
  const int k0 = org + 32 * kblk, ktok = k0 + n;
  const bool kvalid = wave_on && ktok >= 0;
  const int ilo = first_query(ktok, causal, npre);
  const int wg_kfirst = max(org + 32 * blk0, 0);
  const int qlo = causal ? (wg_kfirst < npre ? 0 : wg_kfirst) : 0;
  const int qb0 = (qlo - org) >> 5;  // the tiles start at this query block
  const int nqt = (nblk - qb0 + KSP - 1) / KSP;

  DmaRows<T, ROWS, DP, W> dma;
  dma.init(Q, p.sq[2], dO, p.sdo[2], N, D, wave, lane);
  const i32x4_t roff = buffer_rsrc(offg, 4u * (uint32_t)N), rdel = buffer_rsrc(delg, 4u * (uint32_t)N);
  auto issue = [&](int t, int buf) {
    const int tok0 = org + 32 * (qb0 + t * KSP);
    dma.issue(tok0, sT[buf][0], sT[buf][1]);
    if (wave < ROWS / 64) {
      const uint32_t vo = 4u * (uint32_t)(tok0 + 64 * wave + lane);  // negative tokens: out of range
      dma4(vo, roff, lds_addr(&sRaw[buf][0][64 * wave]));
      if constexpr (SOFTMAX) dma4(vo, rdel, lds_addr(&sRaw[buf][1][64 * wave]));
    }
  };
  issue(0, 0);

  frag kf[KS], vf[KS];
  float nckn = 0.f;  // -c * 0.5||k||^2
#pragma unroll
  for (int t = 0; t < KS; ++t) {
    const bool ok = kvalid && 16 * t + 8 * h < D;
    kf[t] = ok ? ld8<T>(K + (int64_t)ktok * p.sk[2] + 16 * t + 8 * h) : zero_frag<T>();
    vf[t] = ok ? ld8<T>(V + (int64_t)ktok * p.sv[2] + 16 * t + 8 * h) : zero_frag<T>();
  }
#pragma unroll
  for (int t = 0; t < KS; ++t) nckn += sumsq8<T>(kf[t]);
  nckn = -c * 0.5f * xhalf_sum(nckn);

  f32x16_t acc[2 * ND];  // dK^T, then dV^T
  float csum = 0.f;
#pragma unroll
  for (int d = 0; d < 2 * ND; ++d) acc[d] = zero16();
  split_pipeline(nqt, issue, [&](int t0, int buf) {
    const int qb = qb0 + t0 * KSP + ki, q0 = org + 32 * qb;
    if (!wave_on || qb >= nblk || !blk_any(q0, k0, causal, npre)) return;
    const T* qt_ = sT[buf][0] + 32 * ki * DP;
    const T* dt_ = sT[buf][1] + 32 * ki * DP;
    const bool ok = q0 + n >= 0;  // padding queries: P = 0
    const float lo = sRaw[buf][0][32 * ki + n], dl = SOFTMAX ? sRaw[buf][1][32 * ki + n] : 0.f;
    f32x16_t s = row_term(ok ? -lo * inv_c : -__builtin_inff(), h, zero16());
    f32x16_t dp = SOFTMAX ? row_term(ok ? -dl : 0.f, h, zero16()) : zero16();
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      s = E::mma(ld8<T>(qt_ + L::off(n, 16 * t + 8 * h)), kf[t], s);
      dp = E::mma(ld8<T>(dt_ + L::off(n, 16 * t + 8 * h)), vf[t], dp);
    }
    if (!blk_nomask(q0, k0, causal, npre)) mask_query_rows(s, q0, h, ilo);
    frag pf[2], sf[2];
    float ds[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float pv = fast_exp2(fmaf(s[i], c, nckn));
      ds[i] = pv * dp[i];
      pf[i >> 3][i & 7] = (T)pv;
      sf[i >> 3][i & 7] = (T)ds[i];
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        acc[ND + d] = E::mma(L::template tr<T>(dt_, 16 * t, 32 * d, lane), pf[t], acc[ND + d]);
        acc[d] = E::mma(L::template tr<T>(qt_, 16 * t, 32 * d, lane), sf[t], acc[d]);
      }
    csum += tree_sum16(ds);
  });
  split_sum<W, KSP, 2 * ND, 1>(acc, &csum, reinterpret_cast<f32x4_t*>(&sT[0][0][0]), sX, wave, lane);

  if (!wave_on || ki != 0) return;
  const float g2 = 2.f * p.gamma;
  const float cs = xhalf_sum(csum);
  if (ktok < 0) return;
  T* dkrow = dK + (int64_t)ktok * p.sdk[2];
  T* dvrow = dV + (int64_t)ktok * p.sdv[2];
  const T* krow = K + (int64_t)ktok * p.sk[2];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * d + 8 * g + 4 * h;
      if (dd < D) {
        float k4[4], a4[4], b4[4];
        ld4f<T>(krow + dd, k4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a4[e] = g2 * (acc[d][4 * g + e] - cs * k4[e]);
          b4[e] = acc[ND + d][4 * g + e];
        }
        st4f<T>(dkrow + dd, a4);
        st4f<T>(dvrow + dd, b4);
      }
    }
}

}  // namespace rbf
