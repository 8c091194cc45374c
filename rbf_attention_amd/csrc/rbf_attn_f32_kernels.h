// fp32 kernels for up to 128 features, on the bf16 matrix instructions.
//
// gfx950's fp32 MFMA (v_mfma_f32_32x32x2f32) runs at a sixteenth of the bf16
// rate, and the fp32 kernels built on it spent 4096 of their cycles per 32 x 32
// block (D = 64, forward) in it.  Here every fp32 operand is cut into three
// bf16 values that add up to it exactly (high and middle by rounding, low what
// is left: 24 significant bits), and a product is the six bf16 products of parts
// whose magnitudes reach the result's last bits (high x high, high x middle,
// middle x high, middle x middle, high x low, low x high), accumulated in fp32,
// smallest first: 2.7x the fp32 MFMA's rate.  (Splitting a product over parts of
// lower precision is Dekker's method; with three bf16 parts it is known as the
// bf16x3 emulation of fp32.)  What is dropped is at most 2^-24 of the product
// (2^-26 in the mean), as much as rounding one fp32 product: |x - high| <= 2^-8
// and |low| <= 2^-17 for 1 <= |x| < 2, so middle x low twice is <= 2^-24.  Each
// bf16 product is exact and one instruction sums sixteen of them, so the result's
// error is that of fp32 accumulation.
//
// The parts are exact as long as the lowest is a normal bf16 number.  So what may be
// small is multiplied by 2^24 (kLift) before it is cut: the operands in which a
// result is linear, P (but the softmax forward's, whose row sums are kept above 2^-60)
// and dS (by way of dP).  That puts all of fp32's normal range above 2^-102, and the
// power of two comes out of the result again.  Results that are not finite -- an
// infinite or NaN input, whose parts make NaN of everything, or magnitudes (2^40 and
// more) that the factor took past fp32's range -- are computed again in plain fp32 by
// the work-group that finds them (the EXACT pass below), which is slow, and rare.
//
// Work-groups of W waves, KSP of them per 32-token block (as the split
// kernels): tiles of 32 * KSP streamed tokens are loaded into registers one
// tile ahead, cut, and stored as three bf16 planes of swizzled rows (SLayout)
// per operand; transposed operands come from the same planes by the transposing
// LDS read, so no transposed copy is stored.
//
// Against the fp32-MFMA kernels (us fwd / dQ / dK/dV on one card, causal softmax;
// relative 2-norm error against 64 bits of O, dQ, dK, dV in units of 1e-6):
//   B2 H4 N132 D64     19 / 25 / 30 -> 13 / 16 / 15       0.67 1.70 1.75 1.67 -> 0.66 1.75 1.72 1.65
//   B1 H4 N4000 D64    362 / 460 / 601 -> 124 / 146 / 177  0.83 1.66 2.25 2.36 -> 0.75 1.62 1.82 1.87
//   B4 H8 N1001 D64, every key visible
//                      99 / 127 / 163 -> 55 / 74 / 121     0.94 1.64 1.98 1.97 -> 0.82 1.56 1.83 1.82
//   B8 H16 N2000 D64   645 / 883 / 1327 -> 374 / 513 / 698 0.71 1.69 2.02 1.99 -> 0.70 1.55 1.80 1.92
//   B4 H8 N1500 D128   245 / 330 / 442 -> 164 / 206 / 273  0.82 1.63 1.92 1.96 -> 0.79 1.58 1.78 1.77
//   B8 H16 N1500 D32   206 / 288 / 360 -> 149 / 184 / 253  0.75 1.68 1.92 1.95 -> 0.75 1.64 1.83 1.81
// The B8 H16 N2000 D64 forward issues 393 GFLOP of bf16 MFMA in 374 us, 1.05
// PFLOP/s: bound by the matrix units (a large bf16 matrix product runs at 1.18
// on the same kind of card).  Rounding the high part, the lifts and the finite
// check cost, over 14 shapes of 16 to 128 features, 2.2 / 3.3 / 6.5 % at the median
// (fwd / dQ / dK/dV) and 9 / 8 / 14 % at most: B4 H8 N1000 D32 29.3 -> 32.0 and 37.9
// -> 43.0 (fwd, dK/dV), B1 H8 N300 D32 11.8 -> 12.7 (dQ).
#pragma once

#include "rbf_attn_kernels.h"
#include "rbf_attn_split_kernels.h"

namespace rbf {

// Eight consecutive fp32 values as three bf16 fragments.
struct Frag3 {
  bf16x8_t h, m, l;
};

__device__ __forceinline__ Frag3 cut8(const float* x) {
  u32x4_t h, m, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bf16x2_t hh = {(__bf16)x[2 * e], (__bf16)x[2 * e + 1]};
    const uint32_t hw = __builtin_bit_cast(uint32_t, hh);
    h[e] = hw;
    const float ra = x[2 * e] - __uint_as_float(hw << 16), rb = x[2 * e + 1] - __uint_as_float(hw & 0xffff0000u);
    const bf16x2_t mm = {(__bf16)ra, (__bf16)rb};
    const uint32_t mw = __builtin_bit_cast(uint32_t, mm);
    m[e] = mw;
    const bf16x2_t ll = {(__bf16)(ra - __uint_as_float(mw << 16)), (__bf16)(rb - __uint_as_float(mw & 0xffff0000u))};
    l[e] = __builtin_bit_cast(uint32_t, ll);
  }
  return {__builtin_bit_cast(bf16x8_t, h), __builtin_bit_cast(bf16x8_t, m), __builtin_bit_cast(bf16x8_t, l)};
}

constexpr float kLift = 0x1p24f;

// cut8 of x * f (f a power of two).
__device__ __forceinline__ Frag3 cut8(const float* x, float f) {
  float y[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = x[e] * f;
  return cut8(y);
}

// Whether one of n accumulators, or x, is infinite or NaN (by the bits: the compiler
// may take a comparison of floats for one without NaN).
__device__ __forceinline__ bool not_finite(const f32x16_t* acc, int n, float x) {
  uint32_t m = __float_as_uint(x) << 1;
#pragma unroll
  for (int d = 0; d < n; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) m = max(m, __float_as_uint(acc[d][i]) << 1);
  return m >= 0xff000000u;
}

__device__ __forceinline__ f32x16_t mma3(const Frag3& a, const Frag3& b, f32x16_t c) {
  typedef Elem<__bf16> E;
  c = E::mma(a.l, b.h, c);
  c = E::mma(a.h, b.l, c);
  c = E::mma(a.m, b.m, c);
  c = E::mma(a.m, b.h, c);
  c = E::mma(a.h, b.m, c);
  return E::mma(a.h, b.h, c);
}

// Row fragment (features 16t + 8h ..) of a register-resident operand's token,
// zeros where !ok; returns the sum of squares of the loaded values.
__device__ __forceinline__ float load8(const float* p, bool ok, float* x) {
  float s = 0.f;
  if (ok) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p), b = *reinterpret_cast<const f32x4_t*>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = a[e];
      x[4 + e] = b[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = 0.f;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) s = fmaf(x[e], x[e], s);
  return s;
}

// Tiles of ROWS tokens of two operands A and B, global -> registers -> three
// bf16 planes each in LDS (planes [A h, A m, A l, B h, B m, B l] of ROWS x DP).
// Work unit: eight features of a token; consecutive threads take consecutive
// features, so loads read whole rows.
template <int ROWS, int DP, int NT>
struct Stage3 {
  static constexpr int CPR = DP / 8, HALF = ROWS * CPR, PER = (2 * HALF + NT - 1) / NT;
  static_assert((2 * HALF) % NT == 0 || 2 * HALF < NT, "whole units per thread");
  float r[PER][8];

  __device__ static __forceinline__ bool place(int j, int tid, bool& second, int& row, int& ch) {
    int u = tid + j * NT;
    if (2 * HALF < NT && u >= 2 * HALF) return false;
    second = HALF % NT == 0 ? j * NT >= HALF : u >= HALF;
    u -= second ? HALF : 0;
    row = u / CPR;
    ch = u % CPR;
    return true;
  }

  __device__ __forceinline__ void load(const float* A, int64_t sa, const float* B, int64_t sb, int tok0, int N, int D, int tid) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      bool second;
      int row, ch;
      if (!place(j, tid, second, row, ch)) continue;
      const int tok = tok0 + row;
      const bool ok = tok >= 0 && tok < N && 8 * ch < D;
      const float* p = second ? B + (int64_t)tok * sb + 8 * ch : A + (int64_t)tok * sa + 8 * ch;
      f32x4_t a = {}, b = {};
      if (ok) {
        a = *reinterpret_cast<const f32x4_t*>(p);
        b = *reinterpret_cast<const f32x4_t*>(p + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r[j][e] = a[e];
        r[j][4 + e] = b[e];
      }
    }
  }

  // The planes are those of LA * A and kLift * B; nrm (where NORMS): LA * -0.5 ||row||^2
  // of A's rows, -inf for tokens outside [0, N).
  template <bool NORMS, bool LIFT_A>
  __device__ __forceinline__ void store(__bf16 (*planes)[ROWS * DP], float* nrm, int tok0, int N, int tid) const {
    constexpr float LA = LIFT_A ? kLift : 1.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      bool second;
      int row, ch;
      if (!place(j, tid, second, row, ch)) continue;
      const Frag3 f = LIFT_A ? cut8(r[j], kLift) : HALF % NT == 0 && !second ? cut8(r[j]) : cut8(r[j], second ? kLift : 1.f);
      __bf16* o = planes[second ? 3 : 0] + SLayout<DP>::off(row, 8 * ch);
      st8<__bf16>(o, f.h);
      st8<__bf16>(o + ROWS * DP, f.m);
      st8<__bf16>(o + 2 * ROWS * DP, f.l);
      if constexpr (NORMS) {
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) s = fmaf(r[j][e], r[j][e], s);
        s = group_sum<CPR>(s);
        const int tok = tok0 + row;
        if (!second && ch == 0) nrm[row] = (tok >= 0 && tok < N) ? -0.5f * LA * s : -__builtin_inff();
      }
    }
  }
};

// Fragment of three planes (plane stride PS elements): row read and transposing
// read, as SLayout's.
template <int DP, int PS>
__device__ __forceinline__ Frag3 row3(const __bf16* t, int n, int col) {
  const __bf16* p = t + SLayout<DP>::off(n, col);
  return {ld8<__bf16>(p), ld8<__bf16>(p + PS), ld8<__bf16>(p + 2 * PS)};
}
template <int DP, int PS>
__device__ __forceinline__ Frag3 tr3(const __bf16* t, int tbase, int fbase, int lane) {
  typedef SLayout<DP> L;
  return {L::template tr<__bf16>(t, tbase, fbase, lane), L::template tr<__bf16>(t + PS, tbase, fbase, lane),
          L::template tr<__bf16>(t + 2 * PS, tbase, fbase, lane)};
}

// ---------------------------------------------------------------------------
// The EXACT pass, at a kernel's end where a result is not finite: a work-group's blocks one
// after another, in fp32 on the VALU: scores in LDS, operands read from global
// memory as they are used, and the output rows themselves as accumulators (element
// e of a block always by the same thread).  Written for few registers (it is part of
// kernels whose loops need them), not for speed: a step with an infinite key value in
// every head takes 13 ms instead of 0.22 at B4 H8 N1001 D64 and 67 instead of 0.72 at
// B4 H8 N1500 D128 (accumulators in registers and scores formed once: 8 and 30 ms, but
// the loops' dK/dV 2-7 % slower).  A masked pair is
// left out, so that an infinity reaches only what it is visible to.
// ---------------------------------------------------------------------------
constexpr int kExactRow = 33;  // floats per row of 32 scores in LDS

// init + sum over the features of a[i] * b[i].
__device__ __forceinline__ float exact_dot(const float* a, const float* b, int D, float init) {
#pragma unroll 1
  for (int i = 0; i < D; i += 4) {
    const f32x4_t x = *reinterpret_cast<const f32x4_t*>(a + i), y = *reinterpret_cast<const f32x4_t*>(b + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) init = fmaf(x[e], y[e], init);
  }
  return init;
}

// A kernel's Params where they are, in the kernel argument segment (their only
// argument), through a pointer the compiler knows nothing of: nothing that the pass
// alone uses stays in registers during the kernel's loop.
typedef const __attribute__((address_space(4))) Params* KernArg;
__device__ __forceinline__ KernArg kern_arg() {
  KernArg p = (KernArg)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// The (b, h) slice's pointers and what the three passes share.
struct ExactArgs {
  const float *Q, *K, *V, *O, *dO;
  int64_t sq, sk, sv, so, sdo;
  int N, D, org, npre, b, hh;
  bool causal;
  float c;
  __device__ __forceinline__ ExactArgs(KernArg p, int bh) {
    b = bh / p->H;
    hh = bh - b * p->H;
    Q = reinterpret_cast<const float*>(p->q) + b * p->sq[0] + hh * p->sq[1];
    K = reinterpret_cast<const float*>(p->k) + b * p->sk[0] + hh * p->sk[1];
    V = reinterpret_cast<const float*>(p->v) + b * p->sv[0] + hh * p->sv[1];
    O = reinterpret_cast<const float*>(p->o) + b * p->so[0] + hh * p->so[1];
    dO = reinterpret_cast<const float*>(p->dout) + b * p->sdo[0] + hh * p->sdo[1];
    sq = p->sq[2];
    sk = p->sk[2];
    sv = p->sv[2];
    so = p->so[2];
    sdo = p->sdo[2];
    N = p->N;
    D = p->D;
    org = p->org;
    npre = p->num_prefix;
    causal = p->causal != 0;
    c = p->c;
  }
};

// lds: 32 * (kExactRow + 3) floats.
template <int DP, int NT, bool SOFTMAX>
__device__ __forceinline__ void exact_fwd_block(KernArg p, float* lds, int bh, int qblk, int tid) {
  const ExactArgs a(p, bh);
  float *S = lds, *rm = S + 32 * kExactRow, *rl = rm + 32, *ra = rl + 32;
  float* O = const_cast<float*>(a.O);
  const int q0 = a.org + 32 * qblk, nblk = p->nblk;
  __syncthreads();
#pragma unroll 1
  for (int e = tid; e < 32 * DP; e += NT)
    if (q0 + e / DP >= 0 && e % DP < a.D) O[(q0 + e / DP) * a.so + e % DP] = 0.f;
  if (tid < 32) {
    const int q = q0 + tid;
    rm[tid] = SOFTMAX ? -__builtin_inff() : q >= 0 ? 0.5f * a.c * exact_dot(a.Q + q * a.sq, a.Q + q * a.sq, a.D, 0.f) : 0.f;
    rl[tid] = 0.f;
    ra[tid] = 1.f;
  }
#pragma unroll 1
  for (int kb = 0; kb < nblk; ++kb) {
    const int k0 = a.org + 32 * kb;
    if (!blk_any(q0, k0, a.causal, a.npre)) continue;
    __syncthreads();
#pragma unroll 1
    for (int e = tid; e < 1024; e += NT) {
      const int r = e >> 5, j = e & 31, q = q0 + r, k = k0 + j;
      float s = -__builtin_inff();
      if (q >= 0 && k >= 0 && k <= last_key(q, a.N, a.causal, a.npre)) {
        const float* kr = a.K + k * a.sk;
        s = exact_dot(a.Q + q * a.sq, kr, a.D, -0.5f * exact_dot(kr, kr, a.D, 0.f));
      }
      S[r * kExactRow + j] = s;
    }
    __syncthreads();
    if (SOFTMAX && tid < 32) {
      float m = rm[tid], l = 0.f;
#pragma unroll 1
      for (int j = 0; j < 32; ++j) m = fmaxf(m, a.c * S[tid * kExactRow + j]);
      const float off = m == -__builtin_inff() ? 0.f : m;
#pragma unroll 1
      for (int j = 0; j < 32; ++j) l += fast_exp2(fmaf(S[tid * kExactRow + j], a.c, -off));
      const float alpha = rm[tid] == -__builtin_inff() ? 0.f : fast_exp2(rm[tid] - off);
      rl[tid] = rl[tid] * alpha + l;
      ra[tid] = alpha;
      rm[tid] = m;
    }
    __syncthreads();
#pragma unroll 1
    for (int e = tid; e < 32 * DP; e += NT) {
      const int r = e / DP, d = e % DP, q = q0 + r;
      if (q < 0 || d >= a.D) continue;
      const int last = last_key(q, a.N, a.causal, a.npre);
      const float off = rm[r] == -__builtin_inff() ? 0.f : rm[r];
      float x = O[q * a.so + d] * ra[r];
#pragma unroll 1
      for (int j = max(0, -k0); j < 32 && k0 + j <= last; ++j)
        x = fmaf(fast_exp2(fmaf(S[r * kExactRow + j], a.c, -off)), a.V[(k0 + j) * a.sv + d], x);
      O[q * a.so + d] = x;
    }
  }
  if constexpr (SOFTMAX) {
#pragma unroll 1
    for (int e = tid; e < 32 * DP; e += NT) {
      const int r = e / DP, d = e % DP, q = q0 + r;
      if (q >= 0 && d < a.D) O[q * a.so + d] /= rl[r];
    }
  }
  if (SOFTMAX && tid < 32 && q0 + tid >= 0) p->lse[(int64_t)bh * a.N + q0 + tid] = rm[tid] + __log2f(rl[tid]);
}

// lds: 32 * (kExactRow + 3) floats.  Delta, or the norm offset, was written by
// the kernel.
template <int DP, int NT, bool SOFTMAX>
__device__ __forceinline__ void exact_dq_block(KernArg p, float* lds, int bh, int qblk, int tid) {
  const ExactArgs a(p, bh);
  float *S = lds, *roff = S + 32 * kExactRow, *rdel = roff + 32, *rsum = rdel + 32;
  float* dQ = reinterpret_cast<float*>(p->dq) + a.b * p->sdq[0] + a.hh * p->sdq[1];
  const int64_t sdq = p->sdq[2];
  const int q0 = a.org + 32 * qblk, nblk = p->nblk;
  __syncthreads();
#pragma unroll 1
  for (int e = tid; e < 32 * DP; e += NT)
    if (q0 + e / DP >= 0 && e % DP < a.D) dQ[(q0 + e / DP) * sdq + e % DP] = 0.f;
  if (tid < 32) {
    const int q = q0 + tid;
    float off = 0.f, del = 0.f;
    if (q >= 0) {
      off = SOFTMAX ? p->lse[(int64_t)bh * a.N + q] : 0.5f * a.c * exact_dot(a.Q + q * a.sq, a.Q + q * a.sq, a.D, 0.f);
      if (SOFTMAX) del = exact_dot(a.O + q * a.so, a.dO + q * a.sdo, a.D, 0.f);
    }
    roff[tid] = off;
    rdel[tid] = del;
    rsum[tid] = 0.f;
  }
#pragma unroll 1
  for (int kb = 0; kb < nblk; ++kb) {
    const int k0 = a.org + 32 * kb;
    if (!blk_any(q0, k0, a.causal, a.npre)) continue;
    __syncthreads();
#pragma unroll 1
    for (int e = tid; e < 1024; e += NT) {
      const int r = e >> 5, j = e & 31, q = q0 + r, k = k0 + j;
      float ds = 0.f;
      if (q >= 0 && k >= 0 && k <= last_key(q, a.N, a.causal, a.npre)) {
        const float* kr = a.K + k * a.sk;
        const float s = exact_dot(a.Q + q * a.sq, kr, a.D, -0.5f * exact_dot(kr, kr, a.D, 0.f));
        ds = fast_exp2(fmaf(s, a.c, -roff[r])) * exact_dot(a.V + k * a.sv, a.dO + q * a.sdo, a.D, -rdel[r]);
      }
      S[r * kExactRow + j] = ds;
    }
    __syncthreads();
#pragma unroll 1
    for (int e = tid; e < 32 * DP; e += NT) {
      const int r = e / DP, d = e % DP, q = q0 + r;
      if (q < 0 || d >= a.D) continue;
      const int last = last_key(q, a.N, a.causal, a.npre);
      float x = dQ[q * sdq + d];
#pragma unroll 1
      for (int j = max(0, -k0); j < 32 && k0 + j <= last; ++j) x = fmaf(S[r * kExactRow + j], a.K[(k0 + j) * a.sk + d], x);
      dQ[q * sdq + d] = x;
    }
    if (!SOFTMAX && tid < 32) {
      float x = 0.f;
#pragma unroll 1
      for (int j = 0; j < 32; ++j) x += S[tid * kExactRow + j];
      rsum[tid] += x;
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int e = tid; e < 32 * DP; e += NT) {
    const int r = e / DP, d = e % DP, q = q0 + r;
    if (q < 0 || d >= a.D) continue;
    const float x = dQ[q * sdq + d];
    dQ[q * sdq + d] = 2.f * p->gamma * (SOFTMAX ? x : x - rsum[r] * a.Q[q * a.sq + d]);
  }
}

// lds: 32 * (2 * kExactRow + 2) floats.
template <int DP, int NT, bool SOFTMAX>
__device__ __forceinline__ void exact_dkdv_block(KernArg p, float* lds, int bh, int kblk, int tid) {
  const ExactArgs a(p, bh);
  float *P = lds, *S = P + 32 * kExactRow, *rnk = S + 32 * kExactRow, *rsum = rnk + 32;
  float* dK = reinterpret_cast<float*>(p->dk) + a.b * p->sdk[0] + a.hh * p->sdk[1];
  float* dV = reinterpret_cast<float*>(p->dv) + a.b * p->sdv[0] + a.hh * p->sdv[1];
  const int64_t sdk = p->sdk[2], sdv = p->sdv[2];
  const int k0 = a.org + 32 * kblk, nblk = p->nblk;
  const float* offg = p->lse + (int64_t)bh * a.N;
  const float* delg = SOFTMAX ? p->delta + (int64_t)bh * a.N : nullptr;
  __syncthreads();
#pragma unroll 1
  for (int e = tid; e < 32 * DP; e += NT)
    if (k0 + e / DP >= 0 && e % DP < a.D) dK[(k0 + e / DP) * sdk + e % DP] = dV[(k0 + e / DP) * sdv + e % DP] = 0.f;
  if (tid < 32) {
    const float* kr = a.K + max(k0 + tid, 0) * a.sk;
    rnk[tid] = -0.5f * a.c * exact_dot(kr, kr, a.D, 0.f);
    rsum[tid] = 0.f;
  }
#pragma unroll 1
  for (int qb = 0; qb < nblk; ++qb) {
    const int q0 = a.org + 32 * qb;
    if (!blk_any(q0, k0, a.causal, a.npre)) continue;
    __syncthreads();
#pragma unroll 1
    for (int e = tid; e < 1024; e += NT) {
      const int r = e >> 5, j = e & 31, k = k0 + r, q = q0 + j;
      float pv = 0.f, ds = 0.f;
      if (k >= 0 && q >= 0 && q < a.N && q >= first_query(k, a.causal, a.npre)) {
        const float s = exact_dot(a.Q + q * a.sq, a.K + k * a.sk, a.D, -offg[q] / a.c);
        pv = fast_exp2(fmaf(s, a.c, rnk[r]));
        ds = pv * exact_dot(a.dO + q * a.sdo, a.V + k * a.sv, a.D, SOFTMAX ? -delg[q] : 0.f);
      }
      P[r * kExactRow + j] = pv;
      S[r * kExactRow + j] = ds;
    }
    __syncthreads();
#pragma unroll 1
    for (int e = tid; e < 32 * DP; e += NT) {
      const int r = e / DP, d = e % DP, k = k0 + r;
      if (k < 0 || d >= a.D) continue;
      float x = dK[k * sdk + d], y = dV[k * sdv + d];
#pragma unroll 1
      for (int j = max(0, first_query(k, a.causal, a.npre) - q0); j < 32 && q0 + j < a.N; ++j) {
        if (q0 + j < 0) continue;
        x = fmaf(S[r * kExactRow + j], a.Q[(q0 + j) * a.sq + d], x);
        y = fmaf(P[r * kExactRow + j], a.dO[(q0 + j) * a.sdo + d], y);
      }
      dK[k * sdk + d] = x;
      dV[k * sdv + d] = y;
    }
    if (tid < 32) {
      float x = 0.f;
#pragma unroll 1
      for (int j = 0; j < 32; ++j) x += S[tid * kExactRow + j];
      rsum[tid] += x;
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int e = tid; e < 32 * DP; e += NT) {
    const int r = e / DP, d = e % DP, k = k0 + r;
    if (k >= 0 && d < a.D) dK[k * sdk + d] = 2.f * p->gamma * (dK[k * sdk + d] - rsum[r] * a.K[k * a.sk + d]);
  }
}

// ---------------------------------------------------------------------------
// Forward: as rbf_fwd_group with the static softmax bound (and its rerun).
// ---------------------------------------------------------------------------
template <int DP, int W, int KSP, bool SOFTMAX>
__global__ __launch_bounds__(64 * W) void rbf_fwd_f32_kernel(const Params p) {
  constexpr int NT = 64 * W, KS = DP / 16, ND = DP / 32, GB = W / KSP, ROWS = 32 * KSP, PS = ROWS * DP;
  __shared__ __attribute__((aligned(1024))) __bf16 sT[6][PS];
  __shared__ __attribute__((aligned(16))) float sKn[ROWS];
  __shared__ float sM[W][32];
  __shared__ float sX[KSP > 1 ? W / 2 : 1][1][64];
  static_assert(KSP == 1 || W / 2 * ND * 4096 <= (int)sizeof(sT), "the partials fit the tiles");

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
  const float* Q = reinterpret_cast<const float*>(p.q) + b * p.sq[0] + hh * p.sq[1];
  const float* K = reinterpret_cast<const float*>(p.k) + b * p.sk[0] + hh * p.sk[1];
  const float* V = reinterpret_cast<const float*>(p.v) + b * p.sv[0] + hh * p.sv[1];
  float* O = reinterpret_cast<float*>(const_cast<void*>(p.o)) + b * p.so[0] + hh * p.so[1];

  const int blk0 = nblk - (ngrp - grp) * GB;
  const int qblk = blk0 + wave / KSP;
  const bool wave_on = qblk >= 0;
  const int q0 = org + 32 * qblk, qtok = q0 + n;
  const bool qvalid = wave_on && qtok >= 0;
  const int jmax = last_key(qtok, N, causal, npre);
  const int hi = min(causal ? max(org + 32 * (blk0 + GB), npre) : N, N);
  const int nkt = ((hi - 1 - org) >> 5) / KSP + 1;

  Stage3<ROWS, DP, NT> st;
  auto load = [&](int kt) __attribute__((always_inline)) { st.load(K, p.sk[2], V, p.sv[2], org + kt * ROWS, N, D, tid); };
  load(0);

  Frag3 qf[KS];
  float qn2 = 0.f;  // c * 0.5 ||q||^2
#pragma unroll
  for (int t = 0; t < KS; ++t) {
    float x[8];
    qn2 += load8(Q + (int64_t)qtok * p.sq[2] + 16 * t + 8 * h, qvalid && 16 * t + 8 * h < D, x);
    qf[t] = cut8(x);
  }
  qn2 = c * 0.5f * xhalf_sum(qn2);

  f32x16_t oacc[ND];
  float lrow, m_run;
  auto run = [&](auto safe_tag) {
    constexpr bool SAFE = decltype(safe_tag)::value;
#pragma unroll
    for (int d = 0; d < ND; ++d) oacc[d] = zero16();
    lrow = 0.f;
    m_run = !SOFTMAX ? qn2 : (SAFE ? -__builtin_inff() : qn2 - kBoundMargin);
    for (int kt = 0; kt < nkt; ++kt) {
      lds_barrier();  // every wave is done with the previous tile
      st.template store<true, false>(sT, sKn, org + kt * ROWS, N, tid);
      lds_barrier();
      if (kt + 1 < nkt) load(kt + 1);
      const int k0 = org + 32 * (kt * KSP + ki);
      if (!wave_on || k0 >= N || !blk_any(q0, k0, causal, npre)) continue;
      const __bf16* kt_ = sT[0] + 32 * ki * DP;
      const __bf16* vt_ = sT[3] + 32 * ki * DP;
      f32x16_t s = ld_rows16(sKn + 32 * ki, h);
#pragma unroll
      for (int t = 0; t < KS; ++t) s = mma3(row3<DP, PS>(kt_, n, 16 * t + 8 * h), qf[t], s);
      if (!blk_nomask(q0, k0, causal, npre)) mask_key_rows(s, k0, h, jmax);
      if constexpr (SOFTMAX && SAFE) {
        const float mt = xhalf_max(tree_max16(s)) * c;
        if (__any(mt > m_run + kTau)) {
          const float mnew = fmaxf(m_run, mt);
          const float alpha = (mnew == -__builtin_inff()) ? 1.f : fast_exp2(m_run - mnew);
#pragma unroll
          for (int d = 0; d < ND; ++d) oacc[d] *= alpha;
          lrow *= alpha;
          m_run = mnew;
        }
      }
      const float moff = (SAFE && m_run == -__builtin_inff()) ? 0.f : m_run;
      float pe[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) pe[i] = fast_exp2(fmaf(s[i], c, -moff));
      if constexpr (SOFTMAX) lrow += tree_sum16(pe);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const Frag3 pf = SOFTMAX ? cut8(pe + 8 * t) : cut8(pe + 8 * t, kLift);
#pragma unroll
        for (int d = 0; d < ND; ++d) oacc[d] = mma3(tr3<DP, PS>(vt_, 16 * t, 32 * d, lane), pf, oacc[d]);
      }
    }
    if constexpr (KSP > 1) {
      if constexpr (SOFTMAX && SAFE) {
        // bring the splits' partials to the block's largest offset
        if (h == 0) sM[wave][n] = m_run;
        __syncthreads();
        float M = m_run;
#pragma unroll
        for (int e = 0; e < KSP; ++e) M = fmaxf(M, sM[wave - ki + e][n]);
        const float w = (m_run == -__builtin_inff()) ? 0.f : fast_exp2(m_run - M);
#pragma unroll
        for (int d = 0; d < ND; ++d) oacc[d] *= w;
        lrow *= w;
        m_run = M;
      }
      split_sum<W, KSP, ND, 1>(oacc, &lrow, reinterpret_cast<f32x4_t*>(&sT[0][0]), sX, wave, lane);
    }
  };

  run(std::false_type{});
  if constexpr (SOFTMAX) {
    const float l = xhalf_sum(lrow);
    const bool bad = qvalid && ki == 0 && !(l >= kSumLow && l <= kSumHigh);
    if (__syncthreads_or(bad)) {
      load(0);
      run(std::true_type{});
    }
  }
  if (__syncthreads_or(qvalid && ki == 0 && not_finite(oacc, ND, lrow))) {
    static_assert(32 * (kExactRow + 3) * 4 <= (int)sizeof(sT), "the pass fits the tiles");
#pragma unroll 1
    for (int g = 0; g < GB; ++g)
      if (blk0 + g >= 0) exact_fwd_block<DP, NT, SOFTMAX>(kern_arg(), reinterpret_cast<float*>(&sT[0][0]), bh, blk0 + g, tid);
    return;
  }

  if (!wave_on || ki != 0) return;
  const float lsum = SOFTMAX ? xhalf_sum(lrow) : 1.f;
  const float inv = SOFTMAX ? 1.f / kLift / lsum : 1.f / kLift / kLift;
  if (qtok < 0) return;
  float* orow = O + (int64_t)qtok * p.so[2];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * d + 8 * g + 4 * h;
      if (dd < D) {
        float v4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v4[e] = oacc[d][4 * g + e] * inv;
        st4f<float>(orow + dd, v4);
      }
    }
  if (SOFTMAX && h == 0) p.lse[(int64_t)bh * N + qtok] = m_run + __log2f(lsum);
}

// ---------------------------------------------------------------------------
// dQ (and Delta, or the non-softmax norm offsets), as rbf_bwd_dq_group.
// ---------------------------------------------------------------------------
template <int DP, int W, int KSP, bool SOFTMAX>
__global__ __launch_bounds__(64 * W) void rbf_bwd_dq_f32_kernel(const Params p) {
  constexpr int NT = 64 * W, KS = DP / 16, ND = DP / 32, GB = W / KSP, ROWS = 32 * KSP, PS = ROWS * DP;
  __shared__ __attribute__((aligned(1024))) __bf16 sT[6][PS];
  __shared__ __attribute__((aligned(16))) float sKn[ROWS];
  __shared__ float sX[KSP > 1 ? W / 2 : 1][1][64];
  static_assert(KSP == 1 || W / 2 * ND * 4096 <= (int)sizeof(sT), "the partials fit the tiles");

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
  const float* Q = reinterpret_cast<const float*>(p.q) + b * p.sq[0] + hh * p.sq[1];
  const float* K = reinterpret_cast<const float*>(p.k) + b * p.sk[0] + hh * p.sk[1];
  const float* V = reinterpret_cast<const float*>(p.v) + b * p.sv[0] + hh * p.sv[1];
  const float* Og = reinterpret_cast<const float*>(p.o) + b * p.so[0] + hh * p.so[1];
  const float* dO = reinterpret_cast<const float*>(p.dout) + b * p.sdo[0] + hh * p.sdo[1];
  float* dQ = reinterpret_cast<float*>(p.dq) + b * p.sdq[0] + hh * p.sdq[1];

  const int blk0 = nblk - (ngrp - grp) * GB;
  const int qblk = blk0 + wave / KSP;
  const bool wave_on = qblk >= 0;
  const int q0 = org + 32 * qblk, qtok = q0 + n;
  const bool qvalid = wave_on && qtok >= 0;
  const int jmax = last_key(qtok, N, causal, npre);
  const int hi = min(causal ? max(org + 32 * (blk0 + GB), npre) : N, N);
  const int nkt = ((hi - 1 - org) >> 5) / KSP + 1;

  Stage3<ROWS, DP, NT> st;
  auto load = [&](int kt) __attribute__((always_inline)) { st.load(K, p.sk[2], V, p.sv[2], org + kt * ROWS, N, D, tid); };
  load(0);

  Frag3 qf[KS], df[KS];  // df: of kLift * dO
  float off, dlt = 0.f, qn2 = 0.f;
#pragma unroll
  for (int t = 0; t < KS; ++t) {
    const bool ok = qvalid && 16 * t + 8 * h < D;
    float x[8], y[8];
    qn2 += load8(Q + (int64_t)qtok * p.sq[2] + 16 * t + 8 * h, ok, x);
    qf[t] = cut8(x);
    load8(dO + (int64_t)qtok * p.sdo[2] + 16 * t + 8 * h, ok, y);
    df[t] = cut8(y, kLift);
    if constexpr (SOFTMAX) {
      load8(Og + (int64_t)qtok * p.so[2] + 16 * t + 8 * h, ok, x);
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) s = fmaf(x[e], y[e], s);
      dlt += s;
    }
  }
  if constexpr (SOFTMAX) {
    dlt = xhalf_sum(dlt);
    off = qvalid ? p.lse[(int64_t)bh * N + qtok] : 0.f;
    if (qvalid && h == 0 && ki == 0) p.delta[(int64_t)bh * N + qtok] = dlt;
  } else {
    off = c * 0.5f * xhalf_sum(qn2);
    if (qvalid && h == 0 && ki == 0) p.lse[(int64_t)bh * N + qtok] = off;
  }

  f32x16_t dqacc[ND];  // times kLift^3; S: kLift times, dP and dS: kLift^2 times
  float rsum = 0.f;
#pragma unroll
  for (int d = 0; d < ND; ++d) dqacc[d] = zero16();
  for (int kt = 0; kt < nkt; ++kt) {
    lds_barrier();
    st.template store<true, true>(sT, sKn, org + kt * ROWS, N, tid);
    lds_barrier();
    if (kt + 1 < nkt) load(kt + 1);
    const int k0 = org + 32 * (kt * KSP + ki);
    if (!wave_on || k0 >= N || !blk_any(q0, k0, causal, npre)) continue;
    const __bf16* kt_ = sT[0] + 32 * ki * DP;
    const __bf16* vt_ = sT[3] + 32 * ki * DP;
    f32x16_t s = ld_rows16(sKn + 32 * ki, h), dp = SOFTMAX ? splat16(-kLift * kLift * dlt) : zero16();
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      s = mma3(row3<DP, PS>(kt_, n, 16 * t + 8 * h), qf[t], s);
      dp = mma3(row3<DP, PS>(vt_, n, 16 * t + 8 * h), df[t], dp);
    }
    if (!blk_nomask(q0, k0, causal, npre)) mask_key_rows(s, k0, h, jmax);
    float ds[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) ds[i] = fast_exp2(fmaf(s[i], c / kLift, -off)) * dp[i];
    if constexpr (!SOFTMAX) rsum += tree_sum16(ds);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const Frag3 sf = cut8(ds + 8 * t);
#pragma unroll
      for (int d = 0; d < ND; ++d) dqacc[d] = mma3(tr3<DP, PS>(kt_, 16 * t, 32 * d, lane), sf, dqacc[d]);
    }
  }
  if constexpr (KSP > 1) split_sum<W, KSP, ND, 1>(dqacc, &rsum, reinterpret_cast<f32x4_t*>(&sT[0][0]), sX, wave, lane);

  if (__syncthreads_or(qvalid && ki == 0 && not_finite(dqacc, ND, rsum))) {
    static_assert(32 * (kExactRow + 3) * 4 <= (int)sizeof(sT), "the pass fits the tiles");
#pragma unroll 1
    for (int g = 0; g < GB; ++g)
      if (blk0 + g >= 0) exact_dq_block<DP, NT, SOFTMAX>(kern_arg(), reinterpret_cast<float*>(&sT[0][0]), bh, blk0 + g, tid);
    return;
  }
  if (!wave_on || ki != 0) return;
  const float g2 = 2.f * p.gamma, unlift2 = 1.f / (kLift * kLift), unlift3 = unlift2 / kLift;
  float rs = 0.f;
  if constexpr (!SOFTMAX) rs = unlift2 * xhalf_sum(rsum);
  if (qtok < 0) return;
  float* drow = dQ + (int64_t)qtok * p.sdq[2];
  const float* qrow = Q + (int64_t)qtok * p.sq[2];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * d + 8 * g + 4 * h;
      if (dd < D) {
        float v4[4], q4[4] = {};
        if constexpr (!SOFTMAX) ld4f<float>(qrow + dd, q4);
#pragma unroll
        for (int e = 0; e < 4; ++e) v4[e] = g2 * (unlift3 * dqacc[d][4 * g + e] - (SOFTMAX ? 0.f : rs * q4[e]));
        st4f<float>(drow + dd, v4);
      }
    }
}

// ---------------------------------------------------------------------------
// dK and dV, as rbf_bwd_dkdv_group.
// ---------------------------------------------------------------------------
template <int DP, int W, int KSP, bool SOFTMAX>
__global__ __launch_bounds__(64 * W) void rbf_bwd_dkdv_f32_kernel(const Params p) {
  constexpr int NT = 64 * W, KS = DP / 16, ND = DP / 32, GB = W / KSP, ROWS = 32 * KSP, PS = ROWS * DP;
  __shared__ __attribute__((aligned(1024))) __bf16 sT[6][PS];
  __shared__ __attribute__((aligned(16))) float sOff[ROWS], sDel[ROWS];  // -kLift * L/c (or -0.5||q||^2), -kLift^2 * Delta
  __shared__ float sX[KSP > 1 ? W / 2 : 1][1][64];
  static_assert(KSP == 1 || W / 2 * 2 * ND * 4096 <= (int)sizeof(sT), "the partials fit the tiles");

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ki = wave % KSP;
  const int N = p.N, D = p.D, org = p.org, nblk = p.nblk;
  const bool causal = p.causal != 0;
  const int npre = p.num_prefix;
  const float c = p.c;
  const float inv_c = 1.f / c;
  const int ngrp = (nblk + GB - 1) / GB;
  int bh, grp;
  split_wg(ngrp, p.hchunk, bh, grp);
  const int b = bh / p.H, hh = bh - b * p.H;
  const float* Q = reinterpret_cast<const float*>(p.q) + b * p.sq[0] + hh * p.sq[1];
  const float* K = reinterpret_cast<const float*>(p.k) + b * p.sk[0] + hh * p.sk[1];
  const float* V = reinterpret_cast<const float*>(p.v) + b * p.sv[0] + hh * p.sv[1];
  const float* dO = reinterpret_cast<const float*>(p.dout) + b * p.sdo[0] + hh * p.sdo[1];
  float* dK = reinterpret_cast<float*>(p.dk) + b * p.sdk[0] + hh * p.sdk[1];
  float* dV = reinterpret_cast<float*>(p.dv) + b * p.sdv[0] + hh * p.sdv[1];
  const float* offg = p.lse + (int64_t)bh * N;
  const float* delg = SOFTMAX ? p.delta + (int64_t)bh * N : nullptr;

  const int blk0 = grp * GB;
  const int kblk = blk0 + wave / KSP;
  const bool wave_on = kblk < nblk;
  const int k0 = org + 32 * kblk, ktok = k0 + n;
  const bool kvalid = wave_on && ktok >= 0;
  const int ilo = first_query(ktok, causal, npre);
  const int wg_kfirst = max(org + 32 * blk0, 0);
  const int qlo = causal ? (wg_kfirst < npre ? 0 : wg_kfirst) : 0;
  const int qb0 = (qlo - org) >> 5;
  const int nqt = (nblk - qb0 + KSP - 1) / KSP;

  Stage3<ROWS, DP, NT> st;
  float offr = 0.f, delr = 0.f;
  auto load = [&](int t) __attribute__((always_inline)) {
    const int tok0 = org + 32 * (qb0 + t * KSP);
    st.load(Q, p.sq[2], dO, p.sdo[2], tok0, N, D, tid);
    if (tid < ROWS) {
      const int tok = tok0 + tid;
      const bool ok = tok >= 0 && tok < N;
      offr = ok ? -offg[tok] * inv_c * kLift : -__builtin_inff();  // padding queries: P = 0
      if constexpr (SOFTMAX) delr = ok ? -kLift * kLift * delg[tok] : 0.f;
    }
  };
  load(0);

  Frag3 kf[KS], vf[KS];  // vf: of kLift * V
  float nckn = 0.f;  // -c * 0.5||k||^2
#pragma unroll
  for (int t = 0; t < KS; ++t) {
    const bool ok = kvalid && 16 * t + 8 * h < D;
    float x[8];
    nckn += load8(K + (int64_t)ktok * p.sk[2] + 16 * t + 8 * h, ok, x);
    kf[t] = cut8(x);
    load8(V + (int64_t)ktok * p.sv[2] + 16 * t + 8 * h, ok, x);
    vf[t] = cut8(x, kLift);
  }
  nckn = -c * 0.5f * xhalf_sum(nckn);

  // dK^T times kLift^3, then dV^T times kLift^2; S: kLift times, dP and dS: kLift^2 times
  f32x16_t acc[2 * ND];
  float csum = 0.f;
#pragma unroll
  for (int d = 0; d < 2 * ND; ++d) acc[d] = zero16();
  for (int t0 = 0; t0 < nqt; ++t0) {
    lds_barrier();
    st.template store<false, true>(sT, nullptr, 0, N, tid);
    if (tid < ROWS) {
      sOff[tid] = offr;
      sDel[tid] = delr;
    }
    lds_barrier();
    if (t0 + 1 < nqt) load(t0 + 1);
    const int qb = qb0 + t0 * KSP + ki, q0 = org + 32 * qb;
    if (!wave_on || qb >= nblk || !blk_any(q0, k0, causal, npre)) continue;
    const __bf16* qt_ = sT[0] + 32 * ki * DP;
    const __bf16* dt_ = sT[3] + 32 * ki * DP;
    f32x16_t s = ld_rows16(sOff + 32 * ki, h), dp = SOFTMAX ? ld_rows16(sDel + 32 * ki, h) : zero16();
#pragma unroll
    for (int t = 0; t < KS; ++t) {
      s = mma3(row3<DP, PS>(qt_, n, 16 * t + 8 * h), kf[t], s);
      dp = mma3(row3<DP, PS>(dt_, n, 16 * t + 8 * h), vf[t], dp);
    }
    if (!blk_nomask(q0, k0, causal, npre)) mask_query_rows(s, q0, h, ilo);
    float pv[16], ds[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      pv[i] = fast_exp2(fmaf(s[i], c / kLift, nckn));
      ds[i] = pv[i] * dp[i];
    }
    csum += tree_sum16(ds);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const Frag3 pf = cut8(pv + 8 * t, kLift), sf = cut8(ds + 8 * t);
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        acc[ND + d] = mma3(tr3<DP, PS>(dt_, 16 * t, 32 * d, lane), pf, acc[ND + d]);
        acc[d] = mma3(tr3<DP, PS>(qt_, 16 * t, 32 * d, lane), sf, acc[d]);
      }
    }
  }
  if constexpr (KSP > 1) split_sum<W, KSP, 2 * ND, 1>(acc, &csum, reinterpret_cast<f32x4_t*>(&sT[0][0]), sX, wave, lane);

  if (__syncthreads_or(kvalid && ki == 0 && not_finite(acc, 2 * ND, csum))) {
    static_assert(32 * (2 * kExactRow + 2) * 4 <= (int)sizeof(sT), "the pass fits the tiles");
#pragma unroll 1
    for (int g = 0; g < GB; ++g)
      if (blk0 + g < nblk) exact_dkdv_block<DP, NT, SOFTMAX>(kern_arg(), reinterpret_cast<float*>(&sT[0][0]), bh, blk0 + g, tid);
    return;
  }
  if (!wave_on || ki != 0) return;
  const float g2 = 2.f * p.gamma, unlift2 = 1.f / (kLift * kLift), unlift3 = unlift2 / kLift;
  const float cs = unlift2 * xhalf_sum(csum);
  if (ktok < 0) return;
  float* dkrow = dK + (int64_t)ktok * p.sdk[2];
  float* dvrow = dV + (int64_t)ktok * p.sdv[2];
  const float* krow = K + (int64_t)ktok * p.sk[2];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * d + 8 * g + 4 * h;
      if (dd < D) {
        float k4[4], a4[4], b4[4];
        ld4f<float>(krow + dd, k4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a4[e] = g2 * (unlift3 * acc[d][4 * g + e] - cs * k4[e]);
          b4[e] = acc[ND + d][4 * g + e] * unlift2;
        }
        st4f<float>(dkrow + dd, a4);
        st4f<float>(dvrow + dd, b4);
      }
    }
}

}  // namespace rbf
