// Launchers of the fp32 kernels for up to 128 features.
#include "rbf_attn_f32_kernels.h"
#include "rbf_attn_launch.h"

namespace rbf {
namespace {

template <int W, int KSP, typename F>
hipError_t launch(F kernel, const Params& p, hipStream_t st) {
  constexpr int GB = W / KSP;
  const long long grid = (long long)p.B * p.H * ((p.nblk + GB - 1) / GB);
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * W), 0, st, p);
  return hipGetLastError();
}

int64_t blocks(const Params& p) { return (int64_t)p.B * p.H * p.nblk; }

// Waves per work-group (W) and per 32-token block (KSP), by the number of
// blocks.  Few blocks want the chain split four ways; enough blocks for every
// SIMD's two waves want one wave per block and eight blocks sharing the work of
// cutting a tile.  Measured at D = 64 (us; W, KSP):
//                            fwd: 4,4 / 8,2 / 8,1   dQ: 4,4 / 8,2 / 8,1   dK/dV: 4,4 / 4,2 / 4,1 / 8,1
//   B1 H8 N300 (80 blocks)   15 / 19 / 27           18 / 24 / 34          20 / 23 / 35 / 44
//   B1 H4 N4000 (500)        112 / 155 / 273        133 / 197 / 356       153 / 208 / 354 / 478
//   B4 H8 N1024 (1024)       71 / 45 / 75           90 / 59 / 97          103 / 72 / 99 / 130
//   the same, all visible    112 / 50 / 77          138 / 68 / 102        160 / 120 / 104 / 136
//   B8 H8 N1024 (2048)       143 / 60 / 77          178 / 79 / 101        209 / 143 / 122 / 131
//   B8 H16 N2000 (8064)      943 / 402 / 362        1128 / 549 / 501      1426 / 1022 / 845 / 685
// Up to 32 features the same limits hold (us fwd / dQ / dK/dV, against the fp32-MFMA
// kernels, which they stay well below on both sides of each): B1 H8 N300 23 / 28 / 33
// -> 11 / 13 / 13, B4 H8 N1000 62 / 77 / 96 -> 32 / 38 / 43, B8 H16 N1500 206 / 288 /
// 360 -> 149 / 184 / 253, B16 H16 N1000 all visible 341 / 480 / 620 -> 244 / 304 / 434.
// With 128 features a wave's fragments and accumulators leave one wave per
// SIMD: four-wave work-groups, two waves per block up to 640 blocks (B2 H8 N700
// 83 -> 55, 98 -> 65, 124 -> 86; at B4 H8 N1500 171 -> 197, 200 -> 230, 256 ->
// 317).
template <int DP, bool SM>
hipError_t fwd(const Params& p, hipStream_t st) {
  const int64_t n = blocks(p);
  if constexpr (DP == 128) {
    return n <= 640 ? launch<4, 2>(rbf_fwd_f32_kernel<DP, 4, 2, SM>, p, st) : launch<4, 1>(rbf_fwd_f32_kernel<DP, 4, 1, SM>, p, st);
  } else {
    if (n <= 640) return launch<4, 4>(rbf_fwd_f32_kernel<DP, 4, 4, SM>, p, st);
    if (n <= 3072) return launch<8, 2>(rbf_fwd_f32_kernel<DP, 8, 2, SM>, p, st);
    return launch<8, 1>(rbf_fwd_f32_kernel<DP, 8, 1, SM>, p, st);
  }
}

template <int DP, bool SM>
hipError_t dq(const Params& p, hipStream_t st) {
  const int64_t n = blocks(p);
  if constexpr (DP == 128) {
    return n <= 640 ? launch<4, 2>(rbf_bwd_dq_f32_kernel<DP, 4, 2, SM>, p, st) : launch<4, 1>(rbf_bwd_dq_f32_kernel<DP, 4, 1, SM>, p, st);
  } else {
    if (n <= 640) return launch<4, 4>(rbf_bwd_dq_f32_kernel<DP, 4, 4, SM>, p, st);
    if (n <= 3072) return launch<8, 2>(rbf_bwd_dq_f32_kernel<DP, 8, 2, SM>, p, st);
    return launch<8, 1>(rbf_bwd_dq_f32_kernel<DP, 8, 1, SM>, p, st);
  }
}

template <int DP, bool SM>
hipError_t dkdv(const Params& p, hipStream_t st) {
  const int64_t n = blocks(p);
  if constexpr (DP == 128) {
    return n <= 640 ? launch<4, 2>(rbf_bwd_dkdv_f32_kernel<DP, 4, 2, SM>, p, st) : launch<4, 1>(rbf_bwd_dkdv_f32_kernel<DP, 4, 1, SM>, p, st);
  } else {
    if (n <= 640) return launch<4, 4>(rbf_bwd_dkdv_f32_kernel<DP, 4, 4, SM>, p, st);
    if (n <= 1280 && p.causal) return launch<4, 2>(rbf_bwd_dkdv_f32_kernel<DP, 4, 2, SM>, p, st);
    if (n <= 3072) return launch<4, 1>(rbf_bwd_dkdv_f32_kernel<DP, 4, 1, SM>, p, st);
    return launch<8, 1>(rbf_bwd_dkdv_f32_kernel<DP, 8, 1, SM>, p, st);
  }
}

}  // namespace

#define RBF_F32_DISPATCH(F)                                                                     \
  do {                                                                                          \
    if (p.D > 128) return hipErrorInvalidValue;                                                 \
    const bool sm = variant == 0;                                                               \
    if (p.D <= 32) return sm ? F<32, true>(p, st) : F<32, false>(p, st);                        \
    if (p.D <= 64) return sm ? F<64, true>(p, st) : F<64, false>(p, st);                        \
    return sm ? F<128, true>(p, st) : F<128, false>(p, st);                                     \
  } while (0)

hipError_t launch_fwd_narrow_fp32(const Params& p, int variant, hipStream_t st) { RBF_F32_DISPATCH(fwd); }
hipError_t launch_bwd_dq_narrow_fp32(const Params& p, int variant, hipStream_t st) { RBF_F32_DISPATCH(dq); }
hipError_t launch_bwd_dkdv_narrow_fp32(const Params& p, int variant, hipStream_t st) { RBF_F32_DISPATCH(dkdv); }

}  // namespace rbf
