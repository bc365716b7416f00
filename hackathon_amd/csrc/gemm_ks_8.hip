// int8 / E4M3 / fp32 instantiations of the small-output GEMM and conv (see gemm_ks.h).
#include "gemm_ks.h"

namespace c3h {
namespace gk {

int launch_ks_i8(Problem p, hipStream_t s, int mode, int out_dtype, int tile) {
  if (mode == 0) return launch_ks_tile<MmaI8, int32_t, kDenseK>(p, s, tile, "qgemm_ks");
  if (mode == 1 || out_dtype == C3H_I8) return launch_ks_tile<MmaI8, int8_t, kDenseK>(p, s, tile, "qgemm_ks");
  if (out_dtype == C3H_F32) return launch_ks_tile<MmaI8, float, kDenseK>(p, s, tile, "qgemm_ks");
  if (out_dtype == C3H_BF16) return launch_ks_tile<MmaI8, bf16_t, kDenseK>(p, s, tile, "qgemm_ks");
  return launch_ks_tile<MmaI8, f16_t, kDenseK>(p, s, tile, "qgemm_ks");
}

int launch_ks_f8(Problem p, hipStream_t s, int out_dtype, int tile) {
  if (out_dtype == C3H_F32) return launch_ordered_tile<MmaF8, float, kDenseK>(p, s, tile, "gemm_fp8_small");
  if (out_dtype == C3H_BF16) return launch_ordered_tile<MmaF8, bf16_t, kDenseK>(p, s, tile, "gemm_fp8_small");
  return launch_ordered_tile<MmaF8, f16_t, kDenseK>(p, s, tile, "gemm_fp8_small");
}

int launch_ks_f32(Problem p, hipStream_t s, int am, int tile) {
  return am == kConvTap ? launch_ks_tile<MmaF32, float, kConvTap>(p, s, tile, "conv_ks")
                        : launch_ks_tile<MmaF32, float, kDenseK>(p, s, tile, "gemm_ks");
}

}  // namespace gk
}  // namespace c3h
