// int8 / E4M3 instantiations of the DMA kernel's 64-column tiles (see
// mid_tile in gemm_kernels.h).
#include "gemm_kernels.h"

namespace c3h {
namespace gk {

int launch_mid_i8(Problem p, hipStream_t s, int mode, int out_dtype, int tile) {
  if (mode == 0) return launch_mid_tile<MmaI8, int32_t, kDenseK>(p, s, tile, "qgemm_mid");
  if (mode == 1 || out_dtype == C3H_I8) return launch_mid_tile<MmaI8, int8_t, kDenseK>(p, s, tile, "qgemm_mid");
  if (out_dtype == C3H_F32) return launch_mid_tile<MmaI8, float, kDenseK>(p, s, tile, "qgemm_mid");
  if (out_dtype == C3H_BF16) return launch_mid_tile<MmaI8, bf16_t, kDenseK>(p, s, tile, "qgemm_mid");
  return launch_mid_tile<MmaI8, f16_t, kDenseK>(p, s, tile, "qgemm_mid");
}

int launch_mid_f8(Problem p, hipStream_t s, int out_dtype, int tile) {
  if (out_dtype == C3H_F32) return launch_mid_tile<MmaF8, float, kDenseK>(p, s, tile, "gemm_fp8_mid");
  if (out_dtype == C3H_BF16) return launch_mid_tile<MmaF8, bf16_t, kDenseK>(p, s, tile, "gemm_fp8_mid");
  return launch_mid_tile<MmaF8, f16_t, kDenseK>(p, s, tile, "gemm_fp8_mid");
}

}  // namespace gk
}  // namespace c3h
