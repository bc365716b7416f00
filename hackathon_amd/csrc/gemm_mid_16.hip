// bf16 / fp16 instantiations of the DMA kernel's 64-column tiles (see
// mid_tile in gemm_kernels.h).
#include "gemm_kernels.h"

namespace c3h {
namespace gk {

namespace {
template <typename Mma, typename T>
int launch_mid_type(Problem p, hipStream_t s, int am, int tile) {
  const bool f32 = p.out_dtype == C3H_F32;
  if (am == kConvTap)
    return f32 ? launch_mid_tile<Mma, float, kConvTap>(p, s, tile, "conv_mid")
               : launch_mid_tile<Mma, T, kConvTap>(p, s, tile, "conv_mid");
  return f32 ? launch_mid_tile<Mma, float, kDenseK>(p, s, tile, "gemm_mid")
             : launch_mid_tile<Mma, T, kDenseK>(p, s, tile, "gemm_mid");
}
template <typename Mma, typename T>
int launch_mid_part(Problem p, hipStream_t s, int tile) {
  return p.out_dtype == C3H_F32 ? launch_mid_tile<Mma, float, kDenseK, true>(p, s, tile, "gemm_mid_splitk")
                                : launch_mid_tile<Mma, T, kDenseK, true>(p, s, tile, "gemm_mid_splitk");
}
}  // namespace

int launch_mid_16(Problem p, hipStream_t s, int in_dtype, int am, int tile) {
  return in_dtype == C3H_BF16 ? launch_mid_type<MmaBF16, bf16_t>(p, s, am, tile)
                              : launch_mid_type<MmaF16, f16_t>(p, s, am, tile);
}

int launch_mid_16_part(Problem p, hipStream_t s, int in_dtype, int tile) {
  return in_dtype == C3H_BF16 ? launch_mid_part<MmaBF16, bf16_t>(p, s, tile)
                              : launch_mid_part<MmaF16, f16_t>(p, s, tile);
}

}  // namespace gk
}  // namespace c3h
