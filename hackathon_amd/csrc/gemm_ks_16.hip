// bf16 / fp16 instantiations of the small-output GEMM and conv (see gemm_ks.h).
#include "gemm_ks.h"

namespace c3h {
namespace gk {

namespace {
template <typename Mma, typename T>
int launch_ks_type(Problem p, hipStream_t s, int am, int tile) {
  const bool f32 = p.out_dtype == C3H_F32;
  if (am == kConvTap)
    return f32 ? launch_ordered_tile<Mma, float, kConvTap>(p, s, tile, "conv_small")
               : launch_ordered_tile<Mma, T, kConvTap>(p, s, tile, "conv_small");
  return f32 ? launch_ordered_tile<Mma, float, kDenseK>(p, s, tile, "gemm_small")
             : launch_ordered_tile<Mma, T, kDenseK>(p, s, tile, "gemm_small");
}
template <typename Mma, typename T>
int launch_ks_part(Problem p, hipStream_t s, int tile) {
  return p.out_dtype == C3H_F32 ? launch_ordered_tile<Mma, float, kDenseK, true>(p, s, tile, "gemm_small_splitk")
                                : launch_ordered_tile<Mma, T, kDenseK, true>(p, s, tile, "gemm_small_splitk");
}
}  // namespace

int launch_ks_16(Problem p, hipStream_t s, int in_dtype, int am, int tile) {
  return in_dtype == C3H_BF16 ? launch_ks_type<MmaBF16, bf16_t>(p, s, am, tile)
                              : launch_ks_type<MmaF16, f16_t>(p, s, am, tile);
}

int launch_ks_16_part(Problem p, hipStream_t s, int in_dtype, int tile) {
  return in_dtype == C3H_BF16 ? launch_ks_part<MmaBF16, bf16_t>(p, s, tile)
                              : launch_ks_part<MmaF16, f16_t>(p, s, tile);
}

}  // namespace gk
}  // namespace c3h
