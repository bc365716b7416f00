#pragma once
// GEMMs with few output tiles: a workgroup computes one small tile, its KW
// waves each taking every KW-th K tile, and the waves' partial tiles are
// summed in LDS (in wave order, so results are deterministic) before the
// common epilogue.
//
// What bounds these shapes is latency and one CU's operand rate: the 128 x
// 128 tiles of a GEMM of a few hundred rows occupy a handful of CUs, each
// walking all of K alone.  Small tiles spread the output over the chip and
// the K split over the waves of a workgroup shortens each one's walk, with
// no fp32 partials in memory and no second launch.  No operand is shared
// between the waves: each moves its own K tiles to its own LDS stages
// (buffer_load ... lds, 8 rows x 128 bytes per instruction) and the main loop
// has no barrier.  (Loading the MFMA fragments straight into registers reads
// 16 rows x 64 bytes per instruction with neighbouring lanes in different
// rows, which the CU takes at 16 B/clk against 54 B/clk for the DMA.)
#include "gemm_kernels.h"

namespace c3h {
namespace gk {

// Columns n .. n + 3 of row m, n < p.n: the accumulators v (int32 bits for
// int8 operands) through the scale / quantization and the epilogue into out.
// wide: all four columns exist and the row's vectors are aligned.
template <typename Mma, typename TO>
__device__ __forceinline__ void ks_finish4(const float4 acc4, int64_t m, int64_t n, bool wide, TO* out, const TO* resp,
                                           const QuantDiv& qd) {
  const KArg<Problem>& p = kernel_arg<Problem>();
  const float acc[4] = {acc4.x, acc4.y, acc4.z, acc4.w};
  const int64_t o = m * p.ldo + n;
  const int cols = wide ? 4 : static_cast<int>(min(static_cast<int64_t>(4), p.n - n));
  if constexpr (std::is_same<TO, int32_t>::value) {
    if (wide) {
      *reinterpret_cast<float4*>(out + o) = acc4;
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < cols) out[o + c] = __float_as_int(acc[c]);
    }
  } else {
    float res[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!std::is_same<TO, int8_t>::value) {
      if (resp && wide) {
        Elem<TO>::load4(resp + o, res);
      } else if (resp) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c < cols) res[c] = Elem<TO>::to_f32(resp[o + c]);
      }
    }
    float v[4];
    int8_t code[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      v[c] = 0.0f;
      code[c] = 0;
      if (c < cols) {
        if constexpr (Mma::kInt) {
          // the arithmetic of store_strip_q
          const int mode = p.qmode;
          const float sa = p.a_scale, sy = p.y_scale, zy = static_cast<float>(p.y_zero);
          const bool requant = mode == 1 || mode == 3;
          const float mult = requant ? (sa * p.b_scale[n + c]) / sy : sa * p.b_scale[n + c];
          v[c] = static_cast<float>(__float_as_int(acc[c])) * mult;
          if (requant) {
            const float y = fminf(fmaxf(rintf(v[c]) + zy, -128.0f), 127.0f);
            v[c] = mode == 1 ? y : (y - zy) * sy;
          }
          if (mode >= 2) v[c] = apply_epilogue(p.epi, v[c], m, n + c, p.n, res[c], 0);
          if constexpr (std::is_same<TO, int8_t>::value)
            code[c] = mode == 1 ? static_cast<int8_t>(v[c]) : qd.code(round_to_dtype(v[c], p.act_dtype), p.q_zero);
        } else {
          v[c] = acc[c];
          if constexpr (Mma::kScaled) v[c] = (v[c] * p.a_rows[m]) * p.b_scale[n + c];
          v[c] = apply_epilogue(p.epi, v[c], m, n + c, p.n, res[c], 0);
        }
      }
    }
    if constexpr (std::is_same<TO, int8_t>::value) {
      if (wide) {
        uint32_t w = 0u;
#pragma unroll
        for (int c = 0; c < 4; ++c) w |= (static_cast<uint32_t>(code[c]) & 0xffu) << (8 * c);
        *reinterpret_cast<uint32_t*>(out + o) = w;
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c < cols) out[o + c] = code[c];
      }
    } else if (wide) {
      Elem<TO>::store4(out + o, v);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < cols) out[o + c] = Elem<TO>::from_f32(v[c]);
    }
  }
}

template <typename Mma, typename TO, int AM, int BM, int BN, int KW>
__global__ void __launch_bounds__(KW * 64) gemm_ks_kernel(Problem p) {
  constexpr int ES = Mma::ES, VE = 16 / ES, BK = 128 / ES;
  constexpr int TM = BM / 16, TN = BN / 16, KS = 8 / Mma::kStep;
  constexpr int GR = (BM + BN) / 8;  // 8-row DMA loads per K tile
  constexpr int S = 2, STAGE = (BM + BN) * 128;
  constexpr int SS = BN + 4;
  constexpr int kSum = KW * BM * SS * 4, kOps = KW * S * STAGE;
  typedef typename Mma::vec vec;
  typedef typename Mma::acc_t acc_t;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kSum > kOps ? kSum : kOps];

  int tm, tn;
  tile_coords_grouped(p, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, lg = lane >> 4;

  const __amdgpu_buffer_rsrc_t rs_a = make_rsrc(p.a, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rs_b = make_rsrc(p.b, p.b_bytes);
  // Byte offset of this lane's row of each load at K = 0 (A and B below 2^31
  // bytes: host check).  Rows past M / N start at kOobOffset, chunks past K
  // add it: either way the load writes zeros.  (Both at once wrap to a small
  // offset: such a value meets only outputs past the edge.)  Conv rows start
  // at tap (0, 0), which may lie in the padding (a negative offset), and keep
  // their input coordinates; rows past M get a coordinate no tap brings into
  // the image.
  const int chunk = (lane & 7) ^ (lane >> 3);  // the K chunk the XOR swizzle puts at this lane's slot
  uint32_t row_off[GR];
  int row_hi[BM / 8], row_wi[BM / 8];
#pragma unroll
  for (int g = 0; g < GR; ++g) {
    const int r = g * 8 + (lane >> 3);
    if (g >= BM / 8) {
      row_off[g] = n0 + r - BM < p.n ? static_cast<uint32_t>((n0 + r - BM) * p.ldb * ES) : kOobOffset;
    } else if (AM == kConvTap) {
      const ConvRow cr = conv_row(p, m0 + r);
      row_off[g] = static_cast<uint32_t>(
          static_cast<int32_t>((cr.base + (static_cast<int64_t>(cr.hi0) * p.cw + cr.wi0) * p.c_stride) * ES));
      row_hi[g] = cr.valid ? cr.hi0 : -0x40000000;
      row_wi[g] = cr.wi0;
    } else {
      row_off[g] = m0 + r < p.m ? static_cast<uint32_t>((m0 + r) * p.lda * ES) : kOobOffset;
    }
  }
  const int k_total = static_cast<int>(p.k);
  // Conv: the tap and channel of the next K tile to load (this wave's tiles
  // are KW apart, each inside one tap: c_pack is a multiple of BK).
  int t_kh = 0, t_kw = 0, t_c0 = 0;
  auto advance = [&](int channels) {
    t_c0 += channels;
    while (t_c0 >= p.c_pack) {
      t_c0 -= p.c_pack;
      if (++t_kw >= p.kw) {
        t_kw = 0;
        ++t_kh;
      }
    }
  };
  if (AM == kConvTap) advance(wave * BK);
  auto issue = [&](int kt, int st) {
    const uint32_t off = kt * BK + chunk * VE < k_total ? static_cast<uint32_t>(kt * 128 + chunk * 16) : kOobOffset;
    const int dh = t_kh * p.dh, dw = t_kw * p.dw;
    const int32_t tap = ((dh * p.cw + dw) * p.c_stride + t_c0) * ES + chunk * 16;
#pragma unroll
    for (int g = 0; g < GR; ++g) {
      const int dst = (wave * S + st) * STAGE + g * 1024;
      uint32_t voff = row_off[g] + off;
      if (g < BM / 8) {
        if (AM == kConvTap) {
          voff = kOobOffset;
          if (static_cast<unsigned>(row_hi[g] + dh) < static_cast<unsigned>(p.ch) &&
              static_cast<unsigned>(row_wi[g] + dw) < static_cast<unsigned>(p.cw))
            voff = row_off[g] + static_cast<uint32_t>(tap);
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (lds_void_ptr)(smem + dst), 16, voff, 0, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_b, (lds_void_ptr)(smem + dst), 16, voff, 0, 0, 0);
      }
    }
    if (AM == kConvTap) advance(KW * BK);
  };

  // This thread's four output columns (at most one such piece per thread).
  // For the common epilogue its operands -- residual, bias, E4M3 scales -- are
  // loaded here, ahead of the operands, so that no memory round trip is left
  // after the main loop.
  constexpr int NC = BN / 4;
  static_assert(BM * NC <= KW * 64, "one piece per thread");
  const int o_row = tid / NC, o_col = tid % NC * 4;
  const int64_t om = m0 + o_row, on = n0 + o_col;
  const bool o_live = tid < BM * NC && om < p.m && on < p.n;
  TO* out = static_cast<TO*>(p.out);
  const TO* resp = static_cast<const TO*>(p.epi.residual);
  constexpr uintptr_t kA = 4 * sizeof(TO) - 1;
  const bool vec_ok = p.ldo % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & kA) == 0 &&
                      (reinterpret_cast<uintptr_t>(resp) & kA) == 0;
  const bool wide = vec_ok && on + 4 <= p.n;
  const bool simple = !Mma::kInt && wide && epilogue_is_simple(kernel_arg<Problem>(), vec_ok, true);
  float res[4] = {0.f, 0.f, 0.f, 0.f}, row_scale = 1.0f;
  float4 bias4 = make_float4(0.f, 0.f, 0.f, 0.f), col_scale = make_float4(1.f, 1.f, 1.f, 1.f);
  if constexpr (!Mma::kInt) {
    if (o_live && simple) {
      if (resp) Elem<TO>::load4(resp + om * p.ldo + on, res);
      if (p.epi.bias_mode == 2) bias4 = *reinterpret_cast<const float4*>(static_cast<const float*>(p.epi.bias) + on);
      if constexpr (Mma::kScaled) {
        row_scale = p.a_rows[om];
        col_scale = *reinterpret_cast<const float4*>(p.b_scale + on);
      }
    }
  }

  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  // This wave's K tiles: wave, wave + KW, ...
  const int nkt = (k_total + BK - 1) / BK;
  const int rounds = wave < nkt ? (nkt - wave + KW - 1) / KW : 0;
  if (rounds > 0) issue(wave, 0);
  if (rounds > 1) issue(wave + KW, 1);
  for (int r = 0; r < rounds; ++r) {
    if (r + 1 < rounds) wait_vmcnt<GR>();
    else wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    const uint8_t* As = smem + (wave * S + (r & 1)) * STAGE;
    const uint8_t* Bs = As + BM * 128;
    vec av[KS][TM], bv[KS][TN];
#pragma unroll
    for (int q = 0; q < KS; ++q) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
        av[q][i] = read_operand<Mma>(As + (16 * i + l16) * 128, 16 * i + l16, q * Mma::kStep, lg);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        bv[q][j] = read_operand<Mma>(Bs + (16 * j + l16) * 128, 16 * j + l16, q * Mma::kStep, lg);
    }
    if (r + S < rounds) {
      wait_lgkmcnt0();  // the fragments are in registers: the stage may be refilled
      asm volatile("" ::: "memory");
      issue(wave + KW * (r + S), r & 1);
    }
#pragma unroll
    for (int q = 0; q < KS; ++q) mma_step<Mma, TM, TN>(acc, av[q], bv[q]);
  }

  // The waves' partial tiles, summed in wave order.
  __syncthreads();  // every wave is done with its stages
  float* stage = reinterpret_cast<float*>(smem);
  float* part = stage + wave * BM * SS;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *reinterpret_cast<float4*>(part + (16 * i + l16) * SS + 16 * j + 4 * lg) =
          __builtin_bit_cast(float4, acc[i][j]);  // C^T accumulators: row l16, columns 4 lg + r
  __syncthreads();
  if (!o_live) return;
  const float* src = stage + o_row * SS + o_col;
  float4 v = *reinterpret_cast<const float4*>(src);
#pragma unroll
  for (int w = 1; w < KW; ++w) {
    const float4 u = *reinterpret_cast<const float4*>(src + w * BM * SS);
    if constexpr (Mma::kInt) {
      v = float4{__int_as_float(__float_as_int(v.x) + __float_as_int(u.x)),
                 __int_as_float(__float_as_int(v.y) + __float_as_int(u.y)),
                 __int_as_float(__float_as_int(v.z) + __float_as_int(u.z)),
                 __int_as_float(__float_as_int(v.w) + __float_as_int(u.w))};
    } else {
      v = float4{v.x + u.x, v.y + u.y, v.z + u.z, v.w + u.w};
    }
  }
  if constexpr (!Mma::kInt) {
    if (simple) {  // ((acc + bias) + residual), then the activation: apply_epilogue's arithmetic
      const float acc4[4] = {v.x, v.y, v.z, v.w}, b4[4] = {bias4.x, bias4.y, bias4.z, bias4.w};
      const float s4[4] = {col_scale.x, col_scale.y, col_scale.z, col_scale.w};
      const int act = p.epi.act;
      const float c0 = p.epi.imm[0], c1 = p.epi.imm[1], c2 = p.epi.imm[2];
      const bool gstd = gelu_std_ok(c0, c1, c2);
      float y[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float t = ((Mma::kScaled ? (acc4[c] * row_scale) * s4[c] : acc4[c]) + b4[c]) + res[c];
        y[c] = act == 1 ? fmaxf(t, 0.0f) : act == 2 ? gelu_act(t, c0, c1, c2, gstd) : t;
      }
      Elem<TO>::store4(out + om * p.ldo + on, y);
      return;
    }
  }
  const QuantDiv qd(Mma::kInt ? p.q_scale : 1.0f);
  ks_finish4<Mma, TO>(v, om, on, wide, out, resp, qd);
}

// Tiles of launch_ks_*: 1 = 16 x 32 with eight waves, 2 = 32 x 32 with four.
template <typename Mma, typename TO, int AM>
int launch_ks_tile(Problem p, hipStream_t s, int tile, const char* what) {
  dim3 grid;
  if (tile == 1) {
    grid_of<16, 32>(p, 1, grid);
    hipLaunchKernelGGL((gemm_ks_kernel<Mma, TO, AM, 16, 32, 8>), grid, dim3(512), 0, s, p);
  } else {
    grid_of<32, 32>(p, 1, grid);
    hipLaunchKernelGGL((gemm_ks_kernel<Mma, TO, AM, 32, 32, 4>), grid, dim3(256), 0, s, p);
  }
  return launch_status(what);
}

}  // namespace gk
}  // namespace c3h
