#pragma once
// GEMMs and convs with few output tiles: a workgroup computes one small tile
// (16 x 32 or 32 x 32).
//
// What bounds these shapes is latency and one CU's operand rate: the 128 x
// 128 tiles of a GEMM of a few hundred rows occupy a handful of CUs, each
// walking all of K alone.  Small tiles spread the output over the chip.  Two
// kernels:
//
// gemm_ordered_kernel (bf16, fp16, E4M3): each output has one accumulator that
//   takes K in order, so its sums are those of every larger tile, bit for
//   bit: a row's result does not depend on how many rows the call has.
// gemm_ks_kernel (fp32, int8): the waves split K -- each takes every KW-th K
//   tile through its own LDS stages, with no barrier in the main loop -- and
//   their partial tiles are summed in LDS in wave order (deterministic).  The
//   fp32 MFMA is 16 times slower than the 16-bit one, so one wave's chain
//   over all of K would be the whole time; int8 sums are exact in any order.
//
// The fp32 sums of a call therefore depend on the tile its shape selects.
//
// Both load by buffer_load ... lds, 8 rows x 128 bytes per instruction.
// (Loading the MFMA fragments straight into registers reads 16 rows x 64
// bytes per instruction with neighbouring lanes in different rows, which the
// CU takes at 16 B/clk against 54 B/clk for the DMA.)
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

// Four output columns of one row: for the common epilogue the operands --
// residual, bias, E4M3 scales -- are loaded ahead of the K walk, so that no
// memory round trip is left after it.
template <typename Mma, typename TO>
struct OutPiece {
  int64_t m, n;
  bool live, wide, simple;
  TO* out;
  const TO* resp;
  float res[4] = {0.f, 0.f, 0.f, 0.f}, row_scale = 1.0f;
  float4 bias4 = make_float4(0.f, 0.f, 0.f, 0.f), col_scale = make_float4(1.f, 1.f, 1.f, 1.f);

  __device__ __forceinline__ void load(int64_t row, int64_t col, bool mine) {
    m = row;
    n = col;
    const KArg<Problem>& p = kernel_arg<Problem>();
    constexpr uintptr_t kA = 4 * sizeof(TO) - 1;
    live = mine && m < p.m && n < p.n;
    out = static_cast<TO*>(p.out);
    resp = static_cast<const TO*>(p.epi.residual);
    const bool vec_ok = p.ldo % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & kA) == 0 &&
                        (reinterpret_cast<uintptr_t>(resp) & kA) == 0;
    wide = vec_ok && n + 4 <= p.n;
    simple = !Mma::kInt && wide && epilogue_is_simple(p, vec_ok, true);
    if constexpr (!Mma::kInt) {
      if (live && simple) {
        if (resp) Elem<TO>::load4(resp + m * p.ldo + n, res);
        if (p.epi.bias_mode == 2) bias4 = *reinterpret_cast<const float4*>(static_cast<const float*>(p.epi.bias) + n);
        if constexpr (Mma::kScaled) {
          row_scale = p.a_rows[m];
          col_scale = *reinterpret_cast<const float4*>(p.b_scale + n);
        }
      }
    }
  }

  __device__ __forceinline__ void finish(const float4 v) const {
    // No contraction: the E4M3 scales' product is rounded before the bias is
    // added, as in the larger tiles.
#pragma clang fp contract(off)
    const KArg<Problem>& p = kernel_arg<Problem>();
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
        Elem<TO>::store4(out + m * p.ldo + n, y);
        return;
      }
    }
    const QuantDiv qd(Mma::kInt ? p.q_scale : 1.0f);
    ks_finish4<Mma, TO>(v, m, n, wide, out, resp, qd);
  }
};

// N of the 8-row loads of a BM x BN tile's K tiles, from load G0 on (load g:
// rows 8 g .. + 7 of A then B), for K tiles that `issue` names in steps of a
// constant number.
template <typename Mma, int AM, int BM, int N, int G0 = 0>
struct TileLoads {
  static constexpr int ES = Mma::ES, VE = 16 / ES, BK = 128 / ES;
  // Byte offset of this lane's row of each load at K = 0 (A and B below 2^31
  // bytes: host check).  Rows past M / N start at kOobOffset, chunks past K
  // add it: either way the load writes zeros.  (Both at once wrap to a small
  // offset: such a value meets only outputs past the edge.)  Conv rows start
  // at tap (0, 0), which may lie in the padding (a negative offset), and keep
  // their input coordinates; rows past M get a coordinate no tap brings into
  // the image.
  uint32_t row_off[N];
  int row_hi[N], row_wi[N];
  int chunk, k_total;
  // Conv: the tap and channel of the next K tile to load (each K tile lies
  // inside one tap: c_pack is a multiple of BK).
  int t_kh = 0, t_kw = 0, t_c0 = 0;

  // first: the index of the first K tile to be issued.
  __device__ __forceinline__ TileLoads(const Problem& p, int64_t m0, int64_t n0, int lane, int first) {
    chunk = (lane & 7) ^ (lane >> 3);  // the K chunk the XOR swizzle puts at this lane's slot
    k_total = static_cast<int>(p.k);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int g = G0 + j, r = g * 8 + (lane >> 3);
      row_hi[j] = row_wi[j] = 0;
      if (g >= BM / 8) {
        row_off[j] = n0 + r - BM < p.n ? static_cast<uint32_t>((n0 + r - BM) * p.ldb * ES) : kOobOffset;
      } else if (AM == kConvTap) {
        const ConvRow cr = conv_row(p, m0 + r);
        row_off[j] = static_cast<uint32_t>(
            static_cast<int32_t>((cr.base + (static_cast<int64_t>(cr.hi0) * p.cw + cr.wi0) * p.c_stride) * ES));
        row_hi[j] = cr.valid ? cr.hi0 : -0x40000000;
        row_wi[j] = cr.wi0;
      } else {
        row_off[j] = m0 + r < p.m ? static_cast<uint32_t>((m0 + r) * p.lda * ES) : kOobOffset;
      }
    }
    if (AM == kConvTap) advance(p, first * BK);
  }

  __device__ __forceinline__ void advance(const Problem& p, int channels) {
    t_c0 += channels;
    while (t_c0 >= p.c_pack) {
      t_c0 -= p.c_pack;
      if (++t_kw >= p.kw) {
        t_kw = 0;
        ++t_kh;
      }
    }
  }

  // K tile kt into the stage at dst; the next call is for tile kt + step.
  // Chunks past K write zeros; a conv's K is whole K tiles, and what a tile
  // past them writes (other input or weights, or zeros) is never multiplied.
  __device__ __forceinline__ void issue(const Problem& p, __amdgpu_buffer_rsrc_t rs_a, __amdgpu_buffer_rsrc_t rs_b,
                                        uint8_t* dst, int kt, int step) {
    // (No test of K for convs: it put branches between their loads, 5 to 10 %
    // of a 32 x 32 tile's time in fp32.)
    const bool k_ok = AM == kConvTap || kt * BK + chunk * VE < k_total;
    const uint32_t off = k_ok ? static_cast<uint32_t>(kt * 128 + chunk * 16) : kOobOffset;
    const int dh = t_kh * p.dh, dw = t_kw * p.dw;
    const int32_t tap = ((dh * p.cw + dw) * p.c_stride + t_c0) * ES + chunk * 16;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      constexpr int kA = BM / 8 - G0;  // loads of A
      const int g = G0 + j;
      uint32_t voff = row_off[j] + off;
      if (j < kA) {
        if (AM == kConvTap) {
          voff = kOobOffset;
          if (static_cast<unsigned>(row_hi[j] + dh) < static_cast<unsigned>(p.ch) &&
              static_cast<unsigned>(row_wi[j] + dw) < static_cast<unsigned>(p.cw))
            voff = row_off[j] + static_cast<uint32_t>(tap);
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (lds_void_ptr)(dst + g * 1024), 16, voff, 0, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_b, (lds_void_ptr)(dst + g * 1024), 16, voff, 0, 0, 0);
      }
    }
    if (AM == kConvTap) advance(p, step * BK);
  }
};

// OM x ON waves own a (BM / OM) x (BN / ON) piece of the tile each and take
// the K tiles in order into its accumulators; NL more waves only load, G K
// tiles a round through S LDS stages.  One barrier per round: an owner reads
// the next round's fragments under the MFMAs of this one's while the loaders
// refill the stage before.  (Owners that also load stall on the issue of
// their loads behind the CU's other loads, with their LDS reads after it: a
// K tile then took 270 clocks in place of 120.)  PART: the accumulators are
// added to a total and restarted after every p.k_part of K -- the fp32
// partials and the ordered sum of a split-K GEMM (splitk_reduce_kernel),
// with neither in memory.
template <typename Mma, typename TO, int AM, int BM, int BN, int OM, int ON, int NL, int G, int S, bool PART>
__global__ void __launch_bounds__((OM * ON + NL) * 64) gemm_ordered_kernel(Problem p) {
  constexpr int BK = 128 / Mma::ES, KS = 8 / Mma::kStep;
  constexpr int TM = BM / OM / 16, TN = BN / ON / 16;
  constexpr int WPT = NL / G, LPW = (BM + BN) / 8 / WPT;  // loaders per K tile, loads per loader and round
  constexpr int TILE = (BM + BN) * 128, STAGE = G * TILE;
  static_assert(NL % G == 0 && (BM + BN) / 8 % WPT == 0, "shape");
  static_assert(S >= 2 && S <= 4 && LPW * (S - 1) < 64, "vmcnt range");
  typedef typename Mma::vec vec;
  typedef typename Mma::acc_t acc_t;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[S * STAGE];

  int tm, tn;
  tile_coords_grouped(p, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, lg = lane >> 4;
  const int nkt = static_cast<int>(ceil_div(p.k, BK)), rounds = (nkt + G - 1) / G;
  // rounds + 1 barriers on either side.
  auto barrier = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  if (wave >= OM * ON) {
    const __amdgpu_buffer_rsrc_t rs_a = make_rsrc(p.a, p.a_bytes);
    const __amdgpu_buffer_rsrc_t rs_b = make_rsrc(p.b, p.b_bytes);
    const int loader = wave - OM * ON, lt = loader / WPT;  // the K tile of a round this wave loads for
    // The loads of all but the `later` newest rounds have landed.
    auto landed = [](int later) { wait_vmcnt_groups<LPW>(later); };
    auto run = [&](auto part_c) {
      TileLoads<Mma, AM, BM, LPW, decltype(part_c)::value * LPW> loads(p, m0, n0, lane, lt);
      auto issue = [&](int round, int st) {
        loads.issue(p, rs_a, rs_b, smem + st * STAGE + lt * TILE, round * G + lt, G);
      };
#pragma unroll
      for (int st = 0; st < S; ++st)
        if (st < rounds) issue(st, st);
      landed(min(S - 1, rounds - 1));
      barrier();
      int st = 0;
      for (int r = 0; r < rounds; ++r) {
        landed(max(0, min(S - 2, rounds - 2 - r)));  // round r + 1
        barrier();                                   // every owner has read round r
        if (r + S < rounds) issue(r + S, st);
        st = st + 1 == S ? 0 : st + 1;
      }
    };
    static_assert(WPT <= 2, "loaders per K tile");
    if (WPT == 1 || loader % WPT == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, WPT - 1>{});
    return;
  }

  const int row0 = wave / ON * 16 * TM, col0 = wave % ON * 16 * TN;  // this wave's piece of the tile
  acc_t acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = acc_t{0, 0, 0, 0};
      total[i][j] = acc_t{-0.0f, -0.0f, -0.0f, -0.0f};  // -0 + x = x
    }
  int left = PART ? p.k_part / BK : 0;
  vec av[2][G][KS][TM], bv[2][G][KS][TN];
  auto read_frags = [&](auto set_c, int st) {
    constexpr int SET = decltype(set_c)::value;
    const uint8_t* base = smem + st * STAGE;
#pragma unroll
    for (int t = 0; t < G; ++t)
#pragma unroll
      for (int q = 0; q < KS; ++q) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int r = row0 + 16 * i + l16;
          av[SET][t][q][i] = read_operand<Mma>(base + t * TILE + r * 128, r, q * Mma::kStep, lg);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int r = col0 + 16 * j + l16;
          bv[SET][t][q][j] = read_operand<Mma>(base + t * TILE + (BM + r) * 128, r, q * Mma::kStep, lg);
        }
      }
  };
  auto mma_tile = [&](auto set_c, int t) {
    constexpr int SET = decltype(set_c)::value;
#pragma unroll
    for (int q = 0; q < KS; ++q) mma_step<Mma, TM, TN>(acc, av[SET][t][q], bv[SET][t][q]);
    if (PART && --left == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = acc_t{0, 0, 0, 0};
        }
      left = p.k_part / BK;
    }
  };
  OutPiece<Mma, TO> piece[TM][TN];  // C^T accumulators: row l16, columns 4 lg + r
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) piece[i][j].load(m0 + row0 + 16 * i + l16, n0 + col0 + 16 * j + 4 * lg, true);
  barrier();
  read_frags(std::integral_constant<int, 0>{}, 0);
  int st = 0;
  auto body = [&](auto set_c, int tiles) {
    constexpr int SET = decltype(set_c)::value;
    wait_lgkmcnt0();  // round r's fragments are in registers
    barrier();        // round r + 1 is in LDS
    st = st + 1 == S ? 0 : st + 1;
    // (past the last round: a stale, in-bounds stage into the unused set)
    read_frags(std::integral_constant<int, SET ^ 1>{}, st);
#pragma unroll
    for (int t = 0; t < G; ++t)
      if (t < tiles) mma_tile(set_c, t);
    __builtin_amdgcn_sched_barrier(0);
  };
  const std::integral_constant<int, 0> set0;
  const std::integral_constant<int, 1> set1;
  const int full = nkt / G, rest = nkt - full * G;
  int r = 0;
  for (; r + 1 < full; r += 2) {
    body(set0, G);
    body(set1, G);
  }
  if (r < full) {
    body(set0, G);
    if (rest) body(set1, rest);
  } else if (rest) {
    body(set0, rest);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      if (piece[i][j].live) piece[i][j].finish(__builtin_bit_cast(float4, PART ? total[i][j] : acc[i][j]));
}

// Tiles of launch_ordered_*: 1 = 16 x 32 (one workgroup per CU: the rule
// gives it no more; six loaders for convs, whose addresses cost more), 2 =
// 32 x 32 (three stages of 16 KB: three workgroups per CU).
// us, K split over the waves as in gemm_ks_kernel (other bits) / here:
// 1 x 512 x 512 3.4 / 3.1, 200 x 512 x 2048 4.7 / 4.5, 333 x 512 x 2048 5.5 /
// 5.5, 1000 x 512 x 2048 9.5 / 8.8, 1000 x 768 x 3072 16.3 / 15.9; 3x3 convs
// 1 x 7 x 7 x 512 6.3 / 6.9, 8 x 14 x 14 x 256 8.4 / 9.4, 16 x 7 x 7 x 512
// 14.5 / 15.5 -- and 128 x 128 tiles 8.6, 21.8, 21.9, 24.7, 35.1; 49.8, 26.5,
// 46.1.
template <typename Mma, typename TO, int AM, bool PART = false>
int launch_ordered_tile(Problem p, hipStream_t s, int tile, const char* what) {
  dim3 grid;
  if (tile == 1) {
    constexpr int NL = AM == kConvTap ? 6 : 4;
    grid_of<16, 32>(p, 1, grid);
    hipLaunchKernelGGL((gemm_ordered_kernel<Mma, TO, AM, 16, 32, 1, 2, NL, NL, 3, PART>), grid, dim3(64 * (2 + NL)), 0,
                       s, p);
  } else {
    grid_of<32, 32>(p, 1, grid);
    hipLaunchKernelGGL((gemm_ordered_kernel<Mma, TO, AM, 32, 32, 2, 2, 4, 2, 3, PART>), grid, dim3(512), 0, s, p);
  }
  return launch_status(what);
}

template <typename Mma, typename TO, int AM, int BM, int BN, int KW>
__global__ void __launch_bounds__(KW * 64) gemm_ks_kernel(Problem p) {
  constexpr int BK = 128 / Mma::ES;
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
  TileLoads<Mma, AM, BM, GR> loads(p, m0, n0, lane, wave);
  auto issue = [&](int kt, int st) { loads.issue(p, rs_a, rs_b, smem + (wave * S + st) * STAGE, kt, KW); };

  // This thread's four output columns (at most one such piece per thread).
  constexpr int NC = BN / 4;
  static_assert(BM * NC <= KW * 64, "one piece per thread");
  const int o_row = tid / NC, o_col = tid % NC * 4;
  OutPiece<Mma, TO> piece;
  piece.load(m0 + o_row, n0 + o_col, tid < BM * NC);

  // fp32: the four MFMAs of a 16-byte chunk sum apart.  One chain per wave
  // rounded K / KW terms in a row, which lost precision to the split-K this
  // kernel replaces (error against 64 bits, split-K / one chain / four, 1e-7:
  // 256 x 512 x 784 in 14 splits 1.54 / 1.87 / 1.14, 16 x 512 x 2048 in 64 1.79 / 2.88 / 1.59).
  constexpr int CH = std::is_same<Mma, MmaF32>::value ? 4 : 1;
  acc_t acc[CH][TM][TN];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[c][i][j] = acc_t{0, 0, 0, 0};

  // This wave's K tiles: wave, wave + KW, ...
  const int nkt = static_cast<int>(ceil_div(p.k, BK));
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
    for (int q = 0; q < KS; ++q) mma_chains<Mma, TM, TN>(acc, av[q], bv[q]);
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
          __builtin_bit_cast(float4, chain_sum<TM, TN>(acc, i, j));  // C^T accumulators: row l16, columns 4 lg + r
  __syncthreads();
  if (!piece.live) return;
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
  piece.finish(v);
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
