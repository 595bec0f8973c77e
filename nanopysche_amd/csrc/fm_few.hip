// Grouped BF16 GEMM for few tokens per expert (a decoding step, a short
// prompt): out[r] = tokens[r] W_e^T for the rows of each expert's group.
//
// What bounds it is streaming the weights of the experts that have tokens, once,
// from memory.  The 256 x 256 tile of fm_gemm.hip gives such a launch too few
// workgroups (88 for 8 experts of 2816 x 2048 rows) and each of them a chain of
// K steps whose loads come two at a time.  Here a workgroup owns 64 weight rows
// of one expert and its 4 waves a quarter of K each, with the loads of two
// 64-deep steps in flight a wave; a wave's step goes through LDS of its own (no
// barrier in the loop) into 16x16x32 MFMA fragments, weights on the row side, 32 tokens at a
// time.  The four partial sums meet in LDS in wave order.
//
// Measured (MI355X, 16 tokens top-2 over 8 experts, captured): gate|up [2816, 2048]
// 41 -> 17.7 us, down [2048, 1408] 29 -> 11.1 us (92 and 46 MB of weights: 5.2 and
// 4.2 TB/s).
#include <type_traits>

#include "fm_common.h"
#include "../../include/fm_hip.h"

namespace fm {

constexpr int kFewRows = 64;     // weight rows of a workgroup
constexpr int kFewTokens = 32;   // tokens of a pass

struct FewArgs {
  const uint16_t* x;       // [rows, ld_x] tokens, expert groups from offsets
  int64_t ld_x;
  const uint16_t* w;       // [E] matrices, pitch ld_w, stride gs: [N][K], or (NN) [K][N]
  const uint16_t* w2;      // rows (NN: K rows) from `split` on, or = w
  int64_t split;
  int64_t ld_w, gs;
  const int32_t* counts;   // [E] rows that hold a token
  const int32_t* offsets;  // [E + 1] group starts
  int64_t N, K, chunk;     // chunk: K of a wave, a multiple of 64
  void* out;               // [rows, ld_out] bf16 or fp32
  int64_t ld_out;
  int out_f32;
  int blocks;              // N / 64
};

template <bool NN>
__global__ __launch_bounds__(256, 2) void few_gemm_kernel(FewArgs a) {
  constexpr int kW = kFewRows * 128, kX = kFewTokens * 128;   // bytes of a wave's step
  __shared__ __attribute__((aligned(16))) uint8_t lds[4][kW + kX];
  const int lane = threadIdx.x & 63, m = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int e = int(blockIdx.x) / a.blocks;
  const int64_t n0 = int64_t(int(blockIdx.x) - e * a.blocks) * kFewRows;
  const int n_e = a.counts[e];
  const int64_t r0 = a.offsets[e], r1 = a.offsets[e + 1];
  uint8_t* mine = lds[wave];
  const int64_t k0 = wave * a.chunk, k1 = k0 + a.chunk < a.K ? k0 + a.chunk : a.K;
  const int lr = lane >> 3, lc = lane & 7;   // staging: 16 bytes lc of row 8 j + lr

  // weights: [N][K] rows n0 + 8 j + lr (a 64-row block lies in one tensor), or K rows k + 8 j + lr
  const bool second = !NN && n0 >= a.split;
  const uint16_t* wb = (second ? a.w2 : a.w) + int64_t(e) * a.gs;
  const uint16_t* wb2 = a.w2 + int64_t(e) * a.gs - a.split * a.ld_w;   // NN: K rows from split on
  const int64_t nr = second ? n0 - a.split : n0;
  auto load_w = [&](fm_u32x4 (&v)[8], int64_t k) {   // k + 64 <= K: K and the chunks are multiples of 64
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint16_t* p;
      if constexpr (NN) p = (k >= a.split ? wb2 : wb) + (k + 8 * j + lr) * a.ld_w + n0 + 8 * lc;
      else p = wb + (nr + 8 * j + lr) * a.ld_w + k + 8 * lc;
      v[j] = *reinterpret_cast<const fm_u32x4*>(p);
    }
  };
  auto stage_w = [&](const fm_u32x4 (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = 8 * j + lr;
      // [N][K]: chunk ^ (r / 2 % 8); [K][N]: the 32-byte pieces ^ (r / 2 % 2 + 2 (r / 8 % 2)),
      // so the rows that one pass of a read touches fall on distinct banks
      const int c = NN ? lc ^ (((r >> 1) & 1) * 2 + ((r >> 3) & 1) * 4) : lc ^ ((r >> 1) & 7);
      *reinterpret_cast<fm_u32x4*>(mine + r * 128 + c * 16) = v[j];
    }
  };
  // fragment f, half h of the step: row 16 f + m, columns 32 h + 8 q .. + 8
  auto frag_w = [&](int f, int h) {
    if constexpr (NN) {
      const int r = 32 * h + 8 * q + (m >> 2);   // lane 4 i + p of a transposing read: K row i, columns 4 p .. + 4
      const int s = ((r >> 1) & 1) * 2 + ((r >> 3) & 1) * 4;
      const uint8_t* p = mine + r * 128 + ((2 * f + ((m & 3) >> 1)) ^ s) * 16 + (m & 1) * 8;
      typedef __attribute__((address_space(3))) v4s16 lds_v4;
      const v4s16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)p);
      const v4s16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(p + 4 * 128));
      return __builtin_bit_cast(v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      const int r = 16 * f + m;
      return *reinterpret_cast<const v8bf*>(mine + r * 128 + (((4 * h + q) ^ (r >> 1)) & 7) * 16);
    }
  };

  auto pass = [&](auto fragments, int t0) {
    constexpr int TF = decltype(fragments)::value;   // fragments of 16 tokens
    const uint16_t* xr[2 * TF];
#pragma unroll
    for (int j = 0; j < 2 * TF; ++j) {
      const int t = t0 + 8 * j + lr;
      xr[j] = a.x + (r0 + (t < n_e ? t : n_e - 1)) * a.ld_x + 8 * lc;
    }
    auto load_x = [&](fm_u32x4 (&v)[2 * TF], int64_t k) {
#pragma unroll
      for (int j = 0; j < 2 * TF; ++j) v[j] = *reinterpret_cast<const fm_u32x4*>(xr[j] + k);
    };
    auto stage_x = [&](const fm_u32x4 (&v)[2 * TF]) {
#pragma unroll
      for (int j = 0; j < 2 * TF; ++j) {
        const int r = 8 * j + lr;
        *reinterpret_cast<fm_u32x4*>(mine + kW + r * 128 + ((lc ^ (r >> 1)) & 7) * 16) = v[j];
      }
    };
    v4f acc[4][TF];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int t = 0; t < TF; ++t) acc[f][t] = v4f{0.f, 0.f, 0.f, 0.f};
    auto compute = [&]() {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v8bf xf[TF];
#pragma unroll
        for (int t = 0; t < TF; ++t) {
          const int r = 16 * t + m;
          xf[t] = *reinterpret_cast<const v8bf*>(mine + kW + r * 128 + (((4 * h + q) ^ (r >> 1)) & 7) * 16);
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const v8bf wf = frag_w(f, h);
#pragma unroll
          for (int t = 0; t < TF; ++t)
            acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[t], acc[f][t], 0, 0, 0);
        }
      }
    };
    fm_u32x4 wa[8], wc[8], xa[2 * TF], xc[2 * TF];
    // loads past the chunk re-read a step inside K and are not staged (a load
    // under a condition keeps these arrays out of the registers)
    auto load = [&](fm_u32x4 (&w)[8], fm_u32x4 (&x)[2 * TF], int64_t k) {
      k = k < a.K - 64 ? k : a.K - 64;
      load_w(w, k);
      load_x(x, k);
    };
    load(wa, xa, k0);
    load(wc, xc, k0 + 64);
    for (int64_t k = k0; k < k1; k += 128) {
      stage_w(wa);
      stage_x(xa);
      load(wa, xa, k + 128);
      compute();
      if (k + 64 >= k1) break;
      stage_w(wc);
      stage_x(xc);
      load(wc, xc, k + 192);
      compute();
    }
    // the waves' sums: [token][64 rows + 4] floats each, over the staging
    constexpr int kPitch = kFewRows + 4;
    static_assert(kFewTokens * kPitch * 4 <= kW + kX, "the sums fit the wave's staging");
    float* red = reinterpret_cast<float*>(mine);
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int t = 0; t < TF; ++t) *reinterpret_cast<v4f*>(red + (16 * t + m) * kPitch + 16 * f + 4 * q) = acc[f][t];
    __syncthreads();
    if (int(threadIdx.x) < 128 * TF) {
      const int t = threadIdx.x >> 3, c = (threadIdx.x & 7) * 8;
      float v[8];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float* p = reinterpret_cast<const float*>(lds[w]) + t * kPitch + c;
        const v4f lo = *reinterpret_cast<const v4f*>(p), hi = *reinterpret_cast<const v4f*>(p + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = w == 0 ? lo[j] : v[j] + lo[j];
          v[4 + j] = w == 0 ? hi[j] : v[4 + j] + hi[j];
        }
      }
      if (t0 + t < n_e) {
        const int64_t o = (r0 + t0 + t) * a.ld_out + n0 + c;
        if (a.out_f32) {
          float* d = static_cast<float*>(a.out) + o;
          st_global(d, make_float4(v[0], v[1], v[2], v[3]));
          st_global(d + 4, make_float4(v[4], v[5], v[6], v[7]));
        } else {
          st_global(static_cast<uint16_t*>(a.out) + o,
                    make_uint4(hw_bf16x2(v[0], v[1]), hw_bf16x2(v[2], v[3]), hw_bf16x2(v[4], v[5]), hw_bf16x2(v[6], v[7])));
        }
      }
    }
    __syncthreads();   // the sums are read before the next pass's staging
  };
  for (int t0 = 0; t0 < n_e; t0 += kFewTokens) {
    if (t0 + 16 < n_e) pass(std::integral_constant<int, 2>{}, t0);
    else pass(std::integral_constant<int, 1>{}, t0);
  }
  // the group's padding rows, as the product of zero rows
  for (int64_t r = r0 + n_e + (threadIdx.x >> 3); r < r1; r += 32) {
    const int64_t o = r * a.ld_out + n0 + (threadIdx.x & 7) * 8;
    if (a.out_f32) {
      float* d = static_cast<float*>(a.out) + o;
      st_global(d, make_float4(0.f, 0.f, 0.f, 0.f));
      st_global(d + 4, make_float4(0.f, 0.f, 0.f, 0.f));
    } else {
      st_global(static_cast<uint16_t*>(a.out) + o, make_uint4(0, 0, 0, 0));
    }
  }
}

}  // namespace fm

using namespace fm;

extern "C" {

int fm_grouped_gemm_few(const FmGemmOperand* tokens, const FmGemmOperand* weights, int weights_kn,
                        const int32_t* counts, const int32_t* offsets, int E, int64_t N, int64_t K, void* out,
                        int out_dtype, int64_t ld_out, void* stream) {
  FM_REQUIRE(tokens && weights && tokens->data && weights->data && counts && offsets && out,
             "fm_grouped_gemm_few: null pointer");
  FM_REQUIRE(E >= 1 && N > 0 && N % 64 == 0 && K > 0 && K % 64 == 0 && int64_t(E) * (N / 64) < (int64_t(1) << 31),
             "fm_grouped_gemm_few: N and K must be positive multiples of 64 (got %lld x %lld)", (long long)N,
             (long long)K);
  FM_REQUIRE(tokens->ld >= K && tokens->ld % 8 == 0 && weights->ld >= (weights_kn ? N : K) && weights->ld % 8 == 0,
             "fm_grouped_gemm_few: operand pitches must cover a row and be multiples of 8");
  FM_REQUIRE(weights->group_stride % 8 == 0 && tokens->data2 == nullptr && aligned16(tokens->data) &&
                 aligned16(weights->data) && aligned16(weights->data2) && aligned16(out),
             "fm_grouped_gemm_few: operands and output must be 16-byte aligned, tokens unsplit");
  FM_REQUIRE(weights->data2 == nullptr || (weights->split_rows > 0 && weights->split_rows % 64 == 0 &&
                                           weights->split_rows < (weights_kn ? K : N)),
             "fm_grouped_gemm_few: the split must be a multiple of 64 inside N ([K][N] weights: K)");
  FM_REQUIRE(out_dtype == FM_DTYPE_BF16 || out_dtype == FM_DTYPE_F32, "fm_grouped_gemm_few: bad out dtype");
  FM_REQUIRE(ld_out >= N && ld_out % 8 == 0, "fm_grouped_gemm_few: output pitch must be >= N and a multiple of 8");
  const int64_t split = weights->data2 ? weights->split_rows : INT64_MAX / 4 / (weights->ld > 0 ? weights->ld : 1);
  const uint16_t* w = static_cast<const uint16_t*>(weights->data);
  const FewArgs a{static_cast<const uint16_t*>(tokens->data), tokens->ld, w,
                  weights->data2 ? static_cast<const uint16_t*>(weights->data2) : w, split, weights->ld,
                  weights->group_stride, counts, offsets, N, K, (K / 64 + 3) / 4 * 64, out, ld_out,
                  out_dtype == FM_DTYPE_F32, int(N / 64)};
  const dim3 grid(unsigned(E * (N / 64))), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (weights_kn) hipLaunchKernelGGL(few_gemm_kernel<true>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(few_gemm_kernel<false>, grid, block, 0, s, a);
  return check_launch("fm_grouped_gemm_few");
}

}  // extern "C"
