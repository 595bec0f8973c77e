// The router gate's three products on the matrix cores for bf16 x:
//   logits = x w^T        (gate_logits_kernel)
//   dx     = dlogits w    (gate_dx_kernel)
//   dw     = dlogits^T x  (gate_dw_kernel)
// with the fp32 operand of each (dlogits, an fp32 gate) as three bf16 pieces
// whose sum is the value exactly (8 + 8 + 8 mantissa bits), so every product
// is exact in the fp32 accumulator and the results are sums of exact products
// as on the VALU, in another order (fp32 within a chain of MFMAs, each section below
// says how the chains' sums are added).
//
// Non-finite values: the two low pieces of an infinity or a NaN are 0, and the
// low pieces' sum is dropped where it is not finite (an infinite factor on
// the other side times a zero low piece is NaN, where the value itself gives
// an infinity): the high pieces alone then give the class of the result.
//
// Measured on MI355X for [4096, 7168] bf16 x and a bf16 gate of 256 experts,
// against FMAs on the VALU (15 GFLOP a product, bound by their issue): logits
// 574 -> 49 us, gating + counts + loss 187 -> 29, dx 1167 -> 63, dw 380 -> 75, the pieces
// themselves 13.  What bounds them now: the logits x's read, the chunk sums'
// write and read (floor 10 us of HBM) and the joins of the MFMA chains' sums (10 us), dx
// and dw their 45 GFLOP of pieces at
// 0.7 PFLOP/s, fragments fetched from the L2.
#pragma once

#include "fm_common.h"

namespace fm {

__device__ __forceinline__ v4f mfma16(const uint4& a, const uint4& b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// v = h + m + l, each a bf16 (truncations; exact unless l is below bf16's
// subnormals); m = l = 0 for a non-finite v, a NaN stays one.
struct Pieces { uint32_t h, m, l; };   // bf16 bits in the high half
__device__ __forceinline__ Pieces split3(float v) {
  const uint32_t u = f2u(v);
  if ((u & 0x7f800000u) == 0x7f800000u)
    return Pieces{(u & 0x007fffffu) ? ((u & 0xffff0000u) | 0x00400000u) : u, 0u, 0u};
  const uint32_t h = u & 0xffff0000u;
  const float r = v - u2f(h);
  const uint32_t m = f2u(r) & 0xffff0000u;
  return Pieces{h, m, f2u(r - u2f(m)) & 0xffff0000u};
}
__device__ __forceinline__ uint32_t pack_hi(uint32_t lo, uint32_t hi) { return (lo >> 16) | (hi & 0xffff0000u); }
__device__ __forceinline__ void split3x8(const float (&v)[8], uint4& h, uint4& m, uint4& l) {
  Pieces p[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) p[i] = split3(v[i]);
  h = make_uint4(pack_hi(p[0].h, p[1].h), pack_hi(p[2].h, p[3].h), pack_hi(p[4].h, p[5].h), pack_hi(p[6].h, p[7].h));
  m = make_uint4(pack_hi(p[0].m, p[1].m), pack_hi(p[2].m, p[3].m), pack_hi(p[4].m, p[5].m), pack_hi(p[6].m, p[7].m));
  l = make_uint4(pack_hi(p[0].l, p[1].l), pack_hi(p[2].l, p[3].l), pack_hi(p[4].l, p[5].l), pack_hi(p[6].l, p[7].l));
}
__device__ __forceinline__ float finite_or_0(float v) { return fabsf(v) <= 3.40282347e38f ? v : 0.f; }

// ------------------------------------------------------------ logits ----
// One wave forms 16 TF tokens x 16 NF experts over one of S chunks of D, in
// steps of 64 columns: the step's rows come as whole 128-byte lines (8 rows an
// instruction) into registers one step ahead, then through LDS of the wave's own
// (no barrier; 16-byte chunk c of row r at c ^ (r / 2 % 8), so a fragment read has
// no bank conflict) into MFMA fragments.  (Fragments read straight from memory
// touch four lines per four lanes: 65 us for [4096, 7168] x 256 experts,
// bound by the L1's tag rate.)  Row i of expert fragment f stands for expert
// e0 + 4 NF (i / 4) + 4 f + i % 4, so a lane ends with 4 NF consecutive experts
// of one token.  The chunks' sums are added in chunk order in 64 bits, by the gating
// kernel (SPLIT: the chunk's sums go to part [S][T][ld_p]) or by this wave over all
// chunks (SPLIT false), with the same bits.
// The MFMA chains are short (gate_group_columns): a chain's sums join the chunk's
// with the remainder of that rounding carried into the next chain (compensated
// summation), where one chain a chunk and fp32 sums of the chunks were less exact
// than the FMAs' 64 lane sums.  Rms error against float64 in units of the logits',
// FMAs / one chain a chunk / now: bf16 gate, 16384 tokens, [1024] x 256 6.8e-8 /
// 1.3e-7 / 5.2e-8, [7168] x 256 9.5e-8 / 3.7e-7 / 6.6e-8, [7168] x 12 9.5e-8 / 1.8e-7 /
// 7.1e-8; fp32 gate, [7168] x 256 2.0e-7 / 5.3e-7 / 9.0e-8.
struct GateLogitsArgs {
  const uint16_t* x;     // bf16 [T, ld_x]
  int64_t ld_x, T, D;
  const void* w;         // [E, ld_w] bf16, or fp32 (W32)
  int64_t ld_w;
  const void* bias;      // [E] in w's dtype, or null
  const float* score_bias;
  int E;
  int64_t S, chunk;      // chunk: a multiple of 64
  int eg, tt;            // expert groups, token tiles
  int group;             // columns of an MFMA chain, less 64 (bits above 6)
  float* out;            // SPLIT: part [S][T][ld_o]; else logits [T, ld_o]
  int64_t ld_o;
};

template <int TF, int NF, bool W32, bool SPLIT>
__global__ __launch_bounds__(256, SPLIT ? 2 : 1) void gate_logits_kernel(GateLogitsArgs a) {
  constexpr int XR = 16 * TF, WR = 16 * NF * (W32 ? 2 : 1);   // 128-byte rows: tokens; experts (fp32: halves of 32 columns)
  __shared__ __attribute__((aligned(16))) uint8_t lds[4][(XR + WR) * 128];
  const int lane = threadIdx.x & 63, m = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int64_t wv = int64_t(blockIdx.x) * 4 + wave;
  const int g = int(wv % a.eg);
  const int64_t rest = wv / a.eg;
  const int64_t tile = rest % a.tt, s0 = SPLIT ? rest / a.tt : 0;
  if (SPLIT ? s0 >= a.S : rest >= a.tt) return;
  const int e0 = g * 16 * NF;
  uint8_t* mine = lds[wave];
  // staging: lane takes 16 bytes lc of row 8 j + lr
  const int lr = lane >> 3, lc = lane & 7;
  const uint16_t* xr[XR / 8];
  const uint8_t* wr[WR / 8];
#pragma unroll
  for (int j = 0; j < XR / 8; ++j) {
    const int64_t t = tile * XR + 8 * j + lr;
    xr[j] = a.x + (t < a.T ? t : a.T - 1) * a.ld_x + 8 * lc;
  }
#pragma unroll
  for (int j = 0; j < WR / 8; ++j) {
    const int r = 8 * j + lr, f = (W32 ? r >> 1 : r) >> 4, i = (W32 ? r >> 1 : r) & 15;
    int e = e0 + 4 * NF * (i >> 2) + 4 * f + (i & 3);
    e = e < a.E ? e : a.E - 1;
    wr[j] = W32 ? reinterpret_cast<const uint8_t*>(static_cast<const float*>(a.w) + e * a.ld_w + 32 * (r & 1) + 4 * lc)
                : reinterpret_cast<const uint8_t*>(static_cast<const uint16_t*>(a.w) + e * a.ld_w + 8 * lc);
  }
  uint4 xv[XR / 8], wx[WR / 8];
  // columns k .. k + 64 (zeros from k1 on; D is a multiple of 8, so a lane's 16 bytes are all in or all out)
  auto load = [&](int64_t k, int64_t k1) {
    const bool whole = k + 64 <= k1;
#pragma unroll
    for (int j = 0; j < XR / 8; ++j)
      xv[j] = whole || k + 8 * lc < k1 ? *reinterpret_cast<const uint4*>(xr[j] + k) : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < WR / 8; ++j) {
      const int64_t c = W32 ? k + 32 * ((8 * j + lr) & 1) + 4 * lc : k + 8 * lc;
      wx[j] = whole || c < k1 ? *reinterpret_cast<const uint4*>(wr[j] + k * (W32 ? 4 : 2)) : make_uint4(0, 0, 0, 0);
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int j = 0; j < XR / 8; ++j) {
      const int r = 8 * j + lr;
      *reinterpret_cast<uint4*>(mine + r * 128 + ((lc ^ (r >> 1)) & 7) * 16) = xv[j];
    }
#pragma unroll
    for (int j = 0; j < WR / 8; ++j) {
      const int r = 8 * j + lr;
      *reinterpret_cast<uint4*>(mine + (XR + r) * 128 + ((lc ^ (r >> (W32 ? 2 : 1))) & 7) * 16) = wx[j];
    }
  };
  auto frag_x = [&](int f, int h) {
    const int r = 16 * f + m;
    return *reinterpret_cast<const uint4*>(mine + r * 128 + (((4 * h + q) ^ (r >> 1)) & 7) * 16);
  };
  // fp32: columns 32 h + 8 q .. + 8 are chunks 2 q, 2 q + 1 of row half h
  auto frag_w = [&](int f, int h, int part) {
    const int e = 16 * f + m, r = W32 ? 2 * e + h : e;
    const int c = W32 ? 2 * q + part : 4 * h + q;
    return *reinterpret_cast<const uint4*>(mine + (XR + r) * 128 + ((c ^ (r >> (W32 ? 2 : 1))) & 7) * 16);
  };
  v4f tot[NF][TF];
  typedef double v4d __attribute__((ext_vector_type(4)));
  v4d all[SPLIT ? 1 : NF][SPLIT ? 1 : TF];   // the chunks' sums (topk_logits adds those of SPLIT, alike)
  for (int64_t s = s0; s < (SPLIT ? s0 + 1 : a.S); ++s) {
    const int64_t k0 = s * a.chunk, k1 = k0 + a.chunk < a.D ? k0 + a.chunk : a.D;
    v4f acc[NF][TF], low[W32 ? NF : 1][W32 ? TF : 1];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int t = 0; t < TF; ++t) {
        acc[f][t] = tot[f][t] = v4f{0.f, 0.f, 0.f, 0.f};
        if constexpr (W32) low[f][t] = v4f{0.f, 0.f, 0.f, 0.f};
      }
    load(k0, k1);
    for (int64_t k = k0; k < k1; k += 64) {
      stage();
      if (k + 64 < k1) load(k + 64, k1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint4 xf[TF];
#pragma unroll
        for (int t = 0; t < TF; ++t) xf[t] = frag_x(t, h);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          if constexpr (W32) {
            const uint4 w0 = frag_w(f, h, 0), w1 = frag_w(f, h, 1);
            const float v[8] = {u2f(w0.x), u2f(w0.y), u2f(w0.z), u2f(w0.w), u2f(w1.x), u2f(w1.y), u2f(w1.z), u2f(w1.w)};
            uint4 wh, wm, wl;
            split3x8(v, wh, wm, wl);
#pragma unroll
            for (int t = 0; t < TF; ++t) {
              low[f][t] = mfma16(wl, xf[t], low[f][t]);
              low[f][t] = mfma16(wm, xf[t], low[f][t]);
              acc[f][t] = mfma16(wh, xf[t], acc[f][t]);
            }
          } else {
            const uint4 wf = frag_w(f, h, 0);
#pragma unroll
            for (int t = 0; t < TF; ++t) acc[f][t] = mfma16(wf, xf[t], acc[f][t]);
          }
        }
      }
      // the chain's sums into the chunk's; what that rounding drops starts the next chain
      // (nothing where a sum is not finite)
      if (((k - k0) & a.group) != a.group && k + 64 < k1) continue;
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int t = 0; t < TF; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = tot[f][t][i] + acc[f][t][i];
            acc[f][t][i] = finite_or_0((tot[f][t][i] - v) + acc[f][t][i]);
            tot[f][t][i] = v;
          }
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int t = 0; t < TF; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (W32) tot[f][t][i] += acc[f][t][i] + finite_or_0(low[f][t][i]);
          if constexpr (!SPLIT) all[f][t][i] = s == s0 ? double(tot[f][t][i]) : all[f][t][i] + double(tot[f][t][i]);
        }
  }
#pragma unroll
  for (int t = 0; t < TF; ++t) {
    const int64_t tok = tile * XR + 16 * t + m;
    if (tok >= a.T) continue;
    const int eb = e0 + 4 * NF * q;
    if constexpr (SPLIT) {   // ld_o holds every group's 16 NF experts
      float* o = a.out + (s0 * a.T + tok) * a.ld_o + eb;
#pragma unroll
      for (int f = 0; f < NF; ++f) *reinterpret_cast<v4f*>(o + 4 * f) = tot[f][t];
    } else {
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = eb + 4 * f + i;
          if (e < a.E) {
            float v = float(all[f][t][i]);
            if (a.bias) v += W32 ? static_cast<const float*>(a.bias)[e] : bf16_to_f32(static_cast<const uint16_t*>(a.bias)[e]);
            if (a.score_bias) v += a.score_bias[e];
            a.out[tok * a.ld_o + e] = v;
          }
        }
    }
  }
}

// The launch's shape: fragments per wave, chunks of D.  About 2048 waves (two
// per SIMD, which is what hides the fragments' latency) where D allows chunks
// of at least 128 columns; more chunks would only add partial sums to write
// and read (4 bytes of part per token, expert and chunk).  The tile leaves two waves
// a SIMD their registers: two sums per output, three with an fp32 gate ([4096, 7168] x 256,
// bf16 gate: 64 x 64 outputs 89 us, 76 with the registers of two waves and spills, 32 x 64 72;
// fp32 gate: 32 x 64 279 and 210, 32 x 32 176).
struct GateShape {
  int tf, nf, eg;
  int64_t tt, S, chunk, ld_p;
};
inline GateShape gate_shape(int64_t T, int64_t D, int E, bool w32) {
  GateShape g;
  g.nf = E <= 16 ? 1 : E <= 32 || w32 ? 2 : E <= 48 ? 3 : 4;
  g.tf = T <= 16 ? 1 : (T <= 32 || w32 || g.nf == 4) ? 2 : 4;
  g.eg = (E + 16 * g.nf - 1) / (16 * g.nf);
  g.tt = (T + 16 * g.tf - 1) / (16 * g.tf);
  int64_t s = 2048 / (g.tt * g.eg);
  s = s < 1 ? 1 : s > 32 ? 32 : s;
  if (D > 0) {
    if (s > D / 128) s = D / 128 < 1 ? 1 : D / 128;
    g.chunk = ((D + s - 1) / s + 63) / 64 * 64;
    g.S = (D + g.chunk - 1) / g.chunk;
  } else {   // the bound over D
    g.chunk = 0;
    g.S = s;
  }
  g.ld_p = int64_t(g.eg) * 16 * g.nf;
  return g;
}

// Columns of an MFMA chain: the longest that leaves the rms error below the FMA kernel's
// (16384 tokens, in units of the logits').  bf16 gate, FMAs | chains of 64 / 128 / 256 columns:
// D 512 6.1e-8 | 5.7e-8 / 7.2e-8 / -, D 1024 6.8e-8 | 5.7e-8, D 2048 7.5e-8 | 5.8e-8 / 7.0e-8 / -, D 4096
// 8.4e-8 | 5.8e-8 / 7.1e-8 / 9.4e-8.  fp32 gate: D 512 8.6e-8 | 5.7e-8 / 6.9e-8 / 9.0e-8, D 2560 1.3e-7 |
// 5.7e-8 / - / 8.9e-8.  A join is five VALU instructions a sum: forward of [4096, 7168] x 256 with
// 64 / 128 / 256 columns 80 / 75 / 72 us.
inline int gate_group_columns(int64_t D, bool w32) { return (D < 2048 ? 64 : 128) << int(w32); }

// ------------------------------------------- pieces for the backward ----
// Tiles of 64 x 64: dlogits [T, E] into its bf16 pieces by token (p, [3][Tp x Ep],
// for dx) and by expert (pt, [3][Ep x Tp], for dw) with the tile's column sums
// (db_part [token tiles][E]); the gate [E, D] into pieces by column (wt,
// [3 or 1][Dp x Ep], for dx).  Ep, Tp, Dp: E up to a multiple of 32, T and D of
// 64, filled with zeros.  All three are stored as MFMA fragments: blocks of 16 rows x
// 32 of the contracted index, 1 KiB each, lane (i, q) = row i, 8 q .. + 8 at 16
// (i + 16 q), the blocks of 16 rows consecutive -- one fragment is one coalesced
// read.  wt's rows are permuted within 64 columns: row i of fragment f is column
// 16 (i / 4) + 4 f + i % 4.
__device__ __forceinline__ int64_t frag_offset(int64_t row, int k, int kblocks) {
  return ((row >> 4) * kblocks + (k >> 5)) * 512 + ((row & 15) + 16 * ((k >> 3) & 3)) * 8;
}
struct GatePieceArgs {
  const float* dl;
  int64_t ld_dl, T, D, Tp, Dp;
  int E, Ep;
  const void* w;
  int64_t ld_w;
  int w_bf16;
  uint16_t* p;         // or null (with wt)
  uint16_t* pt;        // or null
  float* db_part;      // or null
  uint16_t* wt;        // or null
  int64_t t_tiles, d_tiles;
};

__global__ __launch_bounds__(256) void gate_pieces_kernel(GatePieceArgs a) {
  __shared__ float tile[64][65];
  const int tid = threadIdx.x, c = tid & 63, r4 = tid >> 6;
  const int e0 = blockIdx.y * 64;
  const bool weights = int64_t(blockIdx.x) >= a.t_tiles;
  if (!weights) {
    const int64_t t0 = int64_t(blockIdx.x) * 64;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t t = t0 + 4 * i + r4;
      tile[4 * i + r4][c] = (t < a.T && e0 + c < a.E) ? a.dl[t * a.ld_dl + e0 + c] : 0.f;
    }
    __syncthreads();
    if (a.db_part && r4 == 0 && e0 + c < a.E) {
      double s = 0.;
      for (int r = 0; r < 64; ++r) s += double(tile[r][c]);
      a.db_part[int64_t(blockIdx.x) * a.E + e0 + c] = float(s);
    }
    const int row = tid >> 2, col = (tid & 3) * 16;
#pragma unroll
    for (int o = 0; o < 16; o += 8) {
      float v[8], u[8];
      uint4 h, m, l;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = tile[row][col + o + i];
        u[i] = tile[col + o + i][row];
      }
      if (a.p && e0 + col + o < a.Ep) {
        split3x8(v, h, m, l);
        uint16_t* d = a.p + frag_offset(t0 + row, e0 + col + o, a.Ep >> 5);
        const int64_t plane = a.Tp * a.Ep;
        *reinterpret_cast<uint4*>(d) = h;
        *reinterpret_cast<uint4*>(d + plane) = m;
        *reinterpret_cast<uint4*>(d + 2 * plane) = l;
      }
      if (a.pt && e0 + row < a.Ep) {
        split3x8(u, h, m, l);
        uint16_t* d = a.pt + frag_offset(e0 + row, int(t0) + col + o, int(a.Tp >> 5));
        const int64_t plane = a.Tp * a.Ep;
        *reinterpret_cast<uint4*>(d) = h;
        *reinterpret_cast<uint4*>(d + plane) = m;
        *reinterpret_cast<uint4*>(d + 2 * plane) = l;
      }
    }
    return;
  }
  const int64_t d0 = (int64_t(blockIdx.x) - a.t_tiles) * 64;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int e = e0 + 4 * i + r4;
    float v = 0.f;
    if (e < a.E && d0 + c < a.D)
      v = a.w_bf16 ? bf16_to_f32(static_cast<const uint16_t*>(a.w)[int64_t(e) * a.ld_w + d0 + c])
                   : static_cast<const float*>(a.w)[int64_t(e) * a.ld_w + d0 + c];
    tile[4 * i + r4][c] = v;
  }
  __syncthreads();
  const int row = tid >> 2, col = (tid & 3) * 16;
#pragma unroll
  for (int o = 0; o < 16; o += 8) {
    float u[8];
    uint4 h, m, l;
#pragma unroll
    for (int i = 0; i < 8; ++i) u[i] = tile[col + o + i][row];
    if (e0 + col + o < a.Ep) {
      split3x8(u, h, m, l);
      const int fr = ((row >> 2) & 3) * 16 + (row >> 4) * 4 + (row & 3);   // column 16 (i / 4) + 4 f + i % 4 -> 16 f + i
      uint16_t* d = a.wt + frag_offset(d0 + fr, e0 + col + o, a.Ep >> 5);
      const int64_t plane = a.Dp * a.Ep;
      *reinterpret_cast<uint4*>(d) = h;
      if (!a.w_bf16) {
        *reinterpret_cast<uint4*>(d + plane) = m;
        *reinterpret_cast<uint4*>(d + 2 * plane) = l;
      }
    }
  }
}

// ---------------------------------------------------------------- dx ----
// A wave forms 64 tokens x 64 columns (4 waves: 128 x 128, the shared fragments
// from the L1), every fragment one coalesced read: K = Ep experts once per pair of pieces, the small pairs first, the
// two high pieces last.  All nine pairs with an fp32 gate: the pieces are
// truncations, so the three smallest pairs have the product's sign and come to
// 2^-21 of it, more than an fp32 rounding.  A lane ends with 16 consecutive
// columns of a token.
struct GateDxArgs {
  const uint16_t* p;     // [3][Tp x Ep] fragments
  const uint16_t* wt;    // [1 or 3][Dp x Ep] fragments
  int64_t T, D, Tp, Dp;
  int Ep;
  uint16_t* dx;          // bf16 [T, ld_dx]
  int64_t ld_dx;
};

template <bool W32>
__global__ __launch_bounds__(256) void gate_dx_kernel(GateDxArgs a) {
  const int lane = threadIdx.x & 63, m = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int64_t t0 = int64_t(blockIdx.x) * 128 + (wave & 1) * 64, d0 = int64_t(blockIdx.y) * 128 + (wave >> 1) * 64;
  if (t0 >= a.T || d0 >= a.D) return;
  const uint16_t* pr[4];
  const uint16_t* wr[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {   // Tp and Dp are multiples of 64
    pr[f] = a.p + (t0 / 16 + f) * (16 * a.Ep) + 8 * lane;
    wr[f] = a.wt + (d0 / 16 + f) * (16 * a.Ep) + 8 * lane;
  }
  const int64_t pp = a.Tp * a.Ep, wp = a.Dp * a.Ep;
  constexpr int kPairs = W32 ? 9 : 3;
  constexpr int kP[9] = {2, 1, W32 ? 2 : 0, 0, 2, 1, 0, 1, 0};   // dlogits piece
  constexpr int kW[9] = {W32 ? 2 : 0, W32 ? 2 : 0, W32 ? 1 : 0, 2, 0, 1, 1, 0, 0};   // gate piece
  v4f acc[4][4];   // [column fragment][token fragment]
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[f][t] = v4f{0.f, 0.f, 0.f, 0.f};
  struct Buf { uint4 p[4], w[4]; } b0, b1;
#pragma unroll
  for (int n = 0; n < kPairs; ++n) {
    const int64_t po = kP[n] * pp, wo = kW[n] * wp;
    if (n == kPairs - 1)
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[f][t][i] = finite_or_0(acc[f][t][i]);
    auto load = [&](Buf& b, int k) {
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        b.p[f] = *reinterpret_cast<const uint4*>(pr[f] + po + 16 * k);
        b.w[f] = *reinterpret_cast<const uint4*>(wr[f] + wo + 16 * k);
      }
    };
    auto step = [&](const Buf& b) {
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[f][t] = mfma16(b.w[f], b.p[t], acc[f][t]);
    };
    load(b0, 0);
    for (int k = 0; k < a.Ep; k += 64) {
      if (k + 32 < a.Ep) load(b1, k + 32);
      step(b0);
      if (k + 64 < a.Ep) load(b0, k + 64);
      if (k + 32 < a.Ep) step(b1);
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int64_t tok = t0 + 16 * t + m;
    if (tok >= a.T) continue;
    uint16_t* o = a.dx + tok * a.ld_dx + d0 + 16 * q;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (d0 + 16 * q + 8 * h < a.D)
        st_global(o + 8 * h, make_uint4(hw_bf16x2(acc[2 * h][t][0], acc[2 * h][t][1]),
                                        hw_bf16x2(acc[2 * h][t][2], acc[2 * h][t][3]),
                                        hw_bf16x2(acc[2 * h + 1][t][0], acc[2 * h + 1][t][1]),
                                        hw_bf16x2(acc[2 * h + 1][t][2], acc[2 * h + 1][t][3])));
  }
}

// ---------------------------------------------------------------- dw ----
// Partial dw of one slice of tokens: a wave forms 64 experts x 128 columns, the
// 4 waves of a workgroup WE expert groups x 4 / WE column groups.  K steps of
// 32 tokens: x through LDS (each token row of 128 columns is 256 bytes; the
// 8-byte pieces of token k of each 64-byte chunk at index ^ (k % 4 + 4 (k / 8 %
// 2)), so the 32 lanes of a transposing read touch all 64 banks once), read
// transposed (ds_read_b64_tr_b16), dlogits' pieces straight from pt's fragments.  Two
// passes over the slice, the low pieces first.  A lane ends with 32
// consecutive columns of an expert.  The slice is the fastest part of the
// workgroup index, so an XCD (workgroups go to them in turn) keeps the pieces of
// one or two slices in its L2: with the column tile fastest every L2 had to hold
// all of pt and the kernel ran at the misses' rate (117 us for 256 x 7168 over 4096
// tokens).
struct GateDwArgs {
  const uint16_t* pt;    // [3][Ep x Tp] fragments
  int64_t Tp;
  int E, Ep;
  const uint16_t* x;     // bf16 [T, ld_x]
  int64_t ld_x, T, D;
  int64_t rows_per_slice, slices;   // rows: a multiple of 32
  float* part;           // [slices][E][D]
};

// (Two waves per SIMD asked for: with more registers to use, the compiler keeps the
// sums in the accumulation half and copies them across in every step.)
template <int WE>
__global__ __launch_bounds__(256, 2) void gate_dw_kernel(GateDwArgs a) {
  constexpr int WD = 4 / WE, NX = 2 * WD;   // NX: 16-byte x loads of a thread per step
  __shared__ __attribute__((aligned(16))) uint8_t xs[2][WD][32][256];
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int e0 = (wave % WE) * 64, wd = wave / WE;
  const int64_t slice = blockIdx.x % a.slices, c0 = (blockIdx.x / a.slices) * (128 * WD);
  const int64_t t_lo = slice * a.rows_per_slice;
  const int64_t t_hi = t_lo + a.rows_per_slice < a.T ? t_lo + a.rows_per_slice : a.T;
  const uint16_t* pr[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int eb = e0 / 16 + f;
    pr[f] = a.pt + int64_t(eb < a.Ep / 16 ? eb : a.Ep / 16 - 1) * (16 * a.Tp) + 8 * lane;
  }
  const int64_t plane = a.Tp * a.Ep;
  // x: thread (row tid / 16 + 16 j, chunk tid % 16) of each column group
  const int xrow = tid >> 4, xc = tid & 15;
  uint4 xv[NX];
  auto load_x = [&](int64_t t) {
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      const int64_t tr = t + xrow + 16 * (j & 1), col = c0 + 128 * (j >> 1) + 8 * xc;
      xv[j] = (tr < t_hi && col < a.D) ? *reinterpret_cast<const uint4*>(a.x + tr * a.ld_x + col)
                                       : make_uint4(0, 0, 0, 0);
    }
  };
  auto store_x = [&](int b) {
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      const int k = xrow + 16 * (j & 1), g = (k & 3) + 4 * ((k >> 3) & 1);
      const uint4 v = xv[j];
      const uint4 u = (g & 1) ? make_uint4(v.z, v.w, v.x, v.y) : v;
      const int slot = (xc & ~3) | ((xc & 3) ^ (g >> 1));
      *reinterpret_cast<uint4*>(&xs[b][j >> 1][k][slot * 16]) = u;
    }
  };
  auto load_p = [&](uint4 (&p)[4], int64_t t, int64_t po) {
#pragma unroll
    for (int f = 0; f < 4; ++f) p[f] = *reinterpret_cast<const uint4*>(pr[f] + po + 16 * t);
  };
  // lane (q, 4 r + p) of a transposing read addresses row 8 q + r (+ 4), columns 32 p + 4 f
  const int kr = 8 * q + (m >> 2), kg = (kr & 3) + 4 * ((kr >> 3) & 1);
  auto frag = [&](int b, int f) {
    const uint8_t* s = &xs[b][wd][kr][(m & 3) * 64 + ((f ^ kg) & 7) * 8];
    typedef __attribute__((address_space(3))) v4s16 lds_v4;
    const v4s16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)s);
    const v4s16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(s + 4 * 256));
    const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
    return make_uint4(l2.x, l2.y, h2.x, h2.y);
  };
  v4f acc[8][4];   // [column fragment][expert fragment]
#pragma unroll
  for (int f = 0; f < 8; ++f)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[f][e] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int64_t pa = pass == 0 ? 2 * plane : 0;
    if (pass == 1)
#pragma unroll
      for (int f = 0; f < 8; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[f][e][i] = finite_or_0(acc[f][e][i]);
    uint4 p0[4], p1[4], n0[4], n1[4];
    load_x(t_lo);
    load_p(n0, t_lo, pa);
    if (pass == 0) load_p(n1, t_lo, plane);
    __syncthreads();   // every wave is done with the buffers of the pass before
    int b = 0;
    for (int64_t t = t_lo; t < t_hi; t += 32, b ^= 1) {
      store_x(b);
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        p0[f] = n0[f];
        if (pass == 0) p1[f] = n1[f];
      }
      // one barrier a step: buffer b was last read two steps ago
      __syncthreads();
      if (t + 32 < t_hi) {
        load_x(t + 32);
        load_p(n0, t + 32, pa);
        if (pass == 0) load_p(n1, t + 32, plane);
      }
      if (e0 < a.E)
#pragma unroll
        for (int f = 0; f < 8; ++f) {
          const uint4 xf = frag(b, f);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            acc[f][e] = mfma16(xf, p0[e], acc[f][e]);
            if (pass == 0) acc[f][e] = mfma16(xf, p1[e], acc[f][e]);
          }
        }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int ex = e0 + 16 * e + m;
    if (ex >= a.E) continue;
    const int64_t col = c0 + 128 * wd + 32 * q;
    float* o = a.part + (slice * a.E + ex) * a.D + col;
#pragma unroll
    for (int f = 0; f < 8; ++f)
      if (col + 4 * f < a.D) *reinterpret_cast<v4f*>(o + 4 * f) = acc[f][e];
  }
}

// dw = the slices' partials summed in slice order (four columns a thread, eight
// slices' loads in flight); an expert's last workgroup its db = the token tiles'
// column sums (lane-strided tiles, then a fixed shuffle tree).  Both in 64 bits,
// as the tiles' column sums: up to 64 partials of a few MFMAs each, and 64 tokens, one
// after the other in fp32 were less exact than the VALU kernels' sums (rms error of dw,
// 16384 tokens, [1024] x 12: 1.6e-7 there, 1.9e-7 in fp32, 1.2e-7 now; db 2 to 3 times).
struct GateDwSumArgs {
  const float* part;
  int64_t S, D;
  int E;
  void* dw;              // [E, ld_dw] or null
  int64_t ld_dw;
  int dw_bf16;
  int vec;               // dw's rows on 16-byte boundaries (bf16: 8)
  const float* db_part;
  int64_t tiles;
  void* db;              // or null
  int db_bf16;
};

__global__ __launch_bounds__(256) void gate_dw_sum_kernel(GateDwSumArgs a) {
  if (blockIdx.x == gridDim.x - 1) {   // every expert's row has a workgroup for its db
    if (a.db == nullptr) return;
    const int lane = threadIdx.x & 63, e = blockIdx.y;
    if (threadIdx.x < 64) {
      double s = 0.;
#pragma unroll 4
      for (int64_t t = lane; t < a.tiles; t += 64) s += double(a.db_part[t * a.E + e]);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
      const float v = float(s);
      if (lane == 0) {
        if (a.db_bf16) static_cast<uint16_t*>(a.db)[e] = f32_to_bf16(v);
        else static_cast<float*>(a.db)[e] = v;
      }
    }
    return;
  }
  const int64_t n = int64_t(a.E) * a.D, col = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (col >= a.D) return;
  const float* p = a.part + int64_t(blockIdx.y) * a.D + col;
  double d4[4] = {0., 0., 0., 0.};
  for (int64_t s = 0; s < a.S; s += 8) {   // eight loads in flight
    v4f u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = *reinterpret_cast<const v4f*>(p + (s + j < a.S ? s + j : s) * n);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s + j < a.S)
#pragma unroll
        for (int i = 0; i < 4; ++i) d4[i] = s + j == 0 ? double(u[0][i]) : d4[i] + double(u[j][i]);
  }
  const v4f v = {float(d4[0]), float(d4[1]), float(d4[2]), float(d4[3])};
  const int64_t o = blockIdx.y * a.ld_dw + col;
  if (a.dw_bf16) {
    uint16_t* d = static_cast<uint16_t*>(a.dw) + o;
    if (a.vec) {
      st_global(d, make_uint2(hw_bf16x2(v[0], v[1]), hw_bf16x2(v[2], v[3])));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = f32_to_bf16(v[j]);
    }
  } else {
    float* d = static_cast<float*>(a.dw) + o;
    if (a.vec) {
      *reinterpret_cast<v4f*>(d) = v;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = v[j];
    }
  }
}

// Which backward: E > 8, and up to 8 experts a long row.  Measured, 8 experts on
// the VALU against 9 here: [16384, 2048] 75 against 80 us, [4096, 2048] 40 / 42,
// [4096, 7168] 94 / 64, [16384, 7168] 236 / 192.  (The VALU pass is one read of x
// and one write of dx; here the pieces come first and a tile of 16 experts is
// half empty, but long rows get their columns in parallel.)
inline bool gate_bwd_mfma(int64_t D, int E) { return E <= 256 && (E > 8 || D > 4096); }

// The backward's layout in the caller's workspace.
struct GateBwdShape {
  int64_t Tp, Dp, t_tiles, slices, rows;
  int Ep, we;
  int64_t part, db, p, pt, wt, bytes;   // byte offsets
};
inline GateBwdShape gate_bwd_shape(int64_t T, int64_t D, int E) {
  GateBwdShape g;
  g.Ep = (E + 31) / 32 * 32;
  g.Tp = (T + 63) / 64 * 64;
  g.Dp = (D + 63) / 64 * 64;
  g.t_tiles = g.Tp / 64;
  g.we = E <= 64 ? 1 : E <= 128 ? 2 : 4;
  // about two workgroups per CU (what the registers allow: a step waits for its
  // loads, not for its MFMAs); at most 64 slices of at least 64 tokens, and 64 MiB of partials
  const int64_t tiles = (D + 512 / g.we - 1) / (512 / g.we);
  int64_t s = 512 / tiles, cap = (64ll << 20) / (int64_t(E) * D * 4);
  s = s > 64 ? 64 : s;
  s = s > cap ? cap : s;
  s = s > (T + 63) / 64 ? (T + 63) / 64 : s;
  s = s >= 8 ? s / 8 * 8 : s;
  s = s < 1 ? 1 : s;
  g.rows = ((T + s - 1) / s + 31) / 32 * 32;
  g.slices = (T + g.rows - 1) / g.rows;
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  g.part = 0;
  g.db = up(g.slices * int64_t(E) * D * 4);
  g.p = g.db + up(g.t_tiles * int64_t(E) * 4);
  g.pt = g.p + up(3 * g.Tp * g.Ep * 2);
  g.wt = g.pt + up(3 * g.Tp * g.Ep * 2);
  g.bytes = g.wt + up(3 * g.Dp * g.Ep * 2);
  return g;
}

}  // namespace fm
