// Pieces of the few-rows products whose blocks own units of four rows of W (gemm_quads.hip, qkv_fused.hip).
//
// The products are those of gemm_skinny.hip to the bit: k-steps of 32 columns on v_mfma_f32_16x16x32_bf16, step s to wave
// s % waves, each wave's steps in order in one accumulator, the waves added in order.  What differs is how the operands
// come: a tile of 16 rows has only four that count, so one load of 64 lanes takes the four rows of FOUR steps (lane
// 16 kq + 4 i + r: row r, step i, piece kq), and step i's operand is that register turned by 4 i lanes within the rows of
// 16 lanes: rows 0 to 3 of the tile are the unit's, the others are other steps' values whose products nobody reads.
// The activations of G = 4 or 8 tokens come in the same way, 16 / G steps to a load.
#pragma once
#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 quad_bf16;
typedef __attribute__((ext_vector_type(4))) float quad_f32;
typedef __attribute__((ext_vector_type(4))) unsigned quad_u32;

// lane c of each row of 16 gets lane c + BY's value
template <int BY>
__device__ __forceinline__ unsigned quad_turn(unsigned v) {
  if constexpr (BY == 0) return v;
  else return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + 16 - BY, 0xF, 0xF, true);   // row_ror
}
template <int BY>
__device__ __forceinline__ quad_u32 quad_turn(quad_u32 v) {
  return quad_u32{quad_turn<BY>(v[0]), quad_turn<BY>(v[1]), quad_turn<BY>(v[2]), quad_turn<BY>(v[3])};
}
template <int BY>
__device__ __forceinline__ float quad_turn(float v) {
  return __builtin_bit_cast(float, quad_turn<BY>(__builtin_bit_cast(unsigned, v)));
}

// the sum over the four lanes 16 apart, in the order of two exchanges (16 lanes away, then 32)
__device__ __forceinline__ float quad_sum_rows(float v) {
  v += __shfl_xor(v, 16, MS_WAVE);
  return v + __shfl_xor(v, 32, MS_WAVE);
}

// The k-steps of one wave.  U units of four rows; G tokens; C loads of W (of four steps) asked for at a time.
template <int U, int G, int C, bool NORM>
struct QuadProduct {
  static constexpr int XL = G / 4;        // loads of activations to one of W
  static constexpr int XS = 16 / G;       // steps of a load of activations
  quad_u32 wv[C][U];
  quad_u32 xv[NORM ? 1 : C][NORM ? 1 : XL];
  quad_f32 xf[NORM ? C : 1][NORM ? XL : 1][2], nw[NORM ? C : 1][NORM ? XL : 1][2];
  quad_f32 acc[U];
  float ss;
  int lane, wave, waves, K, mine;   // mine: this wave's k-steps

  __device__ __forceinline__ QuadProduct(int lane, int wave, int waves, int K) : ss(0.f), lane(lane), wave(wave), waves(waves), K(K), mine(((K + 31) / 32 - wave + waves - 1) / waves) {
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = quad_f32{0.f, 0.f, 0.f, 0.f};
  }
  // first column of this lane's piece: step i of the wave's
  __device__ __forceinline__ int column(int i) const { return (wave + waves * i) * 32 + (lane >> 4) * 8; }
  __device__ __forceinline__ int w_step(int i0, int c) const { return i0 + 4 * c + ((lane >> 2) & 3); }
  __device__ __forceinline__ int x_step(int i0, int c, int j) const { return i0 + 4 * c + j * XS + (lane & 15) / G; }

  // Every load of a lane without a condition (one behind a condition is waited for by itself): past K the last piece
  // once more, masked where it is used.  A load of which no step is this wave's is left out as a whole.  x: this lane's token's row.
  __device__ __forceinline__ void ask(int i0, const bf16* const (&w)[U], const void* x, const float* norm_w) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (c > 0 && i0 + 4 * c >= mine) break;
      const int kw = min(column(w_step(i0, c)), K - 8);
#pragma unroll
      for (int u = 0; u < U; ++u) wv[c][u] = *reinterpret_cast<const quad_u32*>(w[u] + kw);
#pragma unroll
      for (int j = 0; j < XL; ++j) {
        if (j > 0 && i0 + 4 * c + j * XS >= mine) break;
        const int kx = min(column(x_step(i0, c, j)), K - 8);
        if constexpr (NORM) {
          xf[c][j][0] = *reinterpret_cast<const quad_f32*>((const float*)x + kx);
          xf[c][j][1] = *reinterpret_cast<const quad_f32*>((const float*)x + kx + 4);
          nw[c][j][0] = *reinterpret_cast<const quad_f32*>(norm_w + kx);
          nw[c][j][1] = *reinterpret_cast<const quad_f32*>(norm_w + kx + 4);
        } else {
          xv[c][j] = *reinterpret_cast<const quad_u32*>((const bf16*)x + kx);
        }
      }
    }
  }

  template <int I>
  __device__ __forceinline__ void step(const quad_u32 (&w)[U], const quad_u32 (&x)[XL], const quad_f32 (&f)[XL][2]) {
    constexpr int J = I / XS, BY = (I % XS) * G;
    if constexpr (NORM) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = quad_turn<BY>(f[J][0][e]), b = quad_turn<BY>(f[J][1][e]);
        ss = fmaf(a, a, ss);
        ss = fmaf(b, b, ss);
      }
    }
    const quad_bf16 xb = __builtin_bit_cast(quad_bf16, quad_turn<BY>(x[J]));
#pragma unroll
    for (int u = 0; u < U; ++u)
      acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(quad_bf16, quad_turn<4 * I>(w[u])), xb, acc[u], 0, 0, 0);
  }

  __device__ __forceinline__ void use(int i0) {
    const quad_u32 zero = {0u, 0u, 0u, 0u};
    const quad_f32 fzero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const bool in = column(w_step(i0, c)) < K;
      quad_u32 w[U], x[XL];
      quad_f32 f[XL][2];
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = in ? wv[c][u] : zero;
#pragma unroll
      for (int j = 0; j < XL; ++j) {
        const bool xin = column(x_step(i0, c, j)) < K;
        f[j][0] = f[j][1] = fzero;
        if constexpr (NORM) {
          f[j][0] = xin ? xf[c][j][0] : fzero;
          f[j][1] = xin ? xf[c][j][1] : fzero;
          quad_bf16 h;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            h[e] = (__bf16)(f[j][0][e] * nw[c][j][0][e]);
            h[4 + e] = (__bf16)(f[j][1][e] * nw[c][j][1][e]);
          }
          x[j] = xin ? __builtin_bit_cast(quad_u32, h) : zero;   // (a load left out may hold anything)
        } else {
          x[j] = xin ? xv[c][j] : zero;
        }
      }
      step<0>(w, x, f);
      step<1>(w, x, f);
      step<2>(w, x, f);
      step<3>(w, x, f);
    }
  }

  __device__ __forceinline__ void run(const bf16* const (&w)[U], const void* x, const float* norm_w) {
    // (the first ask is the caller's, before whatever else it asks for)
    for (int i = 0; i < mine; i += 4 * C) {
      use(i);
      if (i + 4 * C < mine) ask(i + 4 * C, w, x, norm_w);
    }
  }
};

}  // namespace
