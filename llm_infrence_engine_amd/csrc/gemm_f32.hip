// C[M,N] (+)= A[M,K] . W[N,K]^T (+ bias[N]) in true 32 bits: float operands, float products and float sums, on the
// matrix cores' float instruction (v_mfma_f32_16x16x4_f32: nothing is rounded below 32 bits).
//
// The order of a sum is the same whatever M is, so a token's result does not depend on what else is in the batch: K is
// cut into at most 16 slices (from K alone, `slice_steps`), a slice is summed 16 values at a time from its start, and the
// slices are added in order.  All kernels keep that order:
//   rows     up to 64 rows, by less than 512 columns and where `choose` takes it: all waves of a block on the same 4 to 16
//            rows of W, the slices dealt out over them and added through LDS.  Bound by reading W.
//   few      up to 8 rows, of these: loads that take four steps at a time.
//   diagonal up to 8 rows: an instruction takes a step of two or four slices; also with the norm of A's rows, the gate, or the rotation
//            and store of a q/k/v product within.
//   slices   32 rows of W by 16, 32 or 48 tokens and the slices dealt out over a block's waves, for tiles too few to fill the chip
//            (`choose`): bound by the way of the operands to the CU, 40 KB a us.
//   tiled    the others: 64 x 64 or 32 x 32 tiles staged through LDS four steps ahead, 4 waves.  Bound by the float matrix rate
//            (157 TFLOP/s nominal), short K by writing C.
// Measured with the 0.5B sizes against the 64 x 64 vector-ALU tile that ran them before (one MI355X): of 3 rows the down
// product (896 x 4,864) 319 -> 16 us (12 with grouped loads), gate/up (9,728 x 896) 63 -> 12 us, q/k/v (1,152 x 896) 63 -> 4.5 us, the head
// (151,936 x 896) 221 -> 100 us, of 64 rows 252 -> 220; of 350 rows down 316 -> 45 us, gate/up 108 -> 75 us.  Of few rows
// down is bound by the steps a CU works off (16 waves, 19 steps each); the tiled steps by the way from one barrier to the next.  C leaves a tile through LDS in whole rows (4,096 x 32,000 x 64: 440 us as the fragments lie, 270 so, 261 before).
#include "common.h"
#include "api.h"
#include "gemm_f32.h"
#include "quads.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int STEP = 16;          // k values a slice is summed by at a time: four MFMAs of four
constexpr int MAX_SLICES = 16;
constexpr int LDS_BYTES = 163840;  // of a CU

__host__ __device__ inline int slice_steps(int K) {
  const int steps = (K + STEP - 1) / STEP;
  const int per = (steps + MAX_SLICES - 1) / MAX_SLICES;
  return per > 4 ? per : 4;
}

// Lane l holds row l % 16 and k values 4 (l / 16) .. + 3 of a step, of either operand: MFMA j of the step then sums the
// k values {j, 4 + j, 8 + j, 12 + j}.
__device__ __forceinline__ f32x4 step16(f32x4 w, f32x4 a, f32x4 acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], a[j], acc, 0, 0, 0);
  return acc;
}

// Loads are never behind a condition (a branch around each would have every one waited for by itself): places past the
// row's end read its last four values, and `masked` makes zeros of them before they are used.  K is a multiple of 4.
__device__ __forceinline__ f32x4 load4(const float* row, int k, int K) {
  return *reinterpret_cast<const f32x4*>(row + min(k, K - 4));
}
__device__ __forceinline__ f32x4 masked(f32x4 v, int k, int K) { return k < K ? v : f32x4{0.f, 0.f, 0.f, 0.f}; }

__device__ __forceinline__ void store(float* C, size_t at, float v, const float* bias, int n, int accumulate) {
  if (bias) v += bias[n];
  if (accumulate) v += C[at];
  C[at] = v;
}

// four results side by side (runs: at an address that fits them), those past the last column of N not
__device__ __forceinline__ void store_run(float* C, size_t at, f32x4 v, const float* bias, int n, int N, int accumulate, int runs) {
  if (runs && n + 3 < N) {
    if (bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += bias[n + e];
    }
    if (accumulate) v += *reinterpret_cast<const f32x4*>(C + at);
    *reinterpret_cast<f32x4*>(C + at) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) store(C, at + e, v[e], bias, n + e, accumulate);
  }
}

// R rows of W a block (lanes of the other rows of the instruction repeat them), NT tiles of 16 tokens, the slices dealt out
// over the block's waves in turn.
template <int R, int NT>
__global__ void __launch_bounds__(MAX_SLICES * MS_WAVE)
gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                     float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc, int accumulate) {
  extern __shared__ __align__(16) float part[];      // [slice][token][row of W]
  constexpr int PART = NT * 256;                     // of a slice
  constexpr int AHEAD = NT == 4 ? 2 : 4;            // steps whose operands are asked for before they are used
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);
  const int r = lane & 15, g = lane >> 4;
  const int per = slice_steps(K), steps = (K + STEP - 1) / STEP, slices = (steps + per - 1) / per;
  const int n0 = blockIdx.x * R;
  const float* wrow = W + (size_t)min(n0 + r % R, N - 1) * ldw;
  const float* arow[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) arow[t] = A + (size_t)min(t * 16 + r, M - 1) * lda;   // columns from M on are not stored

  for (int slice = wave; slice < slices; slice += blockDim.x / MS_WAVE) {
    const int first = slice * per, last = min(steps, first + per);
    f32x4 acc[NT] = {};
    f32x4 w[AHEAD], a[AHEAD][NT];
    // steps past the slice's end ask for its last step again, which the cache has
    auto fetch = [&](int u, int step) {
      const int k = min(step, last - 1) * STEP + 4 * g;
      w[u] = load4(wrow, k, K);
#pragma unroll
      for (int t = 0; t < NT; ++t) a[u][t] = load4(arow[t], k, K);
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) fetch(u, first + u);
    for (int s = first; s < last; s += AHEAD) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int k = (s + u) * STEP + 4 * g;
        const f32x4 wu = masked(w[u], k, K);
        f32x4 au[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) au[t] = masked(a[u][t], k, K);
        if (s + AHEAD < last) fetch(u, s + u + AHEAD);
        if (s + u < last) {
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[t] = step16(wu, au[t], acc[t]);
        }
      }
    }
    // the accumulators hold W's row 4 g + i and the token r
#pragma unroll
    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(&part[slice * PART + (t * 16 + r) * 16 + 4 * g]) = acc[t];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < NT * 16 * R; e += blockDim.x) {
    const int m = e / R, n = n0 + e % R, at = m * 16 + e % R;
    if (m >= M || n >= N) continue;
    float v = part[at];
    for (int s = 1; s < slices; ++s) v += part[s * PART + at];
    store(C, (size_t)m * ldc + n, v, bias, n, accumulate);
  }
}

// Up to G = 4 or 8 tokens: the same products in the same order, with fewer loads.  A block of the kernel above spends its time on
// issuing loads (some 70 cycles of its CU each, 38 of them to a wave for 19 steps), and most lanes of these repeat others: 4 rows
// of W and 3 of A fill a quarter of the lanes.  Here one load takes FOUR steps of four rows (of eight rows two steps, of 16 one;
// lane 16 g + X i + r: row r, step i, piece g), and the operand of a step is that register turned by X i lanes within the
// rows of 16; the instruction's other rows and columns hold other steps' values, whose products nobody reads.
template <int X>
struct StepRows {
  static constexpr int LOADS = X / 4, STEPS = 16 / X;      // loads to four steps, steps to a load
  f32x4 v[LOADS];
  __device__ __forceinline__ void fetch(const float* row, int step, int last, int lane, int K) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int k = min(step + j * STEPS + (lane & 15) / X, last) * STEP + 4 * (lane >> 4);
      v[j] = load4(row, k, K);
      if (k >= K) v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  template <int I> __device__ __forceinline__ f32x4 at() const {
    return __builtin_bit_cast(f32x4, quad_turn<(I % STEPS) * X>(__builtin_bit_cast(quad_u32, v[I / STEPS])));
  }
};

template <int R, int G>
__global__ void __launch_bounds__(MAX_SLICES * MS_WAVE)
gemm_f32_few_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                    float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc, int accumulate) {
  extern __shared__ __align__(16) float part[];      // [slice][token][row of W]
  constexpr int PART = G * R, AHEAD = 2;             // groups of four steps asked for before they are used
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);
  const int waves = blockDim.x / MS_WAVE;
  const int per = slice_steps(K), steps = (K + STEP - 1) / STEP, slices = (steps + per - 1) / per, groups = (per + 3) / 4;
  const int n0 = blockIdx.x * R;
  const float* wrow = W + (size_t)min(n0 + (lane & (R - 1)), N - 1) * ldw;
  const float* arow = A + (size_t)min(lane & (G - 1), M - 1) * lda;
  StepRows<R> w[AHEAD];
  StepRows<G> a[AHEAD];
  // the groups of the wave's slices in one row
  const int mine = (slices - wave + waves - 1) / waves * groups;
  int ahead = wave, ahead_at = 0;                    // slice and group of the next loads
  auto fetch = [&](int u) {
    const int step = ahead * per + 4 * ahead_at;
    w[u].fetch(wrow, step, steps - 1, lane, K);
    a[u].fetch(arow, step, steps - 1, lane, K);
    if (++ahead_at == groups) { ahead_at = 0; ahead += waves; }
  };
#pragma unroll
  for (int u = 0; u < AHEAD; ++u)
    if (u < mine) fetch(u);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int slice = wave, at = 0;
  for (int s = 0; s < mine; s += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (s + u >= mine) break;
      const StepRows<R> wu = w[u];
      const StepRows<G> au = a[u];
      if (s + u + AHEAD < mine) fetch(u);
      const int left = min(per, steps - slice * per) - 4 * at;      // steps of this group and the slice's later ones
      auto step = [&](auto index) {
        constexpr int I = decltype(index)::value;
        if (I < left) acc = step16(wu.template at<I>(), au.template at<I>(), acc);
      };
      step(std::integral_constant<int, 0>{});
      step(std::integral_constant<int, 1>{});
      step(std::integral_constant<int, 2>{});
      step(std::integral_constant<int, 3>{});
      if (++at == groups) {
        // lane 16 g + token holds W's rows 4 g .. + 3
        if ((lane & 15) < G && (lane >> 4) * 4 < R) *reinterpret_cast<f32x4*>(&part[slice * PART + (lane & 15) * R + (lane >> 4) * 4]) = acc;
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
        at = 0;
        slice += waves;
      }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < M * R; e += blockDim.x) {
    const int m = e / R, n = n0 + e % R;
    if (n >= N) continue;
    float v = part[e];
    for (int t = 1; t < slices; ++t) v += part[t * PART + e];
    store(C, (size_t)m * ldc + n, v, bias, n, accumulate);
  }
}

// Up to X tokens (4 or 8), R rows of W a block (R <= X): the same products in the same order, S = 16 / X slices by one instruction.
// The instruction's 16 rows are the block's rows at the same step of S slices, its 16 columns the tokens at that step of
// these slices; rows and columns of one slice meet in the blocks on the diagonal, and what else comes out nobody reads.  So a step
// costs 1 / S of the instructions and of the loads, and of both operands every lane's load is its own: 4 rows by 4,864 columns are 19
// dependent steps of four waves, all asked for within the first few (sixteen waves of 76 instructions each are 4 us of the CU's
// matrix pipes alone).
//
// NORM: A is the residual stream, and the rows are normed on their way (NORM pieces of 256 columns at most), by every block for
// itself while its rows of W are on their way; the arithmetic and its order are rms_norm_kernel's.  EPI says what becomes of the sums.
// 3 tokens: gate/up 9,728 x 896 with norm and gate 21.2 us in three kernels -> 13.3, q/k/v 1,152 x 896 with norm, rotation and store
// 13 -> 6.9, 4 rows a block and no norm: see diagonal_rows.  What bounds it then: 64-byte pieces of 16 rows hold the CU's cache up for 70
// cycles a load.  Whole lines through LDS and a ring a wave took 16 to 19 us for gate/up (few waves, each waiting for LDS), 9.4 against 8.4 for
// 896 x 4,864, but 4.0 against 4.4 for 896 x 896.
enum { F32_STORE = 0, F32_SWIGLU = 1, F32_QKV = 2 };

template <int NORM>
__device__ __forceinline__ void norm_rows(const float* __restrict__ x, const float* __restrict__ weight, float eps, float* h, int ldh, int M, int K) {
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = threadIdx.x / MS_WAVE, waves = blockDim.x / MS_WAVE;
  const bool wide = K >= 1024;                       // rms_norm_kernel's blocks: 256 threads, else 128; a lane is two or four of them
  for (int m = wave; m < M; m += waves) {
    float4 v[NORM], w[NORM];
#pragma unroll
    for (int c = 0; c < NORM; ++c) {
      const int i = min(c * 256 + lane * 4, K - 4);
      v[c] = *reinterpret_cast<const float4*>(x + (size_t)m * K + i);
      w[c] = *reinterpret_cast<const float4*>(weight + i);
    }
    float ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NORM; ++c) {
      if (c * 256 + lane * 4 >= K) continue;
      const float t = v[c].x * v[c].x + v[c].y * v[c].y + v[c].z * v[c].z + v[c].w * v[c].w;
      if (wide) ss[c & 3] += t;
      else ss[c & 1] += t;
    }
    float total = 0.f;
    total += wave_sum(ss[0]);
    total += wave_sum(ss[1]);
    if (wide) {
      total += wave_sum(ss[2]);
      total += wave_sum(ss[3]);
    }
    const float inv = 1.0f / sqrtf(total / (float)K + eps);
#pragma unroll
    for (int c = 0; c < NORM; ++c) {
      const int i = c * 256 + lane * 4;
      if (i < K)
        *reinterpret_cast<float4*>(h + m * ldh + i) =
            make_float4(w[c].x * (v[c].x * inv), w[c].y * (v[c].y * inv), w[c].z * (v[c].z * inv), w[c].w * (v[c].w * inv));
    }
  }
}

template <int R, int X, int EPI, int NORM>
__global__ void __launch_bounds__(X * MS_WAVE, X == 4 ? 1 : NORM > 4 ? 2 : NORM ? 4 : 5)
gemm_f32_diagonal_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                    float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc, int accumulate, F32Norm norm, F32Front front) {
  extern __shared__ __align__(16) float part[];      // [slice][token][row of W], behind them (NORM) the normed rows
  constexpr int S = 16 / X, AHEAD = X == 4 ? 10 : 8;
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);
  const int waves = blockDim.x / MS_WAVE;
  const int r = lane & 15, g = lane >> 4;
  const int per = slice_steps(K), steps = (K + STEP - 1) / STEP, slices = (steps + per - 1) / per, groups = (slices + S - 1) / S;
  const int n0 = blockIdx.x * R;
  // the row of W that is the product's row n0 + i (q/k/v: the first halves of R / 2 rotary pairs, then the second)
  auto row_of_w = [&](int i) {
    if constexpr (EPI == F32_QKV) {
      const int half = front.d / 2, p = n0 / 2 + i % (R / 2), head = p / half;
      return head * front.d + p - head * half + (i / (R / 2)) * half;
    }
    return min(n0 + i, N - 1);
  };
  const float* wrow = W + (size_t)row_of_w(r % X % R) * ldw;
  const float* arow = A + (size_t)min(r % X, M - 1) * lda;
  float* h = part + slices * X * R;
  const int ldh = K + 4;
  const float* hrow = h + min(r % X, M - 1) * ldh;
  const int jump = (waves * S - 1) * per * STEP + STEP;   // from a group's last step to the first of the wave's next
  const int mine = (groups - wave + waves - 1) / waves * per;
  f32x4 w[AHEAD], a[NORM ? 1 : AHEAD];
  int ahead = 0, ahead_k = (wave * S + r / X) * per * STEP + 4 * g;      // step in its group and column of the next loads
  auto fetch = [&](int u) {
    w[u] = load4(wrow, ahead_k, K);
    if constexpr (!NORM) a[u] = load4(arow, ahead_k, K);
    if (++ahead == per) { ahead = 0; ahead_k += jump; }
    else ahead_k += STEP;
  };
#pragma unroll
  for (int u = 0; u < AHEAD; ++u)
    if (u < mine) fetch(u);
  if constexpr (NORM > 0) {
    norm_rows<NORM>(A, norm.weight, norm.eps, h, ldh, M, K);
    __syncthreads();
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int group = wave, at = 0, k = (wave * S + r / X) * per * STEP + 4 * g;
  for (int s = 0; s < mine; s += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (s + u >= mine) break;
      const f32x4 wu = masked(w[u], k, K);
      f32x4 au;
      if constexpr (NORM > 0) au = masked(*reinterpret_cast<const f32x4*>(hrow + min(k, K - 4)), k, K);
      else au = masked(a[u], k, K);
      if (s + u + AHEAD < mine) fetch(u);
      acc = step16(wu, au, acc);
      k += STEP;
      if (++at == per) {
        // lane 16 g + c holds W's rows 4 g .. + 3 of the instruction (slice 4 g / X of the group) and token c % X of slice c / X
        const int slice = group * S + r / X;
        if (4 * g / X == r / X && 4 * g % X < R && slice < slices)
          *reinterpret_cast<f32x4*>(&part[(slice * X + r % X) * R + 4 * g % X]) = acc;
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
        at = 0;
        group += waves;
        k += jump - STEP;
      }
    }
  }
  __syncthreads();
  auto sum = [&](int m, int i) {                     // of the product's row n0 + i
    const int e = m * R + i;
    float v = part[e];
    for (int t = 1; t < slices; ++t) v += part[t * X * R + e];
    return v;
  };
  if constexpr (EPI == F32_STORE) {
    for (int e = threadIdx.x; e < M * R; e += blockDim.x) {
      const int m = e / R, n = n0 + e % R;
      if (n < N) store(C, (size_t)m * ldc + n, sum(m, e % R), bias, n, accumulate);
    }
  } else if constexpr (EPI == F32_SWIGLU) {          // rows 2 i and 2 i + 1: gate and up of feature i
    for (int e = threadIdx.x; e < M * R / 2; e += blockDim.x) {
      const int m = e / (R / 2), i = e % (R / 2) * 2;
      if (n0 + i >= N) continue;
      const float gate = sum(m, i), up = sum(m, i + 1);
      C[(size_t)m * ldc + (n0 + i) / 2] = gate / (1.0f + expf(-gate)) * up;
    }
  } else {
    for (int e = threadIdx.x; e < M * R / 2; e += blockDim.x) {
      const int m = e / (R / 2), i = e % (R / 2), n = row_of_w(i), half = front.d / 2, head = n / front.d, j = n - head * front.d;
      float x1 = sum(m, i), x2 = sum(m, i + R / 2);
      if (bias) { x1 += bias[n]; x2 += bias[n + half]; }
      if (head < front.nh + front.nkv) {
        float sn, cs;
        sincosf((float)front.positions[m] * front.inv_freq[j], &sn, &cs);
        const float a1 = x1, a2 = x2;
        x1 = a1 * cs - a2 * sn;
        x2 = a2 * cs + a1 * sn;
      }
      if (head < front.nh) {
        C[(size_t)m * ldc + n] = x1;
        C[(size_t)m * ldc + n + half] = x2;
        continue;
      }
      const long long slot = front.slots[m];
      if (slot < 0) continue;
      const long long page = slot / front.page_size;
      const int off = (int)(slot - page * front.page_size);
      const bool is_v = head >= front.nh + front.nkv;
      const int kvh = head - front.nh - (is_v ? front.nkv : 0);
      const size_t base = ((size_t)page * front.nkv + kvh) * front.page_size * front.d;
      if (is_v && front.v_transposed) {
        front.v_pages[base + (size_t)j * front.page_size + off] = x1;
        front.v_pages[base + (size_t)(j + half) * front.page_size + off] = x2;
      } else {
        float* to = (is_v ? front.v_pages : front.k_pages) + base + (size_t)off * front.d + j;
        to[0] = x1;
        to[half] = x2;
      }
    }
  }
}

// T x T tile: 4 waves of (T / 2) x (T / 2), F x F fragments each.
template <int T>
__global__ void __launch_bounds__(256)
gemm_f32_tiled_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                      float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc, int accumulate, int runs) {
  constexpr int BK = 32, LD = BK + 4;               // rows 36 floats apart: 16 rows' 16-byte reads meet every bank once
  constexpr int F = T / 32, L = T / 32;             // fragments a wave and side, 16-byte loads a thread and operand
  constexpr int AHEAD = 4;                          // steps asked for ahead: one step is 0.1 us of products, a load takes longer
  __shared__ float lds[2][2][T][LD];                // [buffer][operand]
  const int tid = threadIdx.x, lane = tid & (MS_WAVE - 1), wave = tid / MS_WAVE;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * T, m0 = blockIdx.y * T;
  const int wn = (wave & 1) * (T / 2), wm = (wave >> 1) * (T / 2);
  const int per = slice_steps(K);
  const int srow = tid >> 3, sk = (tid & 7) * 4;    // what this thread stages: rows srow + 32 i
  f32x4 total[F][F] = {}, acc[F][F] = {};
  f32x4 wreg[AHEAD][L] = {}, areg[AHEAD][L] = {};

  const float *wrow[L], *arow[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {      // rows past the end repeat the last one and are not stored
    wrow[i] = W + (size_t)min(n0 + srow + 32 * i, N - 1) * ldw;
    arow[i] = A + (size_t)min(m0 + srow + 32 * i, M - 1) * lda;
  }
  auto fetch = [&](int u, int k0) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      wreg[u][i] = load4(wrow[i], k0 + sk, K);
      areg[u][i] = load4(arow[i], k0 + sk, K);
    }
  };
  auto put = [&](int u, int b, int k0) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      *reinterpret_cast<f32x4*>(&lds[b][0][srow + 32 * i][sk]) = masked(wreg[u][i], k0 + sk, K);
      *reinterpret_cast<f32x4*>(&lds[b][1][srow + 32 * i][sk]) = masked(areg[u][i], k0 + sk, K);
    }
  };

#pragma unroll
  for (int u = 0; u < AHEAD; ++u)
    if (u * BK < K) fetch(u, u * BK);
  put(0, 0, 0);
  __syncthreads();
  int left = per;
  for (int base = 0; base < K; base += AHEAD * BK) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {               // AHEAD is even: step u of a round lies in buffer u % 2
      const int k0 = base + u * BK, b = u & 1;
      if (k0 < K) {
        fetch(u, k0 + AHEAD * BK);                  // (nothing is read past K)
#pragma unroll
        for (int kk = 0; kk < BK; kk += STEP) {
          f32x4 wf[F], af[F];
#pragma unroll
          for (int i = 0; i < F; ++i) {
            wf[i] = *reinterpret_cast<const f32x4*>(&lds[b][0][wn + 16 * i + r][kk + 4 * g]);
            af[i] = *reinterpret_cast<const f32x4*>(&lds[b][1][wm + 16 * i + r][kk + 4 * g]);
          }
#pragma unroll
          for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j) acc[i][j] = step16(wf[i], af[j], acc[i][j]);
          if (--left == 0) {      // a slice ends
            left = per;
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
              for (int j = 0; j < F; ++j) { total[i][j] += acc[i][j]; acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
          }
        }
        put((u + 1) % AHEAD, b ^ 1, k0 + BK);           // the other buffer was last read before the barrier that began this step
        __syncthreads();
      }
    }
  }
  // C goes out in rows of the tile (a wave's fragments are 64 bytes of 16 rows each): short K is bound by writing it
  constexpr int LC = T + 4;
  float* tile = &lds[0][0][0][0];                   // (nobody reads operands any more)
  static_assert(T * LC <= 2 * 2 * T * LD, "the tile of C fits where the operands lay");
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
      *reinterpret_cast<f32x4*>(&tile[(wm + 16 * j + r) * LC + wn + 16 * i + 4 * g]) = total[i][j] + acc[i][j];
  __syncthreads();
  const int c = tid % (T / 4) * 4, n = n0 + c;
#pragma unroll
  for (int p = 0; p < T * T / 1024; ++p) {
    const int row = tid / (T / 4) + p * (1024 / T), m = m0 + row;
    if (m >= M) break;
    f32x4 v = *reinterpret_cast<const f32x4*>(&tile[row * LC + c]);
    const size_t at = (size_t)m * ldc + n;
    store_run(C, at, v, bias, n, N, accumulate, runs);
  }
}

int g_kernel = 0;      // measurements: 1 the kernel of up to 64 rows, 2 and 3 the tiled one with tiles of 64 and 32, 4 and 5 that of up to 8 with blocks of 4 and 8 rows of W, 6 to 8 the slices of 16, 32 and 48 tokens; 0 leaves the choice

// Rows of W to a block of the kernel of slices side by side, for a plain product; 0: another kernel is as fast or faster.  Time with four steps to a
// load over that so, W in no cache (64 to 64,000 rows, 256 to 18,944 columns).  4 rows a block, a block a CU: up to 4 tokens from 692 columns on 0.97 to 1.5
// (896 x 4,864 with 3 tokens 11.4 | 8.5 us; 512 columns 0.94 to 1.0), 5 to 8 tokens by 1,028 to 4,864 0.94 to 1.2 (4,992 on 0.9 to 1.1, up to 1,024 0.9 to
// 1.02).  8 rows, up to 4 tokens by 1,028 to 4,864 columns 0.98 to 1.24 (4,992 on 0.88 to 1.08), 5 to 8 by up to 1,536 0.95 to 1.2 (2,048 0.93 to 1.05): a
// block a CU, or where 16 rows a block would be more than one; between these (2,049 to 4,096 rows) 0.67 to 1.0.  Up to three blocks a CU (9,728 rows 0.9 to
// 1.2 up to 4 tokens, 0.86 to 1.1 with 8).
int diagonal_rows(int M, int N, int K) {
  const int cus = ms_compute_units();
  if (M > 8) return 0;
  if ((N + 3) / 4 <= cus) return M <= 4 ? (K > 640 ? 4 : 0) : K > 1024 && K <= 4864 ? 4 : 0;
  const int blocks = (N + 7) / 8;
  return (blocks <= cus || ((N + 15) / 16 > cus && blocks <= 3 * cus)) && K > 1024 && K <= (M <= 4 ? 4864 : 1536) ? 8 : 0;
}

// Floats of LDS.
int diagonal_lds(int M, int K, int R, int X, bool normed) {
  const int steps = (K + STEP - 1) / STEP, per = slice_steps(K);
  return (steps + per - 1) / per * X * R + (normed ? M * (K + 4) : 0);
}

template <int R, int X, int EPI, int NORM>
int launch_diagonal_as(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc,
                       int accumulate, const F32Norm& norm, const F32Front& front, hipStream_t stream) {
  const int steps = (K + STEP - 1) / STEP, per = slice_steps(K), slices = (steps + per - 1) / per;
  const int groups = (slices + 16 / X - 1) / (16 / X), blocks = (N + R - 1) / R;
  const int waves = groups > 4 && blocks > 2 * ms_compute_units() ? 4 : groups;
  gemm_f32_diagonal_kernel<R, X, EPI, NORM><<<blocks, waves * MS_WAVE, diagonal_lds(M, K, R, X, NORM > 0) * sizeof(float), stream>>>(
      A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, norm, front);
  return ms_launch_status();
}

// M <= 8, R rows of W a block.
template <int EPI, int NORM>
int launch_diagonal(int R, const float* A, const float* W, const float* bias, float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc,
                    int accumulate, const F32Norm& norm, const F32Front& front, hipStream_t stream) {
#define GO(R_, X_) return launch_diagonal_as<R_, X_, EPI, NORM>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, norm, front, stream)
  if (R == 4 && M <= 4) GO(4, 4);
  if (R == 4) GO(4, 8);
  GO(8, 8);
#undef GO
}

// TM tokens by 32 rows of W a block, a wave for two slices.  Nothing is shared before the sums: a wave stages its slices' columns, 32
// at a time and the next 32 ahead, in LDS of its own (whole lines of eight rows a load) and waits for its own loads by count.
template <int TM>
__global__ void __launch_bounds__(MAX_SLICES / 2 * MS_WAVE)
gemm_f32_slices_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                       float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc, int accumulate, int runs) {
  constexpr int TN = 32, BK = 32, FN = TN / 16, FM = TM / 16, LOADS = (TN + TM) / 8, LC = TN + 4;
  extern __shared__ __align__(16) float lds[];       // [wave][2][row][8 pieces of 16 bytes]; then [slice][token][LC]
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * TN, m0 = blockIdx.y * TM;
  const int per = slice_steps(K), slices = ((K + STEP - 1) / STEP + per - 1) / per;
  const int begin = 2 * wave * per * STEP, end = min(K, begin + 2 * per * STEP);
  f32x4* mine = reinterpret_cast<f32x4*>(lds) + wave * (2 * LOADS * MS_WAVE);
  // lane l of a load takes row l / 8 of its eight, piece (l % 8) ^ (l / 8): reads of 16 rows by four pieces then meet every bank once
  const int sub = lane >> 3, piece = ((lane & 7) ^ sub) * 4;
  const float* row[LOADS];
#pragma unroll
  for (int p = 0; p < LOADS; ++p)                    // rows past the end repeat the last one and are not stored
    row[p] = p < TN / 8 ? W + (size_t)min(n0 + p * 8 + sub, N - 1) * ldw : A + (size_t)min(m0 + p * 8 - TN + sub, M - 1) * lda;
  auto ask = [&](int b, int k) {                     // (nothing is read past K)
#pragma unroll
    for (int p = 0; p < LOADS; ++p)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(row[p] + min(k + piece, K - 4)),
                                       (__attribute__((address_space(3))) void*)(mine + (b * LOADS + p) * MS_WAVE), 16, 0, 0);
  };
  f32x4 acc[FN][FM] = {}, before[FN][FM] = {};       // of the second slice, when it has begun, and the first
  int left = per, b = 0;
  bool second = false;
  ask(0, begin);
  if (begin + BK < end) ask(1, begin + BK);
  for (int k = begin; k < end; k += BK, b ^= 1) {
    f32x4 wf[2][FN], af[2][FM];
    if (k + BK < end) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = r * 8 + ((4 * h + g) ^ (r & 7));
#pragma unroll
      for (int i = 0; i < FN; ++i) wf[h][i] = mine[b * LOADS * MS_WAVE + i * 128 + at];
#pragma unroll
      for (int j = 0; j < FM; ++j) af[h][j] = mine[b * LOADS * MS_WAVE + (FN + j) * 128 + at];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // read: it may be filled again
    if (k + 2 * BK < end) ask(b, k + 2 * BK);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (k + h * STEP >= end) break;                // the same for the whole wave
      if (k + (h + 1) * STEP > K) {                  // columns past the last: nothing
#pragma unroll
        for (int i = 0; i < FN; ++i) wf[h][i] = masked(wf[h][i], k + h * STEP + 4 * g, K);
#pragma unroll
        for (int j = 0; j < FM; ++j) af[h][j] = masked(af[h][j], k + h * STEP + 4 * g, K);
      }
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = step16(wf[h][i], af[h][j], acc[i][j]);
      if (--left == 0 && !second) {                  // the first slice ends
        second = true;
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
          for (int j = 0; j < FM; ++j) { before[i][j] = acc[i][j]; acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
      }
    }
  }
  __syncthreads();
  float* sum = &lds[(2 * wave * TM + r) * LC + 4 * g];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      *reinterpret_cast<f32x4*>(sum + 16 * j * LC + 16 * i) = second ? before[i][j] : acc[i][j];
      if (2 * wave + 1 < slices) *reinterpret_cast<f32x4*>(sum + (TM + 16 * j) * LC + 16 * i) = acc[i][j];
    }
  __syncthreads();
  for (int e = threadIdx.x; e < TM * TN / 4; e += blockDim.x) {
    const int tok = e / (TN / 4), c = e % (TN / 4) * 4, m = m0 + tok, n = n0 + c;
    if (m >= M) break;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < slices; ++s) v += *reinterpret_cast<const f32x4*>(&lds[(s * TM + tok) * LC + c]);
    store_run(C, (size_t)m * ldc + n, v, bias, n, N, accumulate, runs);
  }
}

int slices_of(int K) { const int steps = (K + STEP - 1) / STEP, per = slice_steps(K); return (steps + per - 1) / per; }
// bytes: two stages of 32 columns a wave, or the slices' sums
int slices_lds(int TM, int slices) { return std::max((slices + 1) / 2 * 2 * (32 + TM) * 32, slices * TM * (32 + 4)) * (int)sizeof(float); }

// The kernel for more than 8 rows by 512 columns and more, by what each was seen to take at 4,600 sizes (64 to 64,000 by 512 to 18,944, 9 to 2,048
// rows; 256 CUs, W in no cache): a start, the reading of W by the MB, and rounds.  `slices` is bound by what a CU reads however many blocks it has at once;
// only their beginnings overlap, one to four to a CU by its LDS.  Of the tiled one's blocks several lie on a CU, and up to one a CU they take as long
// as one.  Rows that are no multiple of 128 bytes cost `slices` 1.1 to 1.45 times the time (`apart`), the first kernel 1.13, the tiles nothing.  The kernel so
// chosen is 0.8 % behind the fastest on average, 21 % at worst (by tiles and slices as if the blocks of a CU did not share it, and W's rows lay on 128 bytes,
// 2.5 % and 7.8 % behind with rows that do and that do not, and twice the time at worst: 9 rows of 401 x 13,188 38 -> 72 -> 38 us, 512 of 64,000 x 512 331 ->
// 571 -> 331, 1,000 of 3,072 x 768 50 -> 76 -> 50).  Before, by the number of tiles alone and with tiled kernels alone | now: 896 x 4,864 at 17, 64, 350, 512 and
// 2,048 rows 24 | 18, 47 | 18, 81 | 45, 82 | 56, 224 | 192 us; 896 x 896 at 64 and 350 12.5 | 6.9, 18.0 | 13.1; 1,152 x 896 at 350 18.1 | 16.8; 4,608 x 3,584 at
// 17 and 128 41 | 25, 80 | 65; 9,728 x 896 as before.
enum { ROWS16 = 16, ROWS32 = 32, ROWS48 = 48, TILE32 = 1, TILE64 = 2, ROWS = 3 };
int rows_a_block(int N, int cus) { return (N + 3) / 4 <= cus ? 4 : (N + 7) / 8 <= cus ? 8 : 16; }
int choose(int M, int N, int K, bool apart, int cus) {
  int best = 0;
  float least = 0.f;
  auto offer = [&](int kind, float us) { if (best == 0 || us < least) { best = kind; least = us; } };
  auto tiles = [&](int T) { return (float)((long long)((N + T - 1) / T) * ((M + T - 1) / T)) / cus; };
  const float k = K * 1e-3f, mb = k * N * 4e-3f, t64 = tiles(64), t32 = tiles(32);
  offer(TILE64, 2.6f + 0.05f * mb + (2.6f + 23.2f * k) * (t64 <= 1.f ? 1.f : std::max(1.63f, 0.43f + 0.73f * t64)));
  offer(TILE32, 2.1f + 0.09f * mb + (1.f + 14.1f * k) * (t32 <= 1.f ? 1.f : std::max(1.19f, 0.44f + 0.433f * t32)));
  const struct { float begin, step, whole, read, begin_apart, step_apart; } kinds[] = {
      {1.7f, 3.09f, 0.71f, 0.169f, 1.29f, 1.39f}, {2.88f, 4.83f, 0.9f, 0.117f, 1.36f, 1.2f}, {3.33f, 7.57f, 0.94f, 0.088f, 1.45f, 1.1f}};
  for (int i = 0; i < 3; ++i) {
    const auto& t = kinds[i];
    const int TM = 16 * (i + 1), at_once = cus * std::min(4, LDS_BYTES / slices_lds(TM, slices_of(K)));
    const long long blocks = (long long)((N + 31) / 32) * ((M + TM - 1) / TM);
    if ((M + TM - 1) / TM > 65535) continue;
    const float begin = t.begin * (apart ? t.begin_apart : 1.f), step = t.step * k * (apart ? t.step_apart : 1.f);
    offer(TM, 2.2f + t.read * mb + begin * ((blocks + at_once - 1) / at_once) +
                  step * (t.whole * ((blocks + cus - 1) / cus) + (1.f - t.whole) * std::max(1.f, (float)blocks / cus)));
  }
  if (M <= 64) {
    const int R = rows_a_block(N, cus), nt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    const float share = (float)((N + R - 1) / R) / cus;
    offer(ROWS, 2.7f + 0.41f * nt + (1.4f + 0.14f * R + 0.111f * M + 0.028f * R * nt) * k * (apart ? 1.13f : 1.f) * (share <= 1.f ? 1.f : 0.72f + 0.9f * share));
  }
  return best;
}

template <int TM>
int launch_slices(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc,
                  int accumulate, int runs, hipStream_t stream) {
  const int slices = slices_of(K);
  static bool raised = false;   // once per instantiation: allow more dynamic LDS than the default 64 KB
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_slices_kernel<TM>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            slices_lds(TM, MAX_SLICES)) != hipSuccess)
      return MS_LAUNCH_FAILED;
    raised = true;
  }
  gemm_f32_slices_kernel<TM><<<dim3((N + 31) / 32, (M + TM - 1) / TM), (slices + 1) / 2 * MS_WAVE, slices_lds(TM, slices), stream>>>(
      A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, runs);
  return ms_launch_status();
}

}  // namespace

// What a decode step's layer makes of up to 8 rows of the residual stream x [M, K] with the norm of its reader, one kernel each:
// the gated product, act [M, N / 2] = silu(gate) * up over interleaved rows of W, and q, k and v with their bias, q to q_out's rows of
// (nh + 2 nkv) d, k and v to their pages.  The bits are those of ms_rms_norm, ms_gemm_generic and ms_silu_mul or ms_rope_store one after the other.
// MS_UNSUPPORTED: sizes or addresses that the kernel does not take.
int ms_gemm_f32_normed(const float* x, const float* W, const float* bias, float* out, int M, int N, int K, const F32Norm& norm,
                       const F32Front* front, hipStream_t stream) {
  if (M > 8 || K % 4 || K > 2048 || ((uintptr_t)x | (uintptr_t)W | (uintptr_t)norm.weight) % 16) return MS_UNSUPPORTED;
  if (front ? front->d % 8 || N != (front->nh + 2 * front->nkv) * front->d : N % 2) return MS_UNSUPPORTED;
  if ((long long)N * K > 32000000) return MS_UNSUPPORTED;      // (64,000 x 1,536 at 8 rows: 119 us so, 101 in the kernel of four steps to a load)
  const int R = (N + 3) / 4 <= 2 * ms_compute_units() ? 4 : 8, X = R == 4 && M <= 4 ? 4 : 8;
  if (diagonal_lds(M, K, R, X, true) * sizeof(float) > 65536) return MS_UNSUPPORTED;      // what a launch may ask for without more ado
  const size_t ldc = front ? N : N / 2;
#define GO(EPI, NORM) return launch_diagonal<EPI, NORM>(R, x, W, bias, out, M, N, K, K, K, ldc, 0, norm, front ? *front : F32Front{}, stream)
  if (front) { if (K <= 1024) GO(F32_QKV, 4); else GO(F32_QKV, 8); }
  if (K <= 1024) GO(F32_SWIGLU, 4); else GO(F32_SWIGLU, 8);
#undef GO
}

namespace {

// Below 512 columns, which writing C bounds: the tiles, the larger ones from two a CU on, but few rows against few of W in the first kernel (of more than 16
// rows every block of it reads all of A, a tile its part once through LDS; 24 rows of 20,000 x 512 17.2 us there, 15.3 in tiles, 32 of 152,064 x 3,584 1,010 and
// 519, 64 of 151,936 x 896 405 and 220, of 6,144 x 2,048 43 and 40, but 33 of them 33 and 40).
int kind_of(int M, int N, int K, bool apart, int cus) {
  if (M <= 8) return ROWS;
  if (K >= 512) return choose(M, N, K, apart, cus);
  if (M <= 16 || (M <= 32 ? N < 64 * cus : M <= 64 && N < 32 * cus)) return ROWS;
  return M > 32 && (long long)((N + 63) / 64) * ((M + 63) / 64) >= 2 * cus ? TILE64 : TILE32;
}

}  // namespace

extern "C" void ms_gemm_f32_force(int kernel) { g_kernel = kernel; }
extern "C" int ms_gemm_f32_kernel(int M, int N, int K) {
  const int side_by_side = diagonal_rows(M, N, K), kind = side_by_side ? 0 : kind_of(M, N, K, K % 32 != 0, ms_compute_units());
  return side_by_side ? 3 + side_by_side / 4 : kind == ROWS ? 1 : kind == TILE64 ? 2 : kind == TILE32 ? 3 : 5 + kind / 16;
}

// The caller has checked sizes; K, lda and ldw are multiples of 4 and A and W lie on 16 bytes.
int ms_gemm_f32_launch(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, size_t lda,
                       size_t ldw, size_t ldc, int accumulate, hipStream_t stream) {
  const int cus = ms_compute_units();
  const int side_by_side = M > 8 ? 0 : g_kernel == 4 ? 4 : g_kernel == 5 ? 8 : g_kernel == 0 ? diagonal_rows(M, N, K) : 0;
  if (side_by_side)
    return launch_diagonal<F32_STORE, 0>(side_by_side, A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, F32Norm{}, F32Front{}, stream);
  const int kind = g_kernel == 1 && M <= 64 ? ROWS : g_kernel == 2 ? TILE64 : g_kernel == 3 ? TILE32 : g_kernel >= 6 ? 16 * (g_kernel - 5)
                   : kind_of(M, N, K, lda % 32 || ldw % 32, cus);
  if (kind == ROWS) {
    // Rows a block: as few as keep the blocks within the CUs, because a CU reads at a rate of its own and 16 bytes a lane
    // fill 64-byte pieces from 4 rows as from 16 (3 rows of 896 x 4,864: 18.3 us as 56 blocks of 16, 17.2 as 224 of 4;
    // q/k/v 6.5 and 6.3).  More tiles than CUs: blocks of four waves, several of them on a CU, instead of one that has a
    // wave for every slice (9,728 x 896: 19.6 us, now 11.9; the head 161, now 100).
    const int R = rows_a_block(N, cus);
    const int steps = (K + STEP - 1) / STEP, per = slice_steps(K), slices = (steps + per - 1) / per;
    const int waves = (N + R - 1) / R > cus && slices > 4 ? 4 : slices;
    dim3 grid((N + R - 1) / R), block(waves * MS_WAVE);
#define ROWS2(R_, NT) gemm_f32_rows_kernel<R_, NT><<<grid, block, (size_t)slices * NT * 256 * sizeof(float), stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate)
#define ROWS(NT) do { if (R == 4) ROWS2(4, NT); else if (R == 8) ROWS2(8, NT); else ROWS2(16, NT); } while (0)
    // Loads of four steps (up to 8 tokens): always where a block has 4 or 8 rows of W (3 tokens: 896 x 896 5.4 -> 4.3 us, 896 x 4,864
    // 15.9 -> 11.8, 2,048 x 2,048 9.1 -> 7.7), with 16 rows, whose loads were full, from more than four steps to a slice on
    // (6,144 x 1,536 16.4 -> 15.0, 64,000 x 1,536 99 -> 85; with four 9,728 x 896 11.8 and 12.4, x 1,024 12.9 and 13.7, others even).
    const bool grouped = M <= 8 && (R < 16 || per > 4);
#define FEW2(R_, G_) gemm_f32_few_kernel<R_, G_><<<grid, block, (size_t)slices * R_ * G_ * sizeof(float), stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate)
#define FEW(G_) do { if (R == 4) FEW2(4, G_); else if (R == 8) FEW2(8, G_); else FEW2(16, G_); } while (0)
    if (grouped && M <= 4) FEW(4);
    else if (grouped) FEW(8);
    else if (M <= 16) ROWS(1);
    else if (M <= 32) ROWS(2);
    else ROWS(4);
#undef ROWS2
#undef FEW2
#undef FEW
#undef ROWS
    return ms_launch_status();
  }
  const int runs = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
#define SLICES(TM) return launch_slices<TM>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, runs, stream)
  if (kind == ROWS16) SLICES(16);
  if (kind == ROWS32) SLICES(32);
  if (kind == ROWS48) SLICES(48);
#undef SLICES
#define TILED(T) gemm_f32_tiled_kernel<T><<<dim3((N + T - 1) / T, (M + T - 1) / T), 256, 0, stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, runs)
  if (kind == TILE64) TILED(64);
  else TILED(32);
#undef TILED
  return ms_launch_status();
}
