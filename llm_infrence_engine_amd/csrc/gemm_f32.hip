// C[M,N] (+)= A[M,K] . W[N,K]^T (+ bias[N]) in true 32 bits: float operands, float products and float sums, on the
// matrix cores' float instruction (v_mfma_f32_16x16x4_f32: nothing is rounded below 32 bits).
//
// The order of a sum is the same whatever M is, so a token's result does not depend on what else is in the batch: K is
// cut into at most 16 slices (from K alone, `slice_steps`), a slice is summed 16 values at a time from its start, and the
// slices are added in order.  Two kernels keep that order:
//   rows     up to 64 rows (a decode step; against very many rows of W up to 16): all waves of a block on the same 4 to 16
//            rows of W, the slices dealt out over them and added through LDS.  Bound by reading W.
//   few      up to 8 rows, of these: loads that take four steps at a time.
//   tiled    the others: 64 x 64 or 32 x 32 tiles staged through LDS four steps ahead, 4 waves; 32 x 32 where the larger
//            tiles would be fewer than two a CU.  Bound by the float matrix rate (157 TFLOP/s nominal), short K by writing C.
// Measured with the 0.5B sizes against the 64 x 64 vector-ALU tile that ran them before (one MI355X): of 3 rows the down
// product (896 x 4,864) 319 -> 16 us (12 with grouped loads), gate/up (9,728 x 896) 63 -> 12 us, q/k/v (1,152 x 896) 63 -> 4.5 us, the head
// (151,936 x 896) 221 -> 100 us, of 64 rows 252 -> 220; of 338 rows down 316 -> 84 us, gate/up 108 -> 88 us.  Down is bound
// by the steps a CU works off (16 waves, 19 steps each), whatever its rows; the tiled steps by the way from one barrier to
// the next.  C leaves a tile through LDS in whole rows (4,096 x 32,000 x 64: 440 us as the fragments lie, 270 so, 261 before).
#include "common.h"
#include "api.h"
#include "quads.h"
#include <type_traits>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int STEP = 16;          // k values a slice is summed by at a time: four MFMAs of four
constexpr int MAX_SLICES = 16;

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
}

int g_kernel = 0;      // measurements: 1 the kernel of few rows, 2 and 3 the tiled one with tiles of 64 and 32; 0 leaves the choice

}  // namespace

extern "C" void ms_gemm_f32_force(int kernel) { g_kernel = kernel; }

// The caller has checked sizes; K, lda and ldw are multiples of 4 and A and W lie on 16 bytes.
int ms_gemm_f32_launch(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, size_t lda,
                       size_t ldw, size_t ldc, int accumulate, hipStream_t stream) {
  const int cus = ms_compute_units();
  // More than 16 rows against many: every block of the first kernel reads all of A, a tile its part once through LDS.  17 to 32
  // rows from 64 features a CU on (24 rows of 20,000 x 512 17.2 us there, 15.3 in tiles; 32 of 152,064 x 3,584 1,010 and 519;
  // of 9,728 x 896 19.3 and 19.1), 33 to 64 from 32 a CU on (64 of 9,728 x 896 33 and 24, of 151,936 x 896 405 and 220, of
  // 6,144 x 2,048 43 and 40, but 33 of them 33 and 40).
  const bool few = M <= 16 || (M <= 32 ? N < 64 * cus : M <= 64 && N < 32 * cus);
  if (g_kernel == 1 ? M <= 64 : g_kernel == 0 && few) {
    // Rows a block: as few as keep the blocks within the CUs, because a CU reads at a rate of its own and 16 bytes a lane
    // fill 64-byte pieces from 4 rows as from 16 (3 rows of 896 x 4,864: 18.3 us as 56 blocks of 16, 17.2 as 224 of 4;
    // q/k/v 6.5 and 6.3).  More tiles than CUs: blocks of four waves, several of them on a CU, instead of one that has a
    // wave for every slice (9,728 x 896: 19.6 us, now 11.9; the head 161, now 100).
    const int R = (N + 3) / 4 <= cus ? 4 : (N + 7) / 8 <= cus ? 8 : 16;
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
  const long long big = (long long)((N + 63) / 64) * ((M + 63) / 64);
  const int runs = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
  if (g_kernel == 2 || (g_kernel != 3 && M > 32 && big >= 2 * cus))
    gemm_f32_tiled_kernel<64><<<dim3((N + 63) / 64, (M + 63) / 64), 256, 0, stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, runs);
  else
    gemm_f32_tiled_kernel<32><<<dim3((N + 31) / 32, (M + 31) / 32), 256, 0, stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate, runs);
  return ms_launch_status();
}
