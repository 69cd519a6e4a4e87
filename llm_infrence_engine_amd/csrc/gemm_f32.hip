// C[M,N] (+)= A[M,K] . W[N,K]^T (+ bias[N]) in true 32 bits: float operands, float products and float sums, on the
// matrix cores' float instruction (v_mfma_f32_16x16x4_f32: nothing is rounded below 32 bits).
//
// The order of a sum is the same whatever M is, so a token's result does not depend on what else is in the batch: K is
// cut into at most 16 slices (from K alone, `slice_steps`), a slice is summed 16 values at a time from its start, and the
// slices are added in order.  Two kernels keep that order:
//   rows     M <= 64 (a decode step): all waves of a block on the same 4 to 16 rows of W, the slices dealt out over them
//            and added through LDS.  Bound by reading W.
//   tiled    more rows: 64 x 64 or 32 x 32 tiles staged through LDS four steps ahead, 4 waves; 32 x 32 where the larger
//            tiles would be fewer than two a CU.  Bound by the float matrix rate (157 TFLOP/s nominal).
// Measured with the 0.5B sizes against the 64 x 64 vector-ALU tile that ran them before (one MI355X): of 3 rows the down
// product (896 x 4,864) 319 -> 17 us, gate/up (9,728 x 896) 63 -> 12 us, q/k/v (1,152 x 896) 63 -> 6.3 us, the head
// (151,936 x 896) 221 -> 100 us; of 338 rows down 316 -> 84 us, gate/up 108 -> 88 us.  Down is bound by the steps a CU
// works off (16 waves, 19 steps each), whatever its rows; the tiled steps by the way from one barrier to the next.
#include "common.h"
#include "api.h"

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
  __shared__ float part[MAX_SLICES][NT * 256];      // [slice][token][row of W]
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
    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(&part[slice][(t * 16 + r) * 16 + 4 * g]) = acc[t];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < NT * 16 * R; e += blockDim.x) {
    const int m = e / R, n = n0 + e % R, at = m * 16 + e % R;
    if (m >= M || n >= N) continue;
    float v = part[0][at];
    for (int s = 1; s < slices; ++s) v += part[s][at];
    store(C, (size_t)m * ldc + n, v, bias, n, accumulate);
  }
}

// T x T tile: 4 waves of (T / 2) x (T / 2), F x F fragments each.
template <int T>
__global__ void __launch_bounds__(256)
gemm_f32_tiled_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                      float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc, int accumulate) {
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
  f32x4 wreg[AHEAD][L], areg[AHEAD][L];

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
  for (int u = 0; u < AHEAD; ++u) fetch(u, u * BK);
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
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) {
      total[i][j] += acc[i][j];
      const int m = m0 + wm + 16 * j + r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + wn + 16 * i + 4 * g + e;
        if (m < M && n < N) store(C, (size_t)m * ldc + n, total[i][j][e], bias, n, accumulate);
      }
    }
}

}  // namespace

// The caller has checked sizes; K, lda and ldw are multiples of 4 and A and W lie on 16 bytes.
int ms_gemm_f32_launch(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, size_t lda,
                       size_t ldw, size_t ldc, int accumulate, hipStream_t stream) {
  if (M <= 64) {
    // Rows a block: as few as keep the blocks within the CUs, because a CU reads at a rate of its own and 16 bytes a lane
    // fill 64-byte pieces from 4 rows as from 16 (3 rows of 896 x 4,864: 18.3 us as 56 blocks of 16, 17.2 as 224 of 4;
    // q/k/v 6.5 and 6.3).  More tiles than CUs: blocks of four waves, several of them on a CU, instead of one that has a
    // wave for every slice (9,728 x 896: 19.6 us, now 11.9; the head 161, now 100).
    const int cus = ms_compute_units();
    const int R = (N + 3) / 4 <= cus ? 4 : (N + 7) / 8 <= cus ? 8 : 16;
    const int steps = (K + STEP - 1) / STEP, per = slice_steps(K), slices = (steps + per - 1) / per;
    const int waves = (N + R - 1) / R > cus && slices > 4 ? 4 : slices;
    dim3 grid((N + R - 1) / R), block(waves * MS_WAVE);
#define ROWS2(R_, NT) gemm_f32_rows_kernel<R_, NT><<<grid, block, 0, stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate)
#define ROWS(NT) do { if (R == 4) ROWS2(4, NT); else if (R == 8) ROWS2(8, NT); else ROWS2(16, NT); } while (0)
    if (M <= 16) ROWS(1);
    else if (M <= 32) ROWS(2);
    else ROWS(4);
#undef ROWS2
#undef ROWS
    return ms_launch_status();
  }
  const long long big = (long long)((N + 63) / 64) * ((M + 63) / 64);
  if (big >= 2 * ms_compute_units())
    gemm_f32_tiled_kernel<64><<<dim3((N + 63) / 64, (M + 63) / 64), 256, 0, stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate);
  else
    gemm_f32_tiled_kernel<32><<<dim3((N + 31) / 32, (M + 31) / 32), 256, 0, stream>>>(A, W, bias, C, M, N, K, lda, ldw, ldc, accumulate);
  return ms_launch_status();
}
