// out[M,N] = A[M,K] . W[N,K]^T for up to 8 rows and a narrow W (decode steps: the output and down projections, the
// pieces of the latent and recurrent layers), bfloat16 in, float accumulation (v_mfma_f32_16x16x32_bf16).
//
// What bounds these is latency, not memory: a launch is 1.6 us, 224 blocks that read 4 MB, pass one barrier and store take
// 2.5 to 2.8, and the tiled kernel took 3.9 for a matrix of 1.6 MB: 56 blocks of 16 rows, whose waves wait for four or five
// loads one after another.  Here a block owns one or two units of FOUR rows, so that there are as many blocks as CUs, and a
// wave's whole share (up to four k-steps a load, three loads in flight) is asked for in one go, each load 1 KB (quads.h says
// how); one barrier, and a lane adds one output.  The sums are those of gemm_skinny.hip, in the same order, to the bit.
// 896 x 896, residual: 3.9 -> 2.8 us at one token (0.6 TB/s; the launch is 1.6), 896 x 4864: 6.1 -> 5.1.  Asking for more
// columns at a time on v_mfma_f32_4x4x4_16b was up to 0.5 us faster still, but adds in another order than more rows do.
#include "common.h"
#include "api.h"
#include "quads.h"

namespace {

// U: units of four rows of W to a block; G: tokens; C: loads of W a wave has in flight
template <int WAVES, int C, int U, int G, int EPI, typename TO, bool NORM>
__global__ void __launch_bounds__(WAVES * MS_WAVE)
gemm_quads_kernel(const void* __restrict__ A, size_t lda, const bf16* __restrict__ W, size_t ldw,
                   const float* __restrict__ bias, TO* __restrict__ out, size_t ldo, int M, int N, int K,
                   const float* __restrict__ norm_w, float eps, const int* __restrict__ rows) {
  __shared__ quad_f32 part[U][WAVES][G];
  __shared__ float part_ss[NORM ? WAVES : 1][G];
  const int lane = threadIdx.x & (MS_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);   // the same for the whole wave
  const int r0 = blockIdx.x * (4 * U);

  const bf16* wrow[U];
#pragma unroll
  for (int u = 0; u < U; ++u) wrow[u] = W + (size_t)min(r0 + 4 * u + (lane & 3), N - 1) * ldw;
  const int xm = min(lane & (G - 1), M - 1);
  const size_t xoff = (size_t)(rows ? rows[xm] : xm) * lda;
  const void* x = NORM ? (const void*)((const float*)A + xoff) : (const void*)((const bf16*)A + xoff);

  QuadProduct<U, G, C, NORM> product(lane, wave, WAVES, K);
  product.ask(0, wrow, x, norm_w);
  // What the epilogue needs from memory arrives under the products: wave u finishes unit u, lane r G + m its row r for
  // token m.
  const int m = lane & (G - 1), r = (lane / G) & 3, n0 = r0 + 4 * min(wave, U - 1);
  const int nc = min(n0 + r, N - 1);
  const float pre = EPI == EPI_RESIDUAL ? reinterpret_cast<const float*>(out)[(size_t)min(m, M - 1) * ldo + nc] : 0.f;
  const float bv = bias && !ms_gated(EPI) && EPI != EPI_XIELU ? bias[nc] : 0.f;
  // the xIELU's two numbers, worked out of what is learned as it is at the time, side by side in two lanes of the waves that finish, while W
  // is on its way (behind the products they were 0.6 us of 3)
  float sp = 0.f;
  if constexpr (EPI == EPI_XIELU) {
    if (wave < U) {
      sp = softplus_f(lane & 1 ? bias[1] : bias[0]);
      asm volatile("" : "+v"(sp));
    }
  }
  product.run(wrow, x, norm_w);

  // rows 0 to 3 of a tile lie in lanes 0 to 15, one token to a lane
  if (lane < G) {
#pragma unroll
    for (int u = 0; u < U; ++u) part[u][wave][lane] = product.acc[u];
  }
  if constexpr (NORM) {
    const float v = quad_sum_rows(product.ss);
    if (lane < G) part_ss[wave][lane] = v;
  }
  __syncthreads();
  if (wave >= U) return;
  const float ap = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sp), 0));
  const float an = 0.5f + __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sp), 1));
  float scale = 1.f;
  if constexpr (NORM) {
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) total += part_ss[w][m];
    scale = 1.0f / sqrtf(total / (float)K + eps);
  }
  if (m >= M) return;
  const float* mine = reinterpret_cast<const float*>(&part[wave][0][m]);
  if constexpr (ms_gated(EPI)) {
    // rows n0, n0+1 are (gate, up) of feature n0/2; rows n0+2, n0+3 of feature n0/2 + 1
    const int p = r & 1;
    float g = 0.f, up = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      g += mine[w * G * 4 + 2 * p];
      up += mine[w * G * 4 + 2 * p + 1];
    }
    if constexpr (NORM) { g *= scale; up *= scale; }
    if (lane < 2 * G && n0 + 2 * p + 1 < N)
      out[(size_t)m * ldo + n0 / 2 + p] = from_float<TO>(ms_gate_value<EPI>(g, up, bias));
  } else {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v += mine[w * G * 4 + r];
    if constexpr (NORM) {
      v *= scale;
      asm("" : "+v"(v));   // rounded here, as in ms_gemm_skinny: not one operation with the bias
    }
    if (lane < 4 * G && n0 + r < N) out[(size_t)m * ldo + n0 + r] = from_float<TO>(EPI == EPI_XIELU ? ms_xielu_value(v, ap, an) : ms_store_value<EPI>(v + bv + pre));
  }
}

// Where this kernel is the faster one (us, before against with it, unless said as before/with).  Narrow matrices gain because
// their blocks elsewhere are few and each a chain of dependent loads; what costs here is that a wave's load of W takes four
// k-steps whether it has four or not, and that every block reads all the activations.  `full`: a wave's steps in sixteenths
// of what its loads could take.
//   One unit a block (a CU for every block): always but for the shortest rows.  896 x 896 at one token 3.9 | 2.8, at 8 4.0 |
//     3.4; 896 x 4864 6.1 | 5.1; 256 columns are even to 5 % worse, 264 even to 6 % better; with the norm, which reads twice the
//     bytes of activations, up to 384 columns 3 to 9 % worse, from 416 on better.
//   Two units a block: rows whose loads are full enough.  1344 x 512 0.97 to 1.02, x 576 1.04 to 1.15, x 896 1.16 to 1.27,
//     x 1024 (half full: two steps to each of 16 waves) 0.92 to 1.01, x 2048 1.12 to 1.23, x 2560 0.93 to 1.03, from 3072 on
//     1.0 to 1.4; where K fills the last step in part, which costs the others more, x 1000 and x 1032 1.05 to 1.15.  5 to 8
//     tokens pay for one round of loads only (896 x 4864: 6.8 | 7.1), 3 or 4 up to 6144 columns (896 x 7296: 7.4 | 8.0).
//     With the norm x 576 1.03 to 1.10 at two tokens, at 4 0.96 to 1.03 (x 640 0.98 to 1.06), at 8 from 896 columns on 1.0
//     to 1.06.
//   Wider ones, measured up to 8 units a CU: full loads of up to 4 tokens (7296 x 896 6.3 | 5.4; 4100 x 992 1.1 to 1.2, x 640
//     0.91 to 1.05, x 1000, where 16 waves have two steps each, 0.84 to 0.93; 8192 x 1024 0.6 to 0.7).
// (9 to 16 tokens stay with ms_gemm_stream and ms_gemm_skinny.)
bool pays(int M, int units, int K, int waves, int loads, bool norm, int cus) {
  if (M > 8) return false;
  const int full = 4 * ((K + 31) / 32) / (waves * loads);
  if (units <= cus) {
    if (norm) return K > 384 && K <= 1024;
    return K > 256 && (M <= 2 || K <= (M <= 4 ? 6144 : 4096));
  }
  if (units <= 2 * cus) {
    const bool part = K % 32 != 0;
    if (waves == 8) return full >= (norm && M > 4 ? 14 : norm && M > 2 ? 10 : 9);
    if (K <= 1024) return part || (norm && M > 4);
    return !norm && M <= 4 && (M <= 2 || K <= 6144) && (part || loads >= 3 || full >= (M > 2 ? 12 : 11));
  }
  return units <= 8 * cus && !norm && M <= 4 && waves == 8 && full >= 13;
}

template <int EPI, typename TO, bool NORM>
int plan(const void* A, size_t lda, const bf16* W, size_t ldw, const float* bias, TO* out, size_t ldo, int M, int N,
         int K, const float* norm_w, float eps, const int* rows, hipStream_t stream) {
  const int cus = ms_compute_units();
  const int units = (N + 3) / 4;
  // waves as ms_gemm_skinny would take for the shape: the order of the sums goes by them
  const int tiles = (N + 15) / 16, skinny_blocks = tiles <= cus ? tiles : cus * ((tiles + 4 * cus - 1) / (4 * cus));
  const int waves = (tiles + skinny_blocks - 1) / skinny_blocks >= 3 || K <= 992 ? 8 : 16;
  const int loads = ((K + 31) / 32 + 4 * waves - 1) / (4 * waves);   // of W to a wave and unit
  if (!pays(M, units, K, waves, loads, NORM, cus)) return MS_UNSUPPORTED;
  const int u = units <= cus ? 1 : 2;
  const int rounds = (loads + (u == 1 ? 2 : 1)) / (u == 1 ? 3 : 2);
  const int c = NORM ? 1 : (loads + rounds - 1) / rounds;
#define GO(WV, CV, UV, GV) \
  if (waves == WV && c == CV && u == UV) { \
    gemm_quads_kernel<WV, CV, UV, GV, EPI, TO, NORM><<<dim3((units + UV - 1) / UV), dim3(WV * MS_WAVE), 0, stream>>>( \
        A, lda, W, ldw, bias, out, ldo, M, N, K, norm_w, eps, rows); \
    return ms_launch_status(); \
  }
  // (those that `pays` can ask for)
#define ONE(GV) GO(8, 1, 1, GV) GO(16, 1, 1, GV) GO(8, 1, 2, GV) GO(16, 1, 2, GV)
  if (M <= 4) { ONE(4) } else { ONE(8) }
  if constexpr (!NORM) {
    if (M <= 4) { GO(16, 2, 1, 4) GO(16, 3, 1, 4) GO(16, 2, 2, 4) } else { GO(16, 2, 1, 8) }
  }
#undef ONE
#undef GO
  return MS_UNSUPPORTED;
}

}  // namespace

// As ms_gemm_stream, for the shapes that it is the faster kernel for; MS_UNSUPPORTED for the others.
extern "C" int ms_gemm_quads(const void* A, long long lda, const int* rows, const float* norm_w, float eps,
                              const void* W, long long ldw, const float* bias, void* out, long long ldo, int M, int N,
                              int K, int epilogue, int out_dtype, int norm, hipStream_t stream) {
  if (M <= 0 || N <= 0) return MS_OK;
  if (K <= 0 || K % 8 || ldw % 8 || lda < K || ldw < K || lda % (norm ? 4 : 8)) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W) % 16 || (norm && ((uintptr_t)norm_w % 16))) return MS_UNSUPPORTED;
  if (norm && !norm_w) return MS_BAD_ARG;
  const bf16* w = (const bf16*)W;
#define RUN(EPI, TO, NORMV) return plan<EPI, TO, NORMV>(A, lda, w, ldw, bias, (TO*)out, ldo, M, N, K, norm_w, eps, rows, stream)
  if (epilogue == EPI_STORE) {
    if (ldo < N) return MS_BAD_ARG;
    if (out_dtype == MS_BF16) { if (norm) RUN(EPI_STORE, bf16, true); else RUN(EPI_STORE, bf16, false); }
    if (out_dtype == MS_F32) { if (norm) RUN(EPI_STORE, float, true); else RUN(EPI_STORE, float, false); }
    return MS_BAD_ARG;
  }
  if (epilogue == EPI_SWIGLU) {
    if (N % 2 || ldo < N / 2 || out_dtype != MS_BF16 || bias) return MS_BAD_ARG;
    if (norm) RUN(EPI_SWIGLU, bf16, true); else RUN(EPI_SWIGLU, bf16, false);
  }
  if (epilogue == EPI_CLAMPED) {
    if (N % 2 || ldo < N / 2 || out_dtype != MS_BF16 || norm || !bias) return MS_BAD_ARG;
    RUN(EPI_CLAMPED, bf16, false);
  }
  if (epilogue == EPI_XIELU) {
    if (ldo < N || out_dtype != MS_BF16 || norm || !bias) return MS_BAD_ARG;
    RUN(EPI_XIELU, bf16, false);
  }
  if (epilogue == EPI_RELU2) {
    if (ldo < N || out_dtype != MS_BF16 || norm) return MS_BAD_ARG;
    RUN(EPI_RELU2, bf16, false);
  }
  if (epilogue == EPI_RESIDUAL) {
    if (ldo < N || out_dtype != MS_F32 || norm) return MS_BAD_ARG;
    RUN(EPI_RESIDUAL, float, false);
  }
#undef RUN
  return MS_BAD_ARG;
}
