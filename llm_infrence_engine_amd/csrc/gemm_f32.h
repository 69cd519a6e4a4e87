// The 32-bit products' entry points within the library (gemm_f32.hip).
#pragma once
#include "common.h"

// The norm that a product's rows are still to pass: scale and epsilon.
struct F32Norm {
  const float* weight;
  float eps;
};

// What the q/k/v product needs beside its operands: W's rows are [q heads | k heads | v heads] of d, turned whole in half-split pairs.
struct F32Front {
  const int *positions, *slots;
  const float* inv_freq;
  float *k_pages, *v_pages;
  int nh, nkv, d, page_size, v_transposed;
};

// The caller has checked sizes; K, lda and ldw are multiples of 4 and A and W lie on 16 bytes.
int ms_gemm_f32_launch(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, size_t lda, size_t ldw, size_t ldc,
                       int accumulate, hipStream_t stream);
int ms_gemm_f32_normed(const float* x, const float* W, const float* bias, float* out, int M, int N, int K, const F32Norm& norm,
                       const F32Front* front, hipStream_t stream);
