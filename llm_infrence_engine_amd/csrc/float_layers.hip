// All layers of a 32-bit step by one call, to the same bits as when every part is asked for by itself: its nine kernels a layer, or, up to 8
// tokens where the products take the norms, the rotation and the gate (ms_gemm_f32_normed: hidden sizes up to 2,048, matrices up to 32 million
// values, rows that fit 64 KB of LDS), five; the q/k/v and the gated product each for itself.  A decode step of the 32-bit path was as slow as its launches were made: 219 of them took 2.62 ms from
// Python (12 us each, of which the launch itself is 4) where the GPU has 1.7 ms of work; with five it has 1.2 (0.5B sizes, 3 tokens behind
// 130: two norms, the rotation and the activation were 15.6 us of a layer's 70, and are 1 to 2 of the products' that took them in).
#include "common.h"
#include "api.h"
#include "gemm_f32.h"

namespace {

// Device addresses of one layer's weights and pages; in host memory.
struct FloatLayer {
  const float *norm1, *w_qkv, *b_qkv, *inv_freq, *w_o, *norm2, *w_gate_up, *w_down;
  float *k_pages, *v_pages;
  float eps1, eps2;
};

// Where the pieces of the scratch begin, in floats, and where the last one ends.  Each on 256 bytes, as an allocation of its own
// would be: which kernel a product takes goes by its rows' addresses, too.
struct Pieces {
  long long sum, h, qkv, heads, gate_up, act, end;
};
Pieces pieces_of(long long N, int H, int num_heads, int num_kv_heads, int head_dim, int I) {
  auto behind = [](long long at, long long floats) { return at + (floats + 63) / 64 * 64; };
  Pieces p;
  p.sum = 0;
  p.h = behind(p.sum, N * H);
  p.qkv = behind(p.h, N * H);
  p.heads = behind(p.qkv, N * (num_heads + 2 * num_kv_heads) * head_dim);
  p.gate_up = behind(p.heads, N * num_heads * head_dim);
  p.act = behind(p.gate_up, N * 2 * I);
  p.end = behind(p.act, N * I);
  return p;
}

}  // namespace

extern "C" int ms_float_layer_bytes() { return (int)sizeof(FloatLayer); }

// Floats of `work` for n_tokens tokens.
extern "C" long long ms_float_layers_work(int n_tokens, int H, int num_heads, int num_kv_heads, int head_dim, int I) {
  return pieces_of(n_tokens, H, num_heads, num_kv_heads, head_dim, I).end;
}

// x float [N, H] in place, but for the last down projection, which is left in work's first [N, H] for whoever adds it.  `work`:
// work_floats floats, at least ms_float_layers_work.  w_gate_up's rows interleaved, heads turned whole, pages as ms_rope_store has
// them; n_live may be null.
extern "C" int ms_float_layers(const void* layers, int n_layers, float* x, float* work, long long work_floats, const int* positions, const int* token_req,
                               const int* slot_mapping, const int* block_table, int table_width, const int* table_rows,
                               const int* n_live, int n_tokens, int H, int I, int num_heads, int num_kv_heads, int head_dim,
                               int page_size, long long num_pages, int v_transposed, float scale, hipStream_t stream) {
  if (n_tokens <= 0) return MS_OK;
  if (!layers || n_layers < 1 || !x || !work || !positions || !token_req || !slot_mapping || !block_table || H <= 0 || I <= 0 ||
      num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || page_size <= 0)
    return MS_BAD_ARG;
  const long long N = n_tokens;
  const int Ko = num_heads * head_dim, Q = (num_heads + 2 * num_kv_heads) * head_dim;
  const Pieces at = pieces_of(N, H, num_heads, num_kv_heads, head_dim, I);
  if (work_floats < at.end) return MS_BAD_ARG;
  float *sum = work + at.sum, *h = work + at.h, *qkv = work + at.qkv, *heads = work + at.heads, *gate_up = work + at.gate_up, *act = work + at.act;
  auto product = [&](const float* a, const float* w, const float* bias, float* out, int n, int k, int accumulate) {
    return ms_gemm_generic(a, w, bias, out, n_tokens, n, k, k, k, n, MS_F32, MS_F32, accumulate, stream);
  };
  // (a product that does not take its norm refuses, and the rows go through the scratch one kernel after the other)
  for (int i = 0; i < n_layers; ++i) {
    const FloatLayer& l = static_cast<const FloatLayer*>(layers)[i];
    const F32Front front{positions, slot_mapping, l.inv_freq, l.k_pages, l.v_pages, num_heads, num_kv_heads, head_dim, page_size, v_transposed};
    int rc = ms_gemm_f32_normed(x, l.w_qkv, l.b_qkv, qkv, n_tokens, Q, H, F32Norm{l.norm1, l.eps1}, &front, stream);
    if (rc == MS_UNSUPPORTED) {
      rc = ms_rms_norm(x, nullptr, MS_F32, 1, N * H, l.norm1, nullptr, h, n_tokens, H, l.eps1, 1, MS_F32, stream);
      if (rc == MS_OK) rc = product(h, l.w_qkv, l.b_qkv, qkv, Q, H, 0);
      if (rc == MS_OK)
        rc = ms_rope_store(qkv, nullptr, positions, l.inv_freq, slot_mapping, l.k_pages, l.v_pages, n_tokens, num_heads, num_kv_heads,
                           head_dim, head_dim, page_size, v_transposed, MS_F32, stream);
    }
    if (rc == MS_OK)
      rc = ms_paged_attention_generic(qkv, Q, l.k_pages, l.v_pages, block_table, table_width, table_rows, n_live, token_req, positions,
                                      heads, Ko, n_tokens, num_heads, num_kv_heads, head_dim, head_dim, page_size, num_pages, scale, 0,
                                      v_transposed, nullptr, 0.f, nullptr, nullptr, 0, 1, 1.f, MS_F32, stream);
    if (rc == MS_OK) rc = product(heads, l.w_o, nullptr, x, H, Ko, 1);
    if (rc == MS_OK) {
      rc = ms_gemm_f32_normed(x, l.w_gate_up, nullptr, act, n_tokens, 2 * I, H, F32Norm{l.norm2, l.eps2}, nullptr, stream);
      if (rc == MS_UNSUPPORTED) {
        rc = ms_rms_norm(x, nullptr, MS_F32, 1, N * H, l.norm2, nullptr, h, n_tokens, H, l.eps2, 1, MS_F32, stream);
        if (rc == MS_OK) rc = product(h, l.w_gate_up, nullptr, gate_up, 2 * I, H, 0);
        if (rc == MS_OK) rc = ms_silu_mul(gate_up, act, n_tokens, I, MS_F32, stream);
      }
    }
    const bool last = i + 1 == n_layers;
    if (rc == MS_OK) rc = product(act, l.w_down, nullptr, last ? sum : x, H, I, !last);
    if (rc != MS_OK) return rc;
  }
  return MS_OK;
}
