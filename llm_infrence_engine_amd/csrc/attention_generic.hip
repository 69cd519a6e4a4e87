// Paged causal attention with grouped heads, any key size and any value size up to 256, for any mix of prompt portions and single decoded tokens.  `sink` (may be null): one number per query
// head whose exponential joins the softmax's denominator; it has no key and no value.  Scores, running
// maximum, exponentials, their sum and the weighted sum of values are all float.  It reads keys and
// values in place through the request's block table and never reads a key beyond the token's own
// position, so what a reused page still holds from an earlier request cannot reach the result.
// block_table int32 [rows, table_stride]; request r of the step has row table_rows[r] (null: row r).
// n_live_tokens (null: all): a device int; tokens from that index on belong to no request and are skipped.
// `softcap` > 0: a score s (already scaled) becomes softcap * tanh(s / softcap).  `slopes` (may be null): one number per
// query head; slope * (distance of the key from the query) is taken off the score, after the cap.  `gate` (may be null):
// `gate_width` numbers per token and query head, 1 (the head's result is multiplied by sigmoid(gate)) or the value size (every
// entry by a sigmoid of its own); `out_scale` multiplies all.
// This is the attention of the 32-bit path and the any-shape fallback of the bfloat16 path.
#include "common.h"
#include "api.h"

namespace {

constexpr int WAVES = 4;
constexpr int MAX_D = 256;

__device__ __forceinline__ void dot4(const float* q, const float* k, float& dot) {
  const float4 v = *reinterpret_cast<const float4*>(k);
  dot = fmaf(q[0], v.x, dot); dot = fmaf(q[1], v.y, dot); dot = fmaf(q[2], v.z, dot); dot = fmaf(q[3], v.w, dot);
}
__device__ __forceinline__ void dot4(const float* q, const bf16* k, float& dot) {
  const uint2 v = *reinterpret_cast<const uint2*>(k);
  dot = fmaf(q[0], __uint_as_float(v.x << 16), dot); dot = fmaf(q[1], __uint_as_float(v.x & 0xffff0000u), dot);
  dot = fmaf(q[2], __uint_as_float(v.y << 16), dot); dot = fmaf(q[3], __uint_as_float(v.y & 0xffff0000u), dot);
}

// A block per (token, query head): its waves take the token's blocks of 64 keys in turn and merge what they found
// through LDS, always in the same order, whatever else is in the step.  A single token's keys are what a decode step
// waits for: with one wave on all of them 135 keys at a head size of 64 took 74 us (3 x 14 items), now 12.4, and prompts of
// 338 tokens 56 us, now 50.  A row of keys is read in pieces of four values, values 32 / C rows at a time.
template <typename T, int C>     // C: values a lane, dv <= 64 C
__global__ void __launch_bounds__(WAVES * MS_WAVE)
paged_attention_generic_kernel(const T* __restrict__ q, size_t q_stride, const T* __restrict__ k_pages,
                               const T* __restrict__ v_pages, const int* __restrict__ block_table, int table_stride,
                               const int* __restrict__ table_rows, const int* __restrict__ n_live_tokens,
                               const int* __restrict__ token_req, const int* __restrict__ positions,
                               T* __restrict__ out, size_t out_stride, int n_tokens, int nh, int nkv, int d, int dv,
                               int page_size, float scale, int window, int v_transposed, int vec,
                               const float* __restrict__ sink, float softcap, const float* __restrict__ slopes,
                               const T* __restrict__ gate, size_t gate_stride, int gate_width, float out_scale) {
  __shared__ float qs[MAX_D];
  __shared__ float ms[WAVES], ls[WAVES], accs[WAVES][C * MS_WAVE];
  constexpr int ROWS = 32 / C;        // rows of values asked for at a time
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);
  const long long item = (long long)blockIdx.y * gridDim.x + blockIdx.x;
  const int n = (int)(item / nh), h = (int)(item - (long long)n * nh);
  if (n >= n_tokens) return;
  if (n_live_tokens && n >= *n_live_tokens) return;   // (the whole block) a token that pads a captured batch
  const int kvh = h / (nh / nkv);
  const int pos = positions[n];
  const int req = token_req[n];
  const int* table = block_table + (size_t)(table_rows ? table_rows[req] : req) * table_stride;

  const T* qp = q + (size_t)n * q_stride + (size_t)h * d;
  for (int i = threadIdx.x; i < d; i += WAVES * MS_WAVE) qs[i] = to_float(qp[i]) * scale;
  __syncthreads();

  int start = 0;
  if (window > 0 && pos - window + 1 > 0) start = pos - window + 1;

  const float slope = slopes ? slopes[h] : 0.f;
  const float inv_cap = softcap > 0.f ? 1.0f / softcap : 0.f;
  float m = -INFINITY, l = 0.f;
  float acc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = 0.f;

  for (int base = start + wave * MS_WAVE; base <= pos; base += WAVES * MS_WAVE) {
    const int j = base + lane;
    const bool valid = j <= pos;
    int row = 0;
    float s = -INFINITY;
    if (valid) {
      const int page = table[j / page_size];
      row = (page * nkv + kvh) * page_size + (j % page_size);
      const T* kp = k_pages + (size_t)row * d;
      float dot = 0.f;
      int i = 0;
      if (vec) {
#pragma unroll 16
        for (; i < d; i += 4) dot4(&qs[i], kp + i, dot);
      }
      for (; i < d; ++i) dot = fmaf(qs[i], to_float(kp[i]), dot);
      s = dot;
      if (softcap > 0.f) s = softcap * tanhf(s * inv_cap);
      if (slopes) s -= slope * (float)(pos - j);
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float ref = m_new == -INFINITY ? 0.f : m_new;      // (a block of nothing but -inf counts for nothing)
    const float p = valid ? expf(s - ref) : 0.f;
    const float corr = expf(m - ref);    // 0 on the first block (m = -inf)
    l = l * corr + wave_sum(p);
    m = m_new;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] *= corr;
    const int count = min(MS_WAVE, pos - base + 1);
    const int vs = v_transposed ? page_size : 1;
    for (int j0 = 0; j0 < count; j0 += ROWS) {
      float v[ROWS][C], pj[ROWS];
#pragma unroll
      for (int u = 0; u < ROWS; ++u) {
        const int jj = min(j0 + u, count - 1);      // (places past the end read the last row and count for nothing)
        pj[u] = j0 + u < count ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), jj)) : 0.f;
        const int vrow = __builtin_amdgcn_readlane(row, jj);
        // value pages are [page][kv head][slot][dim], or transposed [page][kv head][dim][slot]
        const T* vp = v_transposed ? v_pages + (size_t)(vrow / page_size) * page_size * dv + vrow % page_size
                                   : v_pages + (size_t)vrow * dv;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const int i = lane + c * MS_WAVE;
          v[u][c] = i < dv ? to_float(vp[(size_t)i * vs]) : 0.f;
        }
      }
#pragma unroll
      for (int u = 0; u < ROWS; ++u) {
        if (j0 + u < count) {
#pragma unroll
          for (int c = 0; c < C; ++c) acc[c] = fmaf(pj[u], v[u][c], acc[c]);
        }
      }
    }
  }
  if (lane == 0) { ms[wave] = m; ls[wave] = l; }
#pragma unroll
  for (int c = 0; c < C; ++c) accs[wave][lane + c * MS_WAVE] = acc[c];
  __syncthreads();
  // the first block of keys is never empty: a token always sees its own key, so the merged maximum is finite
  float top = ms[0];
  for (int w = 1; w < WAVES; ++w) top = fmaxf(top, ms[w]);
  float factor[WAVES];
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    factor[w] = expf(ms[w] - top);      // 0 for a wave that had no keys
    total += ls[w] * factor[w];
  }
  if (sink) total += expf(sink[h] - top);
  float inv = out_scale / total;
  const T* gp = gate ? gate + (size_t)n * gate_stride + (size_t)h * gate_width : nullptr;
  if (gate && gate_width == 1) { inv /= 1.0f + expf(-to_float(*gp)); gp = nullptr; }
  T* op = out + (size_t)n * out_stride + (size_t)h * dv;
  for (int i = threadIdx.x; i < dv; i += WAVES * MS_WAVE) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o = fmaf(accs[w][i], factor[w], o);
    op[i] = from_float<T>(gp ? o * inv / (1.0f + expf(-to_float(gp[i]))) : o * inv);
  }
}

}  // namespace

extern "C" int ms_paged_attention_generic(const void* q, long long q_stride, const void* k_pages, const void* v_pages,
                                          const int* block_table, int table_stride, const int* table_rows,
                                          const int* n_live_tokens, const int* token_req,
                                          const int* positions, void* out, long long out_stride, int n_tokens,
                                          int num_heads, int num_kv_heads, int head_dim, int value_dim, int page_size,
                                          long long num_pages, float scale, int window, int v_transposed,
                                          const float* sink, float softcap, const float* slopes, const void* gate,
                                          long long gate_stride, int gate_width, float out_scale, int dtype,
                                          hipStream_t stream) {
  if (n_tokens <= 0) return MS_OK;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || page_size <= 0 || table_stride <= 0)
    return MS_BAD_ARG;
  if (head_dim <= 0 || head_dim > MAX_D || value_dim <= 0 || value_dim > MAX_D) return MS_UNSUPPORTED;
  if (gate != nullptr && gate_width != 1 && gate_width != value_dim) return MS_BAD_ARG;
  if (num_pages * num_kv_heads * page_size >= (1ll << 31)) return MS_UNSUPPORTED;  // row index is an int
  const long long items = (long long)n_tokens * num_heads;
  const long long across = items < (1ll << 20) ? items : (1ll << 20);
  if ((items + across - 1) / across > 65535) return MS_UNSUPPORTED;
  dim3 grid((unsigned)across, (unsigned)((items + across - 1) / across)), block(WAVES * MS_WAVE);
  const size_t vec_bytes = dtype == MS_F32 ? 16 : 8;      // a row of keys in pieces of four values
  const int vec = head_dim % 4 == 0 && (uintptr_t)k_pages % vec_bytes == 0;
#define LAUNCH_C(T, C) paged_attention_generic_kernel<T, C><<<grid, block, 0, stream>>>((const T*)q, (size_t)q_stride, (const T*)k_pages, (const T*)v_pages, block_table, table_stride, table_rows, n_live_tokens, token_req, positions, (T*)out, (size_t)out_stride, n_tokens, num_heads, num_kv_heads, head_dim, value_dim, page_size, scale, window, v_transposed, vec, sink, softcap, slopes, (const T*)gate, (size_t)gate_stride, gate_width, out_scale)
#define LAUNCH(T) do { if (value_dim <= 64) LAUNCH_C(T, 1); else if (value_dim <= 128) LAUNCH_C(T, 2); else LAUNCH_C(T, 4); } while (0)
  if (dtype == MS_F32) LAUNCH(float);
  else if (dtype == MS_BF16) LAUNCH(bf16);
  else return MS_BAD_ARG;
#undef LAUNCH_C
#undef LAUNCH
  return ms_launch_status();
}
