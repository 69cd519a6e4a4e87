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
#include <type_traits>

namespace {

constexpr int WAVES = 4, STREAMS = 4;
constexpr int MAX_D = 256;

__device__ __forceinline__ void dot4(const float* q, const float4 v, float& dot) {
  dot = fmaf(q[0], v.x, dot); dot = fmaf(q[1], v.y, dot); dot = fmaf(q[2], v.z, dot); dot = fmaf(q[3], v.w, dot);
}
__device__ __forceinline__ void dot4(const float* q, const float* k, float& dot) { dot4(q, *reinterpret_cast<const float4*>(k), dot); }
__device__ __forceinline__ void dot4(const float* q, const bf16* k, float& dot) {
  const uint2 v = *reinterpret_cast<const uint2*>(k);
  dot = fmaf(q[0], __uint_as_float(v.x << 16), dot); dot = fmaf(q[1], __uint_as_float(v.x & 0xffff0000u), dot);
  dot = fmaf(q[2], __uint_as_float(v.y << 16), dot); dot = fmaf(q[3], __uint_as_float(v.y & 0xffff0000u), dot);
}

// A token's blocks of 64 keys go to STREAMS runs in turn, each with its maximum, sum and weighted values, and the runs are
// merged in order: so a result depends neither on how many waves W a (token, query head) gets nor on what else is in the
// step.  W = 4, a run to a wave, is for steps that would leave the chip idle: a decode step waits for one token's keys (3 x
// 14 items behind 135 keys at a head size of 64: 74 us with one wave that kept one run, 9.1 with four).  With W = 1 a wave
// works its item's runs off by itself and waits for nothing but its own loads: for steps that fill the chip (8 prompts of 64
// tokens, 14 heads of 64 dims: float 61.5 us while every item had four waves, 23.6 so, bfloat16 86 and 19.3).
// What bounds it is the latency of a wave's loads: a lane reads its own key's row, the wave one row of values after another.
// Values are asked for R rows at a time and never behind a condition (each load would be waited for by itself, which was 3
// of the 7 us of a token with one key): lanes past the value size read its last entry, places past the keys the last row.
//
// ONCE (float, heads of 64 dims, few items): a lane's key and the block's values are asked for together, one trip to memory where
// the key and four times 16 rows of values were five: 8 tokens behind 1,000 keys, 14 heads 32.4 -> 26.9 us, 3 behind 135 9.2 -> 8.1.  Up to an
// item a CU: its registers leave room for three blocks, 64 tokens behind 200 keys 20.5 -> 24.2, 140 tokens of a prompt 17.6 -> 21.7.
template <typename T, int C, int W, bool ONCE>     // C: values a lane, dv <= 64 C
__global__ void __launch_bounds__(WAVES * MS_WAVE, W == 1 ? 4 : 1)
paged_attention_generic_kernel(const T* __restrict__ q, size_t q_stride, const T* __restrict__ k_pages,
                               const T* __restrict__ v_pages, const int* __restrict__ block_table, int table_stride,
                               const int* __restrict__ table_rows, const int* __restrict__ n_live_tokens,
                               const int* __restrict__ token_req, const int* __restrict__ positions,
                               T* __restrict__ out, size_t out_stride, int n_tokens, int nh, int nkv, int d, int dv,
                               int page_size, float scale, int window, int v_transposed, int vec,
                               const float* __restrict__ sink, float softcap, const float* __restrict__ slopes,
                               const T* __restrict__ gate, size_t gate_stride, int gate_width, float out_scale) {
  constexpr int ITEMS = WAVES / W;    // of a block
  constexpr int R = C == 4 || W == 1 ? 8 : 16;
  __shared__ float qs[ITEMS][MAX_D];
  __shared__ float ms[ITEMS][STREAMS], ls[ITEMS][STREAMS], accs[ITEMS][STREAMS][C * MS_WAVE];
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);
  const int slot = wave / W, part = wave % W;
  // last tokens first: those of a prompt see the most keys
  const long long item = (long long)n_tokens * nh - 1 - (((long long)blockIdx.y * gridDim.x + blockIdx.x) * ITEMS + slot);
  if (item < 0) return;      // (all waves of an item leave together)
  const int n = item >> 32 ? (int)(item / nh) : (int)((unsigned)item / (unsigned)nh), h = (int)(item - (long long)n * nh);
  if (n_live_tokens && n >= *n_live_tokens) return;   // a token that pads a captured batch
  const int kvh = h / (nh / nkv);
  const int pos = positions[n];
  const int req = token_req[n];
  const int* table = block_table + (size_t)(table_rows ? table_rows[req] : req) * table_stride;

  int start = 0;
  if (window > 0 && pos - window + 1 > 0) start = pos - window + 1;
  const int streams = min(STREAMS, (pos - start) / MS_WAVE + 1);
  const bool alone = streams == 1;      // one run: one wave, nothing to merge; the others of a block of one item leave
  if (alone && part > 0) return;
  // the item's waves have written what they read next
  auto meet = [&] {
    if (W > 1 && !alone) __syncthreads();
    else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  };

  const T* qp = q + (size_t)n * q_stride + (size_t)h * d;
  if (part == 0)
    for (int i = lane; i < d; i += MS_WAVE) qs[slot][i] = to_float(qp[i]) * scale;
  meet();

  const float slope = slopes ? slopes[h] : 0.f;
  const float inv_cap = softcap > 0.f ? 1.0f / softcap : 0.f;
  const int vs = v_transposed ? page_size : 1;
  int entry[C];      // this lane's entries of a row of values
#pragma unroll
  for (int c = 0; c < C; ++c) entry[c] = min(lane + c * MS_WAVE, dv - 1) * vs;

  float m, l, acc[C];
  for (int s = part; s < streams; s += W) {
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = 0.f;
    for (int base = start + s * MS_WAVE; base <= pos; base += STREAMS * MS_WAVE) {
      const int j = base + lane;
      const bool valid = j <= pos;
      size_t row = 0, vrow = 0;       // of the key among the rows of keys, of its first value
      float score = -INFINITY;
      const int count = min(MS_WAVE, pos - base + 1);
      float values[ONCE ? MS_WAVE : 1];
      if constexpr (ONCE) {
        const int jj = min(j, pos), page = jj / page_size, off = jj - page * page_size;      // (lanes past the keys read the last one)
        const size_t head = (size_t)table[page] * nkv + kvh;
        row = head * page_size + off;
        vrow = v_transposed ? head * dv * page_size + off : row * dv;
        const float4* kp = reinterpret_cast<const float4*>(k_pages + row * 64);
        float4 key[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) key[i] = kp[i];
#pragma unroll
        for (int u0 = 0; u0 < MS_WAVE; u0 += 16) {
          if (u0 >= count) break;
#pragma unroll
          for (int u = u0; u < u0 + 16; ++u) {
            const unsigned lo = __builtin_amdgcn_readlane((unsigned)vrow, u), hi = __builtin_amdgcn_readlane((unsigned)(vrow >> 32), u);
            values[u] = to_float((v_pages + (((size_t)hi << 32) | lo))[entry[0]]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        float dot = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) dot4(&qs[slot][4 * i], key[i], dot);
        score = dot;
        if (softcap > 0.f) score = softcap * tanhf(score * inv_cap);
        if (slopes) score -= slope * (float)(pos - j);
        if (!valid) score = -INFINITY;
      } else if (valid) {
        const int page = j / page_size, off = j - page * page_size;
        const size_t head = (size_t)table[page] * nkv + kvh;
        row = head * page_size + off;
        // value pages are [page][kv head][slot][dim], or transposed [page][kv head][dim][slot]
        vrow = v_transposed ? head * dv * page_size + off : row * dv;
        const T* kp = k_pages + row * d;
        float dot = 0.f;
        int i = 0;
        if (vec) {
#pragma unroll (W == 1 && sizeof(T) == 2 ? 8 : 16)
          for (; i < d; i += 4) dot4(&qs[slot][i], kp + i, dot);
        }
#pragma unroll 4
        for (; i < d; ++i) dot = fmaf(qs[slot][i], to_float(kp[i]), dot);
        score = dot;
        if (softcap > 0.f) score = softcap * tanhf(score * inv_cap);
        if (slopes) score -= slope * (float)(pos - j);
      }
      const float m_new = fmaxf(m, wave_max(score));
      const float ref = m_new == -INFINITY ? 0.f : m_new;      // (a block of nothing but -inf counts for nothing)
      const float p = valid ? expf(score - ref) : 0.f;
      const float corr = expf(m - ref);    // 0 on the first block (m = -inf)
      l = l * corr + wave_sum(p);
      m = m_new;
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] *= corr;
      if constexpr (ONCE) {
#pragma unroll
        for (int u = 0; u < MS_WAVE; ++u)
          if (u < count) acc[0] = fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), u)), values[u], acc[0]);
        continue;
      }
      auto rows = [&](auto size, int j0) __attribute__((always_inline)) {
        constexpr int N = decltype(size)::value;
        float v[N][C], pj[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const int jj = min(j0 + u, count - 1);      // (places past the end read the last row and count for nothing)
          pj[u] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), jj));
          const unsigned lo = __builtin_amdgcn_readlane((unsigned)vrow, jj), hi = __builtin_amdgcn_readlane((unsigned)(vrow >> 32), jj);
          const T* vp = v_pages + (((size_t)hi << 32) | lo);
#pragma unroll
          for (int c = 0; c < C; ++c) v[u][c] = to_float(vp[entry[c]]);
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
          if (j0 + u < count) {
#pragma unroll
            for (int c = 0; c < C; ++c) acc[c] = fmaf(pj[u], v[u][c], acc[c]);
          }
        }
      };
      int j0 = 0;
      for (; count - j0 > 4; j0 += R) rows(std::integral_constant<int, R>{}, j0);
      if (count - j0 > 1) rows(std::integral_constant<int, 4>{}, j0);
      else if (count > j0) rows(std::integral_constant<int, 1>{}, j0);
    }
    if (alone) break;
    if (lane == 0) { ms[slot][s] = m; ls[slot][s] = l; }
#pragma unroll
    for (int c = 0; c < C; ++c) accs[slot][s][lane + c * MS_WAVE] = acc[c];
  }
  float top = m, total = l, factor[STREAMS];
  if (!alone) {
    meet();
    // the first run is never empty: a token always sees its own key, so the merged maximum is finite
    top = ms[slot][0];
    for (int s = 1; s < streams; ++s) top = fmaxf(top, ms[slot][s]);
    total = 0.f;
#pragma unroll
    for (int s = 0; s < STREAMS; ++s) {
      factor[s] = 0.f;
      if (s < streams) {
        factor[s] = expf(ms[slot][s] - top);
        total += ls[slot][s] * factor[s];
      }
    }
  }
  if (sink) total += expf(sink[h] - top);
  float inv = out_scale / total;
  const T* gp = gate ? gate + (size_t)n * gate_stride + (size_t)h * gate_width : nullptr;
  if (gate && gate_width == 1) { inv /= 1.0f + expf(-to_float(*gp)); gp = nullptr; }
  T* op = out + (size_t)n * out_stride + (size_t)h * dv;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (!alone && c % W != part) continue;
    const int i = lane + c * MS_WAVE;
    float o = acc[c];
    if (!alone) {
      o = 0.f;
#pragma unroll
      for (int s = 0; s < STREAMS; ++s)
        if (s < streams) o = fmaf(accs[slot][s][i], factor[s], o);
    }
    if (i < dv) op[i] = from_float<T>(gp ? o * inv / (1.0f + expf(-to_float(gp[i]))) : o * inv);
  }
}

int g_waves = 0;      // measurements: 1 or 4 force the waves to a (token, query head), 0 leaves the choice

}  // namespace

extern "C" void ms_attention_generic_force(int waves) { g_waves = waves; }

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
  const size_t vec_bytes = dtype == MS_F32 ? 16 : 8;      // a row of keys in pieces of four values
  const int vec = head_dim % 4 == 0 && (uintptr_t)k_pages % vec_bytes == 0;
  const long long most_keys = window > 0 ? window : (long long)table_stride * page_size;
  // Four waves an item up to 8 items a CU, where more than one block of keys can be visible (6 heads of 32 dims, float, one
  // prompt of 338 tokens, 2,028 items: 38 us with one wave, 28 with four; 8 prompts of 64, 3,072 items: 11.2 and 12.9); values
  // of more than 64 dims, whose merge the waves share out too: up to 16, whatever is visible (8 heads of 128, 4 x 128 tokens,
  // 4,096 items: 47 and 36; one token of 256 dims 6.9 and 5.5).
  const bool wide = value_dim > MS_WAVE;
  int waves = items <= (wide ? 16LL : 8LL) * ms_compute_units() && (wide || most_keys > MS_WAVE) ? 4 : 1;
  if (g_waves) waves = g_waves;
  const long long blocks = waves == 4 ? items : (items + WAVES - 1) / WAVES;
  const long long across = blocks < (1ll << 20) ? blocks : (1ll << 20);
  if ((blocks + across - 1) / across > 65535) return MS_UNSUPPORTED;
  dim3 grid((unsigned)across, (unsigned)((blocks + across - 1) / across)), block(WAVES * MS_WAVE);
#define LAUNCH_W(T, C, W, ONCE) paged_attention_generic_kernel<T, C, W, ONCE><<<grid, block, 0, stream>>>((const T*)q, (size_t)q_stride, (const T*)k_pages, (const T*)v_pages, block_table, table_stride, table_rows, n_live_tokens, token_req, positions, (T*)out, (size_t)out_stride, n_tokens, num_heads, num_kv_heads, head_dim, value_dim, page_size, scale, window, v_transposed, vec, sink, softcap, slopes, (const T*)gate, (size_t)gate_stride, gate_width, out_scale)
#define LAUNCH_C(T, C) do { if (waves == 4) LAUNCH_W(T, C, 4, false); else LAUNCH_W(T, C, 1, false); } while (0)
#define LAUNCH(T) do { if (value_dim <= 64) LAUNCH_C(T, 1); else if (value_dim <= 128) LAUNCH_C(T, 2); else LAUNCH_C(T, 4); } while (0)
  if (dtype == MS_F32 && vec && head_dim == 64 && value_dim <= 64 && waves == 4 && items <= ms_compute_units()) LAUNCH_W(float, 1, 4, true);
  else if (dtype == MS_F32) LAUNCH(float);
  else if (dtype == MS_BF16) LAUNCH(bf16);
  else return MS_BAD_ARG;
#undef LAUNCH_C
#undef LAUNCH_W
#undef LAUNCH
  return ms_launch_status();
}
