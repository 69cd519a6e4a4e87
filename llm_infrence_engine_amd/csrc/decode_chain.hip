// What lies between two attentions of a decode step, for up to 8 tokens of a narrow model, as ONE kernel (CHAIN), or all layers of
// the step with their attentions (FIRST, WHOLE).  In phases:
//
//   o       x1 = x + attention . Wo^T                              (float residual stream)
//   gate    act = silu(norm(x1) . Wg^T) * (norm(x1) . Wu^T)        (gate and up rows interleaved)
//   down    x2 = x1 + act . Wd^T
//   front   the next layer's q, k, v from norm(x2): bias, rotation, k and v into their pages
//   (attention to the keys in the pages and the step's own, WHOLE)
//
// As kernels of their own these are bound by latency: a launch is 1.6 us, and every kernel starts with blocks that wait for
// weights which could have been on their way all along (0.5B, 30 MB of weights: 2.9 + 8.2 + 4.7 + 4.4 = 20.1 us at one token,
// 24.6 at 8, and an attention of 4.1 and, at 577 keys, 7.5).  Here a block is one item of one phase, all phases' blocks are
// launched at once, and a block asks for its weights (into registers) before it waits for the phase before it.  What is left
// of a phase is the way of its results to the blocks that need all of them, about 1.5 us, its sums, and its share of reading
// the weights.  CHAIN: 13.1 us at one token, 14.0 at 4, 15.5 at 8.  WHOLE, with the attention: 14.9, 16.3 and 21.4 a layer.
//
// The way of a result.  Every result travels in a 64-bit word of its own with a tag: 32 bits of value (a float, or two
// bfloat16) and the 32-bit number of this launch.  Words are stored and loaded past the L2s (relaxed, agent scope), and a
// reader polls the very words it is going to use, so there is no flag, no fence and no order between words to rely on.  The
// number differs from launch to launch: `epoch` has a counter for each of a step's launches, which the launch after it in
// the step counts up (the first one counts up the last one's), so nobody writes a counter that its own launch reads.
// Words lie in the order in which a reader's lanes take them, whole runs of 64 bytes and more.
//
// Waiting.  Blocks are dispatched in order, so those that a block waits for run already or will run as soon as there is
// room; but other waiting kernels (another engine's, on another stream) may hold that room.  So no block waits for ever: one that has
// polled `limit` times in vain gives its item up and ends, unless it is the only one that has given up: that one stays and
// works off, as their inputs come in, the items that others gave up.  So a launch needs room for one block to end.  Words that never
// come (a launch out of its turn left them out) end the one that stays, too: after `patience` tries in a row of which none got on, it
// says so behind the list and to the host, and from then on nobody stays.
//
// A row's sums are the same whatever else is in the batch: k-step s belongs to wave s % 8, where it stands decides which lanes
// hold its products, and lanes and waves are added in a fixed order.
#include "common.h"
#include "api.h"
#include "quads.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef unsigned long long u64;

constexpr int WAVES = 8;              // of a block
constexpr int STEPS = 4;              // k-steps of a wave in o, gate and front: up to 1,024 columns
constexpr int DOWN_WAVES = 16;        // runs of k-steps in down, two to a wave
constexpr int DOWN_LOADS = 3;         // loads of four k-steps to such a run: up to 6,144 columns
constexpr int NT = 3;                 // tiles of 16 interleaved gate/up rows to a block
constexpr int UO = 2, UF = 2;         // units of four rows to a block in o and front
constexpr int HEAD = 64;              // dims of a head in WHOLE, two k-steps
constexpr int SHARES = HEAD / 16;     // blocks of attention to a token and key/value head: each has all keys and 16 dims of the values
constexpr int KEYS = 4;               // blocks of 32 keys to a wave: contexts up to 1,024
constexpr int LIST = 32767;           // items that can be given up, the blocks of a launch (the first has no place: it stays)
constexpr int MAX_LAUNCHES = 1024;    // of a step

// What a kernel holds: one layer's chain (its attention before it, the next layer's after it, as kernels of their own), the front
// of the first layer alone, or a step's layers whole, from the first one's attention to the last one's down.
enum { CHAIN = 0, FIRST = 1, WHOLE = 2 };

// One layer's weights and pages; `w_front` to `inv_freq` and `front_k`, `front_v`: of the layer after it.  Device addresses.
struct Layer {
  u64 w_o, w_gu, w_down, w_front, norm2, norm1, b_front, inv_freq, k_pages, v_pages, front_k, front_v;
  float eps2, eps1;
};

struct ChainArgs {
  Layer one;                          // CHAIN, FIRST
  u64 layers;                         // WHOLE: Layer [n_layers] in device memory
  const bf16* attn;                   // CHAIN: the attention's result
  bf16* q_out;                        // CHAIN: the next layer's queries
  float* x;
  const int *positions, *slots, *contexts, *table, *table_rows;
  u64 *x1, *x2, *act, *heads, *qkv;   // words
  unsigned *given_up;                 // how many items, then the items; [LIST]: not 0 if a launch was broken off
  int *told;                          // that, in host memory (or null)
  unsigned *epoch;
  long long ld_attn, ldx;
  float inv_H, scale_log2;
  int M, H, Ko, I, nh, nkv, d, page_size, page_shift, v_transposed, table_width;
  int n_layers, n_attn, n_o, n_gate, n_down, n_front;   // blocks of each phase of a layer
  int gate_units, gate_more;          // units of four gate/up rows to a block of gate, and how many blocks have one more
  int per_head;                       // blocks of front to a head
  int launch, launches;
  unsigned limit, patience;
};

template <typename T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* global(u64 address) {
  return (const __attribute__((address_space(1))) T*)address;
}
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* global_out(u64 address) {
  return (__attribute__((address_space(1))) T*)address;
}
template <typename T, typename P>
__device__ __forceinline__ T load(P p) { return *(const __attribute__((address_space(1))) T*)p; }
template <typename T, typename V>
__device__ __forceinline__ void store(T* p, V v) { *(__attribute__((address_space(1))) T*)p = v; }
// Arguments and layers are read where a phase needs them: all of them at once are more than the scalar registers hold.
typedef const __attribute__((address_space(4))) ChainArgs Args;
typedef const __attribute__((address_space(4))) Layer LayerArgs;

// ---- words
__device__ __forceinline__ void put(u64* word, unsigned value, unsigned tag) {
  __hip_atomic_store((__attribute__((address_space(1))) u64*)word, ((u64)tag << 32) | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 look(const u64* word) {
  return __hip_atomic_load((const __attribute__((address_space(1))) u64*)word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Word of x1 or x2 for column k of token m: a lane of wave (k / 32) % 8 takes 8 columns, in four loads of two words.
__device__ __forceinline__ int stream_word(int k, int m, int M) {
  const int s = k >> 5, e = k & 7;
  return 2 * (((((s % WAVES) * STEPS + s / WAVES) * 4 + e / 2) * 4 + ((k >> 3) & 3)) * M + m) + (e & 1);
}
// Word of act for columns k, k + 1 (k even): a lane takes 8 columns in two loads of two words.
__device__ __forceinline__ int act_word(int k, int m, int M) {
  const int s = k >> 5, p = (k & 7) >> 1;
  return 2 * (((((s % DOWN_WAVES) * (4 * DOWN_LOADS) + s / DOWN_WAVES) * 2 + p / 2) * 4 + ((k >> 3) & 3)) * M + m) + (p & 1);
}
// Word of an attention result's columns k, k + 1 (k even), as act's, in 8 runs.
__device__ __forceinline__ int head_word(int k, int m, int M) {
  const int s = k >> 5, p = (k & 7) >> 1;
  return 2 * (((((s % WAVES) * STEPS + s / WAVES) * 2 + p / 2) * 4 + ((k >> 3) & 3)) * M + m) + (p & 1);
}
// Words of q's features f, f + 1 of head c of the group that shares key/value head g, of k's and of v's (HEAD dims): mg = m * nkv + g.
__device__ __forceinline__ int q_word(int mg, int c, int f, int group) {
  const int p = (f & 7) >> 1;
  return 2 * ((((mg * (HEAD / 32) + f / 32) * 2 + p / 2) * 4 + ((f >> 3) & 3)) * group + c) + (p & 1);
}
__device__ __forceinline__ int k_word(int mg, int f) {
  const int p = (f & 7) >> 1;
  return 2 * (((mg * (HEAD / 32) + f / 32) * 2 + p / 2) * 4 + ((f >> 3) & 3)) + (p & 1);
}

// Reads of two words each, at base + the lane's offset in bytes, past the L2; the wait is in the same block, so nothing is in
// flight behind it.  The hardware wants five wait states between a vector instruction that writes a scalar register (the
// compiler's v_readlane, where it keeps a base in a vector register's lanes) and a memory instruction that reads it, and the
// compiler does not count them for instructions in assembly.
#define SGPRS_READY "s_nop 4\n\t"
#define RD(n, a, b) "global_load_dwordx4 %" #n ", %" #a ", %" #b " sc1\n\t"
__device__ __forceinline__ void read_words(const char* b0, const char* b1, const char* b2, const char* b3, const unsigned (&at)[1], quad_u32 (&v)[4]) {
  asm volatile(SGPRS_READY RD(0, 4, 5) RD(1, 4, 6) RD(2, 4, 7) RD(3, 4, 8) "s_waitcnt vmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
               : "v"(at[0]), "s"(b0), "s"(b1), "s"(b2), "s"(b3) : "memory");
}
__device__ __forceinline__ void read_words(const char* b0, const char* b1, const char* b2, const char* b3, const unsigned (&at)[2], quad_u32 (&v)[8]) {
  asm volatile(SGPRS_READY RD(0, 8, 10) RD(1, 8, 11) RD(2, 8, 12) RD(3, 8, 13) RD(4, 9, 10) RD(5, 9, 11) RD(6, 9, 12) RD(7, 9, 13)
               "s_waitcnt vmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
               : "v"(at[0]), "v"(at[1]), "s"(b0), "s"(b1), "s"(b2), "s"(b3) : "memory");
}
__device__ __forceinline__ void read_words(const char* b0, const char* b1, const unsigned (&at)[6], quad_u32 (&v)[12]) {
  asm volatile(SGPRS_READY RD(0, 12, 18) RD(1, 12, 19) RD(2, 13, 18) RD(3, 13, 19) RD(4, 14, 18) RD(5, 14, 19) RD(6, 15, 18) RD(7, 15, 19)
               RD(8, 16, 18) RD(9, 16, 19) RD(10, 17, 18) RD(11, 17, 19) "s_waitcnt vmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]),
                 "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
               : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "v"(at[4]), "v"(at[5]), "s"(b0), "s"(b1)
               : "memory");
}
// four reads of queries, four of a key and one word of a value
__device__ __forceinline__ void read_words(const char* q, unsigned q_step, unsigned q_at, const char* k, unsigned k_at, const char* v, unsigned v_at,
                                           quad_u32 (&w)[8], u64& value) {
  asm volatile(SGPRS_READY RD(0, 9, 12) RD(1, 9, 13) RD(2, 9, 14) RD(3, 9, 15) RD(4, 10, 16) RD(5, 10, 17) RD(6, 10, 18) RD(7, 10, 19)
               "global_load_dwordx2 %8, %11, %20 sc1\n\t" "s_waitcnt vmcnt(0)"
               : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7]), "=&v"(value)
               : "v"(q_at), "v"(k_at), "v"(v_at), "s"(q), "s"(q + q_step), "s"(q + 2 * q_step), "s"(q + 3 * q_step), "s"(k), "s"(k + 64),
                 "s"(k + 128), "s"(k + 192), "s"(v)
               : "memory");
}
__device__ __forceinline__ void read_words(const char* b0, const char* b1, const unsigned (&at)[1], quad_u32 (&v)[2]) {
  asm volatile(SGPRS_READY RD(0, 2, 3) RD(1, 2, 4) "s_waitcnt vmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]) : "v"(at[0]), "s"(b0), "s"(b1) : "memory");
}
__device__ __forceinline__ void read_words(const char* b0, const char* b1, const unsigned (&at)[2], quad_u32 (&v)[4]) {
  asm volatile(SGPRS_READY RD(0, 4, 6) RD(1, 4, 7) RD(2, 5, 6) RD(3, 5, 7) "s_waitcnt vmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at[0]), "v"(at[1]), "s"(b0), "s"(b1) : "memory");
}
__device__ __forceinline__ void read_words(const char* b0, const char* b1, const unsigned (&at)[3], quad_u32 (&v)[6]) {
  asm volatile(SGPRS_READY RD(0, 6, 9) RD(1, 6, 10) RD(2, 7, 9) RD(3, 7, 10) RD(4, 8, 9) RD(5, 8, 10) "s_waitcnt vmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5])
               : "v"(at[0]), "v"(at[1]), "v"(at[2]), "s"(b0), "s"(b1) : "memory");
}
#undef RD
#undef SGPRS_READY
template <int N>
__device__ __forceinline__ bool all_tagged(const quad_u32 (&v)[N], unsigned tag) {
  unsigned other = 0u;
#pragma unroll
  for (int i = 0; i < N; ++i) other |= (v[i][1] ^ tag) | (v[i][3] ^ tag);
  return __all(other == 0u);
}

// ---- sums over lanes, on the vector ALU
template <int CONTROL>
__device__ __forceinline__ float lanes_moved(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CONTROL, 0xF, 0xF, true));
}
template <int BY> __device__ __forceinline__ float turned(float v) { return lanes_moved<0x120 + BY>(v); }   // within rows of 16
// row 1 += row 0, row 3 += row 2 (of values that are the same throughout a row)
__device__ __forceinline__ float onto_odd_rows(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xA, 0xF, false));
}
__device__ __forceinline__ float sum_of_row(float v) {
  v += turned<8>(v);
  v += turned<4>(v);
  v += turned<2>(v);
  return v + turned<1>(v);
}
// 1 / sqrt(v), with one step of Newton's on the hardware's estimate
__device__ __forceinline__ float inverse_root(float v) {
  const float y = __builtin_amdgcn_rsqf(v);
  return y * fmaf(-0.5f * v * y, y, 1.5f);
}

// The operands of units of four rows lie as quads.h has them: one register takes four k-steps i of four rows r (lane 16 kq +
// 4 i + r), one or two registers the four steps of G tokens m (lane 16 kq + G i + m, 16 / G steps to a register).  Multiplied
// as they are, every product of a row and a token at the same step stands in one of the 16 x 16 results, and the others are
// read by nobody: four k-steps to an instruction and nothing to turn.  Lane group g has the rows at step g.
template <int G>
__device__ __forceinline__ quad_f32 own_step(const quad_f32 (&acc)[G / 4], int lane) {
  if constexpr (G == 4) return acc[0];
  else return lane < 32 ? acc[0] : acc[1];
}
template <int G>
__device__ __forceinline__ bool has_own_step(int lane) { return ((lane & 15) / G) == ((lane >> 4) & (16 / G - 1)); }

struct Shared {
  quad_f32 part[NT * WAVES * 4 * 8];   // gate: [tile][wave][row group * G + token]; else [unit][token][wave * 4 + step]
  float part_ss[8][WAVES];              // [token]
  int late[3];                          // somebody gave up: waiting for the first word, for the others, for a phase before the one before
  int next, position;
  unsigned in_vain;                     // tries in a row
  unsigned done[(LIST + 32) / 32];
};

// One word of the phase before, by one wave, so that blocks far ahead of their inputs disturb nobody.  Whole block; false: not
// within `limit` looks.  SLOT: the word of sh.late, another for each wait of an item: no barrier lies between a wave's read of it
// and the store of the wait that follows.
template <int SLOT = 0>
__device__ __forceinline__ bool wait_first(Shared& sh, const u64* word, unsigned tag, unsigned limit) {
  if (threadIdx.x < MS_WAVE) {
    int late = 1;
    for (unsigned n = 0; n < limit; ++n) {
      if ((unsigned)(look(word) >> 32) == tag) { late = 0; break; }
      __builtin_amdgcn_s_sleep(1);
    }
    if (threadIdx.x == 0) { sh.late[SLOT] = late; sh.late[1] = 0; }
  }
  __syncthreads();
  return sh.late[SLOT] == 0;
}

// A wave's share of the float stream's rows (one load's worth of four k-steps, G tokens), with the norm's weights.
template <int G>
struct StreamRows {
  static constexpr int XL = G / 4, XS = 16 / G;
  quad_f32 nw[XL][2];
  quad_u32 x[XL];          // bfloat16(x * norm weight)
  unsigned at[XL];
  bool in[XL];
  float ss[XL];            // squares of the lane's values

  __device__ __forceinline__ void ask_norm(const __attribute__((address_space(1))) float* norm_w, int lane, int wave, int M, int H) {
    const int mine = (H / 32 - wave + WAVES - 1) / WAVES, m = min(lane & (G - 1), M - 1);
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int i = j * XS + (lane & 15) / G, there = mine > 0 ? min(i, mine - 1) : 0, run = mine > 0 ? wave : 0;
      in[j] = i < mine;
      at[j] = 16u * ((((run * STEPS + there) * 4) * 4 + (lane >> 4)) * M + m);
      const auto w = norm_w + (run + WAVES * there) * 32 + (lane >> 4) * 8;
      nw[j][0] = load<quad_f32>(w);
      nw[j][1] = load<quad_f32>(w + 4);
    }
  }
  __device__ __forceinline__ bool poll(const u64* words, int M, unsigned tag, unsigned limit) {
    const char* b = (const char*)words;
    quad_u32 v[4 * XL];
    for (unsigned n = 0;; ++n) {
      if (n == limit) return false;
      read_words(b, b + 64 * M, b + 128 * M, b + 192 * M, at, v);
      if (all_tagged(v, tag)) break;
      __builtin_amdgcn_s_sleep(1);
    }
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = __uint_as_float(v[4 * j + e / 2][2 * (e & 1)]);
      take(j, f);
    }
    return true;
  }
  // the rows as they lie in memory, from before this launch
  __device__ __forceinline__ void read(const float* x, long long ldx, int lane, int wave, int M, int H) {
    const int mine = (H / 32 - wave + WAVES - 1) / WAVES, m = min(lane & (G - 1), M - 1);
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int i = j * XS + (lane & 15) / G, there = mine > 0 ? min(i, mine - 1) : 0, run = mine > 0 ? wave : 0;
      const float* p = x + (size_t)m * ldx + (run + WAVES * there) * 32 + (lane >> 4) * 8;
      const quad_f32 lo = load<quad_f32>(p), hi = load<quad_f32>(p + 4);
      const float f[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      take(j, f);
    }
  }
  __device__ __forceinline__ void take(int j, const float (&values)[8]) {
    ss[j] = 0.f;
    quad_bf16 h;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = in[j] ? values[e] : 0.f;
      ss[j] = fmaf(f, f, ss[j]);
      h[e] = (__bf16)(f * nw[j][e / 4][e & 3]);
    }
    x[j] = __builtin_bit_cast(quad_u32, h);
  }
  // the wave's squares of token m, in every lane with lane % G = m: steps 0 + 2 and 1 + 3, then both, whatever G is
  __device__ __forceinline__ float squares() const {
    float v;
    if constexpr (G == 4) {
      v = ss[0] + turned<8>(ss[0]);
      v += turned<4>(v);
    } else {
      v = ss[0] + ss[1];
      v += turned<8>(v);
    }
    return quad_sum_rows(v);
  }
};

// Writes a wave's share of U units' sums; `finish_units` has, behind a barrier, for pair p = unit * M + token the four rows'
// sums in lanes 16 to 31 (p = 2 wave) and 48 to 63 (p = 2 wave + 1).
template <int U, int G>
__device__ __forceinline__ void leave_units(Shared& sh, const quad_f32 (&acc)[U][G / 4], int lane, int wave) {
  if (has_own_step<G>(lane)) {
#pragma unroll
    for (int u = 0; u < U; ++u) sh.part[(u * G + (lane & (G - 1))) * (4 * WAVES) + wave * 4 + (lane >> 4)] = own_step<G>(acc[u], lane);
  }
}
__device__ __forceinline__ quad_f32 finish_units(const Shared& sh, int u, int G, int m, int lane) {
  quad_f32 v = sh.part[(u * G + m) * (4 * WAVES) + (lane & 31)];
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = onto_odd_rows(sum_of_row(v[r]));
  return v;
}
__device__ __forceinline__ unsigned two_bf16(float lo, float hi) {
  return (unsigned)__builtin_bit_cast(unsigned short, from_float<bf16>(lo)) | (unsigned)__builtin_bit_cast(unsigned short, from_float<bf16>(hi)) << 16;
}
// unit and token of pair p = unit * M + token of at most two units (a token within the batch for a pair beyond them, too)
__device__ __forceinline__ void pair_of(int p, int M, int& unit, int& token) {
  unit = p >= 2 * M ? 2 : p >= M ? 1 : 0;
  token = min(p - unit * M, M - 1);
}
__device__ __forceinline__ float row_of(const quad_f32& v, int r) { return r & 2 ? (r & 1 ? v[3] : v[2]) : (r & 1 ? v[1] : v[0]); }
__device__ __forceinline__ quad_f32 product(const quad_u32& w, const quad_u32& x, const quad_f32& acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(quad_bf16, w), __builtin_bit_cast(quad_bf16, x), acc, 0, 0, 0);
}

// A CU's loads come back in the order they were asked for, so another block's weights hold up a block that looks for its words.
// Where blocks have a layer's time to fetch theirs, a wave asks for two loads at a time (0.5B, a layer of one token 15.9 us
// without this, 15.1 for three or six loads at a time, 14.9; one at a time comes too late, 16.8; 8 tokens 23.6 -> 21.4).
template <int MODE>
__device__ __forceinline__ void paced() {
  if constexpr (MODE == WHOLE) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
}

// The tokens' attention to the keys of one key/value head, by one block for each 16 dims of the values: every wave up to four
// blocks of 32 keys, which it asks for before anything is known of the queries (they lie in the pages since earlier steps);
// the step's own key comes in words, as the queries do, and goes to the wave whose turn it would be.
__device__ __forceinline__ bool run_attention(Args& a, Shared& sh, LayerArgs& L, int b, int lane, int wave, unsigned tag, unsigned limit) {
  const int share = b % SHARES, mg = b / SHARES, m = mg / a.nkv, g = mg - m * a.nkv, group = a.nh / a.nkv;
  const int col = lane & 15, kq = lane >> 4;
  const int pos = load<int>(a.contexts + m) - 1, blocks = min((max(pos, 0) + 31) >> 5, WAVES * KEYS);   // of 32 old keys
  const int* table = a.table + (size_t)(a.table_rows ? load<int>(a.table_rows + m) : m) * a.table_width;
  const auto k_pages = global<bf16>(L.k_pages), v_pages = global<bf16>(L.v_pages);
  quad_u32 kf[KEYS][2][2];
  u64 vf[KEYS][2];
#pragma unroll
  for (int i = 0; i < KEYS; ++i) {
    const int block = wave + WAVES * i;
    if (block < blocks) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int key = min(block * 32 + t * 16, (pos - 1) & ~15);      // (of a tile behind the last key, the last one's)
        const int at = key >> a.page_shift, off = key & (a.page_size - 1);
        const size_t page = (size_t)load<int>(table + at) * a.nkv + g;
#pragma unroll
        for (int s = 0; s < 2; ++s) kf[i][t][s] = load<quad_u32>(k_pages + (page * a.page_size + off + col) * HEAD + s * 32 + kq * 8);
        vf[i][t] = load<u64>(v_pages + (page * HEAD + share * 16 + col) * a.page_size + off + kq * 4);
      }
    }
  }
  const u64 *q = a.qkv, *k = q + (size_t)a.M * a.nh * (HEAD / 2), *v = k + (size_t)a.M * a.nkv * (HEAD / 2);
  if (!wait_first(sh, q + q_word(mg, 0, 0, group), tag, limit)) return false;
  const bool own = wave == (blocks & (WAVES - 1));     // the step's own key is this wave's
  quad_u32 qf[2], kn[2];
  unsigned vn = 0u;
  bool ok = true;
  {
    const unsigned step = 64u * (unsigned)group;
    const char *qb = (const char*)q + (size_t)mg * 4 * step, *kb = (const char*)k + (size_t)mg * 256, *vb = (const char*)(v + (size_t)mg * (HEAD / 2));
    quad_u32 w[8];
    u64 value;
    for (unsigned n = 0;; ++n) {
      if (n == limit) { ok = false; break; }
      read_words(qb, step, 16u * (unsigned)(kq * group + min(col, group - 1)), kb, 16u * (unsigned)kq, vb, 4u * (unsigned)(share * 16 + (col & ~1)), w, value);
      if (all_tagged(w, tag) && __all((unsigned)(value >> 32) == tag)) break;
      __builtin_amdgcn_s_sleep(1);
    }
    vn = (unsigned)value >> (16 * (col & 1)) & 0xFFFFu;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      qf[s] = quad_u32{w[2 * s][0], w[2 * s][2], w[2 * s + 1][0], w[2 * s + 1][2]};
      kn[s] = quad_u32{w[4 + 2 * s][0], w[4 + 2 * s][2], w[5 + 2 * s][0], w[5 + 2 * s][2]};
      if (col != 0) kn[s] = quad_u32{0u, 0u, 0u, 0u};     // row 0 of a tile of keys
    }
  }
  const quad_f32 none = {0.f, 0.f, 0.f, 0.f};
  const float low = -__builtin_inff();
  quad_f32 sc[KEYS][2];
  float sn = low, mx = low;
#pragma unroll
  for (int i = 0; i < KEYS; ++i) {
    const int block = wave + WAVES * i;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[i][t] = quad_f32{low, low, low, low};
      if (block < blocks) {
        const quad_f32 z = product(kf[i][t][1], qf[1], product(kf[i][t][0], qf[0], none));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (block * 32 + t * 16 + kq * 4 + r < pos) sc[i][t][r] = z[r] * a.scale_log2;
          mx = fmaxf(mx, sc[i][t][r]);
        }
      }
    }
  }
  if (own) {
    const quad_f32 z = product(kn[1], qf[1], product(kn[0], qf[0], none));
    if (kq == 0) sn = z[0] * a.scale_log2;
    mx = fmaxf(mx, sn);
  }
  mx = fmaxf(mx, __shfl_xor(mx, 16, MS_WAVE));
  mx = fmaxf(mx, __shfl_xor(mx, 32, MS_WAVE));
  const float ref = mx == low ? 0.f : mx;
  const quad_u32 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  quad_f32 out = none, sum = none;
#pragma unroll
  for (int i = 0; i < KEYS; ++i) {
    const int block = wave + WAVES * i;
    if (block < blocks) {
      quad_bf16 p;
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = (__bf16)__builtin_amdgcn_exp2f(sc[i][e / 4][e & 3] - ref);
      if (block * 32 + 32 > pos) {     // what lies behind the last key may be anything
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int there = pos - (block * 32 + t * 16 + kq * 4);
          vf[i][t] &= there >= 4 ? ~0ull : there <= 0 ? 0ull : (1ull << (16 * there)) - 1;
        }
      }
      const quad_u32 values = {(unsigned)vf[i][0], (unsigned)(vf[i][0] >> 32), (unsigned)vf[i][1], (unsigned)(vf[i][1] >> 32)};
      const quad_u32 w = __builtin_bit_cast(quad_u32, p);
      out = product(values, w, out);
      sum = product(ones, w, sum);
    }
  }
  if (own) {
    quad_bf16 p = {0, 0, 0, 0, 0, 0, 0, 0};
    if (kq == 0) p[0] = (__bf16)__builtin_amdgcn_exp2f(sn - ref);
    const quad_u32 w = __builtin_bit_cast(quad_u32, p);
    out = product(quad_u32{kq == 0 ? vn : 0u, 0u, 0u, 0u}, w, out);
    sum = product(ones, w, sum);
  }
  if (!ok && lane == 0) sh.late[1] = 1;
  float* stats = reinterpret_cast<float*>(&sh.part[WAVES * MS_WAVE]);     // [wave][col]: reference, and behind them sums
  sh.part[wave * MS_WAVE + lane] = out;
  if (kq == 0) {
    stats[wave * 16 + col] = mx;
    stats[WAVES * 16 + wave * 16 + col] = sum[0];
  }
  __syncthreads();
  const bool late = sh.late[1] != 0;
  if (!late && wave == 0) {
    float top = low;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) top = fmaxf(top, stats[w * 16 + col]);
    quad_f32 o = none;
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(stats[w * 16 + col] - top);
      o += f * sh.part[w * MS_WAVE + lane];
      l = fmaf(f, stats[WAVES * 16 + w * 16 + col], l);
    }
    o *= 1.0f / l;
    if (col < group) {
      u64* word = a.heads + head_word((g * group + col) * HEAD + share * 16 + kq * 4, m, a.M);
#pragma unroll
      for (int h = 0; h < 2; ++h) put(word + h, two_bf16(o[2 * h], o[2 * h + 1]), tag);
    }
  }
  return !late;
}

template <int G, int MODE>
__device__ __forceinline__ bool run_o(Args& a, Shared& sh, LayerArgs& L, int layer, int b, int lane, int wave, unsigned tag, unsigned limit) {
  constexpr int XL = G / 4, XS = 16 / G;
  const int r0 = b * 4 * UO, kq = lane >> 4, mine = (a.Ko / 32 - wave + WAVES - 1) / WAVES, run = mine > 0 ? wave : 0;
  const quad_u32 zero = {0u, 0u, 0u, 0u};
  quad_u32 w[UO], x[XL];
  const int iw = (lane >> 2) & 3;
  const size_t kw = (size_t)(run + WAVES * (mine > 0 ? min(iw, mine - 1) : 0)) * 32 + kq * 8;
#pragma unroll
  for (int u = 0; u < UO; ++u) w[u] = load<quad_u32>(global<bf16>(L.w_o) + (size_t)(r0 + 4 * u + (lane & 3)) * a.Ko + kw);
  // pair 2 wave + (lane / 32) is finished here, its row lane % 4
  int u, m;
  pair_of(2 * wave + (lane >> 5), a.M, u, m);
  const int n = r0 + 4 * min(u, UO - 1) + (lane & 3);
  const bool mine_to_store = u < UO && (lane & 31) >= 16 && (lane & 31) < 20;
  float pre = 0.f;
  bool ok = true;
  if (MODE == CHAIN || layer == 0) pre = mine_to_store ? load<float>(a.x + (size_t)m * a.ldx + n) : 0.f;
  if constexpr (MODE == CHAIN) {
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int i = j * XS + (lane & 15) / G, mt = min(lane & (G - 1), a.M - 1);
      x[j] = load<quad_u32>(a.attn + (size_t)mt * a.ld_attn + (run + WAVES * (mine > 0 ? min(i, mine - 1) : 0)) * 32 + kq * 8);
    }
  } else {
    if (!wait_first(sh, a.heads + head_word((b * 8) % a.Ko, 0, a.M), tag, limit)) return false;
    if (layer > 0 && 2 * wave < UO * a.M) {      // the stream before (there long before the heads are)
      const u64* word = a.x2 + stream_word(n, m, a.M);
      ok = false;
      for (unsigned t = 0; t < limit && !ok; ++t) {
        const u64 v = look(word);
        pre = __uint_as_float((unsigned)v);
        ok = __all((unsigned)(v >> 32) == tag - 1u);
      }
    }
    unsigned at[XL];
    quad_u32 v[2 * XL];
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int i = j * XS + (lane & 15) / G;
      at[j] = 16u * ((((run * STEPS + (mine > 0 ? min(i, mine - 1) : 0)) * 2) * 4 + kq) * a.M + min(lane & (G - 1), a.M - 1));
    }
    const char* words = (const char*)a.heads;
    for (unsigned t = 0; ok; ++t) {
      if (t == limit) { ok = false; break; }
      read_words(words, words + 64 * a.M, at, v);
      if (all_tagged(v, tag)) break;
      __builtin_amdgcn_s_sleep(1);
    }
#pragma unroll
    for (int j = 0; j < XL; ++j) x[j] = quad_u32{v[2 * j][0], v[2 * j][2], v[2 * j + 1][0], v[2 * j + 1][2]};
    if (!ok && lane == 0) sh.late[1] = 1;
  }
#pragma unroll
  for (int j = 0; j < XL; ++j)
    if (j * XS + (lane & 15) / G >= mine) x[j] = zero;
  quad_f32 acc[UO][XL];
#pragma unroll
  for (int v = 0; v < UO; ++v) {
    if (iw >= mine) w[v] = zero;
#pragma unroll
    for (int j = 0; j < XL; ++j) acc[v][j] = product(w[v], x[j], quad_f32{0.f, 0.f, 0.f, 0.f});
  }
  leave_units<UO, G>(sh, acc, lane, wave);
  __syncthreads();
  const bool late = MODE != CHAIN && sh.late[1];
  if (!late && 2 * wave < UO * a.M) {
    const quad_f32 sum = finish_units(sh, min(u, UO - 1), G, m, lane);
    if (mine_to_store) put(a.x1 + stream_word(n, m, a.M), __float_as_uint(row_of(sum, lane) + pre), tag);
  }
  return !late;
}

template <int G, int MODE>
__device__ __forceinline__ bool run_gate(Args& a, Shared& sh, LayerArgs& L, int b, int lane, int wave, unsigned tag, unsigned limit) {
  constexpr int XS = 16 / G;
  const int col = lane & 15, kq = lane >> 4;
  const int steps = a.H / 32, mine = (steps - wave + WAVES - 1) / WAVES;
  const int n0 = 4 * (b * a.gate_units + min(b, a.gate_more)), rows_here = 4 * (a.gate_units + (b < a.gate_more ? 1 : 0));
  const int nt = (rows_here + 15) / 16;
  quad_u32 w[STEPS][NT];
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int k = min(wave + WAVES * i, steps - 1) * 32 + kq * 8;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      w[i][u] = load<quad_u32>(global<bf16>(L.w_gu) + (size_t)(n0 + min(u * 16 + col, rows_here - 1)) * a.H + k);
      paced<MODE>();
    }
  }
  StreamRows<G> rows;
  rows.ask_norm(global<float>(L.norm2), lane, wave, a.M, a.H);
  // In a launch of its own o is short: its words are polled as they are (waiting for one first: 0.4 to 1.2 us more).
  if (MODE == CHAIN) {
    if (threadIdx.x == 0) sh.late[1] = 0;
    __syncthreads();
  } else if (!wait_first(sh, a.x1 + stream_word((b * 8) % a.H, 0, a.M), tag, limit)) return false;
  quad_f32 acc[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) acc[u] = quad_f32{0.f, 0.f, 0.f, 0.f};
  float squares = 0.f;
  if (rows.poll(a.x1, a.M, tag, limit)) {
    squares = rows.squares();
    auto step = [&](auto index) {
      constexpr int i = decltype(index)::value, J = i / XS, BY = (i % XS) * G;
      if (i >= mine) return;       // the same for the whole wave
      const quad_u32 x = quad_turn<BY>(rows.x[J]);
#pragma unroll
      for (int u = 0; u < NT; ++u) acc[u] = product(w[i][u], x, acc[u]);
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
  } else if (lane == 0) {
    sh.late[1] = 1;
  }
  if (col < G) {
#pragma unroll
    for (int u = 0; u < NT; ++u) sh.part[(u * WAVES + wave) * 4 * G + kq * G + col] = acc[u];
    if (kq == 0) sh.part_ss[col][wave] = squares;
  }
  __syncthreads();
  const bool late = sh.late[1] != 0;
  if (!late && wave < nt && col < a.M && wave * 16 + kq * 4 < rows_here) {
    // tile `wave`: this lane has rows kq * 4 .. + 3 of it for token col: gate and up of two features
    float total = 0.f;
    quad_f32 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < WAVES; ++v) {
      total += sh.part_ss[col][v];
      sum += sh.part[(wave * WAVES + v) * 4 * G + kq * G + col];
    }
    sum *= inverse_root(fmaf(total, a.inv_H, L.eps2));
    put(a.act + act_word((n0 + wave * 16 + kq * 4) / 2, col, a.M), two_bf16(fast_silu(sum[0]) * sum[1], fast_silu(sum[2]) * sum[3]), tag);
  }
  return !late;
}

// P: pairs of loads of act asked for at a time
template <int G, int UD, int P, int MODE>
__device__ __forceinline__ bool run_down(Args& a, Shared& sh, LayerArgs& L, bool last, int b, int lane, int wave, unsigned tag, unsigned limit) {
  constexpr int XL = G / 4, XS = 16 / G, C = DOWN_LOADS;
  const int r0 = b * 4 * UD, kq = lane >> 4, steps = a.I / 32;
  const quad_u32 zero = {0u, 0u, 0u, 0u};
  // Where there are as many blocks as CUs, their weights would come ahead of x1 on the way to gate's blocks: they wait for x1 (one
  // token 13.5 -> 13.1 us; half as many blocks lose 0.3).
  if constexpr (UD == 1 && MODE == CHAIN) {
    if (!wait_first<2>(sh, a.x1 + stream_word((b * 8) % a.H, 0, a.M), tag, limit)) return false;
  }
  // runs `wave` and `wave` + 8 of the 16, C loads of four steps each
  quad_u32 w[2][C][UD];
  int mine[2], run[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    mine[h] = (steps - (wave + h * WAVES) + DOWN_WAVES - 1) / DOWN_WAVES;
    run[h] = mine[h] > 0 ? wave + h * WAVES : 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = min(4 * c + ((lane >> 2) & 3), max(mine[h], 1) - 1);
#pragma unroll
      for (int u = 0; u < UD; ++u) {
        w[h][c][u] = load<quad_u32>(global<bf16>(L.w_down) + (size_t)(r0 + 4 * u + (lane & 3)) * a.I + (run[h] + DOWN_WAVES * i) * 32 + kq * 8);
        paced<MODE>();
      }
    }
  }
  int pu, pm;
  pair_of(2 * wave + (lane >> 5), a.M, pu, pm);
  const int n = r0 + 4 * min(pu, UD - 1) + (lane & 3);
  if (!wait_first(sh, a.act + act_word((b * 32) % a.I, 0, a.M), tag, limit)) return false;
  // the stream before, of this lane's row (there long before act is)
  bool ok = true;
  float pre = 0.f;
  if (2 * wave < UD * a.M) {
    const u64* word = a.x1 + stream_word(n, pm, a.M);
    ok = false;
    for (unsigned t = 0; t < limit && !ok; ++t) {
      const u64 v = look(word);
      pre = __uint_as_float((unsigned)v);
      ok = __all((unsigned)(v >> 32) == tag);
    }
  }
  quad_f32 acc[UD][XL];
#pragma unroll
  for (int u = 0; u < UD; ++u)
#pragma unroll
    for (int j = 0; j < XL; ++j) acc[u][j] = quad_f32{0.f, 0.f, 0.f, 0.f};
  // act in rounds of P pairs of loads; six are both runs of up to 4 tokens, or one run of 8.  A step past a run's last takes that one's words
  // again, a run without any (short rows) the first run's; neither counts.
  const char* words = (const char*)a.act;
#pragma unroll
  for (int first = 0; first < 2 * C * XL; first += P) {
    unsigned at[P];
    quad_u32 v[2 * P];
#pragma unroll
    for (int l = 0; l < P; ++l) {
      const int h = (first + l) / (C * XL), c = (first + l) / XL % C, j = (first + l) % XL;
      const int i = min(4 * c + j * XS + (lane & 15) / G, max(mine[h], 1) - 1);
      at[l] = 16u * ((((run[h] * 4 * C + i) * 2) * 4 + kq) * a.M + min(lane & (G - 1), a.M - 1));
    }
    for (unsigned t = 0; ok; ++t) {
      if (t == limit) { ok = false; break; }
      read_words(words, words + 64 * a.M, at, v);
      if (all_tagged(v, tag)) break;
      __builtin_amdgcn_s_sleep(1);
    }
    if (!ok) break;
#pragma unroll
    for (int l = 0; l < P; ++l) {
      const int h = (first + l) / (C * XL), c = (first + l) / XL % C, j = (first + l) % XL;
      quad_u32 x = {v[2 * l][0], v[2 * l][2], v[2 * l + 1][0], v[2 * l + 1][2]};
      if (4 * c + 4 > mine[h]) {      // (the same for the whole wave)
        if (4 * c + j * XS + (lane & 15) / G >= mine[h]) x = zero;
        if (4 * c + ((lane >> 2) & 3) >= mine[h]) {
#pragma unroll
          for (int u = 0; u < UD; ++u) w[h][c][u] = zero;
        }
      }
#pragma unroll
      for (int u = 0; u < UD; ++u) acc[u][j] = product(w[h][c][u], x, acc[u][j]);
    }
  }
  if (!ok && lane == 0) sh.late[1] = 1;
  leave_units<UD, G>(sh, acc, lane, wave);
  __syncthreads();
  const bool late = sh.late[1] != 0;
  if (!late && 2 * wave < UD * a.M) {
    const quad_f32 sum = finish_units(sh, min(pu, UD - 1), G, pm, lane);
    if (pu < UD && (lane & 31) >= 16 && (lane & 31) < 20) {
      const float v = row_of(sum, lane) + pre;
      if (MODE == CHAIN ? a.n_front > 0 : !last) put(a.x2 + stream_word(n, pm, a.M), __float_as_uint(v), tag);
      if (MODE == CHAIN || last) store(a.x + (size_t)pm * a.ldx + n, v);
    }
  }
  return !late;
}

template <int G, int MODE>
__device__ __forceinline__ bool run_front(Args& a, Shared& sh, LayerArgs& L, int b, int lane, int wave, unsigned tag, unsigned limit) {
  constexpr int XL = G / 4;
  const int d = a.d, half = d / 2, head = b / a.per_head, j0 = (b - head * a.per_head) * 2 * UF;
  const int kq = lane >> 4, mine = (a.H / 32 - wave + WAVES - 1) / WAVES, run = mine > 0 ? wave : 0, iw = (lane >> 2) & 3;
  const quad_u32 zero = {0u, 0u, 0u, 0u};
  quad_u32 w[UF];
  const size_t kw = (size_t)(run + WAVES * (mine > 0 ? min(iw, mine - 1) : 0)) * 32 + kq * 8;
#pragma unroll
  for (int u = 0; u < UF; ++u)
    w[u] = load<quad_u32>(global<bf16>(L.w_front) + ((size_t)head * d + j0 + 2 * u + (lane & 1) + ((lane >> 1) & 1) * half) * a.H + kw);
  StreamRows<G> rows;
  rows.ask_norm(global<float>(L.norm1), lane, wave, a.M, a.H);
  // pair 2 wave + (lane / 32), a unit and a token, is finished here; lane % 4 = r stores row r (0, 1: lower features, 2, 3: partners)
  int unit, m;
  pair_of(2 * wave + (lane >> 5), a.M, unit, m);
  const int pu = min(unit, UF - 1), r = lane & 3;
  const int j = j0 + 2 * pu + (r & 1);
  const auto bias = global<float>(L.b_front);
  const float b_lo = L.b_front ? bias[head * d + j] : 0.f, b_hi = L.b_front ? bias[head * d + half + j] : 0.f;
  // where this lane's results go: a word of this launch's attention, its place in the pages or among the queries
  const int f = r < 2 ? j : j + half;   // this lane's feature within the head
  const int kind = head < a.nh ? 0 : head < a.nh + a.nkv ? 1 : 2, kv = head - a.nh - (kind == 2 ? a.nkv : 0);
  u64* word = a.qkv;
  if constexpr (MODE != CHAIN) {
    const int group = a.nh / a.nkv, of = head / group;
    if (kind == 0) word += q_word(m * a.nkv + of, head - of * group, f, group);
    else if (kind == 1) word += (size_t)a.M * a.nh * (HEAD / 2) + k_word(m * a.nkv + kv, f);
    else word += (size_t)a.M * (a.nh + a.nkv) * (HEAD / 2) + (m * a.nkv + kv) * (HEAD / 2) + f / 2;
  }
  u64 place = 0;
  if (kind == 0) {
    if constexpr (MODE == CHAIN) place = (u64)(a.q_out + ((size_t)m * a.nh + head) * d + f);
  } else {
    const long long slot = load<int>(a.slots + m);
    const bool pow2 = (a.page_size & (a.page_size - 1)) == 0;   // no division then
    const long long page = pow2 ? slot >> (31 - __builtin_clz(a.page_size)) : slot / a.page_size;
    const int off = pow2 ? (int)(slot & (a.page_size - 1)) : (int)(slot % a.page_size);
    const size_t row = (size_t)page * a.nkv + kv;
    if (kind == 1) place = L.front_k + 2 * ((row * a.page_size + off) * d + f);
    else place = L.front_v + 2 * (a.v_transposed ? (row * d + f) * a.page_size + off : (row * a.page_size + off) * d + f);
    if (slot < 0) place = 0;
  }
  float sn = 0.f, cs = 1.f;
  if (head < a.nh + a.nkv) ms_sincos_rot((float)load<int>(a.positions + m) * global<float>(L.inv_freq)[j], &sn, &cs);   // q and k heads turn
#pragma unroll
  for (int u = 0; u < UF; ++u)
    if (iw >= mine) w[u] = zero;
  bool ok = true;
  if constexpr (MODE == FIRST) {
    rows.read(a.x, a.ldx, lane, wave, a.M, a.H);
  } else {
    if (!wait_first(sh, a.x2 + stream_word((b * 8) % a.H, 0, a.M), tag, limit)) return false;
    ok = rows.poll(a.x2, a.M, tag, limit);
  }
  quad_f32 acc[UF][XL];
  float squares = 0.f;
  if (ok) {
    squares = rows.squares();
#pragma unroll
    for (int u = 0; u < UF; ++u)
#pragma unroll
      for (int l = 0; l < XL; ++l) acc[u][l] = product(w[u], rows.x[l], quad_f32{0.f, 0.f, 0.f, 0.f});
  } else if (lane == 0) {
    sh.late[1] = 1;
  }
  leave_units<UF, G>(sh, acc, lane, wave);
  if (lane < G) sh.part_ss[lane][wave] = squares;
  __syncthreads();
  const bool late = MODE != FIRST && sh.late[1];
  if (!late && 2 * wave < UF * a.M) {
    const quad_f32 sum = finish_units(sh, pu, G, m, lane);
    if (unit < UF && (lane & 31) >= 16 && (lane & 31) < 20) {
      float total = 0.f;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) total += sh.part_ss[m][v];
      const float inv = inverse_root(fmaf(total, a.inv_H, L.eps1));
      const float lo = (r & 1 ? sum[1] : sum[0]) * inv + b_lo, hi = (r & 1 ? sum[3] : sum[2]) * inv + b_hi;
      const float value = r < 2 ? lo * cs - hi * sn : hi * cs + lo * sn;
      if constexpr (MODE != CHAIN) {        // features f and f + 1 from neighbouring lanes
        const unsigned both = two_bf16(value, lanes_moved<0xB1>(value));
        if (!(r & 1)) put(word, both, tag + 1u);
      }
      if (place) *global_out<unsigned short>(place) = __builtin_bit_cast(unsigned short, __float2bfloat16(value));
    }
  }
  return !late;
}

// Thread 0 of the one block that stays: the next item to try, or -1 when every item that was given up is done.
__device__ int next_given_up(unsigned* given_up, Shared& sh, int own) {
  for (;;) {
    const unsigned n = __hip_atomic_load(given_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int at = -1;
    for (unsigned i = 1; i <= n; ++i) {
      const unsigned p = (sh.position + i) % n;
      if (!((sh.done[p / 32] >> (p % 32)) & 1)) { at = (int)p; break; }
    }
    if (at == 0) { sh.position = 0; return own; }
    if (at > 0) {
      unsigned item = 0;     // its owner counted itself and stores its item next: it is running
      while (item == 0) item = __hip_atomic_load(given_up + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sh.position = at;
      return (int)item - 1;
    }
    // all n are done: leave the list empty, unless somebody came meanwhile
    for (unsigned i = 1; i < n; ++i) __hip_atomic_store(given_up + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);
    unsigned expected = n;
    if (__hip_atomic_compare_exchange_strong(given_up, &expected, 0u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return -1;
  }
}

template <int G, int UD, int P, int MODE>
__device__ __forceinline__ bool run_item(Shared& sh, int item, unsigned tag, unsigned limit) {
  int lane = threadIdx.x & (MS_WAVE - 1);
  int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);   // the same for the whole wave
  Args* args = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
  // what a phase works out from these belongs into that phase, not ahead of all of them
  asm volatile("" : "+v"(lane), "+s"(wave), "+s"(args));
  Args& a = *args;
  if constexpr (MODE == FIRST) {
    return run_front<G, MODE>(a, sh, a.one, item, lane, wave, tag, limit);
  } else {
    int layer = 0, b = item;
    if constexpr (MODE == WHOLE) {
      const int of_a_layer = a.n_attn + a.n_o + a.n_gate + a.n_down + a.n_front;
      layer = item / of_a_layer;
      b = item - layer * of_a_layer;
      tag += (unsigned)layer;
    }
    LayerArgs& L = MODE == WHOLE ? *((LayerArgs*)a.layers + layer) : a.one;
    if constexpr (MODE == WHOLE) {
      if (b < a.n_attn) return run_attention(a, sh, L, b, lane, wave, tag, limit);
      b -= a.n_attn;
    }
    if (b < a.n_o) return run_o<G, MODE>(a, sh, L, layer, b, lane, wave, tag, limit);
    if ((b -= a.n_o) < a.n_gate) return run_gate<G, MODE>(a, sh, L, b, lane, wave, tag, limit);
    if ((b -= a.n_gate) < a.n_down) return run_down<G, UD, P, MODE>(a, sh, L, layer == a.n_layers - 1, b, lane, wave, tag, limit);
    return run_front<G, MODE>(a, sh, L, b - a.n_down, lane, wave, tag, limit);
  }
}

// The number of a launch (WHOLE: of its first layer; FIRST: the one before that, of the WHOLE launch that follows it).
__device__ __forceinline__ unsigned first_tag(const ChainArgs& a, int mode) {
  if (mode == CHAIN) return a.epoch[a.launch] * (unsigned)a.launches + (unsigned)a.launch + 1u;
  const unsigned step = mode == FIRST ? a.epoch[0] + 1u : a.epoch[1];
  return step * (unsigned)(a.n_layers + 1) + (mode == FIRST ? 0u : 1u);
}

template <int G, int UD, int MODE>
__global__ void __launch_bounds__(WAVES * MS_WAVE, 4)
decode_chain_kernel(ChainArgs a) {
  __shared__ Shared sh;
  const unsigned tag = first_tag(a, MODE);
  if (blockIdx.x == 0 && threadIdx.x == 0) a.epoch[a.launch == 0 ? a.launches - 1 : a.launch - 1] += 1;
  if (run_item<G, UD, 6, MODE>(sh, blockIdx.x, tag, a.limit)) return;
  if constexpr (MODE != FIRST) {      // (which waits for nothing)
    // given up: end, or stay if nobody has yet (and no launch was broken off: then nothing is listed any more, either)
    if (threadIdx.x == 0) {
      unsigned before = 1;
      if (!__hip_atomic_load(a.given_up + LIST, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        before = __hip_atomic_fetch_add(a.given_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (before > 0) __hip_atomic_store(a.given_up + before, blockIdx.x + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      for (unsigned& d : sh.done) d = 0;
      sh.position = 0;
      sh.in_vain = 0;
      sh.next = before > 0 ? -1 : (int)blockIdx.x;
    }
    __syncthreads();
    while (sh.next >= 0) {      // (three pairs at a time: the loop needs registers of its own)
      const bool ok = run_item<G, UD, 3, MODE>(sh, sh.next, tag, 64);
      __syncthreads();
      if (threadIdx.x == 0) {
        if (ok) {
          sh.done[sh.position / 32] |= 1u << (sh.position % 32);
          sh.in_vain = 0;
        }
        sh.next = ++sh.in_vain > a.patience ? -1 : next_given_up(a.given_up, sh, (int)blockIdx.x);
      }
      __syncthreads();
    }
    if (threadIdx.x == 0 && sh.in_vain > a.patience) {      // (the list stays as it is: at most this launch's other blocks are on it)
      __hip_atomic_store(a.given_up + LIST, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (a.told) __hip_atomic_store(a.told, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

size_t round_up(size_t n) { return (n + 255) / 256 * 256; }
size_t stream_bytes(int M) { return round_up((size_t)WAVES * STEPS * 32 * M * 8); }
size_t act_bytes(int M) { return round_up((size_t)DOWN_WAVES * 4 * DOWN_LOADS * 16 * M * 8); }
size_t heads_bytes(int M) { return round_up((size_t)WAVES * STEPS * 16 * M * 8); }
size_t qkv_bytes(int M, int heads) { return round_up((size_t)M * heads * (HEAD / 2) * 8); }
constexpr size_t LIST_BYTES = 4 * (1 + LIST), EPOCH_BYTES = 4 * MAX_LAUNCHES;

unsigned g_limit = 2048;         // looks of a waiting block, each about 0.8 us
unsigned g_patience = 400000;    // tries of the block that stays, of 64 looks or more each: 20 s in which no block of the launch ended

int down_units(int M, bool whole) { return M <= 2 && !whole ? 1 : 2; }

// The sizes and what follows from them; false: not taken.
bool sizes_into(ChainArgs& a, int M, int H, int I, int nh, int nkv, int d, int n_layers) {
  if (M < 1 || M > 8 || H <= 0 || nh <= 0 || nkv <= 0 || d <= 0 || I <= 0 || n_layers < 0) return false;
  const long long Ko = (long long)nh * d;
  if (H % 32 || Ko % 32 || I % 32 || d % (4 * UF) || H > 32 * WAVES * STEPS || Ko > 32 * WAVES * STEPS || nkv > nh ||
      I > 32 * DOWN_WAVES * 4 * DOWN_LOADS)
    return false;
  if (n_layers && (d != HEAD || nh % nkv || nh / nkv > 16)) return false;
  a.M = M; a.H = H; a.Ko = (int)Ko; a.I = I; a.nh = nh; a.nkv = nkv; a.d = d;
  a.n_layers = n_layers ? n_layers : 1;
  a.n_attn = n_layers ? M * nkv * SHARES : 0;
  a.n_o = H / (4 * UO);
  a.n_gate = std::max((I / 2 + 4 * NT - 1) / (4 * NT), std::min(I / 2, 256));
  a.n_down = H / (4 * down_units(M, n_layers > 0));
  a.n_front = (nh + 2 * nkv) * (d / 2) / (2 * UF);
  a.gate_units = I / 2 / a.n_gate; a.gate_more = I / 2 % a.n_gate;
  a.per_head = d / (4 * UF);
  a.inv_H = 1.0f / (float)H;
  return (long long)a.n_layers * (a.n_attn + a.n_o + a.n_gate + a.n_down + a.n_front) <= LIST;
}
void workspace_into(ChainArgs& a, void* workspace, int* told) {
  char* ws = (char*)workspace;
  a.given_up = (unsigned*)ws; ws += LIST_BYTES;
  a.epoch = (unsigned*)ws; ws += EPOCH_BYTES;
  a.x1 = (u64*)ws; ws += stream_bytes(a.M);
  a.x2 = (u64*)ws; ws += stream_bytes(a.M);
  a.act = (u64*)ws; ws += act_bytes(a.M);
  a.heads = (u64*)ws; ws += heads_bytes(a.M);
  a.qkv = (u64*)ws;
  a.told = told;
  a.limit = g_limit;
  a.patience = g_patience;
}
template <int MODE>
int launch_chain(const ChainArgs& a, int blocks, hipStream_t stream) {
  const dim3 grid(blocks), block(WAVES * MS_WAVE);
  if constexpr (MODE == FIRST) {
    if (a.M <= 4) decode_chain_kernel<4, 1, MODE><<<grid, block, 0, stream>>>(a);
    else decode_chain_kernel<8, 1, MODE><<<grid, block, 0, stream>>>(a);
  } else {
    if (MODE == CHAIN && a.M <= 2) decode_chain_kernel<4, 1, CHAIN><<<grid, block, 0, stream>>>(a);
    else if (a.M <= 4) decode_chain_kernel<4, 2, MODE><<<grid, block, 0, stream>>>(a);
    else decode_chain_kernel<8, 2, MODE><<<grid, block, 0, stream>>>(a);
  }
  return ms_launch_status();
}
int shift_of(int page_size) { return page_size > 0 && (page_size & (page_size - 1)) == 0 ? 31 - __builtin_clz(page_size) : -1; }

}  // namespace

// Tests: how many times a waiting block looks before it gives its item up; 0 restores the choice.
extern "C" void ms_decode_chain_limit(int limit) { g_limit = limit > 0 ? (unsigned)limit : 2048u; }
// And how many tries in a row may be in vain before the block that stays breaks the launch off; 0 restores the choice.
extern "C" void ms_decode_chain_patience(int tries) { g_patience = tries > 0 ? (unsigned)tries : 400000u; }

// Bytes of a workspace, to be zeroed once and then left to launches of ONE batch size, one step after the other, 0 where the
// kernels do not take the sizes: for ms_decode_chain (n_layers 0), or for ms_decode_first and ms_decode_layers of n_layers layers.
extern "C" int ms_decode_chain_workspace(int M, int H, int num_heads, int num_kv_heads, int head_dim, int I, int n_layers) {
  ChainArgs a;
  if (!sizes_into(a, M, H, I, num_heads, num_kv_heads, head_dim, n_layers)) return 0;
  const size_t chain = LIST_BYTES + EPOCH_BYTES + 2 * stream_bytes(M) + act_bytes(M);
  return (int)(n_layers ? chain + heads_bytes(M) + qkv_bytes(M, num_heads + 2 * num_kv_heads) : chain);
}

// attn bfloat16 [M, num_heads head_dim] (M <= 8), x float [M, H] (in place), weights bfloat16 with contiguous rows: w_o [H, num_heads
// head_dim], w_gate_up [2 I, H] interleaved, w_down [H, I]; w_qkv (or null: no front) [(nh + 2 nkv) d, H], q_out, pages and so on
// as in ms_qkv_rope_store.  `launch` of `launches` (2 to 1,024) chains of the step.
extern "C" int ms_decode_chain(const void* attn, long long ld_attn, const void* w_o, float* x, long long ldx, const float* norm2,
                               float eps2, const void* w_gate_up, const void* w_down, const float* norm1, float eps1,
                               const void* w_qkv, const float* b_qkv, const int* positions, const float* inv_freq,
                               const int* slot_mapping, void* q_out, void* k_pages, void* v_pages, int M, int H, int I,
                               int num_heads, int num_kv_heads, int head_dim, int page_size, int v_transposed, void* workspace,
                               int* told, int launch, int launches, hipStream_t stream) {
  if (M <= 0) return MS_OK;
  ChainArgs a = {};
  if (!sizes_into(a, M, H, I, num_heads, num_kv_heads, head_dim, 0)) return MS_UNSUPPORTED;
  if (launches < 2 || launches > MAX_LAUNCHES || launch < 0 || launch >= launches || !workspace || !attn || !w_o || !x || !norm2 ||
      !w_gate_up || !w_down || ld_attn < a.Ko || ldx < H)
    return MS_BAD_ARG;
  if (ld_attn % 8 || (((uintptr_t)attn | (uintptr_t)w_o | (uintptr_t)w_gate_up | (uintptr_t)w_down | (uintptr_t)norm2) % 16) ||
      ((uintptr_t)workspace % 256))
    return MS_UNSUPPORTED;
  if (w_qkv) {
    if (!norm1 || !positions || !inv_freq || !slot_mapping || !q_out || !k_pages || !v_pages || page_size <= 0) return MS_BAD_ARG;
    if (((uintptr_t)w_qkv | (uintptr_t)norm1) % 16) return MS_UNSUPPORTED;
  } else {
    a.n_front = 0;
  }
  a.attn = (const bf16*)attn; a.ld_attn = ld_attn;
  a.x = x; a.ldx = ldx;
  a.one = Layer{(u64)w_o, (u64)w_gate_up, (u64)w_down, (u64)w_qkv, (u64)norm2, (u64)norm1, (u64)b_qkv, (u64)inv_freq, 0, 0,
                (u64)k_pages, (u64)v_pages, eps2, eps1};
  a.positions = positions; a.slots = slot_mapping; a.q_out = (bf16*)q_out;
  a.page_size = page_size; a.v_transposed = v_transposed;
  a.launch = launch; a.launches = launches;
  workspace_into(a, workspace, told);
  return launch_chain<CHAIN>(a, a.n_o + a.n_gate + a.n_down + a.n_front, stream);
}

// A whole step's layers in two launches, in this order on one workspace: ms_decode_first is the first layer's norm, q/k/v, rotation
// and cache store of x float [M, H]; ms_decode_layers everything from its attention to the last layer's down projection, into x.
// Values' pages transposed, pages of a power of two from 16 tokens on, contexts (with the step's token) of at most 1,024 keys.
extern "C" int ms_decode_first(const float* x, long long ldx, const float* norm1, float eps1, const void* w_qkv, const float* b_qkv,
                               const int* positions, const float* inv_freq, const int* slot_mapping, void* k_pages, void* v_pages,
                               int M, int H, int I, int num_heads, int num_kv_heads, int head_dim, int page_size, int n_layers,
                               void* workspace, hipStream_t stream) {
  if (M <= 0) return MS_OK;
  ChainArgs a = {};
  if (n_layers < 1 || !sizes_into(a, M, H, I, num_heads, num_kv_heads, head_dim, n_layers)) return MS_UNSUPPORTED;
  if (!x || !norm1 || !w_qkv || !positions || !inv_freq || !slot_mapping || !k_pages || !v_pages || !workspace || ldx < H) return MS_BAD_ARG;
  if (shift_of(page_size) < 4 || ldx % 4 || (((uintptr_t)x | (uintptr_t)norm1 | (uintptr_t)w_qkv) % 16) || (uintptr_t)workspace % 256)
    return MS_UNSUPPORTED;
  a.x = const_cast<float*>(x); a.ldx = ldx;
  a.one = Layer{0, 0, 0, (u64)w_qkv, 0, (u64)norm1, (u64)b_qkv, (u64)inv_freq, 0, 0, (u64)k_pages, (u64)v_pages, 0.f, eps1};
  a.positions = positions; a.slots = slot_mapping;
  a.page_size = page_size; a.page_shift = shift_of(page_size); a.v_transposed = 1;
  a.launch = 0; a.launches = 2;
  workspace_into(a, workspace, nullptr);
  return launch_chain<FIRST>(a, a.n_front, stream);
}

// layers: n_layers records of ms_decode_layer_bytes() bytes in device memory (struct Layer above; the last one's w_front and what
// follows from it are not read).  context_lens [M] counts the step's token; table int32 [rows, table_width], table_rows [M] or null.
extern "C" int ms_decode_layer_bytes() { return (int)sizeof(Layer); }
extern "C" int ms_decode_layers(const void* layers, float* x, long long ldx, const int* positions, const int* slot_mapping,
                                const int* context_lens, const int* table, const int* table_rows, int table_width, float scale,
                                int M, int H, int I, int num_heads, int num_kv_heads, int head_dim, int page_size, int n_layers,
                                void* workspace, int* told, hipStream_t stream) {
  if (M <= 0) return MS_OK;
  ChainArgs a = {};
  if (n_layers < 1 || !sizes_into(a, M, H, I, num_heads, num_kv_heads, head_dim, n_layers)) return MS_UNSUPPORTED;
  if (!layers || !x || !positions || !slot_mapping || !context_lens || !table || table_width <= 0 || !workspace || ldx < H) return MS_BAD_ARG;
  if (shift_of(page_size) < 4 || (uintptr_t)layers % 8 || (uintptr_t)workspace % 256) return MS_UNSUPPORTED;
  a.layers = (u64)layers;
  a.x = x; a.ldx = ldx;
  a.positions = positions; a.slots = slot_mapping; a.contexts = context_lens; a.table = table; a.table_rows = table_rows;
  a.table_width = table_width;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.page_size = page_size; a.page_shift = shift_of(page_size); a.v_transposed = 1;
  a.launch = 1; a.launches = 2;
  workspace_into(a, workspace, told);
  return launch_chain<WHOLE>(a, n_layers * (a.n_attn + a.n_o + a.n_gate + a.n_down + a.n_front) - a.n_front, stream);
}
