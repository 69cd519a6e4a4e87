// The products between two attentions of a decode step, for up to 8 tokens of a narrow model, as ONE kernel:
//
//   o       x1 = x + attention . Wo^T                              (float residual stream)
//   gate    act = silu(norm(x1) . Wg^T) * (norm(x1) . Wu^T)        (gate and up rows interleaved)
//   down    x2 = x1 + act . Wd^T, back into x
//   front   the next layer's q, k, v from norm(x2): bias, rotation, q to its buffer, k and v into their pages
//
// As four kernels these are bound by latency: a launch is 1.6 us, and every kernel starts with blocks that wait for weights
// which could have been on their way all along (0.5B, 30 MB of weights: 2.9 + 8.2 + 4.7 + 4.4 = 20.1 us at one token, 24.6 at 8).
// Here a block is one item of one phase, all phases' blocks are launched at once, and a block asks for its weights (into
// registers) before it waits for the phase before it.  What is left of a phase is the way of its results to the blocks that
// need all of them, about 1.5 us, its sums, and its share of reading the weights: 13.1 us at one token, 14.0 at 4, 15.5 at 8.
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
// works off, as their inputs come in, the items that others gave up.  So a launch needs room for one block to end.
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
constexpr int LIST = 1151;            // items that can be given up: the sizes above make 1,024 at most
constexpr int MAX_LAUNCHES = 1024;    // of a step

struct ChainArgs {
  const bf16* attn;
  const bf16 *w_o, *w_gu, *w_down, *w_front;
  float* x;
  const float *norm2, *norm1, *b_front, *inv_freq;
  const int *positions, *slots;
  bf16 *q_out, *k_pages, *v_pages;
  u64 *x1, *x2, *act;
  unsigned *given_up;                 // [1 + LIST]: how many, then the items
  unsigned *epoch;
  long long ld_attn, ldx;
  float eps2, eps1, inv_H;
  int M, H, Ko, I, nh, nkv, d, page_size, v_transposed;
  int n_o, n_gate, n_down, n_front;   // blocks of each phase
  int gate_units, gate_more;          // units of four gate/up rows to a block of gate, and how many blocks have one more
  int per_head;                       // blocks of front to a head
  int launch, launches;
  unsigned limit;
};

// ---- words
__device__ __forceinline__ void put(u64* word, unsigned value, unsigned tag) {
  __hip_atomic_store(word, ((u64)tag << 32) | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 look(const u64* word) {
  return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
  int late[2];                          // somebody gave up: waiting for the first word, for the others
  int next, position;
  unsigned done[(LIST + 32) / 32];
};

// One word of the phase before, by one wave, so that blocks far ahead of their inputs disturb nobody.  Whole block; false: not
// within `limit` looks.
__device__ __forceinline__ bool wait_first(Shared& sh, const u64* word, unsigned tag, unsigned limit) {
  if (threadIdx.x < MS_WAVE) {
    int late = 1;
    for (unsigned n = 0; n < limit; ++n) {
      if ((unsigned)(look(word) >> 32) == tag) { late = 0; break; }
      __builtin_amdgcn_s_sleep(1);
    }
    if (threadIdx.x == 0) { sh.late[0] = late; sh.late[1] = 0; }
  }
  __syncthreads();
  return sh.late[0] == 0;
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

  __device__ __forceinline__ void ask_norm(const float* norm_w, int lane, int wave, int M, int H) {
    const int mine = (H / 32 - wave + WAVES - 1) / WAVES, m = min(lane & (G - 1), M - 1);
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int i = j * XS + (lane & 15) / G, there = mine > 0 ? min(i, mine - 1) : 0, run = mine > 0 ? wave : 0;
      in[j] = i < mine;
      at[j] = 16u * ((((run * STEPS + there) * 4) * 4 + (lane >> 4)) * M + m);
      const float* w = norm_w + (run + WAVES * there) * 32 + (lane >> 4) * 8;
      nw[j][0] = *reinterpret_cast<const quad_f32*>(w);
      nw[j][1] = *reinterpret_cast<const quad_f32*>(w + 4);
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
      ss[j] = 0.f;
      quad_bf16 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = in[j] ? __uint_as_float(v[4 * j + e / 2][2 * (e & 1)]) : 0.f;
        ss[j] = fmaf(f, f, ss[j]);
        h[e] = (__bf16)(f * nw[j][e / 4][e & 3]);
      }
      x[j] = __builtin_bit_cast(quad_u32, h);
    }
    return true;
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
// unit and token of pair p = unit * M + token of at most two units (a token within the batch for a pair beyond them, too)
__device__ __forceinline__ void pair_of(int p, int M, int& unit, int& token) {
  unit = p >= 2 * M ? 2 : p >= M ? 1 : 0;
  token = min(p - unit * M, M - 1);
}
__device__ __forceinline__ float row_of(const quad_f32& v, int r) { return r & 2 ? (r & 1 ? v[3] : v[2]) : (r & 1 ? v[1] : v[0]); }
__device__ __forceinline__ quad_f32 product(const quad_u32& w, const quad_u32& x, const quad_f32& acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(quad_bf16, w), __builtin_bit_cast(quad_bf16, x), acc, 0, 0, 0);
}

template <int G>
__device__ __forceinline__ void run_o(const ChainArgs& a, Shared& sh, int b, int lane, int wave, unsigned tag) {
  constexpr int XL = G / 4, XS = 16 / G;
  const int r0 = b * 4 * UO, kq = lane >> 4, mine = (a.Ko / 32 - wave + WAVES - 1) / WAVES, run = mine > 0 ? wave : 0;
  const quad_u32 zero = {0u, 0u, 0u, 0u};
  quad_u32 w[UO], x[XL];
  const int iw = (lane >> 2) & 3;
  const size_t kw = (size_t)(run + WAVES * (mine > 0 ? min(iw, mine - 1) : 0)) * 32 + kq * 8;
#pragma unroll
  for (int u = 0; u < UO; ++u) w[u] = *reinterpret_cast<const quad_u32*>(a.w_o + (size_t)(r0 + 4 * u + (lane & 3)) * a.Ko + kw);
#pragma unroll
  for (int j = 0; j < XL; ++j) {
    const int i = j * XS + (lane & 15) / G, m = min(lane & (G - 1), a.M - 1);
    x[j] = *reinterpret_cast<const quad_u32*>(a.attn + (size_t)m * a.ld_attn + (run + WAVES * (mine > 0 ? min(i, mine - 1) : 0)) * 32 + kq * 8);
    if (i >= mine) x[j] = zero;
  }
  // pair 2 wave + (lane / 32) is finished here, its row lane % 4
  int u, m;
  pair_of(2 * wave + (lane >> 5), a.M, u, m);
  const int n = r0 + 4 * u + (lane & 3);
  const bool mine_to_store = u < UO && (lane & 31) >= 16 && (lane & 31) < 20;
  const float pre = mine_to_store ? a.x[(size_t)m * a.ldx + n] : 0.f;
  quad_f32 acc[UO][XL];
#pragma unroll
  for (int v = 0; v < UO; ++v) {
    if (iw >= mine) w[v] = zero;
#pragma unroll
    for (int j = 0; j < XL; ++j) acc[v][j] = product(w[v], x[j], quad_f32{0.f, 0.f, 0.f, 0.f});
  }
  leave_units<UO, G>(sh, acc, lane, wave);
  __syncthreads();
  if (2 * wave >= UO * a.M) return;
  const quad_f32 sum = finish_units(sh, min(u, UO - 1), G, m, lane);
  if (mine_to_store) put(a.x1 + stream_word(n, m, a.M), __float_as_uint(row_of(sum, lane) + pre), tag);
}

template <int G>
__device__ __forceinline__ bool run_gate(const ChainArgs& a, Shared& sh, int b, int lane, int wave, unsigned tag, unsigned limit) {
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
    for (int u = 0; u < NT; ++u)
      w[i][u] = *reinterpret_cast<const quad_u32*>(a.w_gu + (size_t)(n0 + min(u * 16 + col, rows_here - 1)) * a.H + k);
  }
  StreamRows<G> rows;
  rows.ask_norm(a.norm2, lane, wave, a.M, a.H);
  // o is short: its words are polled as they are (waiting for one first: 0.4 to 1.2 us more)
  if (threadIdx.x == 0) sh.late[1] = 0;
  __syncthreads();
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
  if (sh.late[1]) return false;
  if (wave >= nt || col >= a.M || wave * 16 + kq * 4 >= rows_here) return true;
  // tile `wave`: this lane has rows kq * 4 .. + 3 of it for token col: gate and up of two features
  float total = 0.f;
  quad_f32 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < WAVES; ++v) {
    total += sh.part_ss[col][v];
    sum += sh.part[(wave * WAVES + v) * 4 * G + kq * G + col];
  }
  sum *= inverse_root(fmaf(total, a.inv_H, a.eps2));
  const bf16 f0 = from_float<bf16>(fast_silu(sum[0]) * sum[1]), f1 = from_float<bf16>(fast_silu(sum[2]) * sum[3]);
  const unsigned both = (unsigned)__builtin_bit_cast(unsigned short, f0) | ((unsigned)__builtin_bit_cast(unsigned short, f1) << 16);
  put(a.act + act_word((n0 + wave * 16 + kq * 4) / 2, col, a.M), both, tag);
  return true;
}

// P: pairs of loads of act asked for at a time
template <int G, int UD, int P>
__device__ __forceinline__ bool run_down(const ChainArgs& a, Shared& sh, int b, int lane, int wave, unsigned tag, unsigned limit) {
  constexpr int XL = G / 4, XS = 16 / G, C = DOWN_LOADS;
  const int r0 = b * 4 * UD, kq = lane >> 4, steps = a.I / 32;
  const quad_u32 zero = {0u, 0u, 0u, 0u};
  // Where there are as many blocks as CUs, their weights would come ahead of x1 on the way to gate's blocks: they wait for x1 (one
  // token 13.5 -> 13.1 us; half as many blocks lose 0.3).
  if constexpr (UD == 1) {
    if (!wait_first(sh, a.x1 + stream_word((b * 8) % a.H, 0, a.M), tag, limit)) return false;
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
      for (int u = 0; u < UD; ++u)
        w[h][c][u] = *reinterpret_cast<const quad_u32*>(a.w_down + (size_t)(r0 + 4 * u + (lane & 3)) * a.I + (run[h] + DOWN_WAVES * i) * 32 + kq * 8);
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
  if (sh.late[1]) return false;
  if (2 * wave >= UD * a.M) return true;
  const quad_f32 sum = finish_units(sh, min(pu, UD - 1), G, pm, lane);
  if (pu >= UD || (lane & 31) < 16 || (lane & 31) >= 20) return true;
  const float v = row_of(sum, lane) + pre;
  if (a.n_front) put(a.x2 + stream_word(n, pm, a.M), __float_as_uint(v), tag);
  a.x[(size_t)pm * a.ldx + n] = v;
  return true;
}

template <int G>
__device__ __forceinline__ bool run_front(const ChainArgs& a, Shared& sh, int b, int lane, int wave, unsigned tag, unsigned limit) {
  constexpr int XL = G / 4;
  const int d = a.d, half = d / 2, head = b / a.per_head, j0 = (b - head * a.per_head) * 2 * UF;
  const int kq = lane >> 4, mine = (a.H / 32 - wave + WAVES - 1) / WAVES, run = mine > 0 ? wave : 0, iw = (lane >> 2) & 3;
  const quad_u32 zero = {0u, 0u, 0u, 0u};
  quad_u32 w[UF];
  const size_t kw = (size_t)(run + WAVES * (mine > 0 ? min(iw, mine - 1) : 0)) * 32 + kq * 8;
#pragma unroll
  for (int u = 0; u < UF; ++u)
    w[u] = *reinterpret_cast<const quad_u32*>(a.w_front + ((size_t)head * d + j0 + 2 * u + (lane & 1) + ((lane >> 1) & 1) * half) * a.H + kw);
  StreamRows<G> rows;
  rows.ask_norm(a.norm1, lane, wave, a.M, a.H);
  // pair 2 wave + (lane / 32), a unit and a token, is finished here; lane % 4 = r stores row r (0, 1: lower features, 2, 3: partners)
  int unit, m;
  pair_of(2 * wave + (lane >> 5), a.M, unit, m);
  const int pu = min(unit, UF - 1), r = lane & 3;
  const int j = j0 + 2 * pu + (r & 1);
  const float b_lo = a.b_front ? a.b_front[head * d + j] : 0.f, b_hi = a.b_front ? a.b_front[head * d + half + j] : 0.f;
  const long long slot = a.slots[m];
  float sn = 0.f, cs = 1.f;
  if (head < a.nh + a.nkv) ms_sincos_rot((float)a.positions[m] * a.inv_freq[j], &sn, &cs);   // q and k heads turn
#pragma unroll
  for (int u = 0; u < UF; ++u)
    if (iw >= mine) w[u] = zero;
  if (!wait_first(sh, a.x2 + stream_word((b * 8) % a.H, 0, a.M), tag, limit)) return false;
  quad_f32 acc[UF][XL];
  float squares = 0.f;
  if (rows.poll(a.x2, a.M, tag, limit)) {
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
  if (sh.late[1]) return false;
  if (2 * wave >= UF * a.M) return true;
  const quad_f32 sum = finish_units(sh, pu, G, m, lane);
  if (unit >= UF || (lane & 31) < 16 || (lane & 31) >= 20) return true;
  float total = 0.f;
#pragma unroll
  for (int v = 0; v < WAVES; ++v) total += sh.part_ss[m][v];
  const float inv = inverse_root(fmaf(total, a.inv_H, a.eps1));
  const float lo = (r & 1 ? sum[1] : sum[0]) * inv + b_lo, hi = (r & 1 ? sum[3] : sum[2]) * inv + b_hi;
  const bf16 v = __float2bfloat16(r < 2 ? lo * cs - hi * sn : hi * cs + lo * sn);
  const int f = r < 2 ? j : j + half;   // this lane's feature within the head
  if (head < a.nh) {
    a.q_out[((size_t)m * a.nh + head) * d + f] = v;
    return true;
  }
  if (slot < 0) return true;
  const bool pow2 = (a.page_size & (a.page_size - 1)) == 0;   // no division then
  const long long page = pow2 ? slot >> (31 - __builtin_clz(a.page_size)) : slot / a.page_size;
  const int off = pow2 ? (int)(slot & (a.page_size - 1)) : (int)(slot % a.page_size);
  const size_t row = (size_t)page * a.nkv;
  if (head < a.nh + a.nkv) a.k_pages[((row + (head - a.nh)) * a.page_size + off) * d + f] = v;
  else if (a.v_transposed) a.v_pages[((row + (head - a.nh - a.nkv)) * d + f) * a.page_size + off] = v;
  else a.v_pages[((row + (head - a.nh - a.nkv)) * a.page_size + off) * d + f] = v;
  return true;
}

// Thread 0 of the one block that stays: the next item to try, or -1 when every item that was given up is done.
__device__ int next_given_up(const ChainArgs& a, Shared& sh, int own) {
  for (;;) {
    const unsigned n = __hip_atomic_load(a.given_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int at = -1;
    for (unsigned i = 1; i <= n; ++i) {
      const unsigned p = (sh.position + i) % n;
      if (!((sh.done[p / 32] >> (p % 32)) & 1)) { at = (int)p; break; }
    }
    if (at == 0) { sh.position = 0; return own; }
    if (at > 0) {
      unsigned item = 0;     // its owner counted itself and stores its item next: it is running
      while (item == 0) item = __hip_atomic_load(a.given_up + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sh.position = at;
      return (int)item - 1;
    }
    // all n are done: leave the list empty, unless somebody came meanwhile
    for (unsigned i = 1; i < n; ++i) __hip_atomic_store(a.given_up + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);
    unsigned expected = n;
    if (__hip_atomic_compare_exchange_strong(a.given_up, &expected, 0u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return -1;
  }
}

template <int G, int UD, int P>
__device__ __forceinline__ bool run_item(const ChainArgs& a, Shared& sh, int item, unsigned tag, unsigned limit) {
  int lane = threadIdx.x & (MS_WAVE - 1);
  int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);   // the same for the whole wave
  asm volatile("" : "+v"(lane), "+s"(wave));   // what a phase works out from them belongs into that phase, not ahead of all
  int b = item;
  if (b < a.n_o) { run_o<G>(a, sh, b, lane, wave, tag); return true; }
  if ((b -= a.n_o) < a.n_gate) return run_gate<G>(a, sh, b, lane, wave, tag, limit);
  if ((b -= a.n_gate) < a.n_down) return run_down<G, UD, P>(a, sh, b, lane, wave, tag, limit);
  return run_front<G>(a, sh, b - a.n_down, lane, wave, tag, limit);
}

template <int G, int UD>
__global__ void __launch_bounds__(WAVES * MS_WAVE, 4)
decode_chain_kernel(ChainArgs a) {
  __shared__ Shared sh;
  const unsigned tag = a.epoch[a.launch] * (unsigned)a.launches + (unsigned)a.launch + 1u;
  if (blockIdx.x == 0 && threadIdx.x == 0) a.epoch[a.launch == 0 ? a.launches - 1 : a.launch - 1] += 1;
  if (run_item<G, UD, 6>(a, sh, blockIdx.x, tag, a.limit)) return;

  // given up: end, or stay if nobody has yet
  if (threadIdx.x == 0) {
    const unsigned before = __hip_atomic_fetch_add(a.given_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before > 0) __hip_atomic_store(a.given_up + before, blockIdx.x + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (unsigned& d : sh.done) d = 0;
    sh.position = 0;
    sh.next = before > 0 ? -1 : (int)blockIdx.x;
  }
  __syncthreads();
  while (sh.next >= 0) {      // (three pairs at a time: the loop needs registers of its own)
    const bool ok = run_item<G, UD, 3>(a, sh, sh.next, tag, 64);
    __syncthreads();
    if (threadIdx.x == 0) {
      if (ok) sh.done[sh.position / 32] |= 1u << (sh.position % 32);
      sh.next = next_given_up(a, sh, (int)blockIdx.x);
    }
    __syncthreads();
  }
}

size_t round_up(size_t n) { return (n + 255) / 256 * 256; }
size_t stream_bytes(int M) { return round_up((size_t)WAVES * STEPS * 32 * M * 8); }
size_t act_bytes(int M) { return round_up((size_t)DOWN_WAVES * 4 * DOWN_LOADS * 16 * M * 8); }
constexpr size_t HEAD_BYTES = 4 * (1 + LIST), EPOCH_BYTES = 4 * MAX_LAUNCHES;

unsigned g_limit = 2048;   // looks of a waiting block, each about 0.8 us

int down_units(int M) { return M <= 2 ? 1 : 2; }
int blocks_of(int M, int H, int I, int nh, int nkv, int d, int* n) {
  n[0] = H / (4 * UO);
  n[1] = std::max((I / 2 + 4 * NT - 1) / (4 * NT), std::min(I / 2, 256));
  n[2] = H / (4 * down_units(M));
  n[3] = (nh + 2 * nkv) * (d / 2) / (2 * UF);
  return n[0] + n[1] + n[2] + n[3];
}

}  // namespace

// Tests: how many times a waiting block looks before it gives its item up; 0 restores the choice.
extern "C" void ms_decode_chain_limit(int limit) { g_limit = limit > 0 ? (unsigned)limit : 2048u; }

// Bytes of a workspace for ms_decode_chain, to be zeroed once and then left to launches of ONE batch size, one step after the
// other; 0 where the kernel does not take the sizes.
extern "C" int ms_decode_chain_workspace(int M, int H, int num_heads, int num_kv_heads, int head_dim, int I) {
  if (M < 1 || M > 8 || H <= 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || I <= 0) return 0;
  const long long Ko = (long long)num_heads * head_dim;
  if (H % 32 || Ko % 32 || I % 32 || head_dim % (4 * UF) || H > 32 * WAVES * STEPS || Ko > 32 * WAVES * STEPS ||
      I > 32 * DOWN_WAVES * 4 * DOWN_LOADS)
    return 0;
  int n[4];
  if (blocks_of(M, H, I, num_heads, num_kv_heads, head_dim, n) > LIST) return 0;
  return (int)(HEAD_BYTES + EPOCH_BYTES + 2 * stream_bytes(M) + act_bytes(M));
}

// attn bfloat16 [M, num_heads head_dim] (M <= 8), x float [M, H] (in place), weights bfloat16 with contiguous rows: w_o [H, num_heads
// head_dim], w_gate_up [2 I, H] interleaved, w_down [H, I]; w_qkv (or null: no front) [(nh + 2 nkv) d, H], q_out, pages and so on
// as in ms_qkv_rope_store.  `launch` of `launches` (2 to 1,024) chains of the step.
extern "C" int ms_decode_chain(const void* attn, long long ld_attn, const void* w_o, float* x, long long ldx, const float* norm2,
                               float eps2, const void* w_gate_up, const void* w_down, const float* norm1, float eps1,
                               const void* w_qkv, const float* b_qkv, const int* positions, const float* inv_freq,
                               const int* slot_mapping, void* q_out, void* k_pages, void* v_pages, int M, int H, int I,
                               int num_heads, int num_kv_heads, int head_dim, int page_size, int v_transposed, void* workspace,
                               int launch, int launches, hipStream_t stream) {
  if (M <= 0) return MS_OK;
  if (!ms_decode_chain_workspace(M, H, num_heads, num_kv_heads, head_dim, I)) return MS_UNSUPPORTED;
  if (launches < 2 || launches > MAX_LAUNCHES || launch < 0 || launch >= launches || !workspace || !attn || !w_o || !x || !norm2 ||
      !w_gate_up || !w_down || ld_attn < num_heads * head_dim || ldx < H)
    return MS_BAD_ARG;
  if (ld_attn % 8 || (((uintptr_t)attn | (uintptr_t)w_o | (uintptr_t)w_gate_up | (uintptr_t)w_down | (uintptr_t)norm2) % 16) ||
      ((uintptr_t)workspace % 256))
    return MS_UNSUPPORTED;
  if (w_qkv) {
    if (!norm1 || !positions || !inv_freq || !slot_mapping || !q_out || !k_pages || !v_pages || page_size <= 0) return MS_BAD_ARG;
    if (((uintptr_t)w_qkv | (uintptr_t)norm1) % 16) return MS_UNSUPPORTED;
  }
  ChainArgs a;
  a.attn = (const bf16*)attn;
  a.w_o = (const bf16*)w_o; a.w_gu = (const bf16*)w_gate_up; a.w_down = (const bf16*)w_down; a.w_front = (const bf16*)w_qkv;
  a.x = x;
  a.norm2 = norm2; a.norm1 = norm1; a.b_front = b_qkv; a.inv_freq = inv_freq;
  a.positions = positions; a.slots = slot_mapping;
  a.q_out = (bf16*)q_out; a.k_pages = (bf16*)k_pages; a.v_pages = (bf16*)v_pages;
  char* ws = (char*)workspace;
  a.given_up = (unsigned*)ws;
  a.epoch = (unsigned*)(ws + HEAD_BYTES);
  a.x1 = (u64*)(ws + HEAD_BYTES + EPOCH_BYTES);
  a.x2 = (u64*)((char*)a.x1 + stream_bytes(M));
  a.act = (u64*)((char*)a.x2 + stream_bytes(M));
  a.ld_attn = ld_attn; a.ldx = ldx;
  a.eps2 = eps2; a.eps1 = eps1;
  a.M = M; a.H = H; a.Ko = num_heads * head_dim; a.I = I;
  a.nh = num_heads; a.nkv = num_kv_heads; a.d = head_dim; a.page_size = page_size; a.v_transposed = v_transposed;
  int n[4];
  blocks_of(M, H, I, num_heads, num_kv_heads, head_dim, n);
  a.n_o = n[0]; a.n_gate = n[1]; a.n_down = n[2]; a.n_front = w_qkv ? n[3] : 0;
  a.gate_units = I / 2 / n[1]; a.gate_more = I / 2 % n[1];
  a.per_head = head_dim / (4 * UF);
  a.inv_H = 1.0f / (float)H;
  a.launch = launch; a.launches = launches;
  a.limit = g_limit;
  const int blocks = a.n_o + a.n_gate + a.n_down + a.n_front;
  const dim3 grid(blocks), block(WAVES * MS_WAVE);
  if (M <= 2) decode_chain_kernel<4, 1><<<grid, block, 0, stream>>>(a);
  else if (M <= 4) decode_chain_kernel<4, 2><<<grid, block, 0, stream>>>(a);
  else decode_chain_kernel<8, 2><<<grid, block, 0, stream>>>(a);
  return ms_launch_status();
}
