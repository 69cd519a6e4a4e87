// out[M,N] = A[M,K] . W[N,K]^T for many tokens (prompt portions), bfloat16 in, float accumulation on the
// matrix cores (v_mfma_f32_16x16x32_bf16), with the gated activation as an epilogue: the product of the
// interleaved gate/up weight never goes to memory, which saves the write of [M, 2I], its read and a kernel.
//
// A block of 4 or 8 waves owns a tile of BN features by BM tokens: as large as registers allow where there are enough of them (256 x 256: a byte
// loaded does 128 multiply-adds), narrower where CUs would be left without one.  Per step of 64 columns the tile's rows of W and A go from memory
// straight to LDS (global_load_lds, 16 bytes a lane: no registers, no LDS write instructions) into SW slots for W and SA for A, SW - 1 and SA steps
// before they are multiplied: with three slots and two the 256 x 256 tile's are all of the CU's 160 KB, tiles of 64 and 96 have up to five of each,
// since a step of theirs is over before its successor's rows have come.  LDS rows are 128 bytes
// with their eight 16-byte pieces permuted by the row number (piece c at place c ^ (row & 7)): fragment reads then run at
// the full LDS rate (measured 237 bytes a clock; rows 144 bytes apart give 116).
//
// What bounds it: with all CUs at work the matrix pipes are busy 60 % of the time at 1.8 GHz (8,192 cubed: 1.36
// PFLOP/s), where the library's kernel has them busy 86 % of the time and the chip then runs at 1.54 GHz (1.57): the power
// the chip may draw is close.  A step of the 256 x 256 tile takes 1.6 us then, 1.15 us with a third of the CUs at work, and
// its products 0.85 us at 2.4 GHz.  One barrier a step with everything drained at it, and reads from LDS that the compiler
// had moved next to their use, took 1.70 and 1.38 us (7B gate/up, 2,048 tokens 525 -> 480 us and 4,096 951 -> 864; 0.5B
// gate/up, 2,048 tokens 47.3 -> 43.0; 8,192 cubed 877 -> 811).
//
// W is the A operand of the MFMA and the tokens the B operand, so a lane ends up with 4 output features of one
// token per tile.  Which 16 features make up a tile is free: tile i of a wave takes, for q = 0..3, the four
// features q * 4 FT + i * 4 .. + 3 of the wave's FT * 16, so that the lane with quarter q holds 4 FT consecutive
// features of its token over its FT tiles and stores them as one run.
#include "common.h"
#include "api.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// beside the epilogues of common.h (without EPI_RESIDUAL): the q/k/v product's, the grouped product's, and EPI_SWIGLU with
// the tanh form of the gelu for the silu
enum { EPI_QKV = 2, EPI_GROUPED = 7, EPI_GEGLU = 4, EPI_SUMS = 8, EPI_LOGITS = 10 };
// float results as they are; EPI_LOGITS: of one tile of tokens, so W is read once and marked as not to be kept
constexpr bool tiled_sums(int epi) { return epi == EPI_SUMS || epi == EPI_LOGITS; }

// the gate's activation of a gated epilogue: g * sigmoid(g), or the tanh form of the gelu with the tanh as
// 1 - 2 / (2^(2 y log2 e) + 1) through the hardware's exp2 and reciprocal (the result is rounded to bfloat16)
template <int EPI> __device__ __forceinline__ float gate_act(float g) {
  if (EPI == EPI_GEGLU) {
    const float y = 0.7978845608028654f * (g + 0.044715f * g * g * g);
    const float t = 1.0f - 2.0f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(2.885390081777927f * y) + 1.0f);
    return 0.5f * g * (1.0f + t);
  }
  return fast_silu(g);
}

// What the grouped product needs beside the operands: the token tiles are tiles of rows that belong to one expert each
// (ms_moe_align's lists), W holds the experts' matrices one after the other, rows of A are gathered and rows of the
// result scattered by the rows' list.
struct GroupedRows {
  const int* rows;          // [m_tiles * BM]: item of every row, < 0: none
  const int* tile_expert;   // [m_tiles]: the tile's expert, < 0: nobody's tile
  size_t expert_stride;     // elements between two experts' matrices
  int in_div;               // > 0: row p of the product reads A[item / in_div]; 0: A[p]
  int out_scatter;          // the result of row p goes to out[item] (else out[p])
  int act;                  // 1: the exact gelu of the product; 2: the clamped gate over interleaved features
  float limit, alpha;       // of the clamped gate (EPI_CLAMPED too)
};

__device__ __forceinline__ float tiled_gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752440f)); }

// What the q/k/v epilogue needs beside the product: W's rows are [q heads | k heads | v heads] of FT * 16 features.
struct QkvEpilogue {
  const float* bias;        // [(nh + 2 nkv) d] or null
  const float2* table;      // [M, d / 2]: (cos, sin) of each token's rotation angles
  const int* slots;         // [M], < 0: the token's k and v are not stored
  bf16* k_pages;            // [pages, nkv, page_size, d]
  bf16* v_pages;            // the same, or [pages, nkv, d, page_size] with v_transposed
  int nh, nkv, page_size, v_transposed;
};

constexpr int BK = 64;                  // columns a step
constexpr int PITCH = BK;               // LDS rows of 128 bytes; piece c of row l lies at place c ^ (l & 7)

// LDS row l of the block's W rows (l < WF * FT * 16) holds this feature of the tile
template <int FT>
__device__ __forceinline__ int feature_of_row(int l) {
  const int wf = l / (FT * 16), rem = l - wf * (FT * 16);
  const int i = rem >> 4, rr = rem & 15;
  return wf * (FT * 16) + (rr >> 2) * (4 * FT) + i * 4 + (rr & 3);
}

// A lane's run of RUN consecutive results goes to memory in the widest pieces that RUN allows (16 bytes for a
// multiple of 8 bfloat16, else 8 or 4), when the row starts at such an address.
template <int RUN>
__device__ __forceinline__ void store_run(bf16* o, const float* v, int valid) {
  constexpr int PIECE = RUN % 8 == 0 ? 8 : (RUN % 4 == 0 ? 4 : (RUN % 2 == 0 ? 2 : 1));
  typedef __attribute__((ext_vector_type(PIECE))) __bf16 piece_t;
  if (PIECE > 1 && valid >= RUN && ((uintptr_t)o % (PIECE * 2)) == 0) {
#pragma unroll
    for (int g = 0; g < RUN; g += PIECE) {
      piece_t pk;
#pragma unroll
      for (int e = 0; e < PIECE; ++e) pk[e] = (__bf16)v[g + e];
      *reinterpret_cast<piece_t*>(o + g) = pk;
    }
  } else {
#pragma unroll
    for (int g = 0; g < RUN; ++g)
      if (g < valid) o[g] = from_float<bf16>(v[g]);
  }
}

__device__ __forceinline__ void store_run_f32(float* o, const float* v, int run, int valid) {
  if (valid >= run && run % 4 == 0 && ((uintptr_t)o % 16) == 0) {
    for (int g = 0; g < run; g += 4) *reinterpret_cast<f32x4*>(o + g) = f32x4{v[g], v[g + 1], v[g + 2], v[g + 3]};
  } else {
    for (int g = 0; g < run; ++g)
      if (g < valid) o[g] = v[g];
  }
}

// WF x WT waves along features and tokens, each with FT x TT tiles of 16 x 16.  K is a multiple of 64.
template <int WF, int WT, int FT, int TT, int SW, int SA, int EPI, typename TO>
__global__ void __launch_bounds__(WF * WT * MS_WAVE)
gemm_tiled_kernel(const bf16* __restrict__ A, size_t lda, const bf16* __restrict__ W, size_t ldw,
                  TO* __restrict__ out, size_t ldo, int M, int N, int K, int m_tiles, int n_tiles, int xm, int parts,
                  QkvEpilogue qkv, GroupedRows grp) {
  constexpr int NWAVES = WF * WT, THREADS = NWAVES * MS_WAVE;
  constexpr int BN = WF * FT * 16, BM = WT * TT * 16;
  static_assert(BN % 8 == 0 && BM % 8 == 0, "a load brings eight rows");
  // loads of 8 rows (1 KB) a wave makes per step at most, of W and of A
  constexpr int LOADS_W = (BN / 8 + NWAVES - 1) / NWAVES, LOADS_A = (BM / 8 + NWAVES - 1) / NWAVES;
  constexpr int SLOT_W = BN * PITCH, SLOT_A = BM * PITCH;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  bf16* lds = reinterpret_cast<bf16*>(lds_raw);          // SW slots of BN rows of W, SA of BM rows of A

  // Blocks with consecutive ids go to consecutive XCDs, each with an L2 of its own.  With xm = 1 the tiles, token tiles running
  // fastest (they share a tile of W at the same time), are dealt out over the XCDs in equal runs: a tile of W is read from memory
  // by one XCD, or by the two at a run's end, every XCD reads all of A, and no XCD has a round of its CUs more than others (by whole rows
  // of tiles, 51 over 8 XCDs, 255 tiles took two: 23.3 us, 15.0 so).  Else the 8 XCDs are laid over the tiles as xm x (8 / xm): an XCD takes every xm-th token tile and
  // every (8 / xm)-th tile of W, which leaves it 1 / xm of A to keep in its L2; the host launches 8 * ceil(m_tiles / xm) *
  // ceil(n_tiles / (8 / xm)) blocks.  One without a tile leaves.
  const int xcd = blockIdx.x & 7;
  const int local = (int)(blockIdx.x >> 3);
  int steps = K / BK;
  int nt = 0, mt = 0;
  if (EPI == EPI_SUMS || (EPI != EPI_GROUPED && xm == 1)) {
    // (partial sums: the runs of the columns one after the other, each with all tiles)
    const int to_a_part = m_tiles * n_tiles, all = to_a_part * parts, per = (all + 7) / 8, id = xcd * per + local;
    if (local >= per || id >= all) return;
    const int part = EPI == EPI_SUMS ? id / to_a_part : 0, tile = id - part * to_a_part;
    nt = tile / m_tiles;
    mt = tile - nt * m_tiles;
    if (EPI == EPI_SUMS) {
      const int from = (int)((long long)steps * part / parts), to = (int)((long long)steps * (part + 1) / parts);
      steps = to - from;
      A += (size_t)from * BK;
      W += (size_t)from * BK;
      out += (size_t)part * M * N;
    }
  } else {
    const int xn = 8 / xm, mi = (m_tiles + xm - 1) / xm;
    nt = (local / mi) * xn + xcd / xm;
    mt = (local % mi) * xm + xcd % xm;
  }
  if (nt >= n_tiles || mt >= m_tiles) return;
  const int n0 = nt * BN, m0 = mt * BM;
  if (EPI == EPI_GROUPED) {     // the token tile is a tile of one expert's rows: its matrix is the W of this block
    const int e = grp.tile_expert[mt];
    if (e < 0) return;
    W += (size_t)e * grp.expert_stride;
  }
  const int lane = threadIdx.x & (MS_WAVE - 1), wave = threadIdx.x / MS_WAVE;
  const int wf = wave % WF, wt = wave / WF;
  const int col = lane & 15, kq = lane >> 4;

  // Load p of a wave fills LDS rows (wave + p * NWAVES) * 8 .. + 7 of a slot: lane l's 16 bytes land at l * 16 of that
  // 1 KB, which is place l & 7 of row l >> 3, so the lane asks memory for the piece that belongs there.  Rows past the
  // end of W or A repeat the last row (their results are not stored).
  const bf16 *src_w[LOADS_W], *src_a[LOADS_A];
#pragma unroll
  for (int p = 0; p < LOADS_W; ++p) {
    const int l = min((wave + p * NWAVES) * 8 + (lane >> 3), BN - 1);   // (past the tile's rows: not loaded)
    src_w[p] = W + (size_t)min(n0 + feature_of_row<FT>(l), N - 1) * ldw + ((lane & 7) ^ (l & 7)) * 8;
  }
#pragma unroll
  for (int p = 0; p < LOADS_A; ++p) {
    const int l = min((wave + p * NWAVES) * 8 + (lane >> 3), BM - 1);
    int r = min(m0 + l, M - 1);
    if (EPI == EPI_GROUPED && grp.in_div > 0) r = max(grp.rows[r], 0) / grp.in_div;   // (a row without an item: any row)
    src_a[p] = A + (size_t)r * lda + ((lane & 7) ^ (l & 7)) * 8;
  }
  typedef __attribute__((address_space(3))) void lds_void;
  typedef const __attribute__((address_space(1))) void global_void;
  // the wave's p-th load of a step's rows of W, or of A, into the slot whose first value in LDS is `slot`
  auto load_w = [&](int p, int step, int slot) {
    if ((p + 1) * NWAVES * 8 <= BN || (wave + p * NWAVES) * 8 < BN)   // the last round may be for some waves only
      __builtin_amdgcn_global_load_lds((global_void*)(src_w[p] + step * BK),
                                       (lds_void*)(lds + slot + (wave + p * NWAVES) * 8 * PITCH), 16, 0, EPI == EPI_LOGITS ? 2 : 0);
  };
  auto load_a = [&](int p, int step, int slot) {
    if ((p + 1) * NWAVES * 8 <= BM || (wave + p * NWAVES) * 8 < BM)
      __builtin_amdgcn_global_load_lds((global_void*)(src_a[p] + step * BK),
                                       (lds_void*)(lds + SW * SLOT_W + slot + (wave + p * NWAVES) * 8 * PITCH), 16, 0, 0);
  };
  constexpr int FEWEST_W = BN / 8 / NWAVES, FEWEST_A = BM / 8 / NWAVES;   // loads every wave makes

  f32x4 acc[FT][TT];
#pragma unroll
  for (int i = 0; i < FT; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // a lane's fragment pieces: columns kq * 8 of the first 32 columns of a step at place kq ^ (row & 7), of the
  // second 32 at that place ^ 4 (rows of a tile start at a multiple of 16, so row & 7 is col & 7)
  static_assert(BK == 64, "a step is two products of 32 columns deep");
  const int place0 = (kq ^ (col & 7)) * 8, place1 = ((kq + 4) ^ (col & 7)) * 8;
  const bf16* w_frag = lds + (wf * FT * 16 + col) * PITCH;
  const bf16* a_frag = lds + SW * SLOT_W + (wt * TT * 16 + col) * PITCH;

  // A step is four blocks of products, two to each half of its columns; a block's fragments of W (a half's FT lie in a ring
  // of FT registers) and, before a half, its TT fragments of the tokens are read beside the first products of the block
  // before it, and waited for at its start only.  The barrier stands before the last block: by then every fragment of the
  // step is in registers, so the wave waits for its share of the next step's rows, the barrier makes all shares visible and
  // says that everybody is done with this step's slots, into which go the step after next of A, during the last block, and
  // the one after that of W, during the next step's first: W, which mostly comes from beyond the L2, has the longer way.
  // The loads are asked for one by one between the products (eight in a row hold up those behind them).  So no read from
  // LDS and no load from memory is waited for with the matrix pipe idle.  The order of the instructions is the written one (sched_barrier), and a step is one straight piece
  // of code: left to itself the compiler moved the reads for the next step behind the branch to it and waited for each on
  // the spot, and a step took twice the time of its products.
  constexpr int HALF = (FT + 1) / 2;      // tiles of W in the first block of a half; the second has the others
  bf16x8 wr[FT], a[2][TT];
  auto read_w = [&](int half, int i, int slot) {
    wr[i] = *reinterpret_cast<const bf16x8*>(w_frag + slot + i * 16 * PITCH + (half ? place1 : place0));
  };
  auto read_a = [&](int half, int j, int slot) {
    a[half][j] = *reinterpret_cast<const bf16x8*>(a_frag + slot + j * 16 * PITCH + (half ? place1 : place0));
  };
  // LEFT: steps that follow, as far as it matters (AHEAD or more: of those to come, W's step SW - 1 on and A's step SA on are asked for)
  constexpr int AHEAD = SA;
  static_assert(SA == SW || SA == SW - 1, "which loads are under way at a barrier is counted for these");
  auto step = [&](auto left_c, int s, int slot_w, int next_w, int free_w, int slot_a, int next_a) {
    constexpr int LEFT = decltype(left_c)::value;
    constexpr bool ASK_W = LEFT >= SW - 1, ASK_A = LEFT >= SA;
    // loads under way that are newer than the next step's: of W and A for the steps behind it, and of W alone for the one asked for first
    constexpr int BEHIND = LEFT >= SA ? SW - 3 + (SA == SW) : LEFT - 1, NEWER = BEHIND * (FEWEST_W + FEWEST_A) + (LEFT >= SA && SA < SW ? FEWEST_W : 0);
#pragma unroll
    for (int block = 0; block < 4; ++block) {
      const int half = block >> 1, i0 = block & 1 ? HALF : 0, i1 = block & 1 ? FT : HALF;
      if constexpr (LEFT > 0) {
        if (block == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NEWER) : "memory");
      }
      // what the next block needs: tiles r0 .. r1 - 1 of W and, when it begins a half, the tokens' fragments
      const int r0 = block & 1 ? 0 : HALF, r1 = block & 1 ? HALF : FT, of_a = block & 1 ? TT : 0;
      const int reads = block == 3 && LEFT == 0 ? 0 : r1 - r0 + of_a, spread = i1 - i0 > 2 ? 2 : 1;
#pragma unroll
      for (int i = i0; i < i1; ++i) {
#pragma unroll
        for (int r = 0; r < reads; ++r) {
          if (r * spread / reads != i - i0) continue;
          const int to = block == 1 ? 1 : block == 3 ? 0 : half;
          if (r < of_a) read_a(to, r, block == 3 ? next_a : slot_a);
          else read_w(to, r0 + r - of_a, block == 3 ? next_w : slot_w);
        }
#pragma unroll
        for (int j = 0; j < TT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[i], a[half][j], acc[i][j], 0, 0, 0);
        if (ASK_W && block == 0) {
#pragma unroll
          for (int p = 0; p < LOADS_W; ++p) if (p * (i1 - i0) / LOADS_W == i - i0) load_w(p, s + SW - 1, free_w);
        }
        if (ASK_A && block == 3) {
#pragma unroll
          for (int p = 0; p < LOADS_A; ++p) if (p * (i1 - i0) / LOADS_A == i - i0) load_a(p, s + SA, slot_a);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // The q/k/v epilogue's inputs (heads of 64): asked for before the first rows of W, so that they have long come when the sums are there.
  constexpr bool EARLY = EPI == EPI_QKV && FT == 4 && TT == 1;
  constexpr int EJ = EARLY ? TT : 1, ER = EARLY ? 4 * FT : 1;
  float2 turns[EJ][ER];
  float biases[ER];
  int slots[EJ];
  if constexpr (EARLY) {
    const int head = (n0 + wf * FT * 16) / (FT * 16);
    const bool live = head < qkv.nh + 2 * qkv.nkv, rotated = head < qkv.nh + qkv.nkv;
    if (live) {
#pragma unroll
      for (int g = 0; g < ER; ++g) biases[g] = qkv.bias ? qkv.bias[(size_t)head * FT * 16 + kq * ER + g] : 0.f;
#pragma unroll
      for (int j = 0; j < EJ; ++j) {
        const int mm = min(m0 + wt * TT * 16 + j * 16 + col, M - 1);
        slots[j] = head < qkv.nh ? -1 : qkv.slots[mm];
        if (rotated) {
          const float2* turn = qkv.table + (size_t)mm * (FT * 8) + (kq & 1) * ER;
#pragma unroll
          for (int g = 0; g < ER; ++g) turns[j][g] = turn[g];
        }
      }
    }
  }
#pragma unroll
  for (int first = 0; first < SA; ++first) {
    if (first < SW - 1 && first < steps) {
#pragma unroll
      for (int p = 0; p < LOADS_W; ++p) load_w(p, first, first * SLOT_W);
    }
    if (first < steps) {
#pragma unroll
      for (int p = 0; p < LOADS_A; ++p) load_a(p, first, first * SLOT_A);
    }
  }
  if (steps >= SA) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((SW - 2) * FEWEST_W + (SA - 1) * FEWEST_A) : "memory");
  else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int j = 0; j < TT; ++j) read_a(0, j, 0);
#pragma unroll
  for (int i = 0; i < HALF; ++i) read_w(0, i, 0);
  int sw = 0, sa = 0;      // the current step's slots
  auto after_w = [&](int slot) { return slot == (SW - 1) * SLOT_W ? 0 : slot + SLOT_W; };
  auto after_a = [&](int slot) { return slot == (SA - 1) * SLOT_A ? 0 : slot + SLOT_A; };
  auto before_w = [&](int slot) { return slot == 0 ? (SW - 1) * SLOT_W : slot - SLOT_W; };
  int at = 0;
  for (; at + AHEAD < steps; ++at) {
    step(std::integral_constant<int, AHEAD>{}, at, sw, after_w(sw), before_w(sw), sa, after_a(sa));
    sw = after_w(sw);
    sa = after_a(sa);
  }
  auto last_steps = [&](auto self, auto left_c) -> void {
    constexpr int LEFT = decltype(left_c)::value;
    // Fewer steps than slots: the pipeline never fills.  (The last step there always is.  Said so to the compiler, the loop of small tiles is 64 to 68
    // instructions; not, it has two copies of their sums and moves all of them over in every step, 99.  Large tiles it makes wait for registers when told.)
    if ((LEFT == 0 && FT * TT <= 4) || steps - at > LEFT) {
      step(left_c, at, sw, after_w(sw), before_w(sw), sa, after_a(sa));
      sw = after_w(sw);
      sa = after_a(sa);
      ++at;
    }
    if constexpr (LEFT > 0) self(self, std::integral_constant<int, LEFT - 1>{});
  };
  last_steps(last_steps, std::integral_constant<int, AHEAD - 1>{});

  // the lane's run of 4 FT features of token m (tile j): acc[i][j][r] is feature f0 + i * 4 + r
  const int f0 = n0 + wf * (FT * 16) + kq * (4 * FT);
  if (EPI == EPI_QKV) {
    // A wave's FT * 16 features are one head, and a lane holds a quarter of it: quarters 0 and 1 are the first
    // half of the head, 2 and 3 the second, so the value that a rotation pairs with lies at the same place in the
    // lane 32 further.  q heads go to out [M, nh d] rotated, k heads rotated and v heads as they are into the pages.
    constexpr int D = FT * 16, RUN = 4 * FT;
    const int head = (n0 + wf * D) / D;
    if (head >= qkv.nh + 2 * qkv.nkv) return;
    const bool rotated = head < qkv.nh + qkv.nkv;
    const int e0 = kq * RUN;
    const bool is_v = !rotated;
    const int kvh = head - qkv.nh - (is_v ? qkv.nkv : 0);
    const float* bias = qkv.bias ? qkv.bias + (size_t)head * D + e0 : nullptr;
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      const int m = m0 + wt * TT * 16 + j * 16 + col;
      const int mm = min(m, M - 1);       // lanes past the last token take part in the exchange and store nothing
      const float2* turn = qkv.table + (size_t)mm * (D / 2) + (kq & 1) * RUN;
      bf16* dst = nullptr;                // a run of the lane's values, or (values transposed) a column of the page
      size_t step = 1;
      if (m < M) {
        if (head < qkv.nh) {
          dst = reinterpret_cast<bf16*>(out) + (size_t)m * ldo + (size_t)head * D + e0;
        } else {
          const long long slot = EARLY ? slots[EARLY ? j : 0] : qkv.slots[m];
          if (slot >= 0) {
            const long long page = slot / qkv.page_size;
            const int off = (int)(slot - page * qkv.page_size);
            if (is_v && qkv.v_transposed) {
              dst = qkv.v_pages + (((size_t)page * qkv.nkv + kvh) * D + e0) * qkv.page_size + off;
              step = (size_t)qkv.page_size;
            } else {
              dst = (is_v ? qkv.v_pages : qkv.k_pages) + (((size_t)page * qkv.nkv + kvh) * qkv.page_size + off) * D + e0;
            }
          }
        }
      }
#pragma unroll
      for (int g0 = 0; g0 < RUN; g0 += 8) {     // eight values at a time: few registers live beside the sums
        bf16x8 pk;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int g = g0 + e;
          float v = acc[g >> 2][j][g & 3] + (EARLY ? biases[EARLY ? g : 0] : bias ? bias[g] : 0.f);
          if (rotated) {
            const float2 cs = EARLY ? turns[EARLY ? j : 0][EARLY ? g : 0] : turn[g];
            const float other = __shfl_xor(v, 32);
            v = kq < 2 ? v * cs.x - other * cs.y : v * cs.x + other * cs.y;
          }
          pk[e] = (__bf16)v;
        }
        if (!dst) continue;
        if (step == 1) {
          *reinterpret_cast<bf16x8*>(dst + g0) = pk;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) reinterpret_cast<__bf16*>(dst)[(size_t)(g0 + e) * step] = pk[e];
        }
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    const int m = m0 + wt * TT * 16 + j * 16 + col;
    if (m >= M) continue;
    if (ms_gated(EPI) || EPI == EPI_GEGLU) {   // features 2g, 2g + 1 are gate g and up g: 2 FT outputs from o0 on
      const int o0 = f0 / 2, n_out = N / 2;
      float v[2 * FT];
#pragma unroll
      for (int i = 0; i < FT; ++i) {
        if (EPI == EPI_CLAMPED) {
          v[2 * i] = fast_clamped_glu(acc[i][j][0], acc[i][j][1], grp.limit, grp.alpha);
          v[2 * i + 1] = fast_clamped_glu(acc[i][j][2], acc[i][j][3], grp.limit, grp.alpha);
        } else {
          v[2 * i] = gate_act<EPI>(acc[i][j][0]) * acc[i][j][1];
          v[2 * i + 1] = gate_act<EPI>(acc[i][j][2]) * acc[i][j][3];
        }
      }
      store_run<2 * FT>(reinterpret_cast<bf16*>(out) + (size_t)m * ldo + o0, v, n_out - o0);
    } else if (EPI == EPI_GROUPED) {
      const int item = grp.rows[m];
      if (item < 0) continue;
      const size_t row = grp.out_scatter ? (size_t)item : (size_t)m;
      if (sizeof(TO) == 2 && grp.act == 2) {      // gate and up of feature f0 / 2 + g
        float v[2 * FT];
#pragma unroll
        for (int g = 0; g < 2 * FT; ++g)
          v[g] = fast_clamped_glu(acc[g >> 1][j][2 * (g & 1)], acc[g >> 1][j][2 * (g & 1) + 1], grp.limit, grp.alpha);
        store_run<2 * FT>(reinterpret_cast<bf16*>(out) + row * ldo + f0 / 2, v, (N - f0) / 2);
        continue;
      }
      float v[4 * FT];
#pragma unroll
      for (int g = 0; g < 4 * FT; ++g) v[g] = grp.act ? tiled_gelu_erf(acc[g >> 2][j][g & 3]) : acc[g >> 2][j][g & 3];
      if (sizeof(TO) == 4) store_run_f32(reinterpret_cast<float*>(out) + row * ldo + f0, v, 4 * FT, N - f0);
      else store_run<4 * FT>(reinterpret_cast<bf16*>(out) + row * ldo + f0, v, N - f0);
    } else if (tiled_sums(EPI)) {
      float v[4 * FT];
#pragma unroll
      for (int g = 0; g < 4 * FT; ++g) v[g] = acc[g >> 2][j][g & 3];
      store_run_f32(reinterpret_cast<float*>(out) + (size_t)m * ldo + f0, v, 4 * FT, N - f0);
    } else {
      float v[4 * FT];
#pragma unroll
      for (int g = 0; g < 4 * FT; ++g) v[g] = ms_store_value<EPI>(acc[g >> 2][j][g & 3]);
      store_run<4 * FT>(reinterpret_cast<bf16*>(out) + (size_t)m * ldo + f0, v, N - f0);
    }
  }
}

int g_xcd_split = 0;   // measurements: 0 leaves the choice, 1, 2, 4, 8 force the number of XCD rows

// Over how many XCDs the token tiles are spread (see the kernel).  Measured at the gate/up shapes of 0.5B to 32B:
// no difference up to 4,096 tokens; at 8,192 tokens of the 0.5B and 1.5B shapes four rows of XCDs take 143 against
// 155 us and 406 against 425 (an XCD then keeps a quarter of A in its L2 instead of fetching all of it again and
// again), two rows lie between.
int choose_xcd_split(int M) {
  if (g_xcd_split) return g_xcd_split;
  return M >= 6144 ? 4 : (M >= 4096 ? 2 : 1);
}

template <int WF, int WT, int FT, int TT, int SW, int SA, int EPI, typename TO>
int launch(const bf16* A, size_t lda, const bf16* W, size_t ldw, TO* out, size_t ldo, int M, int N, int K,
           hipStream_t stream, const QkvEpilogue& qkv = QkvEpilogue{}, const GroupedRows& grp = GroupedRows{}, int parts = 1) {
  constexpr int BN = WF * FT * 16, BM = WT * TT * 16;
  constexpr size_t lds = (size_t)(SW * BN + SA * BM) * PITCH * sizeof(bf16);
  static bool raised = false;   // once per instantiation: allow more dynamic LDS than the default 64 KB
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tiled_kernel<WF, WT, FT, TT, SW, SA, EPI, TO>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return MS_LAUNCH_FAILED;
    raised = true;
  }
  const int n_tiles = (N + BN - 1) / BN, m_tiles = (M + BM - 1) / BM;
  const int xm = choose_xcd_split(M);
  const long long blocks = EPI == EPI_SUMS || xm == 1 ? ((long long)m_tiles * n_tiles * parts + 7) / 8 * 8
                                                      : 8LL * ((m_tiles + xm - 1) / xm) * ((n_tiles + 8 / xm - 1) / (8 / xm));
  if (blocks > 0x7fffffffLL) return MS_UNSUPPORTED;
  gemm_tiled_kernel<WF, WT, FT, TT, SW, SA, EPI, TO><<<dim3((unsigned)blocks), dim3(WF * WT * MS_WAVE), lds, stream>>>(
      A, lda, W, ldw, out, ldo, M, N, K, m_tiles, n_tiles, xm, parts, qkv, grp);
  return ms_launch_status();
}

// The grouped product: tiles of 256 features by 256 rows (TT = 4) or 128 rows (TT = 2), the rows' tiles those of
// ms_moe_align.  The XCDs are laid over the tiles of W alone (xm = 1), row tiles running fastest on an XCD:
// neighbouring row tiles mostly belong to one expert and then share its slab of W in that XCD's L2 at the same time.
// With the loads waited for by count 128 sizes (1 to 100 tiles, 512 to 5,632 features, 256 to 3,584 columns) take 0.72 to 0.94 of
// the time that everything drained at a barrier a step took: 16 experts of 5,632 x 2,048, 100 tiles of 256 rows 590.8 -> 526.7 us,
// 2,048 x 2,816, 32 tiles of 128 rows 72.5 -> 61.6.
constexpr int GROUPED_TT = 4;
template <typename TO, int TT>
int launch_grouped(const bf16* A, size_t lda, const bf16* W, TO* out, size_t ldo, int tiles, int N, int K,
                   const GroupedRows& grp, hipStream_t stream) {
  constexpr int WF = 2, WT = 4, FT = 8;
  constexpr int BN = WF * FT * 16, BM = WT * TT * 16;
  constexpr size_t lds = (size_t)(3 * BN + 2 * BM) * PITCH * sizeof(bf16);
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tiled_kernel<WF, WT, FT, TT, 3, 2, EPI_GROUPED, TO>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return MS_LAUNCH_FAILED;
    raised = true;
  }
  const int n_tiles = (N + BN - 1) / BN;
  const long long blocks = 8LL * tiles * ((n_tiles + 7) / 8);
  if (blocks > 0x7fffffffLL) return MS_UNSUPPORTED;
  gemm_tiled_kernel<WF, WT, FT, TT, 3, 2, EPI_GROUPED, TO><<<dim3((unsigned)blocks), dim3(WF * WT * MS_WAVE), lds, stream>>>(
      A, lda, W, (size_t)K, out, ldo, tiles * BM, N, K, tiles, n_tiles, 1, 1, QkvEpilogue{}, grp);
  return ms_launch_status();
}

// The tiles.  1 to 3 are as large as registers and LDS allow a block that has a CU to itself, two to a CU, four to a CU; 4 and 5 fill
// rounds that 1 would not.  6 to 12 are for products that would leave CUs without a block, or one block to a CU: there a step is as long as its
// loads take to come, so these have narrower tiles, that more CUs get one of, and as many slots as LDS holds.
enum { T256 = 1, T128 = 2, T64 = 3, T192X256 = 4, T160X256 = 5, T64_DEEP = 6, T160X128 = 7, T192X128 = 8, T128X256 = 9, T96X128 = 10, T64X128 = 11, T128_DEEP = 12 };

int g_tile = 0;   // measurements: 0 leaves the choice of tile, 1 to 12 force one

// What takes a tile: us of a launch, of a round of tiles over the CUs, of a step of 64 columns in every round, and of a step with
// all CUs at work beyond that.
struct TileKind { int tile, features, tokens, to_a_cu; double fixed, round, step, busy; };
constexpr TileKind KINDS[] = {{T256, 256, 256, 1, 0.06, 5.93, 0.98, 0.52},     {T128, 128, 128, 2, 2.02, 1.02, 0.46, 0.13},
                              {T64, 64, 64, 4, 3.20, 0.00, 0.23, 0.01},        {T192X256, 192, 256, 1, 0.28, 5.24, 0.75, 0.44},
                              {T160X256, 160, 256, 1, 0.58, 4.77, 0.73, 0.36}, {T64_DEEP, 64, 64, 2, 2.61, 0.25, 0.25, 0.00},
                              {T160X128, 160, 128, 1, 1.58, 2.63, 0.49, 0.20}, {T192X128, 192, 128, 1, 1.56, 2.65, 0.51, 0.25},
                              {T128X256, 128, 256, 1, 1.04, 3.31, 0.58, 0.31}, {T96X128, 96, 128, 1, 1.58, 2.21, 0.32, 0.16},
                              {T64X128, 64, 128, 1, 1.62, 1.64, 0.25, 0.13}};

struct TileChoice { int tile, features, tokens; double us; long long tiles, slots; };

// Of the tiles with two steps ahead alone, by what they were measured to take (a start and end of 3 us and a step by its tile, rounds over the CUs).
TileChoice choose_older(int M, int N, int K) {
  const long long cus = ms_compute_units();
  const double steps = (double)((K + BK - 1) / BK);
  const long long small = (long long)((N + 127) / 128) * ((M + 127) / 128);
  if (small < cus) return {T64, 64, 64, 0.0, (long long)((N + 63) / 64) * ((M + 63) / 64), 4 * cus};
  TileChoice best{T128, 128, 128, ((double)small / (double)(2 * cus) + 0.3) * 1.15 * steps, small, (small + 2 * cus - 1) / (2 * cus) * 2 * cus};
  const struct { int tile, features; double step_us; } wide[] = {{T256, 256, 1.60}, {T192X256, 192, 1.30}, {T160X256, 160, 1.30}};
  for (const auto& w : wide) {
    const long long tiles = (long long)((N + w.features - 1) / w.features) * ((M + 255) / 256), rounds = (tiles + cus - 1) / cus;
    const double us = (double)rounds * (3.0 + steps * w.step_us);
    if (us < best.us) best = {w.tile, w.features, 256, us, tiles, rounds * cus};
  }
  return best;
}

// The tile that takes the least time by a model of the measurements: 200 sizes (65 to 4,096 tokens, 1,152 to 37,888 features,
// 256 to 3,584 columns), every tile timed at each, every product by a W that lies in no cache.  Its times lie within 0.77 and 1.28 of the measured
// ones (tiles with a CU to themselves 0.81 to 1.14), and the tile it takes is 0.4 % behind the best one on average, 12 % at worst; with 1 to 5 alone
// the best is 9 % behind on average and up to 42 (0.5B gate/up, 9,728 x 896: 128 tokens 11.1 -> 9.3 us, 256 13.9 -> 10.9, 512 18.4 -> 13.6, 768 17.7 ->
// 16.3, from 1,024 on the same; 5,632 x 2,048 at 256 tokens 20.8 -> 15.8, 37,888 x 3,584 at 128 80 -> 56).  (The tiles of 64 x 64 have become a
// little faster since, 0.1 to 0.8 us a product; at 171 sizes down to 64 features it is 2.2 % behind the best one.)
TileChoice choose_tile(int M, int N, int K) {
  // What the model was measured at ends here.  Taken there all the same it was 0.71 to 1.13 times as fast as those below up to 192 columns and 0.62 to 1.2
  // beyond 4,096 tokens (146 sizes): 12,558 x 128 at 1,188 tokens 23.9 and 28.5 us, 980 x 128 at 10,455 15.4 and 22.4.
  if (K < 256 || M >= 6144) return choose_older(M, N, K);
  const long long cus = ms_compute_units();
  const double steps = (double)((K + BK - 1) / BK);
  const int xm = choose_xcd_split(M);
  TileChoice best{0, 0, 0, 1e30, 0, 0};
  for (const TileKind& k : KINDS) {
    const long long n_tiles = (N + k.features - 1) / k.features, m_tiles = (M + k.tokens - 1) / k.tokens;
    // (laid over the XCDs in whole rows, as many as the XCD with the most has, eight times: 512 x 768 at 4,926 tokens took 96 x 128, 15.2 us, and
    // takes 128 x 128, 9.5; 26 sizes from 4,096 tokens on 0.94 -> 1.10 times as fast as by choose_older)
    const long long tiles = xm == 1 ? n_tiles * m_tiles : 8 * ((n_tiles + 8 / xm - 1) / (8 / xm)) * ((m_tiles + xm - 1) / xm), rounds = (tiles + cus - 1) / cus;
    if (k.tile == T64 ? tiles <= 2 * cus : k.tile == T64_DEEP && tiles > 2 * cus) continue;      // (two of the deep ones share a CU)
    const double share = (double)tiles / (double)cus;
    const double us = k.fixed + (double)rounds * (k.round + steps * k.step) + steps * k.busy * (k.to_a_cu == 1 ? share : std::min(1.0, share));
    const long long places = cus * k.to_a_cu;
    if (us < best.us) best = {k.tile, k.features, k.tokens, us, tiles, (tiles + places - 1) / places * places};
  }
  return best;
}

// Tile and column parts of a product in partial sums: the least time, with the norm that adds them up, by a model of 4,200 measurements (150
// sizes, 896 to 5,120 features, 896 to 18,944 columns, 65 to 1,000 tokens, five tiles, one to eight parts): 0.8 % behind the best on average, 8 % at
// most (a model of the three older tiles, without the norm, 2.8 % and 30): a launch and the norm; rounds of blocks, a step of one and what its
// neighbours on the CU and the other CUs add to it; the sums and the result, written and read.  896 x 4,864 at 100 and 400 tokens 11.1 -> 10.7 and
// 18.0 -> 17.7 us, 3,584 x 18,944 at 150 65 -> 50, 1,536 x 8,960 at 128 20.0 -> 16.7.  Few rows of a large W are read faster by two blocks to a CU
// (5,120 x 13,824 at 65 tokens 40.5 us, 44.0 in the deep tiles).
struct SumsChoice { int tile, parts; double us; long long blocks; };

SumsChoice choose_sums(int M, int N, int K) {
  const long long cus = ms_compute_units();
  const int steps = K / BK;
  const struct { int tile, size, to_a_cu; double start, round, step, beside, over, busy, sums, result; } kinds[] = {
      {T256, 256, 1, 0.19, 5.74, 1.15, 0.00, 0.00, 0.24, 1.40, 0.33},     {T128, 128, 2, 7.16, 0.15, 0.48, 0.61, 0.20, 0.23, 1.13, 0.04},
      {T64, 64, 4, 5.44, 0.00, 0.30, 2.24, 0.00, 0.10, 1.78, 0.02},       {T64_DEEP, 64, 2, 5.87, 0.03, 0.28, 0.48, 0.54, 0.06, 1.39, 0.04},
      {T128_DEEP, 128, 1, 7.12, 0.37, 0.43, 0.00, 0.00, 0.09, 1.52, 0.02}};
  // More parts than W is read in save nothing (8,072 x 10,880 at 123 tokens 8 parts 62 us, 4 57), and sums in rows that do not begin on four values go out
  // and come back one by one (7,749 x 10,240 at 127 tokens 8 parts 140 us, 4 103; 103 such sizes 13 % behind the best parts without, 2.5 % so).
  const double reading = 2e-6 * N * K / 5.5, apart = N % 4 ? 5. : 1.;
  SumsChoice best{0, 1, 1e30, 0};
  for (const auto& k : kinds) {
    if (k.tile == T128_DEEP && M <= 128 && (long long)N * K >= 40000000) continue;
    const long long tiles = (long long)((N + k.size - 1) / k.size) * ((M + k.size - 1) / k.size), places = cus * k.to_a_cu;
    for (int p = 1; p <= 8 && (p == 1 || p * 2 <= steps); ++p) {
      const long long blocks = tiles * p, deep = (blocks + cus - 1) / cus;
      const double share = (double)blocks / (double)cus;
      const double rounds = k.to_a_cu == 1 ? (double)deep : blocks <= places ? 1. : share / k.to_a_cu + k.over;
      const double step = k.step * (1. + k.beside * (double)(std::min<long long>(deep, k.to_a_cu) - 1)) + k.busy * std::min(1., share);
      const double us = k.start + std::max(rounds * (k.round + (steps + p - 1) / p * step), reading) + (k.sums * p * apart + k.result) * M * N * 8 / 5e6;
      if (us < best.us) best = {k.tile, p, us, blocks};
    }
  }
  return best;
}

}  // namespace

extern "C" void ms_gemm_tiled_force(int tile) { g_tile = tile; }
extern "C" int ms_gemm_tiled_tile(int M, int N, int K) { return choose_tile(M, N, K).tile; }
extern "C" void ms_gemm_tiled_force_xcd_split(int xm) { g_xcd_split = xm; }

// What of the tiles' places the product fills: tiles in whole rounds over the CUs.
static double full(int M, int N, const TileChoice& c) { return (double)M * N / ((double)c.slots * c.features * c.tokens); }
// The same with the rounds counted for the XCD with the most tiles, where these are laid over the XCDs in whole rows.
static double full_in_rows(int M, int N, const TileChoice& c) {
  const int to_a_cu = c.tile == T128 ? 2 : c.tile == T64 ? 4 : 1, xm = choose_xcd_split(M), xn = 8 / xm, cus = ms_compute_units();
  const long long n_tiles = (N + c.features - 1) / c.features, m_tiles = (M + c.tokens - 1) / c.tokens;
  const long long most = ((n_tiles + xn - 1) / xn) * ((m_tiles + xm - 1) / xm), places = (long long)(cus + 7) / 8 * to_a_cu;
  return (double)M * N / ((double)((most + places - 1) / places) * places * 8 * c.features * c.tokens);
}

// Products whose result has to stay in 32 bits up to what reads it.  Where gate and up, or the addend of a norm, have been held in float by this
// kernel, the library's product in its place would round them to bfloat16 first, which nobody asked for: so the sizes below, which the tiles
// with two steps ahead (256, 192 or 160 features by 256 tokens, 128 x 128, 64 x 64) were given by their own measurements, stay here also where
// the library is expected to be faster now (and the squared relu's are these alone).  Of 1.4 million sizes (65 to 8,192 tokens) that is 11 % of the gated
// ones, most of them by more than 5,120 columns, and 0.02 % of the sums'; time of the library and the next kernel over this one's at 65 of them, W in
// no cache: 0.84 to 1.63, 1.05 on average, and 0.82 to 1.88, 1.05.
static bool rounds_full(int M, const TileChoice& older) { return older.tile != T64 && M <= 2048 && older.tiles * 10 >= older.slots * 9; }
static bool gate_in_float(int M, int N, int K) {
  const TileChoice c = choose_older(M, N, K);
  if (c.tile == T64) return false;
  if (rounds_full(M, c)) return true;
  const double f = full_in_rows(M, N, c);
  if (K <= 3584) return c.tile == T192X256 || c.tile == T160X256 || f >= 0.65 || (c.tile == T128 && f <= 0.4);
  return K <= 5120 && M > 512 && f >= 0.8;
}

// Parts of a product in partial sums, by the same older tiles; 0: a bfloat16 addend, as ever.
static SumsChoice choose_older_sums(int M, int N, int K) {
  const long long cus = ms_compute_units();
  const int steps = K / BK;
  const struct { int tile, size, to_a_cu; double start_us[4], step_us[4]; } kinds[] = {
      {T256, 256, 1, {12.}, {1.05}}, {T128, 128, 2, {9., 13.}, {0.55, 1.0}}, {T64, 64, 4, {7., 7., 7., 8.}, {0.30, 0.43, 0.63, 0.82}}};
  SumsChoice best{0, 1, 1e30, 0};
  for (const auto& k : kinds) {
    const long long tiles = (long long)((N + k.size - 1) / k.size) * ((M + k.size - 1) / k.size), places = cus * k.to_a_cu;
    for (int p = 1; p <= 8 && (p == 1 || p * 4 <= steps); ++p) {
      const long long blocks = tiles * p;
      const int at = (int)(blocks >= places ? k.to_a_cu : (blocks + cus - 1) / cus) - 1;
      double rounds = (double)((blocks + places - 1) / places);
      if (k.to_a_cu > 1 && rounds > 1) rounds = (double)blocks / (double)places + 0.3;
      const double step = k.step_us[at] + (k.to_a_cu == 1 ? 0.5 * (double)(blocks < cus ? blocks : cus) / (double)cus : 0.);
      const double us = rounds * (k.start_us[at] + (steps + p - 1) / p * step) + (double)p * M * N * 8 / 5e6;
      if (us < best.us) best = {k.tile, p, us, blocks};
    }
  }
  return best;
}
// (of sizes that ms_gemm_tiled_sums_parts considers)
static int sums_in_float(int M, int N, int K) {
  if (M > 512 && M <= 1024 && K <= 8192) return 0;
  const SumsChoice c = choose_older_sums(M, N, K);
  const int cus = ms_compute_units();
  if (M > 256 && M <= 512 && K > 4096 && K <= 8192 && c.parts == 1) return 0;
  if (M > 1024 && (c.tile != T256 || c.parts == 1 || c.blocks >= cus || c.blocks * 6 < cus * 5)) return 0;
  return c.parts;
}

// Whether the gated product of M tokens is faster here than as the library's product and an activation kernel.  Time of these over
// this kernel's, a different W every call, with silu (the gelu and the clamped gate, whose kernels cost more: 1.08 times that), at 190 sizes
// of up to 2,048 tokens (65 on, 5,632 to 55,296 rows, 1,600 to 5,120 columns) and with the larger tiles at 687 of up to 4,096:
//   up to 1,536 columns 1.02 to 2 (65 to 8,192 tokens);
//   up to 2,048 tokens by up to 2,560 columns and up to 192 tokens by up to 3,584 1.03 to 2.1 (128 to 11,008 rows, 65 to 2,048 tokens, 2,300
//     sizes); not: 2,304 columns and more that are a multiple of 256, by so few rows and tokens that the library splits them, products of up to 131,072 values,
//     from 2,816 columns on 262,144 of up to 2,048 rows (2,560 for 96 tokens): 0.75 to 1.06 (512 x 3,584 at 192 tokens 18.7 us and 14.0);
//   by up to 5,120 where the model expects 0.81 PFLOP/s and more, or by up to 4,096 with tiles that are 0.72 full, 0.94 to 1.44, 1.11 on average (37,888 x 3,584 at 512 tokens 1.17, 900 1.23);
//     not: tiles of 128 beyond 512 tokens at less than 0.92 PFLOP/s (0.84 to 1.0: what the library takes for 513 to 580 tokens is little more
//     than for 512); beyond 1,024 tokens by more than 4,096 columns less full than 0.8 (0.95 to 1.12);
//   in all 0.6 % behind the better way on average (250 sizes), 7 % by the tiles' fill alone;
//   beyond, with the tiles counted in whole rows over the XCDs (as they lay when these were measured): up to 3,584 columns tiles of 192 or 160
//     features, the others from 0.65 on, 0.92 to 1.60; 4,096 to 5,120 columns from 0.8 on 0.91 to 1.58;
//   8,192 columns 0.96 to 1.03, in this kernel only where gate and up have been held in float.
extern "C" int ms_gemm_tiled_pays(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % BK) return 0;
  if (K <= 1536 || gate_in_float(M, N, K)) return 1;
  if (K > 5120) return 0;
  if (M <= 2048 && (K <= 2560 || (K <= 3584 && M <= 192)))
    return !(K > 2048 && K % 256 == 0 &&
             (K <= 2560 ? (long long)M * N <= 1 << 17 : (long long)M * N <= 1 << 18 && N <= (M <= 96 ? 2560 : 2048)));
  const TileChoice c = choose_tile(M, N, K);
  if (M <= 2048) {
    const double rate = 2e-9 * M * N * K / c.us;       // PFLOP/s
    if (c.tile == T128 && M > 512 && rate < 0.92) return 0;
    if (K <= 4096) return rate >= 0.81 || full(M, N, c) >= 0.72;
    return M <= 1024 ? rate >= 0.81 : full(M, N, c) >= 0.8;
  }
  const double f = full_in_rows(M, N, c);
  if (K <= 3584) return c.tile == T192X256 || c.tile == T160X256 || f >= 0.65;
  return f >= 0.8;
}

// The same question for the squared relu, whose product is written whole and whose own kernel costs little: the sizes that the
// gated product takes beyond 2,048 tokens or with rounds not full are 0.69 to 1.4 here, a quarter of them below 0.97.  The narrower tiles
// move few of them: 11 sizes that their rounds would fill were 0.84 to 1.36, half of them below 0.97 (4,694 x 3,072 at 1,212 tokens 54 us and 46).
extern "C" int ms_gemm_tiled_relu2_pays(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % BK) return 0;
  return K <= 1536 || rounds_full(M, choose_older(M, N, K));
}

// A bfloat16 [M, lda], W bfloat16 [N, ldw] (rows of K, K a multiple of 64), out bfloat16.
// epilogue 0: out[M, N] = product;  epilogue 1: out[M, N / 2] = silu(gate) * up over interleaved rows of W;
// epilogue 4: the same with the tanh form of the gelu for the silu; epilogue 5: max(product, 0)^2; epilogue 6: as 1 with the
// clamped gate (limit, alpha).
extern "C" int ms_gemm_tiled(const void* A, long long lda, const void* W, long long ldw, void* out, long long ldo, int M,
                             int N, int K, int epilogue, float limit, float alpha, hipStream_t stream) {
  if (M <= 0 || N <= 0) return MS_OK;
  if (K <= 0 || K % BK || lda % 8 || ldw % 8 || lda < K || ldw < K) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W) % 16) return MS_UNSUPPORTED;
  const bool gated = ms_gated(epilogue) || epilogue == EPI_GEGLU;
  if (gated ? (N % 2 || ldo < N / 2) : ((epilogue != EPI_STORE && epilogue != EPI_RELU2) || ldo < N)) return MS_BAD_ARG;
  GroupedRows numbers{};
  numbers.limit = limit;
  numbers.alpha = alpha;
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  bf16* o = (bf16*)out;
  int tile = g_tile;
  if (tile == 0) tile = choose_tile(M, N, K).tile;
#define GO(WF, WT, FT, TT, SW, SA) return epilogue == EPI_SWIGLU ? launch<WF, WT, FT, TT, SW, SA, EPI_SWIGLU, bf16>(a, lda, w, ldw, o, ldo, M, N, K, stream) \
                                : epilogue == EPI_GEGLU ? launch<WF, WT, FT, TT, SW, SA, EPI_GEGLU, bf16>(a, lda, w, ldw, o, ldo, M, N, K, stream)  \
                                : epilogue == EPI_RELU2 ? launch<WF, WT, FT, TT, SW, SA, EPI_RELU2, bf16>(a, lda, w, ldw, o, ldo, M, N, K, stream)  \
                                : epilogue == EPI_CLAMPED ? launch<WF, WT, FT, TT, SW, SA, EPI_CLAMPED, bf16>(a, lda, w, ldw, o, ldo, M, N, K, stream, QkvEpilogue{}, numbers)  \
                                                        : launch<WF, WT, FT, TT, SW, SA, EPI_STORE, bf16>(a, lda, w, ldw, o, ldo, M, N, K, stream)
  switch (tile) {      // features x tokens, slots of W and of A
    case T256: GO(2, 4, 8, 4, 3, 2);
    case T64: GO(1, 4, 4, 1, 3, 2);
    case T192X256: GO(2, 4, 6, 4, 3, 2);
    case T160X256: GO(2, 4, 5, 4, 3, 2);
    case T64_DEEP: GO(1, 4, 4, 1, 5, 4);
    case T160X128: GO(2, 4, 5, 2, 4, 3);
    case T192X128: GO(2, 4, 6, 2, 4, 3);
    case T128X256: GO(2, 4, 4, 4, 4, 3);
    case T96X128: GO(2, 4, 3, 2, 5, 5);
    case T64X128: GO(1, 8, 4, 1, 5, 5);
    default: GO(2, 4, 4, 2, 3, 2);
  }
#undef GO
}

// Column parts for a product whose reader adds partial sums up itself (the norm that follows a down projection), 0 where the
// library's product, or this kernel's whole one, is the faster way.  Few features leave a product of whole columns fewer
// tiles than CUs: 2,048 tokens by 3,584 x 18,944 are 112 tiles of 256 for 256 CUs; in two parts 235 us + 30 for the norm that adds
// them up, the library 363 + 17.  Time of the other way and its norm over this, 3,565 sizes (512 to 8,192 features, 768 to
// 28,672 columns, 65 to 4,096 tokens; every product by a W that lies in no cache: with W at hand the whole product of a narrow
// model looks better than it is in a model, 896 x 896 by 512 tokens 0.95 where it is 1.05), inside and outside the lines:
//   up to 128 tokens 1.05 to 4.1, 1.6 on average;
//   up to 256 tokens by 4,096 columns and more or up to 1,024 0.95 to 3.6, 1.5 on average;
//   up to 512 tokens by more than 8,192 columns 1.0 to 3.1; by more than 4,096 in several parts, up to 5,120 features, 0.90 to 1.8,
//     not two blocks of up to three parts a CU at less than 0.485 PFLOP/s, 1.13 on average; by up to 1,024 for up to 1,024 features 0.96 to 1.11.  Not: whole columns (4,480 x 6,784 at 429 tokens 0.82), more
//     features (0.81 to 1.2), 4,096 columns (0.93 to 1.12), 1,024 and fewer for more features (0.87 to 1.0);
//   up to 1,024 tokens by more than 8,192 columns, up to 5,120 features or by 16,384 columns and more, 0.92 to 3.2, 1.33 on average;
//     else 0.88 to 2.0, 1.08 on average (8,192 columns 0.89 to 1.17);
//   up to 1,000 tokens by 4,096 to 8,192 columns for up to 2,048 features, in three parts and more or, from 5,600 columns on, in two of
//     the tiles of 128, 0.94 to 1.35, 1.08 on average (300 sizes with the norm; 896 x 4,864 by 640 and 768 tokens 24.3 -> 20.6 and 24.9 ->
//     22.6 us).  Not: whole columns (0.81 to 0.83), two parts of fewer columns (0.95 to 1.06) or of tiles of 64 (0.95 to 1.02), rows that do not
//     begin on four values (1,710 x 7,936 at 711 tokens 0.93); 1,000 is where this was measured up to (1,001 to 1,100 tokens are 0.95 to 1.5, too);
//   in all 12 of 3,416 below 0.97;
//   beyond, by 16,384 columns and more where one round of blocks in parts fills 5/6 of the CUs, but not all: 0.96 to 2.0, 1.4 on
//     average (3,584 x 18,944 at 1,281 to 1,536 tokens and at 1,793 to 2,304).  With every CU taken 0.96 to 1.02 (4,096 x 28,672 at 2,048
//     tokens); elsewhere 0.74 to 1.47 (3,584 x 18,944 1.08 at 1,600 tokens, 1.4 at 1,200 and 2,560, 0.80 at 2,816): what the library
//     takes there changes by a factor of two from one number of tokens to the next.
extern "C" int ms_gemm_tiled_sums_parts(int M, int N, int K) {
  if (M <= 64 || N <= 0 || K < 768 || K % BK || N > 8192) return 0;
  if (M > 128 && (M <= 256 ? K > 1024 && K < 4096
                  : M <= 512 ? K <= 8192 && (K <= 4096 || N > 5120) && (K > 1024 || N > 1024)
                  : M <= 1000 && N <= 2048 && K > 4096 ? false
                  : M <= 1024 ? K <= 8192 || (N > 5120 && K < 16384) : K < 16384)) return 0;   // (asked for twice a layer: before the choice)
  const SumsChoice c = choose_sums(M, N, K);
  const int cus = ms_compute_units();
  const bool slower =
      (M > 256 && M <= 512 && K > 4096 && K <= 8192 &&
       (c.parts == 1 || c.blocks > 2 * cus || (c.tile != T64_DEEP && c.blocks > cus && c.parts <= 3 && 2e-9 * M * N * K < 0.485 * c.us))) ||
      (M > 512 && M <= 1024 && K <= 8192 && (N % 4 || (c.parts < 3 && (c.parts == 1 || K < 5600 || c.tile == T64 || c.tile == T64_DEEP)))) ||
      (M > 1024 && (c.tile != T256 || c.parts == 1 || c.blocks >= cus || c.blocks * 6 < cus * 5));
  return slower ? sums_in_float(M, N, K) : c.parts;
}

// Partial sums of the plain product over `parts` runs of the columns: float [parts, M, N].
extern "C" int ms_gemm_tiled_sums(const void* A, long long lda, const void* W, long long ldw, float* partial, int M, int N, int K,
                                  int parts, hipStream_t stream) {
  if (M <= 0 || N <= 0) return MS_OK;
  if (K <= 0 || K % BK || lda % 8 || ldw % 8 || lda < K || ldw < K) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W | (uintptr_t)partial) % 16) return MS_UNSUPPORTED;
  if (parts < 1 || parts > K / BK) return MS_BAD_ARG;
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  int tile = g_tile;
  if (tile == 0) tile = choose_sums(M, N, K).tile;
#define GO(WF, WT, FT, TT, SW, SA) return launch<WF, WT, FT, TT, SW, SA, EPI_SUMS, float>(a, lda, w, ldw, partial, (size_t)N, M, N, K, stream, QkvEpilogue{}, GroupedRows{}, parts)
  switch (tile) {
    case T256: GO(2, 4, 8, 4, 3, 2);
    case T64: GO(1, 4, 4, 1, 3, 2);
    case T64_DEEP: GO(1, 4, 4, 1, 5, 4);
    case T128_DEEP: GO(2, 4, 4, 2, 5, 4);
    default: GO(2, 4, 4, 2, 3, 2);
  }
#undef GO
}

// out [M, N] float = A . W^T for 17 to 64 tokens by very many short rows (a narrow model's head), which ms_gemm_slab leaves alone: its slabs
// pay a start and an end each.  us of ms_gemm_panel | so: 151,936 x 896 at 17 tokens 65 | 51, 32 68 | 58, 64 81 | 68 (of W 5.3 to 4.0 TB/s; the
// results are 39 MB more); x 1,536 105 | 85, 110 | 95, 132 | 113.  MS_UNSUPPORTED for what it does not take.
extern "C" int ms_gemm_tiled_logits(const void* A, long long lda, const void* W, long long ldw, float* out, long long ldo, int M, int N, int K,
                                    hipStream_t stream) {
  if (M <= 0 || N <= 0) return MS_OK;
  if (M > 64 || K <= 0 || K % BK || lda % 8 || ldw % 8 || lda < K || ldw < K || ldo < N) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W) % 16) return MS_UNSUPPORTED;
  return launch<1, 4, 4, 1, 5, 4, EPI_LOGITS, float>((const bf16*)A, lda, (const bf16*)W, ldw, out, ldo, M, N, K, stream);
}

// The grouped product of routed experts on this kernel: for every tile t of tile_rows rows (ms_gemm_tiled_grouped_rows()
// or half of that) with an expert e and each of its rows p (item = rows[p] >= 0): out[out_scatter ? item : p] =
// act(W[e] . A[in_div ? item / in_div : p]); W [experts, N, K] bfloat16 with K a multiple of 64, out bfloat16 or float.
// MS_UNSUPPORTED for what it does not take.
extern "C" int ms_gemm_tiled_grouped_rows() { return 4 * GROUPED_TT * 16; }
extern "C" int ms_gemm_tiled_grouped(const void* A, long long lda, const void* W, const int* rows, const int* tile_expert,
                                     void* out, long long ldo, int tiles, int tile_rows, int N, int K, int in_div,
                                     int out_scatter, int act, float limit, float alpha, int out_dtype, hipStream_t stream) {
  if (tiles <= 0 || N <= 0) return MS_OK;
  if (act == 2 && (N % 2 || out_dtype != MS_BF16)) return MS_BAD_ARG;
  if (K <= 0 || K % BK || lda % 8 || lda < K || ldo < (act == 2 ? N / 2 : N) || in_div < 0) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W) % 16) return MS_UNSUPPORTED;
  const bool whole = tile_rows == ms_gemm_tiled_grouped_rows();
  if (!whole && tile_rows * 2 != ms_gemm_tiled_grouped_rows()) return MS_UNSUPPORTED;
  if (out_dtype != MS_BF16 && out_dtype != MS_F32) return MS_BAD_ARG;
  const GroupedRows grp{rows, tile_expert, (size_t)N * (size_t)K, in_div, out_scatter, act, limit, alpha};
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
#define GO(TO, TT) return launch_grouped<TO, TT>(a, (size_t)lda, w, (TO*)out, (size_t)ldo, tiles, N, K, grp, stream)
  if (out_dtype == MS_BF16) { if (whole) GO(bf16, GROUPED_TT); else GO(bf16, GROUPED_TT / 2); }
  if (whole) GO(float, GROUPED_TT); else GO(float, GROUPED_TT / 2);
#undef GO
}

// Whether a plain product of M tokens should run here rather than in the library.  On the GPU the library's
// kernels are as fast or faster; but a call into the library costs the host 19 us and a call here 5, and a
// portion of up to about a thousand tokens of a narrow model is over on the GPU before the host has enqueued
// its 200 launches.  Measured at the 0.5B shape with the q/k/v and o products here: a prompt of up to 512 tokens
// 3.3 -> 2.7 ms, of 1,024 tokens 3.3 -> 3.15, of 1,536 tokens 3.4 -> 3.5 (so not beyond 1,024); the down projection's
// long rows take this kernel three times as long as the library and stay there.
extern "C" int ms_gemm_tiled_plain_pays(int M, int N, int K) {
  return M > 0 && M <= 1024 && N > 0 && N <= 2048 && K > 0 && K <= 1024 && K % BK == 0;
}


// The q/k/v product of a prompt portion with what follows it as the epilogue: bias, rotation of the q and k heads
// (pairs (j, j + d/2) turned by the angle whose cosine and sine rope_table[token][j] holds: ms_rope_table makes
// them once a step for all layers) and the store of k and v into the cache pages, so the projection of k and v
// never goes to memory as a matrix and q is written once.
// A [M, lda] bfloat16, W [(nh + 2 nkv) d, ldw], q_out [M, nh d]; head_dim 64 or 128 (a wave's features are one
// head), rotation over the whole head.  Pays where the plain product here keeps up with the library's: narrow
// models (ms_gemm_tiled_qkv_pays).
extern "C" int ms_gemm_tiled_qkv_pays(int M, int N, int K, int head_dim) {
  return M > 0 && N > 0 && K > 0 && K % BK == 0 && K <= 1024 && N <= 2048 && (head_dim == 64 || head_dim == 128);
}

// A wave's features are a head.  As long as a tile of 64 tokens (then of 128) to every head is not more than a CU's worth, these with as many slots
// as LDS holds; then tiles that share a CU.  Heads of 64 (18 of them by 896, us of the tiles of 64 | the taken one): 512 tokens 10.3 | 8.9, 1,024
// 11.5 | 10.7, 1,536 12.6 | 10.9, 2,048 19.7 in a second round, 15.3 in tiles of 64.  Of many tiles of 64 a CU those of 128 x 128 have less to read:
// from 8 on by more than 960 columns and from 14 on by 768 and more 0.76 to 1.02 of the time (32 heads by 1,024 at 8,192 tokens 62 us, 79 in tiles of 64;
// 18 by 896 at 16,384 78 and 84); below 0.95 to 2.2 (8 heads to 32, 1,024 to 16,384 tokens, 128 to 1,024 columns), by 512 columns 1.06 to 2.1.
// Heads of 128 (12 by 1,024; 256 features by 128 tokens before; with 256 tokens the epilogue does not fit the registers): 100 to 1,024 tokens 32
// to 34 | 16, 2,048 35 | 24, 4,096 36.
extern "C" int ms_gemm_tiled_qkv_tile(int M, int K, int heads, int head_dim) {
  const long long cus = ms_compute_units(), of_64 = (long long)heads * ((M + 63) / 64);
  if (of_64 <= cus) return T64_DEEP;
  if ((long long)heads * ((M + 127) / 128) <= cus) return T64X128;
  return head_dim == 64 && (K <= 960 ? K < 768 || of_64 < 14 * cus : of_64 < 8 * cus) ? T64 : T128;
}

extern "C" int ms_gemm_tiled_qkv(const void* A, long long lda, const void* W, long long ldw, const float* bias,
                                 const float* rope_table, const int* slot_mapping, void* q_out,
                                 void* k_pages, void* v_pages, int M, int K, int nh, int nkv, int head_dim, int page_size,
                                 int v_transposed, hipStream_t stream) {
  if (M <= 0) return MS_OK;
  if (nh <= 0 || nkv <= 0 || page_size <= 0 || !rope_table || !slot_mapping || !q_out || !k_pages || !v_pages)
    return MS_BAD_ARG;
  if (head_dim != 64 && head_dim != 128) return MS_UNSUPPORTED;
  if (K <= 0 || K % BK || lda % 8 || ldw % 8 || lda < K || ldw < K) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W | (uintptr_t)q_out | (uintptr_t)k_pages | (uintptr_t)v_pages | (uintptr_t)rope_table) % 16) return MS_UNSUPPORTED;
  const int N = (nh + 2 * nkv) * head_dim;
  const QkvEpilogue e{bias, (const float2*)rope_table, slot_mapping, (bf16*)k_pages, (bf16*)v_pages, nh, nkv, page_size,
                      v_transposed};
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  bf16* o = (bf16*)q_out;
  const size_t ldo = (size_t)nh * head_dim;
#define GO(WF, WT, FT, TT, SW, SA) return launch<WF, WT, FT, TT, SW, SA, EPI_QKV, bf16>(a, lda, w, ldw, o, ldo, M, N, K, stream, e)
  int tile = g_tile;
  if (tile == 0) tile = ms_gemm_tiled_qkv_tile(M, K, nh + 2 * nkv, head_dim);
  if (head_dim == 128) {
    if (tile == T64_DEEP) GO(1, 4, 8, 1, 5, 4);
    if (tile == T64X128) GO(1, 8, 8, 1, 3, 3);
    GO(2, 4, 8, 2, 3, 2);
  }
  if (tile == T64_DEEP) GO(1, 4, 4, 1, 5, 4);
  if (tile == T64X128) GO(1, 8, 4, 1, 5, 5);
  if (tile == T64) GO(1, 4, 4, 1, 3, 2);
  GO(2, 4, 4, 2, 3, 2);
#undef GO
}
