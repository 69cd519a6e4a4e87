// Paged causal attention of prompt portions on the matrix cores (v_mfma_f32_16x16x32_bf16), bfloat16 in, float softmax:
// the columns, score and value products and the lazily moving reference of csrc/attention_mfma.hip, with the keys and
// values staged in LDS.
//
// Why: a wave of the unstaged kernel draws 16 KB for 32 keys of 128 dims and does 0.2 us of products with them, and eight
// waves on a CU ask for more than the 45 bytes a clock that a CU gets from its L2 (320 to 400 TFLOP/s at 128 dims).  Here
// the four waves of a block own neighbouring tiles of 32 columns and walk the same keys, 64 at a time: those go from the
// pages straight to LDS (global_load_lds), a tile of keys ahead of their use, and every wave reads all of them there.  Two
// blocks share a CU (64 KB of LDS each), one barrier a tile.  What is left is the softmax on the vector pipe (16
// exponentials of 16 clocks per 32 x 32 scores) beside the products: 870 TFLOP/s at 4,096 tokens of 28 heads of 128 dims,
// 990 behind 4,096 more, where the unstaged kernel has 380 and 400.
//
// A unit is 32 keys.  Row r of the u-th score product of a unit is its key 8 (r / 4) + 4 u + r % 4, so that a lane (quarter
// kq) has the scores of the eight consecutive keys 8 kq .. + 7, which it needs as one 16-byte read of a value's row.
// Rounding: the probabilities meet the values as bfloat16, and those that are powers of two lose nothing by it.  The four
// waves that share a tile in the other kernel have a reference each, the largest score of their first 32 keys; a column here
// has one (two at 64 dims), and where that stayed with its first 64 keys the result lay 2 to 9 % farther from 64 bits (28
// heads of 128 dims, 16 x 130 tokens, scores of spread 2: 0.00180 of the norm for 0.00175; 14 of 64 dims: 0.00189 for
// 0.00176).  So over the wave's first 128 keys the reference goes with the maximum of every unit of 32, down too, and later
// it moves at a smaller distance than there: 0.00175 and 0.00176, and no farther than the other kernel from 64 to 8,192 keys
// at spreads of 1 to 5.  Price: 1 to 6 % of a long prompt's time (2,048 tokens of 28 heads of 128 dims 58.5 -> 61.2 us),
// while short ones gain as much from the exchange of maxima without LDS (16 x 100: 13.9 -> 13.3).
// LDS: keys in rows of D, their 16-byte pieces permuted so that the 16 rows of a product meet every bank once (piece p of
// key k at place p ^ f(k)); values as they lie in a page of 16, [dim][16 keys], the two halves of a row swapped for every
// other eight dims.
#include "attention_tiles.h"
#include "api.h"
#include <algorithm>
#include <cmath>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

constexpr int GROUP = 4;              // waves that walk the same keys
constexpr int KEYS = 64;              // keys a tile: one chunk of 16 for every wave to bring

constexpr int WIDE = GROUP * 2 * 16;  // columns a block of the wide kind
// kinds: two tiles of columns a wave; one; and twice the groups of waves (two tiles at 64 dims, one at 128)
enum { PROMPT_WIDE = 1, PROMPT_NARROW = 2, PROMPT_NARROW_GROUPS = 3 };

constexpr int FOLLOWED = 128;         // keys over which the reference goes with every unit's maximum ..
constexpr float FOLLOW_DOWN = 4.f;    // .. unless that is further below it: sums grow by 2^16 at most on the way down
// log2 units by which a maximum may run ahead of its reference afterwards (64 dims: two references a column)
template <int D> constexpr float SLACK = D == 64 ? 4.f : 3.f;

template <int D> __device__ __forceinline__ int permute(int key) {     // f of a key's number in its unit
  return D == 128 ? (key & 3) | ((key >> 1) & 12) : ((key >> 1) & 1) | ((key >> 2) & 6);
}

// The maximum over the four lanes, 16 apart, that share a column.
__device__ __forceinline__ float column_max(float x) {
  const unsigned u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned w = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// KG groups of waves own the same columns and take the tiles of keys in turn, each with its own place in LDS; at the end
// they merge what they have, each for its share of the dims.  NT tiles of 16 columns a wave: with one, a block's columns and its
// share of the softmax are half as many, a turn takes 0.6 of the time and twice as many blocks share the work out.
template <int D, int KG, int NT>
__global__ void __launch_bounds__(KG * GROUP * MS_WAVE, D == 64 ? 4 : 2)
attention_prompt_kernel(const bf16* __restrict__ q, size_t q_stride, const bf16* __restrict__ k_pages,
                        const bf16* __restrict__ vt_pages, const int* __restrict__ block_table, int table_stride,
                        const int* __restrict__ table_rows, const int* __restrict__ q_start,
                        const int* __restrict__ context_lens, bf16* __restrict__ out, size_t out_stride, int nh, int nkv,
                        int page_size, float scale_log2e, int window, int n_requests, int pair_order) {
  constexpr int COLS = GROUP * NT * 16;               // columns a block
  constexpr int CT = D / 16, PIECES = D / 8;
  constexpr int CHUNK = 16 * D;                       // values of a chunk of 16 keys, of keys as of values
  constexpr int STAGE = 2 * 4 * CHUNK;                // a tile: four chunks of keys, four of values
  constexpr int LOADS = CHUNK * 2 / 1024;             // wave loads of 1 KB a chunk
  extern __shared__ __align__(16) unsigned char lds_raw[];
  bf16* lds = reinterpret_cast<bf16*>(lds_raw);       // [KG][2 tiles][STAGE]
  static_assert(CT % KG == 0, "the groups share the dims out");
  const int lane = threadIdx.x & (MS_WAVE - 1);
  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x / (GROUP * MS_WAVE));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE) - kg * GROUP;   // in its group
  const int col16 = lane & 15, kq = lane >> 4;
  const int g = blockIdx.x, rep = nh / nkv;

  int r, rank, n_tiles;
  find_tile(q_start, n_requests, rep, COLS, blockIdx.y, lane, r, rank, n_tiles);
  if (r < 0) return;
  const int* table = block_table + (size_t)(table_rows ? table_rows[r] : r) * table_stride;
  const int q0 = q_start[r], qlen = q_start[r + 1] - q0, start_pos = context_lens[r] - qlen, ncols = qlen * rep;
  // Late tiles see the most keys: they go first, and where all blocks fit on the chip at once the later half goes first,
  // latest tile first, then the earlier half, earliest first, so that a long tile's companion on its CU is a short one.
  const int half = pair_order ? (n_tiles + 1) / 2 : n_tiles;
  const int tile = rank < half ? n_tiles - 1 - rank : rank - half;
  const int b0 = tile * COLS, c0 = b0 + wave * NT * 16;       // first column of the block, of the wave
  const int key_hi = start_pos + (min(ncols, b0 + COLS) - 1) / rep;
  const int key_lo = window > 0 ? max(0, start_pos + b0 / rep - window + 1) : 0;
  const int t_begin = key_lo / KEYS, t_end = key_hi / KEYS + 1;
  // the wave's own columns; without any it still brings its chunks
  const bool works = c0 < ncols;
  const int first_pos = start_pos + min(c0, ncols - 1) / rep, last_pos = start_pos + (min(ncols, c0 + NT * 16) - 1) / rep;
  const bool full = c0 + NT * 16 <= ncols;
  const int wave_lo = window > 0 ? max(0, first_pos - window + 1) : 0, follow_end = (wave_lo + FOLLOWED - 1) / KEYS + 1;

  // ---- bringing a tile: the wave's chunk of keys and of values
  const int k_lane = lane * 8;                                 // this lane's first value in a load's 1 KB
  int k_src[LOADS], v_src[LOADS];                              // what it asks for, from the chunk's first value in the page
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int at = j * 512 + k_lane, key = at / D, place = (at % D) / 8;
    k_src[j] = key * D + (place ^ permute<D>((wave & 1) * 16 + key)) * 8;
    const int dim = at / 16, vh = (at >> 3) & 1;
    v_src[j] = dim * page_size + (vh ^ ((dim >> 3) & 1)) * 8;
  }
  auto page_of = [&](int t) {        // the page of the wave's chunk of tile t; past the context: the null page
    const int key = t * KEYS + wave * 16;
    return key <= key_hi ? __builtin_amdgcn_readfirstlane(table[key / page_size]) : 0;
  };
  auto bring = [&](int t, int page, int stage) {
    const int off = (t * KEYS + wave * 16) % page_size;
    const size_t head = ((size_t)page * nkv + g) * page_size * D;
    const bf16* kp = k_pages + head + (size_t)off * D;
    const bf16* vp = vt_pages + head + off;
    bf16* to = lds + (kg * 2 + stage) * STAGE + wave * CHUNK;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) __builtin_amdgcn_global_load_lds((global_void*)(kp + k_src[j]), (lds_void*)(to + j * 512), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < LOADS; ++j) __builtin_amdgcn_global_load_lds((global_void*)(vp + v_src[j]), (lds_void*)(to + 4 * CHUNK + j * 512), 16, 0, 0);
  };
  if (t_begin + kg < t_end) bring(t_begin + kg, page_of(t_begin + kg), 0);
  int page_next = t_begin + kg + KG < t_end ? page_of(t_begin + kg + KG) : 0;

  // ---- this lane's columns
  int pos[NT];      // -1: an idle column (sees no key; its result is not written)
  bf16x8 qv[NT][D / 32];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int c = c0 + t * 16 + col16, cc = min(c, ncols - 1);
    pos[t] = c < ncols ? start_pos + cc / rep : -1;
    const bf16* qp = q + (size_t)(q0 + cc / rep) * q_stride + (size_t)(g * rep + cc % rep) * D + kq * 8;
#pragma unroll
    for (int s = 0; s < D / 32; ++s) qv[t][s] = *reinterpret_cast<const bf16x8*>(qp + s * 32);
  }
  // The sums of the exponentials: at 128 dims one more product, of P^T with ones (the matrix pipe has the time there), at 64
  // added up in float on the vector pipe, a lane's share at a time, as the other kernel's tile at either size has them.
  constexpr bool SUMS_BY_MATRIX = D == 128;
  float m[NT], lvec[NT] = {};
  f32x4 o[CT][NT] = {}, lsum[SUMS_BY_MATRIX ? NT : 1] = {};
#pragma unroll
  for (int t = 0; t < NT; ++t) m[t] = -INFINITY;
  bf16x8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.0f;

  // where a lane's fragments lie: key rows of the u-th product of a unit, value rows of 16 dims
  int k_row[2], k_perm[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int key = (col16 >> 2) * 8 + u * 4 + (col16 & 3);
    k_row[u] = (key >> 4) * CHUNK + (key & 15) * D;
    k_perm[u] = permute<D>(key);
  }
  const int v_row = 4 * CHUNK + (kq >> 1) * CHUNK + col16 * 16 + (((kq & 1) ^ (col16 >> 3)) * 8);

  // the queries have arrived (said here, where the compiler sees it: otherwise it waits for them, and with them for the
  // loads to LDS, before the first product of every turn)
  __builtin_amdgcn_s_waitcnt(0x0F70);
  const int turns = (t_end - t_begin + KG - 1) / KG;
  for (int turn = 0; turn < turns; ++turn) {
    const int t = t_begin + turn * KG + kg, stage = turn & 1;
    // This tile has landed (vmcnt), and the wave's reads of the one before it have ended (lgkmcnt: what uses them need not
    // stand before this), so that its place may be filled again.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t + KG < t_end) {
      bring(t + KG, page_next, stage ^ 1);
      page_next = t + 2 * KG < t_end ? page_of(t + 2 * KG) : 0;
    }
    if (!works || t >= t_end) continue;      // the same for the whole wave
    const float slack = t < follow_end ? -FOLLOW_DOWN : SLACK<D>;
#pragma unroll
    for (int unit = 0; unit < 2; ++unit) {
      const int base = t * KEYS + unit * 32;
      if (base > last_pos) break;
      const bf16* st = lds + (kg * 2 + stage) * STAGE + unit * 2 * CHUNK;

      // scores: s[u][t] holds keys base + kq*8 + u*4 + (0..3) of column t*16 + col16
      f32x4 s[2][NT];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int t2 = 0; t2 < NT; ++t2) s[u][t2] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(st + k_row[u] + (((ks * 4 + kq) ^ k_perm[u]) & (PIECES - 1)) * 8);
#pragma unroll
          for (int t2 = 0; t2 < NT; ++t2) s[u][t2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qv[t2][ks], s[u][t2], 0, 0, 0);
        }
      }

      const bool unmasked = full && base + 31 <= first_pos && (window <= 0 || base > last_pos - window);
      if (!unmasked) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int t2 = 0; t2 < NT; ++t2)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = base + kq * 8 + u * 4 + i;
              if (key > pos[t2] || (window > 0 && key <= pos[t2] - window)) s[u][t2][i] = -INFINITY;
            }
      }
      float bmax[NT];
      bool ahead = false;
#pragma unroll
      for (int t2 = 0; t2 < NT; ++t2) {
        float bm = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) bm = fmaxf(bm, s[u][t2][i]);
        bmax[t2] = bm;
        ahead |= bm * scale_log2e > m[t2] + slack;
      }
      if (__builtin_amdgcn_ballot_w64(ahead) != 0) {      // some column's reference moves: rare once the first keys are past
#pragma unroll
        for (int t2 = 0; t2 < NT; ++t2) {
          const float bm = column_max(bmax[t2]) * scale_log2e;
          const bool step = bm > m[t2] + slack;
          const float corr = step ? fast_exp2(m[t2] - bm) : 1.0f;      // m = -inf: 0
          if (step) m[t2] = bm;
          if (SUMS_BY_MATRIX) lsum[t2] *= corr; else lvec[t2] *= corr;
#pragma unroll
          for (int c = 0; c < CT; ++c) o[c][t2] *= corr;
        }
      }
      float ref[NT];
#pragma unroll
      for (int t2 = 0; t2 < NT; ++t2) ref[t2] = m[t2] == -INFINITY ? 0.f : m[t2];
      // values past the wave's last visible key may be anything a reused page still holds: they count as zeros
      const bool clean = base + 31 <= last_pos;
      bf16x8 p[NT];
#pragma unroll
      for (int t2 = 0; t2 < NT; ++t2) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float e = fast_exp2(fmaf(s[u][t2][i], scale_log2e, -ref[t2]));
            if (!SUMS_BY_MATRIX) lvec[t2] += e;
            p[t2][u * 4 + i] = (__bf16)e;
          }
        if (SUMS_BY_MATRIX) lsum[t2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, p[t2], lsum[t2], 0, 0, 0);
      }
#pragma unroll
      for (int c4 = 0; c4 < CT; c4 += 4) {
        bf16x8 v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = *reinterpret_cast<const bf16x8*>(st + v_row + (c4 + c) * 256);
        if (!clean) {
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (base + kq * 8 + i > last_pos) {
#pragma unroll
              for (int c = 0; c < 4; ++c) v[c][i] = (__bf16)0.0f;
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int t2 = 0; t2 < NT; ++t2) o[c4 + c][t2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[c], p[t2], o[c4 + c][t2], 0, 0, 0);
      }
    }
  }

  constexpr int OWN = CT / KG;
  float l[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (SUMS_BY_MATRIX) {
      l[t] = lsum[t][0];      // every row of the product of ones is the column's sum
    } else {                  // a column's sum is spread over the four lane groups
      l[t] = lvec[t] + __shfl_xor(lvec[t], 16, MS_WAVE);
      l[t] += __shfl_xor(l[t], 32, MS_WAVE);
    }
  }
  if constexpr (KG > 1) {
    __shared__ float sm_m[KG][COLS], sm_l[KG][COLS];
    f32x4* sm_o = reinterpret_cast<f32x4*>(lds);        // [group of the sums][wave][tile of dims][NT][64]
    static_assert((size_t)KG * GROUP * CT * NT * MS_WAVE * 16 <= (size_t)KG * 2 * STAGE * 2, "all sums fit");
    __syncthreads();                                    // nobody reads keys or values any more
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = (wave * NT + t) * 16 + col16;
      if (kq == 0) { sm_m[kg][c] = m[t]; sm_l[kg][c] = l[t]; }
#pragma unroll
      for (int d = 0; d < CT; ++d)
        if (d / OWN != kg) sm_o[(((kg * GROUP + wave) * CT + d) * NT + t) * MS_WAVE + lane] = o[d][t];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = (wave * NT + t) * 16 + col16;
      float big = m[t];
#pragma unroll
      for (int k = 1; k < KG; ++k) big = fmaxf(big, sm_m[(kg + k) % KG][c]);
      const float safe = big == -INFINITY ? 0.f : big, mine = fast_exp2(m[t] - safe);
      l[t] *= mine;
#pragma unroll
      for (int d = 0; d < CT; ++d)
        if (d / OWN == kg) o[d][t] *= mine;
#pragma unroll
      for (int k = 1; k < KG; ++k) {
        const int other = (kg + k) % KG;
        const float theirs = fast_exp2(sm_m[other][c] - safe);
        l[t] += sm_l[other][c] * theirs;
#pragma unroll
        for (int d = 0; d < CT; ++d)
          if (d / OWN == kg) o[d][t] += sm_o[(((other * GROUP + wave) * CT + d) * NT + t) * MS_WAVE + lane] * theirs;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (pos[t] < 0) continue;
    const int c = c0 + t * 16 + col16;
    const float inv = 1.0f / l[t];
    bf16* op = out + (size_t)(q0 + c / rep) * out_stride + (size_t)(g * rep + c % rep) * D + kq * 4;
#pragma unroll
    for (int d = 0; d < CT; ++d) {
      if (KG > 1 && d / OWN != kg) continue;
      bf16x4 w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = (__bf16)(o[d][t][i] * inv);
      *reinterpret_cast<bf16x4*>(op + d * 16) = w;
    }
  }
}

template <int D, int KG, int NT>
int launch(dim3 grid, dim3 block, const bf16* q, size_t q_stride, const bf16* k, const bf16* vt, const int* table, int table_stride,
           const int* table_rows, const int* q_start, const int* ctx, bf16* out, size_t out_stride, int nh, int nkv, int page_size,
           float scale_log2e, int window, int n_requests, int pair_order, hipStream_t stream) {
  constexpr size_t bytes = (size_t)KG * 2 * 2 * KEYS * D * sizeof(bf16);
  static bool raised = false;   // once per instantiation: allow more dynamic LDS than the default 64 KB
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_prompt_kernel<D, KG, NT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
      return MS_LAUNCH_FAILED;
    raised = true;
  }
  attention_prompt_kernel<D, KG, NT><<<grid, block, bytes, stream>>>(q, q_stride, k, vt, table, table_stride, table_rows, q_start, ctx, out, out_stride, nh, nkv, page_size, scale_log2e, window, n_requests, pair_order);
  return ms_launch_status();
}

}  // namespace

// Whether a step's attention is the faster way here than on ms_paged_attention_mfma (a launch's constants: a captured
// graph's are its capacities).  A block's time is a chain of tiles of 64 keys, 1.9 us each (two groups at 64 dims: half as
// many), where the other kernel spreads a tile's keys over four waves.  So this one pays once its blocks fill the chip and
// the step is long beside its longest chain: the last tile of a portion has twice the keys of the mean one where nothing lies
// before it, fewer than that behind cached keys, so what counts is the blocks a CU times (2 - portion / context), `fills`; with a
// window all tiles have about its keys.
// A single token behind a long context is one block with the whole chain: in a step of several requests the contexts may be
// no longer than twice the step.  Time of the other kernel over this one's, at 1,500 steps with 1 to 64 query heads a
// key/value head times 1 to 16 of those, 1 to 64 requests, contexts up to 14,000 keys (most gain; the ends of each range):
//   128 dims, from 7/8 of a block a CU on.  One request: 1.0 to 2.4 from fills 1.35 on (28 heads on 4: 2,048 tokens 91 us / 54)
//     or with at most 400 keys; 0.74 to 1.4 else (4 on 4, 7,777 tokens 183 / 237; 16 on 8, 1,880 tokens 52 / 65).  Several: 0.94
//     to 2.3 from 1.6 on or with at most 600 keys (400 where one portion has a third of the tokens); 0.70 to 1.5 else.
//   64 dims, where a tile draws half as much.  One request: 1.06 to 1.54 from 4,096 keys, 1.7 blocks a CU and fills 2.3 on (14 on
//     2, 4,096 tokens behind 4,096: 143 / 120); 0.94 to 1.3 below.  Several, no portion over a third of the tokens: 0.93 to 1.5
//     from 7/16 of a block a CU on with contexts of at most 288 keys or 9/8 of the portion, 0.8 to 1.4 with longer ones up to
//     1.5 blocks a CU (13 requests of up to 307 tokens behind up to 2,577 keys, 16 on 16: 58 / 72), 0.94 to 1.6 above.
extern "C" int ms_attention_prompt_pays(int n_requests, int n_tokens, int max_q_len, int max_context_len, int num_heads,
                                        int num_kv_heads, int head_dim, int page_size, int window) {
  if ((head_dim != 64 && head_dim != 128) || page_size % 16 || num_kv_heads <= 0) return 0;
  if (n_requests > 1 && (long long)max_context_len > 2LL * n_tokens) return 0;
  const long long blocks = (long long)n_tokens * (num_heads / num_kv_heads) / WIDE * num_kv_heads, cus = ms_compute_units();
  const bool uneven = n_requests == 1 || 3LL * max_q_len > n_tokens;
  long long chain = max_context_len, keys = 2LL * max_context_len - max_q_len;    // of the last tile, of a mean one twice
  if (window > 0) {
    chain = std::min<long long>(chain, (long long)window + WIDE / std::max(1, num_heads / num_kv_heads));
    keys = std::min(keys, 2 * std::min<long long>(window, chain));
  }
  const auto fills = [&](long long twentieths) { return blocks * keys * 20 >= twentieths * cus * chain; };
  if (head_dim == 128)
    return blocks * 8 >= cus * 7 && (chain <= (uneven ? 400 : 600) || fills(n_requests == 1 ? 27 : 32));
  if (n_requests == 1) return blocks * 10 >= cus * 17 && max_context_len >= 4096 && fills(46);
  const bool short_chains = chain <= 288 || 8LL * max_context_len <= 9LL * max_q_len;
  return !uneven && blocks * 16 >= cus * (short_chains ? 7 : 24);
}

// Which kernel a step's attention should take: 0 ms_paged_attention_mfma, else a kind of this one.  exact: the two maxima are the
// step's own; 0: bounds, as a captured step has them, which say nothing of the requests that will be in it.  Between the other
// kernel and the wide kind ms_attention_prompt_pays decides; the narrow kinds take what they were seen to win over that choice,
// in 16,000 random exact steps and 6,600 with a capture's bounds (64 and 128 dims; alone, 2 to 48 even or ragged portions, beside
// single tokens, behind up to 14,000 keys; a quarter with a window).  What decides is how far the wide kind's blocks fill the chip,
// `fill` a CU: up to one or two all run at once and a CU waits for the longest, which blocks of half the columns cut short, while
// beyond that they only start and stream the keys twice as often.  Time over that of the choice without:
//   64 dims, where the other kernel would run: the narrow kind always, 0.63 to 1.05, 0.79 in the middle (with a capture's bounds
//     0.63 to 0.98); one request that fills 1.5 with 2,048 keys a mean tile twice the groups, 0.82 to 0.98 (3,883 tokens behind
//     7,000, 14 heads on 2: 201 us, 204 narrow, 176).
//   64 dims, where the wide kind would: narrow up to a fill of one, 0.69 to 1.02, 0.93 in the middle; beyond 0.73 to 1.28 (8 portions
//     of 512 tokens, 14 on 2, fill 1.75: 19.1 us wide, 22.2 narrow).
//   128 dims, where the wide kind would: one portion with most of the tokens and few keys before it, whose tiles are short and
//     long, up to a fill of two, 0.62 to 1.02, 0.76 in the middle (2,059 tokens of 28 heads on 4 71.9 -> 55.3 us); beyond up to 1.26, and
//     even portions 0.64 to 1.25.
//   128 dims, where the other kernel would, whose waves share a long chain: narrow from a fill of 7/8 or of a 512th of the longest
//     tile's keys (even portions; 0.51 to 1.01, 0.78 in the middle, 1.11 in one of 1,155), 1.5 (one of several with most tokens; 0.57 to
//     0.88), one (one alone; 0.58 to 0.88) or 5/8 (alone behind its own length of keys and more, or with a window; 0.53 to 0.99), and
//     alone between 5/8 and one twice the groups (0.62 to 0.89).  Below up to 1.9.
//   128 dims, several requests with more keys than their longest portion explains, or with bounds: as without.  A single token may
//     hold them (40 heads on 8, 945 tokens beside 8 decoding ones with 3,535 keys: 57 us, 76 narrow; bounds 0.6 to 1.8).
// Steps of a few tokens a request stay with the other kernel (30 requests of 2 tokens 5.4 and 6.0 us).
extern "C" int ms_attention_prompt_kind(int n_requests, int n_tokens, int max_q_len, int max_context_len, int num_heads,
                                        int num_kv_heads, int head_dim, int page_size, int window, int exact) {
  if ((head_dim != 64 && head_dim != 128) || page_size % 16 || num_kv_heads <= 0 || num_heads % num_kv_heads) return 0;
  const int plain = ms_attention_prompt_pays(n_requests, n_tokens, max_q_len, max_context_len, num_heads, num_kv_heads, head_dim, page_size, window)
                        ? PROMPT_WIDE : 0;
  const double rep = num_heads / num_kv_heads;
  if (max_q_len <= 16 || (double)n_tokens * rep / (WIDE / 2) + n_requests > 65535) return plain;
  double chain = max_context_len, mean = max_context_len - max_q_len / 2.0;    // keys of the longest tile and of the mean one
  if (window > 0) {
    chain = std::min(chain, window + WIDE / std::max(1.0, rep));
    mean = std::min(mean, (double)window);
  }
  const bool alone = n_requests == 1, most = alone || 2LL * n_tokens <= (long long)n_requests * max_q_len;
  // wide blocks a CU: the portions are of one length, unless one holds most of the tokens
  const auto blocks = [&](double tokens) { return std::ceil(tokens * rep / WIDE); };
  const double fill = (alone ? blocks(n_tokens)
                       : most ? blocks(max_q_len) + (n_requests - 1) * blocks((double)std::max(n_tokens - max_q_len, 1) / (n_requests - 1))
                              : n_requests * blocks((double)n_tokens / n_requests)) * num_kv_heads / ms_compute_units();
  if (head_dim == 64) {
    if (plain) return exact && !alone && fill <= 1.0 ? PROMPT_NARROW : plain;
    return exact && alone && fill >= 1.5 && mean >= 2048 ? PROMPT_NARROW_GROUPS : PROMPT_NARROW;
  }
  if (!exact || (!alone && chain > 1.5 * max_q_len)) return plain;
  const bool from_start = chain >= max_context_len && mean <= 0.6 * chain;
  if (plain) return most && from_start && fill <= 2.0 ? PROMPT_NARROW : plain;
  if (alone) return fill < 0.625 ? plain : from_start && fill < 1.0 ? PROMPT_NARROW_GROUPS : PROMPT_NARROW;
  if (most) return from_start && fill >= 1.5 ? PROMPT_NARROW : plain;
  return fill >= 0.875 || chain <= 512 * fill ? PROMPT_NARROW : plain;
}

// The arguments of ms_paged_attention_mfma's general shape, for plain scores (no sink, cap, slopes, gate; values of the
// keys' size), on the kind that ms_attention_prompt_kind names.  MS_UNSUPPORTED for what it does not take.
extern "C" int ms_attention_prompt_as(int kind, const void* q, long long q_stride, const void* k_pages, const void* vt_pages,
                                   const int* block_table, int table_stride, const int* table_rows, const int* q_start,
                                   const int* context_lens, void* out, long long out_stride, int n_requests, int n_tokens,
                                   int max_q_len, int num_heads, int num_kv_heads, int head_dim, int page_size, float scale,
                                   int window, hipStream_t stream) {
  if (n_requests <= 0 || max_q_len <= 0 || n_tokens <= 0) return MS_OK;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || table_stride <= 0) return MS_BAD_ARG;
  if (!(scale > 0.f)) return MS_BAD_ARG;   // maxima are taken of the raw scores
  if (q_stride % 8 || out_stride % 4 || ((uintptr_t)q % 16) || ((uintptr_t)out % 8)) return MS_UNSUPPORTED;
  if (num_kv_heads > 65535 || page_size <= 0) return MS_UNSUPPORTED;
  if (head_dim != 64 && head_dim != 128) return MS_UNSUPPORTED;
  if (page_size % 16 || ((uintptr_t)k_pages | (uintptr_t)vt_pages) % 16) return MS_UNSUPPORTED;
  const int rep = num_heads / num_kv_heads;
  if (kind < PROMPT_WIDE || kind > PROMPT_NARROW_GROUPS) return MS_BAD_ARG;
  const int cols = kind == PROMPT_NARROW || (kind == PROMPT_NARROW_GROUPS && head_dim == 128) ? WIDE / 2 : WIDE;
  long long tiles = (long long)n_tokens * rep / cols + n_requests;
  tiles = std::min(tiles, (((long long)max_q_len * rep + cols - 1) / cols) * n_requests);
  if (tiles > 65535 || (long long)max_q_len * rep > 0x7fffffffLL) return MS_UNSUPPORTED;
  const int groups = (head_dim == 64 ? 2 : 1) * (kind == PROMPT_NARROW_GROUPS ? 2 : 1);
  // two blocks share a CU, but for the most groups, whose tiles take its LDS
  const int pair_order = tiles * num_kv_heads <= 2LL * ms_compute_units() && kind != PROMPT_NARROW_GROUPS ? 1 : 0;
  dim3 grid(num_kv_heads, (unsigned)tiles), block(groups * GROUP * MS_WAVE);
#define GO(D, KG, NT) return launch<D, KG, NT>(grid, block, (const bf16*)q, (size_t)q_stride, (const bf16*)k_pages, (const bf16*)vt_pages, block_table, table_stride, table_rows, q_start, context_lens, (bf16*)out, (size_t)out_stride, num_heads, num_kv_heads, page_size, scale * 1.4426950408889634f, window, n_requests, pair_order, stream)
  if (head_dim == 64) {
    if (kind == PROMPT_NARROW) GO(64, 2, 1);
    if (kind == PROMPT_NARROW_GROUPS) GO(64, 4, 2);
    GO(64, 2, 2);
  }
  if (kind == PROMPT_NARROW) GO(128, 1, 1);
  if (kind == PROMPT_NARROW_GROUPS) GO(128, 2, 1);
  GO(128, 1, 2);
#undef GO
}

// The wide kind by name (tests, measurements).
extern "C" int ms_attention_prompt(const void* q, long long q_stride, const void* k_pages, const void* vt_pages,
                                   const int* block_table, int table_stride, const int* table_rows, const int* q_start,
                                   const int* context_lens, void* out, long long out_stride, int n_requests, int n_tokens,
                                   int max_q_len, int num_heads, int num_kv_heads, int head_dim, int page_size, float scale,
                                   int window, hipStream_t stream) {
  return ms_attention_prompt_as(PROMPT_WIDE, q, q_stride, k_pages, vt_pages, block_table, table_stride, table_rows, q_start,
                                context_lens, out, out_stride, n_requests, n_tokens, max_q_len, num_heads, num_kv_heads, head_dim,
                                page_size, scale, window, stream);
}
