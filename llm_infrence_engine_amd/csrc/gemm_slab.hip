// out[M,N] = A[M,K] . W[N,K]^T for 5 to 64 tokens (a decode step of a batch) and a W that has to be read from memory,
// bfloat16 in, float accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16).
//
// What bounds it: reading W once.  A block owns a slab of up to 160 rows of W (or a run of their columns, where the rows are
// few: then it leaves partial sums), and its waves share the slab's columns, 64 at a time: a slice.  A slice's columns of all
// tokens are needed by one wave alone, so nothing is shared and no barrier is passed before the sums are added up: every wave
// has a ring of its own in LDS, waits for its own loads by count, and goes through the slab's tiles of 16 rows with the slice's
// tokens in registers and the sums of all tiles in accumulators.  W goes memory -> LDS (global_load_lds, 16 bytes a lane), eight
// rows by 128 bytes a load: every line is asked for whole and once, marked as not to be kept.  The tokens' next slice comes the same way while this one is
// multiplied; a slab of 148 rows (37,888 over 256 CUs) asks L2 for 0.4 bytes of them per byte of W.
//
// An element's sum runs in an order that goes by the shape of W and the number of column parts.
//
// us before | with it, at 64 and at 24 tokens (before: gemm_panel, whose blocks hold all tokens in LDS, by columns in turn, and
// read W as operands, 16 rows by 64 bytes a load; for narrow W with the columns split and a kernel that adds up): 37,888 x 3,584
// 71 | 52, 59 | 48; 4,608 x 3,584 19.6 | 15.5, 17.4 | 11.7; 3,584 x 3,584 18.6 | 12.7, 14.8 | 10.0, and 11.4, 9.2 as four partial
// sums; 3,584 x 18,944 50 | 33.4, 44 | 27.4 as four; 152,064 x 3,584 268 | 225, 212 | 193; 55,296 x 5,120 124 | 112, 119 | 95;
// 9,728 x 896 11.6 | 8.9, 9.3 | 7.2; 896 x 4,864 11.6 | 6.4, 11.2 | 5.0 as four.  4.8 to 5.2 TB/s of W (64 tokens) and 5.6 to 6.0
// (24) for the largest three.
// The other split, all waves on one slice with a barrier a slice, took 50 us for 37,888 x 3,584, but 29 for 3,584 x 3,584 and
// 126 for 3,584 x 18,944 (0.45 us a step of 64 columns, whatever the slab): its fragments are read by several waves.  Asking for
// neighbouring slices by neighbouring waves, or starting blocks at different columns, changed nothing.
#include "common.h"
#include "api.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;   // a 16-byte piece: 8 bfloat16
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

constexpr int WAVES = 8;
constexpr int SLICE = 64;              // columns: 128 bytes, 8 pieces, of every row
constexpr int NOT_KEPT = 2;            // cache policy of a load: nt
constexpr int LDS_PIECES = 160 * 64;   // all of the CU's
constexpr int MAX_ROWS = 64;           // tokens
constexpr int MAX_TILES = 10;          // tiles of 16 rows of a slab
constexpr long long MAX_STRIDE = 1 << 22;   // values of a row: byte offsets within a slab fit 32 bits

template <typename T, int V> struct alignas(sizeof(T) * V) Row { T v[V]; };

// no more than so many of the wave's loads are under way
template <int LOADS> __device__ __forceinline__ void wait_for() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory"); }
// two times n of them, n up to RING; more: nothing to wait for
template <int RING> __device__ __forceinline__ void wait_for_items(int n) {
  if (n > RING) return;
  if (n == RING) wait_for<2 * RING>();
  else if constexpr (RING > 0) wait_for_items<RING - 1>(n);
}

enum { EPI_QKV = 2 };                  // the front of an attention layer: see QkvFront

// What the q/k/v product's epilogue needs: bias, rotation (half-split pairs, float angles) and the store of k and v into their
// pages, as ms_qkv_rope_store.  W's rows are [q heads | k heads | v heads] of d; the product takes them as pairs (j, j + d/2),
// so that a lane holds two whole rotary pairs of its token.
struct QkvFront {
  const int *positions, *slots;
  const float* inv_freq;
  bf16 *k_pages, *v_pages;
  int nh, nkv, d, page_size, v_transposed;
  unsigned d_inv;
};

// i / d for i below 2^16 by the host's ceil(2^32 / d), d > 1
__device__ __forceinline__ int div_by(int i, unsigned inverse, int d) { return d == 1 ? i : (int)__umulhi((unsigned)i, inverse); }

// TT: tiles of 16 tokens.  FT: tiles of 16 rows of W a slab has at most.
template <int TT, int FT, int EPI, typename TO>
__global__ void __launch_bounds__(WAVES * MS_WAVE)
gemm_slab_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W, int ldw, const float* __restrict__ bias,
                 TO* __restrict__ out, size_t ldo, int M, int N, int K, int q, int rem, int parts, int k_per, int whole_stores,
                 QkvFront front) {
  constexpr int XL = 2 * TT;                                 // loads of the tokens' slice, 1 KB (eight rows) each
  constexpr int OWN = LDS_PIECES / WAVES;                    // a wave's pieces of LDS: the tokens' slice, the ring of items
  constexpr int ITEM = 2;                                    // loads of an item, 16 rows of W by 64 columns
  constexpr int RING = (OWN - XL * 64) / (ITEM * 64);        // items in the ring: 6 to 8
  extern __shared__ u32x4 smem[];
  const int lane = threadIdx.x & (MS_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);
  const int col = lane & 15, kq = lane >> 4;
  // blocks with consecutive ids lie on consecutive XCDs: with 2, 4 or 8 parts an XCD sees the tokens' columns of its part alone
  const int part = blockIdx.x % parts, b = blockIdx.x / parts;
  const int n0 = 4 * (b * q + min(b, rem));
  const int R = min(N, n0 + 4 * (q + (b < rem ? 1 : 0))) - n0;       // this block's rows of W
  const int k0 = part * k_per, k1 = min(K, k0 + k_per);
  const int S = (k1 - k0 + SLICE - 1) / SLICE;
  const int lo = S * FT * wave / WAVES, end = S * FT * (wave + 1) / WAVES;   // this wave's items, a slice's tiles side by side
  u32x4* xst = smem + wave * OWN;
  u32x4* ring = xst + XL * 64;

  // Lane l of a load takes row l / 8 of its eight, piece (l % 8) ^ (l / 8) of its 128 bytes: the fragment reads, 16 rows by four
  // pieces, then run at the full LDS rate.  Rows past the last repeat it, columns past K its last piece.
  const char* wbase = reinterpret_cast<const char*>(EPI == EPI_QKV ? W : W + (size_t)n0 * ldw);   // 32 bits reach over the rows
  const char* abase = reinterpret_cast<const char*>(A);
  const int sub = lane >> 3, piece = ((lane & 7) ^ sub) * 8;
  // the row of W that is the product's row n (q/k/v: the two rows of a rotary pair side by side)
  auto row_of_w = [&](int n) {
    const int head = div_by(n, front.d_inv, front.d), f = n - head * front.d;
    return head * front.d + (f >> 1) + (f & 1) * (front.d / 2);
  };
  int a_tile = lo % FT, a_slice = lo / FT, a_slot = 0;               // the next item to ask for
  auto ask = [&]() {
    const int k = min(k0 + a_slice * SLICE + piece, K - 8);
    u32x4* to = ring + a_slot * (ITEM * 64);
#pragma unroll
    for (int p = 0; p < ITEM; ++p) {
      const int row = min(a_tile * 16 + p * 8 + sub, R - 1);
      const unsigned at = ((unsigned)(EPI == EPI_QKV ? row_of_w(n0 + row) : row) * (unsigned)ldw + (unsigned)k) * 2u;
      __builtin_amdgcn_global_load_lds((global_void*)(wbase + at), (lds_void*)(to + p * 64), 16, 0, NOT_KEPT);
    }
    a_slot = a_slot + 1 == RING ? 0 : a_slot + 1;
    if (++a_tile == FT) { a_tile = 0; ++a_slice; }
  };
  auto ask_tokens = [&](int slice) {
    const int k = min(k0 + slice * SLICE + piece, K - 8);
#pragma unroll
    for (int p = 0; p < XL; ++p) {
      const unsigned at = (unsigned)(min(p * 8 + sub, M - 1) * lda + k) * 2u;
      __builtin_amdgcn_global_load_lds((global_void*)(abase + at), (lds_void*)(xst + p * 64), 16, 0, 0);
    }
  };

  f32x4 acc[FT][TT];
#pragma unroll
  for (int f = 0; f < FT; ++f)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int frag[2] = {col * 8 + (kq ^ (col & 7)), col * 8 + ((4 + kq) ^ (col & 7))};   // row col's pieces kq and 4 + kq
  const u32x4 zero = {0u, 0u, 0u, 0u};

  if (lo < end) {
    const int first = lo / FT, last = (end - 1) / FT;
    ask_tokens(first);
#pragma unroll
    for (int s = 0; s < RING; ++s)
      if (lo + s < end) ask();
    int slot = 0, i = lo, since = RING;                      // since: items asked for since the tokens' slice was
    for (int slice = first; slice <= last; ++slice) {
      // Loads arrive in order: the slice is there when no more loads than the items asked for behind it are under way.  (With
      // more of them than the ring holds an item behind it has been waited for.)
      if (i + RING > end) wait_for<0>();
      else if (slice > first + 1 && FT <= RING) wait_for<FT * ITEM>();
      else wait_for_items<RING>(since);
      u32x4 xb[2][TT];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < TT; ++t) xb[s][t] = xst[t * 128 + frag[s]];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // read: it may be filled again
      ask_tokens(min(slice + 1, last));                                        // (the last one once more, for nothing: the count of loads stays)
      const bool ends = (slice + 1) * SLICE > k1 - k0;       // columns past the last: nothing
      const int gone = k1 - k0 - slice * SLICE - kq * 8;
      if (ends) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
          if (gone - s * 32 <= 0) {
#pragma unroll
            for (int t = 0; t < TT; ++t) xb[s][t] = zero;
          }
      }
      since = 0;
#pragma unroll
      for (int f = 0; f < FT; ++f) {
        const int at = slice * FT + f;
        if (at < lo || at >= end) continue;                  // the same for the whole wave
        // newer than the item: the rest of the ring, and the tokens' next slice if the item was asked for before it
        if (i + RING > end) wait_for<0>();
        else if (f < RING) wait_for<(RING - 1) * ITEM + XL>();
        else wait_for<(RING - 1) * ITEM>();
        u32x4 wa[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) wa[s] = ring[slot * (ITEM * 64) + frag[s]];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (i + RING < end) ask();
        if (ends) {
#pragma unroll
          for (int s = 0; s < 2; ++s)
            if (gone - s * 32 <= 0) wa[s] = zero;
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int t = 0; t < TT; ++t)
            acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wa[s]), __builtin_bit_cast(bf16x8, xb[s][t]), acc[f][t], 0, 0, 0);
        slot = slot + 1 == RING ? 0 : slot + 1;
        ++i;
        ++since;
      }
    }
    wait_for<0>();                                           // nothing comes in any more
  }

  // The waves' sums are added in wave order, as many tiles at a time as LDS holds; each wave adds up every eighth of them.
  constexpr int PER = OWN / 64 / TT < FT ? OWN / 64 / TT : FT;
  f32x4* red = reinterpret_cast<f32x4*>(smem);
  if (parts > 1) out += (size_t)part * M * N;                // partial sums (EPI_STORE, float)
#pragma unroll
  for (int f0 = 0; f0 < FT; f0 += PER) {
    __syncthreads();
#pragma unroll
    for (int f = f0; f < f0 + PER && f < FT; ++f)
#pragma unroll
      for (int t = 0; t < TT; ++t) red[(wave * PER * TT + (f - f0) * TT + t) * MS_WAVE + lane] = acc[f][t];
    __syncthreads();
    for (int id = wave; id < min(PER, FT - f0) * TT; id += WAVES) {
      const int f = f0 + id / TT, tok = (id % TT) * 16 + col, r0 = f * 16 + kq * 4, nb = n0 + r0;
      f32x4 v = red[id * MS_WAVE + lane];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) v += red[(w * PER * TT + id) * MS_WAVE + lane];
      if (tok >= M || r0 >= R) continue;
      const bool whole = whole_stores && r0 + 3 < R;         // four values at an address that fits them
      if constexpr (EPI == EPI_QKV) {
        const int slot = front.slots[tok];
        const float pos = (float)front.positions[tok];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          if (r0 + 2 * p >= R) continue;
          const int head = div_by(nb + 2 * p, front.d_inv, front.d), j = (nb + 2 * p - head * front.d) >> 1, half = front.d / 2;
          const int at = head * front.d + j;
          float lo = v[2 * p] + (bias ? bias[at] : 0.f), hi = v[2 * p + 1] + (bias ? bias[at + half] : 0.f);
          if (head < front.nh + front.nkv) {                 // q and k heads turn by position * inv_freq[j]
            float sn, cs;
            ms_sincos_rot(pos * front.inv_freq[j], &sn, &cs);
            const float x1 = lo, x2 = hi;
            lo = x1 * cs - x2 * sn;
            hi = x2 * cs + x1 * sn;
          }
          TO *to = out + (size_t)tok * ldo + at, *to_hi = to + half;
          if (head >= front.nh) {
            if (slot < 0) continue;
            const bool is_v = head >= front.nh + front.nkv;
            const int kvh = head - front.nh - (is_v ? front.nkv : 0), page = slot / front.page_size, off = slot - page * front.page_size;
            const size_t base = ((size_t)page * front.nkv + kvh) * front.page_size * front.d;
            if (is_v && front.v_transposed) {
              to = front.v_pages + base + (size_t)j * front.page_size + off;
              to_hi = to + (size_t)half * front.page_size;
            } else {
              to = (is_v ? front.v_pages : front.k_pages) + base + (size_t)off * front.d + j;
              to_hi = to + half;
            }
          }
          *to = from_float<TO>(lo);
          *to_hi = from_float<TO>(hi);
        }
      } else if constexpr (ms_gated(EPI)) {
        // rows nb, nb+1 are (gate, up) of feature nb/2; rows nb+2, nb+3 of feature nb/2 + 1
        TO* o = out + (size_t)tok * ldo + nb / 2;
        const float g0 = ms_gate_value<EPI>(v[0], v[1], bias), g1 = ms_gate_value<EPI>(v[2], v[3], bias);
        if (whole) {
          *reinterpret_cast<Row<TO, 2>*>(o) = Row<TO, 2>{{from_float<TO>(g0), from_float<TO>(g1)}};
        } else {
          o[0] = from_float<TO>(g0);                         // (N is even)
          if (r0 + 3 < R) o[1] = from_float<TO>(g1);
        }
      } else {
        TO* o = out + (size_t)tok * ldo + nb;
        Row<TO, 4> old, to;
        if (EPI == EPI_RESIDUAL && whole) old = *reinterpret_cast<const Row<TO, 4>*>(o);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (r0 + r >= R) continue;
          float u = v[r] + (bias ? bias[nb + r] : 0.f);
          if (EPI == EPI_RESIDUAL) u += to_float(whole ? old.v[r] : o[r]);
          to.v[r] = from_float<TO>(ms_store_value<EPI>(u));
          if (!whole) o[r] = to.v[r];
        }
        if (whole) *reinterpret_cast<Row<TO, 4>*>(o) = to;
      }
    }
  }
}

template <int TT, int FT, int EPI, typename TO>
int launch(const bf16* A, size_t lda, const bf16* W, size_t ldw, const float* bias, TO* out, size_t ldo, int M, int N, int K,
           int blocks, int q, int rem, int parts, int k_per, const QkvFront& front, hipStream_t stream) {
  constexpr int lds = LDS_PIECES * 16;
  static bool raised = false;   // once per instantiation: allow more dynamic LDS than the default 64 KB
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_slab_kernel<TT, FT, EPI, TO>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return MS_LAUNCH_FAILED;
    raised = true;
  }
  const int per = ms_gated(EPI) ? 2 : 4;                     // results a lane stores side by side
  const int whole_stores = ldo % per == 0 && (uintptr_t)out % (per * sizeof(TO)) == 0 && (parts == 1 || (size_t)M * N % per == 0);
  gemm_slab_kernel<TT, FT, EPI, TO><<<dim3(blocks * parts), dim3(WAVES * MS_WAVE), lds, stream>>>(
      A, (int)lda, W, (int)ldw, bias, out, ldo, M, N, K, q, rem, parts, k_per, whole_stores, front);
  return ms_launch_status();
}

int k_per_part(int K, int parts) { return ((K + parts - 1) / parts + SLICE - 1) / SLICE * SLICE; }

template <int EPI, typename TO>
int plan(const bf16* A, size_t lda, const bf16* W, size_t ldw, const float* bias, TO* out, size_t ldo, int M, int N, int K,
         int parts, hipStream_t stream, const QkvFront& front = QkvFront{}) {
  // rows of W in units of four, dealt out evenly over as many blocks as the chip has CUs for each of the column parts; a W of
  // more rows than slabs hold takes a whole number of rounds
  const int units = (N + 3) / 4, cus = ms_compute_units();
  int blocks = cus / parts;
  if (blocks < 1) return MS_UNSUPPORTED;
  if (units < blocks) blocks = units;
  const int most = MAX_TILES * 4;                            // units of the highest slab
  const int rounds = ((units + blocks - 1) / blocks + most - 1) / most;
  blocks *= rounds;
  const int q = units / blocks, rem = units % blocks, R = 4 * (q + (rem ? 1 : 0));
  const int ft = (R + 15) / 16, tt = (M + 15) / 16;
  const int k_per = parts > 1 ? k_per_part(K, parts) : K;
#define GO(TTV, FTV) if (tt <= TTV && ft == FTV) return launch<TTV, FTV, EPI, TO>(A, lda, W, ldw, bias, out, ldo, M, N, K, blocks, q, rem, parts, k_per, front, stream)
#define TILES(TTV) GO(TTV, 1); GO(TTV, 2); GO(TTV, 3); GO(TTV, 4); GO(TTV, 5); GO(TTV, 6); GO(TTV, 7); GO(TTV, 8); GO(TTV, 9); GO(TTV, 10)
  TILES(2);
  TILES(4);
#undef TILES
#undef GO
  return MS_UNSUPPORTED;
}

}  // namespace

// The column parts this kernel is to take for a product of M rows with W[N, K], 0 where another kernel is the faster one.
// With a reader that adds sums up from 9 rows on, and by rows of 8,192 columns and more from 5 (a layer's norms and four
// products, the norms folded in and W ringed or streamed | here: 896 wide 22.3 | 25.7 us at 8 rows, 26.3 | 25.6 at 9, 29.1 | 26.0 at 16;
// 2,048 wide 51.2 | 47.4 at 4, 59.2 | 48.8 at 16; 3,584 wide 97 | 95 at 8, 115 | 95 at 16; 5,120 wide 188 | 179 and 229 | 181); other
// products from 17 on, and from 9 on by a W of 8 million values (9,728 x 896 7.0 us at 16 rows, 7.6 with the norm folded in).
// The lines on W change at 5, 9 and 17 rows only: between these edges a row's bits do not hang on how many others there are, across
// them another kernel sums in another order, and a norm may be folded in or not.  The plain product from 4 million values of W on
// (896 x 4,864: 8.5 against 11.3 us at 17 tokens, 12.0 against 11.6 at 64; 1,152 x 896 3.9 | 4.0 and 5.0 | 5.5, 896 x 896 4.2 | 4.1
// and 5.4 | 4.2), but for short rows in several slabs to a CU, whose start and end each pays for
// (151,936 x 896: 64 to 85 against 65 to 83).  Four parts for a reader that adds sums up itself from 896 x 896 on (4.0 against
// 4.2, and no read of the residual stream), as long as a slab of four takes the rows; rows of 8,192 columns and more
// go in four parts even when a kernel has to add them up (3,584 x 18,944: 33.4 + 5 us against 55.8 whole).
extern "C" int ms_gemm_slab_parts(int M, int N, int K, int sums) {
  if (M <= (sums && K >= 8192 ? 4 : 8) || M > MAX_ROWS || N <= 0 || K <= 0 || K % 8 || K > MAX_STRIDE) return 0;
  const long long values = (long long)N * K;
  if (sums ? (values < 750000 || K < 768) : values < (M <= 16 ? 8000000 : 4000000)) return 0;
  const int cus = ms_compute_units();
  if (N > cus * MAX_TILES * 16 && K < 2048) return 0;
  if (N > cus * MAX_TILES * 4 || (!sums && K < 8192)) return 1;
  return (4 - 1) * k_per_part(K, 4) < K ? 4 : 1;
}

// As ms_gemm_panel without a norm.  parts > 1: the columns are split over that many blocks as well, and float partial sums
// [parts][M][N] go to `out` (epilogue 0, float, no bias, ldo = N).
extern "C" int ms_gemm_slab(const void* A, long long lda, const void* W, long long ldw, const float* bias, void* out,
                            long long ldo, int M, int N, int K, int epilogue, int out_dtype, int parts, hipStream_t stream) {
  if (M <= 0 || N <= 0) return MS_OK;
  if (M > MAX_ROWS) return MS_UNSUPPORTED;
  if (K <= 0 || K % 8 || ldw % 8 || lda < K || ldw < K || lda % 8) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W) % 16 || lda > MAX_STRIDE || ldw > MAX_STRIDE) return MS_UNSUPPORTED;
  if (parts < 1 || (parts > 1 && ((parts - 1) * k_per_part(K, parts) >= K || epilogue != EPI_STORE || out_dtype != MS_F32 || bias || ldo != N)))
    return MS_BAD_ARG;
  const bf16 *a = (const bf16*)A, *w = (const bf16*)W;
#define RUN(EPI, TO) return plan<EPI, TO>(a, lda, w, ldw, bias, (TO*)out, ldo, M, N, K, parts, stream)
  if (epilogue == EPI_STORE) {
    if (ldo < N) return MS_BAD_ARG;
    if (out_dtype == MS_BF16) RUN(EPI_STORE, bf16);
    if (out_dtype == MS_F32) RUN(EPI_STORE, float);
    return MS_BAD_ARG;
  }
  if (epilogue == EPI_SWIGLU) {
    if (N % 2 || ldo < N / 2 || out_dtype != MS_BF16 || bias) return MS_BAD_ARG;
    RUN(EPI_SWIGLU, bf16);
  }
  if (epilogue == EPI_CLAMPED) {
    if (N % 2 || ldo < N / 2 || out_dtype != MS_BF16 || !bias) return MS_BAD_ARG;
    RUN(EPI_CLAMPED, bf16);
  }
  if (epilogue == EPI_RELU2) {
    if (ldo < N || out_dtype != MS_BF16) return MS_BAD_ARG;
    RUN(EPI_RELU2, bf16);
  }
  if (epilogue == EPI_RESIDUAL) {
    if (ldo < N || out_dtype != MS_F32) return MS_BAD_ARG;
    RUN(EPI_RESIDUAL, float);
  }
#undef RUN
  return MS_BAD_ARG;
}

// The front of an attention layer: q, k, v = A . W^T + bias with q and k rotated and k and v stored into their pages, as
// ms_qkv_rope_store, whose arguments these are but for A, the normed rows in bfloat16.
extern "C" int ms_gemm_slab_qkv(const void* A, long long lda, const void* W, long long ldw, const float* bias,
                                const int* positions, const float* inv_freq, const int* slot_mapping, void* q_out,
                                void* k_pages, void* v_pages, int M, int K, int num_heads, int num_kv_heads, int head_dim,
                                int page_size, int v_transposed, hipStream_t stream) {
  if (M <= 0) return MS_OK;
  if (num_heads <= 0 || num_kv_heads <= 0 || page_size <= 0 || !positions || !inv_freq || !slot_mapping || !q_out || !k_pages || !v_pages)
    return MS_BAD_ARG;
  const long long N = (long long)(num_heads + 2 * num_kv_heads) * head_dim;
  if (M > MAX_ROWS || head_dim <= 1 || head_dim % 2 || N > 0xffff || N * ldw > 0x7fffffffLL) return MS_UNSUPPORTED;
  if (K <= 0 || K % 8 || ldw % 8 || lda < K || ldw < K || lda % 8 || lda > MAX_STRIDE || ldw > MAX_STRIDE) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W) % 16) return MS_UNSUPPORTED;
  const QkvFront front{positions, slot_mapping, inv_freq, (bf16*)k_pages, (bf16*)v_pages, num_heads, num_kv_heads, head_dim,
                       page_size, v_transposed, (unsigned)((0x100000000ull + head_dim - 1) / head_dim)};
  return plan<EPI_QKV, bf16>((const bf16*)A, lda, (const bf16*)W, ldw, bias, (bf16*)q_out, (size_t)num_heads * head_dim, M, (int)N, K,
                             1, stream, front);
}
