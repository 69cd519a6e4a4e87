// out[M,N] = A[M,K] . W[N,K]^T for one group of tokens (M <= 16, a decode step of a small batch) and a large W, bfloat16 in,
// float accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16).
//
// What bounds it: reading W once.  A plain read of 100 to 600 MB reaches 6.2 TB/s here, one marked as not to be kept 6.8, and
// reads shaped like MFMA operands, 16 rows by 64 bytes a load, 5.5 to 5.9 (5.0 when so marked: the other half of a 128-byte
// line is then fetched again).  So W goes memory -> LDS (global_load_lds, 16 bytes a lane, no registers) as four rows by 256
// bytes a load, each line whole and marked; 16 rows by 128 columns, four loads, are an item, and the operands are read from
// LDS.  Nothing of W is shared, so every wave has a ring of its own (8 to 15 KB, the next items in flight while one is
// multiplied) and waits for its own loads by count: no barrier but one before and two behind the whole product.
//
// The rows of W are dealt out in units of two over the CUs, one block each; a block's tiles of up to 16 rows are cut into
// items of 128 columns, and its waves take equal runs of the items, tile after tile.  A tile that several waves share is added up
// through LDS in wave order by the one that holds its first columns: the order of a sum goes by the shape of W alone.
//
// The activations: with the RMS norm folded in (see gemm_skinny.hip) they are made bfloat16 once and lie whole in LDS;
// without, an item brings its 128 columns of all tokens along, from L2 (long rows would not fit, and a narrow W uses
// each of them once or twice only).
//
// us before | with it (before: gemm_panel, whose operands go to registers 16 rows by 64 bytes a load; at one and at 8 tokens): 55,296 x 5,120
// 104 | 87, 107 | 93; 37,888 x 3,584 55 | 45, 57 | 49; 152,064 x 3,584 186 | 163, 192 | 179; 151,936 x 896 54 | 45, 64 | 50;
// 5,120 x 27,648 (two kernels before) 59 | 45, 61 | 50; 3,584 x 18,944 31 | 25, 32 | 26.  6.0 to 6.7 TB/s
// for the largest at one token, 5.4 to 6.1 at 8.
#include "common.h"
#include "api.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;   // a 16-byte piece: 8 bfloat16
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

constexpr int WAVES = 8;
constexpr int STRIP = 128;            // columns of an item: 256 bytes, 16 pieces, of each of its rows
constexpr int NOT_KEPT = 2;           // cache policy of a load: nt
constexpr int LDS_BUDGET = 156 * 1024;
// KB of a wave's ring: 8 beside the whole activations; more where the items carry theirs, which come from nearby
constexpr int ring_kb(int xl) { return xl ? 15 : 8; }

enum { EPI_QKV = 2 };                 // the front of an attention layer: see QkvFront

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

// L: loads of four rows of W an item takes, the height of a tile over four.  XL: loads of four tokens it takes (0: the
// activations lie in LDS).
template <int L, int XL, int EPI, typename TO, bool NORM>
__global__ void __launch_bounds__(WAVES * MS_WAVE)
gemm_ring_kernel(const void* __restrict__ Av, size_t lda, const bf16* __restrict__ W, size_t ldw,
                 const float* __restrict__ bias, TO* __restrict__ out, size_t ldo, int M, int N, int K,
                 const float* __restrict__ norm_w, float eps, const int* __restrict__ rows, int q, int rem,
                 unsigned strips_inv, unsigned parts_inv, QkvFront front) {
  constexpr int LOADS = L + XL, SLOT = LOADS * 64;             // of an item; pieces of its slot
  constexpr int RING = ring_kb(XL) / LOADS;                    // items in the ring
  constexpr int H = 4 * L;                                     // rows of a tile
  static_assert(NORM == (XL == 0), "the folded norm keeps the activations in LDS, the others bring them along");
  static_assert(RING >= 1, "an item fits the ring");
  extern __shared__ u32x4 smem[];
  const int lane = threadIdx.x & (MS_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MS_WAVE);   // the same for the whole wave
  const int col = lane & 15, kq = lane >> 4;
  const int b = blockIdx.x;
  const int n0 = 2 * (b * q + min(b, rem));
  const int n1 = min(N, n0 + 2 * (q + (b < rem ? 1 : 0)));     // this block's rows of W
  const int S = (K + STRIP - 1) / STRIP;
  const int T = (n1 - n0 + H - 1) / H;
  const int total = T * S;                                     // items, a tile's strips side by side
  const int i0 = total * wave / WAVES, n = total * (wave + 1) / WAVES - i0;   // this wave's
  const int first_tile = div_by(i0, strips_inv, S), first_strip = i0 - first_tile * S;
  const int last_tile = n ? div_by(i0 + n - 1, strips_inv, S) : 0;
  u32x4* ring = smem + wave * (RING * SLOT);
  u32x4* xst = smem + WAVES * RING * SLOT;                     // NORM: the activations [M][pitch]
  const int pitch = S * (STRIP / 8) + 2;                       // rows an odd number of 32 bytes apart
  const int parts = (K / 8 + 63) / 64;                         // loads of 512 columns per row
  float* ss_part = reinterpret_cast<float*>(xst + M * pitch);  // NORM: [M][parts]

  // the row of W that is the product's row n (q/k/v: the two rows of a rotary pair side by side)
  auto row_of_w = [&](int n) {
    if constexpr (EPI != EPI_QKV) return n;
    const int head = div_by(n, front.d_inv, front.d), f = n - head * front.d;
    return head * front.d + (f >> 1) + (f & 1) * (front.d / 2);
  };

  // What the epilogue of the wave's last tile needs from memory is asked for now; most have no other.
  f32x4 pre = {0.f, 0.f, 0.f, 0.f}, bv = {0.f, 0.f, 0.f, 0.f};
  auto epilogue_values = [&](int tile, f32x4& bias_v, f32x4& old_v) {
    const int nb = n0 + tile * H + kq * 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (kq * 4 >= H || nb + r >= n1 || col >= M) continue;
      if (bias && !ms_gated(EPI)) bias_v[r] = bias[row_of_w(nb + r)];
      if (EPI == EPI_RESIDUAL) old_v[r] = reinterpret_cast<const float*>(out)[(size_t)col * ldo + nb + r];
    }
  };
  if (n) epilogue_values(last_tile, bv, pre);
  const int pos = EPI == EPI_QKV ? front.positions[min(col, M - 1)] : 0;
  const int page_slot = EPI == EPI_QKV ? front.slots[min(col, M - 1)] : -1;

  // Lane l of load p takes row 4 p + l / 16 of the tile, piece (l % 16) ^ (that row) of its 256 bytes: the fragment reads, 16
  // rows by four pieces, then meet every bank once.  Rows past the block's last repeat it, columns past K its last piece.
  const int sub = lane >> 4, place = lane & 15;
  int a_tile = first_tile, a_strip = first_strip, a_slot = 0;  // the next item to ask for
  const bf16 *wsrc[L], *xsrc[XL ? XL : 1];
  auto rows_of = [&](int tile) {
#pragma unroll
    for (int p = 0; p < L; ++p) wsrc[p] = W + (size_t)row_of_w(min(n0 + tile * H + 4 * p + sub, n1 - 1)) * ldw;
  };
  auto ask = [&]() {
    u32x4* to = ring + a_slot * SLOT;
#pragma unroll
    for (int p = 0; p < LOADS; ++p) {
      const bool of_w = p < L;
      const int r = 4 * (of_w ? p : p - L) + sub;
      const int k = min(a_strip * STRIP + (place ^ r) * 8, K - 8);
      if (of_w) __builtin_amdgcn_global_load_lds((global_void*)(wsrc[of_w ? p : 0] + k), (lds_void*)(to + p * 64), 16, 0, NOT_KEPT);
      else __builtin_amdgcn_global_load_lds((global_void*)(xsrc[of_w ? 0 : p - L] + k), (lds_void*)(to + p * 64), 16, 0, 0);
    }
    a_slot = a_slot + 1 == RING ? 0 : a_slot + 1;
    if (++a_strip == S) {
      a_strip = 0;
      rows_of(++a_tile);
    }
  };
  auto fill = [&]() {
#pragma unroll
    for (int s = 0; s < RING; ++s) if (s < n) ask();
  };
  rows_of(a_tile);
  if constexpr (!NORM) {
#pragma unroll
    for (int p = 0; p < XL; ++p) {
      const int tok = min(4 * p + sub, M - 1);
      xsrc[p] = (const bf16*)Av + (size_t)(rows ? rows[tok] : tok) * lda;
    }
    fill();
  }

  const int xrow = min(col, M - 1);
  float scale = 1.f;
  if constexpr (NORM) {
    // (token, 512 columns) by waves; the ring is filled behind the first of these loads
    const float* X = (const float*)Av;
    constexpr int PB = 2;
    const int ids = M * parts;
    for (int base = wave; base < ids || base == wave; base += WAVES * PB) {
      f32x4 xf[PB][2], nw[PB][2];
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const int id = base + i * WAVES;
        if (id >= ids) break;   // the same for the whole wave
        const int tok = div_by(id, parts_inv, parts), c = min(((id - tok * parts) * 64 + lane) * 8, K - 8);
        const size_t at = (size_t)(rows ? rows[tok] : tok) * lda + c;
        xf[i][0] = *reinterpret_cast<const f32x4*>(X + at);
        xf[i][1] = *reinterpret_cast<const f32x4*>(X + at + 4);
        nw[i][0] = *reinterpret_cast<const f32x4*>(norm_w + c);
        nw[i][1] = *reinterpret_cast<const f32x4*>(norm_w + c + 4);
      }
      if (base == wave) fill();
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const int id = base + i * WAVES;
        if (id >= ids) break;
        const int tok = div_by(id, parts_inv, parts), c = (id - tok * parts) * 64 + lane;
        const bool in = c * 8 < K;
        bf16x8 h;
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x0 = in ? xf[i][0][e] : 0.f, x1 = in ? xf[i][1][e] : 0.f;
          ss = fmaf(x0, x0, ss);
          ss = fmaf(x1, x1, ss);
          h[e] = (__bf16)(x0 * nw[i][0][e]);
          h[4 + e] = (__bf16)(x1 * nw[i][1][e]);
        }
        ss = wave_sum(ss);
        if (lane == 0) ss_part[id] = ss;
        if (c < S * (STRIP / 8)) xst[tok * pitch + c] = in ? __builtin_bit_cast(u32x4, h) : u32x4{0u, 0u, 0u, 0u};
      }
    }
    asm volatile("s_waitcnt vmcnt(63) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (loads of W under way are their waves' own)
    float squares = 0.f;
    for (int p = 0; p < parts; ++p) squares += ss_part[xrow * parts + p];
    scale = 1.0f / sqrtf(squares / (float)K + eps);
  }

  // lane (col, kq) holds out[token col][n0 + tile * H + kq * 4 + (0..3)]
  auto finish = [&](int tile, f32x4 v, const f32x4& bias_v, const f32x4& old_v) {
    const int nb = n0 + tile * H + kq * 4;
    if constexpr (NORM) v *= scale;
    if (col >= M || kq * 4 >= H) return;
    if constexpr (EPI == EPI_QKV) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if (nb + 2 * p >= n1) continue;
        const int head = div_by(nb + 2 * p, front.d_inv, front.d), j = (nb + 2 * p - head * front.d) >> 1, half = front.d / 2;
        float lo = v[2 * p] + bias_v[2 * p], hi = v[2 * p + 1] + bias_v[2 * p + 1];
        if (head < front.nh + front.nkv) {   // q and k heads turn by position * inv_freq[j]
          float sn, cs;
          ms_sincos_rot((float)pos * front.inv_freq[j], &sn, &cs);
          const float x1 = lo, x2 = hi;
          lo = x1 * cs - x2 * sn;
          hi = x2 * cs + x1 * sn;
        }
        bf16 *to = out + (size_t)col * ldo + head * front.d + j, *to_hi = to + half;
        if (head >= front.nh) {
          if (page_slot < 0) continue;
          const bool is_v = head >= front.nh + front.nkv;
          const int kvh = head - front.nh - (is_v ? front.nkv : 0), page = page_slot / front.page_size, off = page_slot - page * front.page_size;
          const size_t base = ((size_t)page * front.nkv + kvh) * front.page_size * front.d;
          if (is_v && front.v_transposed) {
            to = front.v_pages + base + (size_t)j * front.page_size + off;
            to_hi = to + (size_t)half * front.page_size;
          } else {
            to = (is_v ? front.v_pages : front.k_pages) + base + (size_t)off * front.d + j;
            to_hi = to + half;
          }
        }
        *to = __float2bfloat16(lo);
        *to_hi = __float2bfloat16(hi);
      }
    } else if (ms_gated(EPI)) {
      // rows nb, nb+1 are (gate, up) of feature nb/2; rows nb+2, nb+3 of feature nb/2 + 1
#pragma unroll
      for (int p = 0; p < 2; ++p)
        if (nb + 2 * p + 1 < n1)
          out[(size_t)col * ldo + nb / 2 + p] = from_float<TO>(ms_gate_value<EPI>(v[2 * p], v[2 * p + 1], bias));
    } else {
      TO* o = out + (size_t)col * ldo + nb;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (nb + r < n1) o[r] = from_float<TO>(ms_store_value<EPI>(v[r] + bias_v[r] + old_v[r]));
    }
  };

  const int wrow = min(col, H - 1);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, carried = acc;   // carried: the share of a tile that another wave began
  int tile = first_tile, strip = first_strip, slot = 0;
  for (int i = 0; i < n; ++i) {
    if (i + RING <= n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 1) * LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const u32x4* at = ring + slot * SLOT;
    u32x4 wa[4], xb[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      wa[s] = at[wrow * 16 + ((s * 4 + kq) ^ wrow)];
      if constexpr (NORM) xb[s] = xst[xrow * pitch + strip * 16 + s * 4 + kq];
      else xb[s] = at[L * 64 + xrow * 16 + ((s * 4 + kq) ^ xrow)];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot is read: it may be filled again
    if (i + RING < n) ask();
    if ((strip + 1) * STRIP > K) {                        // past the last column lies nothing of these rows
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (strip * STRIP + s * 32 + kq * 8 >= K) wa[s] = xb[s] = zero;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wa[s]), __builtin_bit_cast(bf16x8, xb[s]), acc, 0, 0, 0);
    slot = slot + 1 == RING ? 0 : slot + 1;
    if (++strip == S) {
      if (tile == first_tile && first_strip) {
        carried = acc;
      } else if (tile == last_tile) {
        finish(tile, acc, bv, pre);
      } else {
        f32x4 bias_v = {0.f, 0.f, 0.f, 0.f}, old_v = bias_v;
        epilogue_values(tile, bias_v, old_v);
        finish(tile, acc, bias_v, old_v);
      }
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
      strip = 0;
      ++tile;
    }
  }

  // tiles that several waves share: the first of them adds the others' sums in wave order
  const bool later = tile == first_tile && first_strip;   // the wave's whole run lies inside a tile begun elsewhere
  if (later) carried = acc;
  __syncthreads();                                         // nobody reads a ring any more
  f32x4* red = reinterpret_cast<f32x4*>(smem);
  if (n && first_strip) red[wave * MS_WAVE + lane] = carried;
  __syncthreads();
  if (!n || strip == 0 || later) return;
  const int end = (tile + 1) * S;
  for (int w = wave + 1; w < WAVES; ++w) {
    const int j0 = total * w / WAVES, j1 = total * (w + 1) / WAVES;
    if (j0 >= end) break;
    if (j1 > j0) acc += red[w * MS_WAVE + lane];
  }
  finish(tile, acc, bv, pre);
}

constexpr unsigned inverse_of(int d) { return d > 1 ? (unsigned)((0x100000000ull + d - 1) / d) : 0u; }

size_t lds_bytes(int M, int K, int loads, int ring, bool norm) {
  const int S = (K + STRIP - 1) / STRIP;
  return (size_t)WAVES * ring * loads * 1024 + (norm ? (size_t)M * (S * 16 + 2) * 16 + (size_t)M * ((K / 8 + 63) / 64) * 4 : 0);
}

template <int L, int XL, int EPI, typename TO, bool NORM>
int launch(const void* A, size_t lda, const bf16* W, size_t ldw, const float* bias, TO* out, size_t ldo, int M, int N,
           int K, const float* norm_w, float eps, const int* rows, int blocks, int q, int rem, const QkvFront& front,
           hipStream_t stream) {
  const size_t lds = lds_bytes(M, K, L + XL, ring_kb(XL) / (L + XL), NORM);
  if (lds > (size_t)LDS_BUDGET) return MS_UNSUPPORTED;
  static bool raised = false;   // once per instantiation: allow more dynamic LDS than the default 64 KB
  if (!raised) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_ring_kernel<L, XL, EPI, TO, NORM>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BUDGET) != hipSuccess)
      return MS_LAUNCH_FAILED;
    raised = true;
  }
  gemm_ring_kernel<L, XL, EPI, TO, NORM><<<dim3(blocks), dim3(WAVES * MS_WAVE), lds, stream>>>(
      A, lda, W, ldw, bias, out, ldo, M, N, K, norm_w, eps, rows, q, rem, inverse_of((K + STRIP - 1) / STRIP),
      inverse_of((K / 8 + 63) / 64), front);
  return ms_launch_status();
}

template <int EPI, typename TO, bool NORM>
int plan(const void* A, size_t lda, const bf16* W, size_t ldw, const float* bias, TO* out, size_t ldo, int M, int N,
         int K, const float* norm_w, float eps, const int* rows, hipStream_t stream, const QkvFront& front = QkvFront{}) {
  const int cus = ms_compute_units();
  const int units = (N + 1) / 2;                        // of two rows (a gate/up pair), dealt out evenly
  const int blocks = units < cus ? units : cus;
  const int q = units / blocks, rem = units % blocks;
  const int R = 2 * (q + (rem ? 1 : 0)), T = (R + 15) / 16;
  const int l = ((R + T - 1) / T + 3) / 4;              // tiles as low as as many of them allow
  if ((long long)(R + 15) * ((K + STRIP - 1) / STRIP) > 0xffff) return MS_UNSUPPORTED;   // (a bound on a block's items)
#define GO(LV, XV) if (l == LV) return launch<LV, XV, EPI, TO, NORM>(A, lda, W, ldw, bias, out, ldo, M, N, K, norm_w, eps, rows, blocks, q, rem, front, stream)
  if constexpr (NORM) {
    GO(1, 0); GO(2, 0); GO(3, 0); GO(4, 0);
  } else {
    if (M <= 4) { GO(1, 1); GO(2, 1); GO(3, 1); GO(4, 1); }
    else if (M <= 8) { GO(1, 2); GO(2, 2); GO(3, 2); GO(4, 2); }
    else { GO(1, 4); GO(2, 4); GO(3, 4); GO(4, 4); }
  }
#undef GO
  return MS_UNSUPPORTED;
}

}  // namespace

// Whether this kernel is the faster one for a product of M rows with W[N, K] (that it can compute): from 24 million values of
// W on.  The line goes by W alone, so that in the calls that come here first (folded norms, and up to 8 rows without: from 9 on slabs
// are asked for before, see ms_gemm_slab_parts) a row's bits do not hang on how many rows there are, but for folded norms of so many
// long rows that they do not fit LDS (M K beyond about 47,000).  Time of the others over this one's, K from 512 to
// 18,944, N from 1,024 to 151,936, 1 to 16 rows, without and with the norm: 0.95 to 1.52 from 24 million on, 1.2 on average (2,048
// x 12,288 with norm, 16 rows 0.91); between 10 and 24 million 0.99 to 1.31 at one row, but with the norm 0.79 to 1.0 at 8 and 16
// rows, whose turn to bfloat16 every block pays for; below, its start (rings, the order of the tiles) is what counts: 896 x
// 4,864 4.9 and 6.0 us.
extern "C" int ms_gemm_ring_pays(int M, int N, int K) {
  return M > 0 && M <= 16 && N > 0 && K > 0 && K % 8 == 0 && (long long)N * K >= 24000000LL;
}

// As ms_gemm_stream; MS_UNSUPPORTED for shapes it does not take: with any_shape = 0 all but those it is the faster kernel for;
// with any_shape = 1 (tests, measurements) only those it cannot compute.
extern "C" int ms_gemm_ring(const void* A, long long lda, const int* rows, const float* norm_w, float eps, const void* W,
                            long long ldw, const float* bias, void* out, long long ldo, int M, int N, int K, int epilogue,
                            int out_dtype, int norm, int any_shape, hipStream_t stream) {
  if (M <= 0 || N <= 0) return MS_OK;
  if (M > 16) return MS_UNSUPPORTED;
  if (K <= 0 || K % 8 || ldw % 8 || lda < K || ldw < K || lda % (norm ? 4 : 8)) return MS_UNSUPPORTED;
  if (((uintptr_t)A | (uintptr_t)W) % 16 || (norm && ((uintptr_t)norm_w % 16))) return MS_UNSUPPORTED;
  if (norm && !norm_w) return MS_BAD_ARG;
  if (!any_shape && !ms_gemm_ring_pays(M, N, K)) return MS_UNSUPPORTED;
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

// ms_qkv_rope_store (qkv_fused.hip), whose checks its arguments have passed, for the sizes that this kernel is the faster one for
// and can compute; MS_UNSUPPORTED for others.  7,168 x 5,120 at one token 22 | 17 us.
extern "C" int ms_gemm_ring_qkv(const float* x, long long ldx, const float* norm_w, float eps, const void* W, const float* bias,
                                const int* positions, const float* inv_freq, const int* slot_mapping, void* q_out,
                                void* k_pages, void* v_pages, int M, int K, int num_heads, int num_kv_heads, int head_dim,
                                int page_size, int v_transposed, hipStream_t stream) {
  const int N = (num_heads + 2 * num_kv_heads) * head_dim;
  if (!ms_gemm_ring_pays(M, N, K) || head_dim % 2 || N > 0xffff) return MS_UNSUPPORTED;
  const QkvFront front{positions, slot_mapping, inv_freq, (bf16*)k_pages, (bf16*)v_pages, num_heads, num_kv_heads, head_dim,
                       page_size, v_transposed, inverse_of(head_dim)};
  return plan<EPI_QKV, bf16, true>(x, ldx, (const bf16*)W, K, bias, (bf16*)q_out, (size_t)num_heads * head_dim, M, N, K, norm_w,
                                   eps, nullptr, stream, front);
}
