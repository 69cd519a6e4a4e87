// What the matrix-core attention kernels share.
#pragma once
#include "common.h"

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

constexpr float REF_SLACK = 8.0f;   // log2 units by which a column's maximum may run ahead of its reference

// Which request the `flat`-th tile of `width` columns belongs to, and which of its tiles it is.  A request owns
// ceil(columns / width) tiles, requests in order, so a launch needs to know only how many tokens and requests a step has,
// not how the tokens are dealt out (a captured graph serves every mix).  The waves of a block find their place alike: a
// lane per request works out its tiles, a prefix sum over the wave and a vote say where the tile falls.  r < 0: the grid
// has room for a partial tile of every request, and this block is surplus.
__device__ __forceinline__ void find_tile(const int* __restrict__ q_start, int n_requests, int rep, int width, int flat,
                                          int lane, int& r, int& rank, int& n_tiles) {
  int before = 0;
  r = -1; rank = 0; n_tiles = 0;
  for (int base = 0; base < n_requests; base += MS_WAVE) {
    const int i = base + lane;
    int mine = 0;
    if (i < n_requests) mine = ((q_start[i + 1] - q_start[i]) * rep + width - 1) / width;
    int upto = mine;   // tiles of the requests base..i
#pragma unroll
    for (int o = 1; o < MS_WAVE; o <<= 1) {
      const int v = __shfl_up(upto, o, MS_WAVE);
      if (lane >= o) upto += v;
    }
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(flat < before + upto);
    if (hit) {
      const int first = __builtin_ctzll(hit);
      r = base + first;
      n_tiles = __shfl(mine, first, MS_WAVE);
      rank = flat - before - (__shfl(upto, first, MS_WAVE) - n_tiles);
      break;
    }
    before += __shfl(upto, MS_WAVE - 1, MS_WAVE);
  }
  r = __builtin_amdgcn_readfirstlane(r);
  rank = __builtin_amdgcn_readfirstlane(rank);
  n_tiles = __builtin_amdgcn_readfirstlane(n_tiles);
}
