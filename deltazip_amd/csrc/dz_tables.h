// Tables of blocks of several deltas (dz_multi_delta_gemm_mixed), made on the device.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/dz_amd.h"

// LDS of dz_segment_tokens.
inline size_t dz_segment_lds(int S) { return (size_t)((S + 2) + (S + 1) + 16 * (S + 1)) * 4; }

// Stable counting sort of tokens by delta id (an id outside [-1, S) counts as -1 and sets bit 0 of *status).  One
// workgroup of 1024 threads; sm: dz_segment_lds(S) bytes, which begin with the S + 2 segment offsets afterwards.  perm
// is written when it returns, for the workgroup.
__device__ __forceinline__ void dz_segment_tokens(const long long* idx, int T, int S, int* perm, unsigned* status, int* sm) {
  // hist[S+2] (exclusive offsets after the scan), running[S+1] (tokens of a key placed by earlier
  // chunks), cnt[16][S+1] (tokens of a key per wavefront of the current chunk)
  int* hist = sm;
  int* running = sm + (S + 2);
  int* cnt = running + (S + 1);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nk = S + 1;
  for (int s = tid; s < S + 2; s += 1024) hist[s] = 0;
  for (int s = tid; s < nk; s += 1024) running[s] = 0;
  __syncthreads();
  bool bad = false;
  for (int t = tid; t < T; t += 1024) {
    long long id = idx[t];
    int key = (id < 0 || id >= S) ? 0 : (int)id + 1;
    bad |= id < -1 || id >= S;
    atomicAdd(&hist[key + 1], 1);
  }
  if (bad && status) atomicOr(status, 1u);
  __syncthreads();
  if (tid == 0) {
    for (int s = 1; s < S + 2; ++s) hist[s] += hist[s - 1];
  }
  __syncthreads();
  // chunks of 1024 tokens in order; inside a chunk a token's place among equal keys is
  // (tokens of that key in earlier wavefronts) + (in lower lanes of its own wavefront)
  for (int base = 0; base < T; base += 1024) {
    for (int c = tid; c < 16 * nk; c += 1024) cnt[c] = 0;
    __syncthreads();
    const int t = base + tid;
    int key = -1;
    if (t < T) {
      long long id = idx[t];
      key = (id < 0 || id >= S) ? 0 : (int)id + 1;
    }
    int rank = 0;
    unsigned long long todo = __builtin_amdgcn_ballot_w64(key >= 0);
    while (todo) {
      const int k = __builtin_amdgcn_readlane(key, __builtin_ctzll(todo));
      const unsigned long long m = __builtin_amdgcn_ballot_w64(key == k);
      if (key == k) rank = __builtin_popcountll(m & ((1ull << lane) - 1ull));
      if (lane == 0) cnt[wave * nk + k] = __builtin_popcountll(m);
      todo &= ~m;
    }
    __syncthreads();
    if (t < T) {
      int before = 0;
      for (int w = 0; w < wave; ++w) before += cnt[w * nk + key];
      perm[hist[key] + running[key] + before + rank] = t;
    }
    __syncthreads();
    for (int k = tid; k < nk; k += 1024) {
      int tot = 0;
      for (int w = 0; w < 16; ++w) tot += cnt[w * nk + k];
      running[k] += tot;
    }
    __syncthreads();
  }
}

// Blocks from segment offsets (segment 0: tokens without a delta, k >= 1: slot k - 1).  Every segment
// starts a new tile of 16 rows; a block holds up to `most` tiles, about as many in each, and up to
// `deltas` deltas; tokens without a delta have blocks of their own.  One workgroup of 1024 threads; off: the offsets, in
// LDS.
__device__ __forceinline__ void dz_build_mixed_blocks(const int* off, const int* perm, int S, int most, int deltas, int* count,
                                                      dz_mixed_block* blocks, int max_blocks) {
  __shared__ int total, n;
  const int tid = threadIdx.x;
  if (tid == 0) total = 0;
  __syncthreads();
  int mine = 0;
  for (int k = tid; k <= S; k += 1024) mine += (off[k + 1] - off[k] + 15) >> 4;
  if (mine) atomicAdd(&total, mine);
  __syncthreads();
  if (tid == 0) {
    const int want = (total + most - 1) / most;
    const int tiles = want > 0 ? (total + want - 1) / want : 1;
    int nd = 0, nt = 0, made = 0;
    dz_mixed_block* b = blocks;
    auto close = [&]() {
      if (nt == 0) return;
      b->nt = nt;
      b->tend[nd - 1] = DZ_MIXED_ROWS / 16;                // (nothing follows the last one)
      ++made;
      b = blocks + min(made, max_blocks - 1);
      nd = nt = 0;
    };
    for (int k = 0; k <= S; ++k) {
      int p = off[k];
      const int hi = off[k + 1];
      while (p < hi) {
        if (nd == deltas) close();
        const int q = min(hi, p + 16 * (tiles - nt));
        nt += (q - p + 15) >> 4;
        b->nd = k > 0 ? nd + 1 : 0;
        b->slot[nd] = k - 1;
        b->lo[nd] = p;
        b->hi[nd] = q;
        b->tend[nd] = nt;
        ++nd;
        p = q;
        if (nt == tiles || k == 0) close();
      }
    }
    close();
    *count = n = made;
  }
  __syncthreads();
  for (int i = tid; i < n * DZ_MIXED_ROWS; i += 1024) {
    const int r = i % DZ_MIXED_ROWS;
    const dz_mixed_block* b = blocks + i / DZ_MIXED_ROWS;
    int t0 = 0, e = 0;
    while (e + 1 < b->nd && (r >> 4) >= b->tend[e]) t0 = b->tend[e++];
    const int pos = b->lo[e] + r - 16 * t0, held = min(pos, b->hi[e] - 1);
    const int row = perm ? perm[held] : held;
    blocks[i / DZ_MIXED_ROWS].row[r] = pos < b->hi[e] ? row : ~row;
  }
}
