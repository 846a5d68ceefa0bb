// Tables of blocks of several deltas (dz_multi_delta_gemm_mixed), made on the device.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/dz_amd.h"

// Blocks from segment offsets (segment 0: tokens without a delta, k >= 1: slot k - 1).  Every segment
// starts a new tile of 16 rows; a block holds up to `most` tiles, about as many in each, and up to
// `deltas` deltas; tokens without a delta have blocks of their own.  One workgroup of 1024 threads; off: S + 2 ints of LDS.
__device__ __forceinline__ void dz_build_mixed_blocks(const int* __restrict__ seg_off, const int* __restrict__ perm, int S,
                                                      int most, int deltas, int* __restrict__ count,
                                                      dz_mixed_block* __restrict__ blocks, int max_blocks, int* off) {
  __shared__ int total, n;
  const int tid = threadIdx.x;
  if (tid == 0) total = 0;
  for (int k = tid; k < S + 2; k += 1024) off[k] = seg_off[k];
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
