// Multi-delta linear layer for batches between decode and prefill, and for prefill batches whose
// tokens are spread over many deltas:
//   y[t, :] (+)= x[t, :] @ w_base^T + x[t, :] @ dequant(delta[slot(t)])^T
// over a table of row blocks of at most 128 tokens, each with one slot.  The same kernel without
// deltas, each block with its own full weight (a few rows of the output projection per delta's own
// table), is dz_gemm_f16_select_rows.  Same products and the same
// summation order as dz_gemm24.hip (2-bit deltas: bit for bit), on a smaller tile.
//
// One workgroup (4 wavefronts) computes 128 output features x one row block; a wavefront owns one
// n-pair (32 features) x all tokens of the block.  With so few tokens a weight operand is used by
// one wavefront only, so base weight and packed delta words go from memory straight into
// registers, a k-block (256 columns) ahead of their use; only the activations, which all four
// wavefronts read, pass through LDS (stages of 128 columns, two buffers).  64 KB of LDS and at most
// 256 registers leave room for two workgroups per CU.  The loop is instantiated per number of
// 16-token tiles: a block of 5 tokens does the work of 16, not of 256.
//
// What bounds it is the way of the weights through the caches, at no one unit's rate: every row block
// reads the base weight and its delta again, 3.85 GB through L2 for 333 tokens of 7 deltas over 5120 x
// 27648 (271 us: 14 TB/s, 28 % of it from beyond L2, 0.52 GB from HBM, matrix cores 30 % busy), 7.8 GB
// for 1999 tokens over 4096 x 22016 (703 us: 11 TB/s, half from beyond L2, matrix cores 35 % busy).
// 5120 x 27648, 2-bit, against the 256 x 256 tiles: 512 tokens of 64 deltas 3470 -> 1369 us, 1024 of 16
// 1000 -> 630, 2048 of 16 1502 -> 1121, 8192 of 64 4993 -> 4299.  (Eight token tiles' operands read two
// at a time: four at a time spilled 40 bytes per lane.)
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/dz_amd.h"
#include "dz_device.h"

namespace {

constexpr int RB = DZ_SHORT_ROWS;                   // tokens per row block
constexpr int BN = 128;                   // features per workgroup
constexpr int SLAB = RB * 64 * 2;         // bytes of 64 columns of activations
constexpr int STAGE = 2 * SLAB;

struct RowsParams {
  const _Float16* x;
  const _Float16* w;             // base weight: [N, K], or in tiles (w_tiled), or nullptr
  const _Float16* w_stack;       // or nullptr; else a block with a slot takes w_stack[slot] in w's place
  long long w_stride;
  const u4_t* codes;
  const u4_t* meta;
  const _Float16* scales;
  long long codes_slot_u4, meta_slot_u4, scales_slot;
  const dz_gemm_tile* tiles;
  const int* perm;
  _Float16* y;
  int K, N, S, G, gslabs, accumulate, ldy, tiles_m, tiles_n, NKB, NP, w_tiled;
};

// One row block [lo, hi), at most 16 * NT tokens.
template <int BITS, int NT>
__device__ __forceinline__ void row_block(const RowsParams& P, unsigned char* smem, int lo, int hi, int slot, int n0) {
  constexpr int NI = (NT + 1) / 2;               // 16-byte requests per thread and slab: 32 rows each
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const uint32_t MAGIC = magic_vgpr();
  const _Float16* const w = P.w_stack && slot >= 0 ? P.w_stack + (size_t)slot * P.w_stride : P.w;
  const bool do_w = w != nullptr, do_d = slot >= 0 && slot < P.S;
  const int np_own = n0 / DZ_NPAIR + wave;
  const int np = min(np_own, P.NP - 1);          // beyond N: the last n-pair again, never stored
  const unsigned Kb = (unsigned)P.K * 2u;

  // base weight: lane (i, g) takes row i of a 16-row tile, columns 32*h + 8*g .. of a slab.  In
  // tiles these sit in fragment g % 2 at position 16 * (2*h + g/2) + i.
  const char* wp;
  unsigned wl, w_a, w_j, w_h, w_kb;
  if (P.w_tiled) {
    wp = (const char*)w + (size_t)np * P.NKB * 16384;
    wl = (unsigned)((lg & 1) * 1024 + ((lg >> 1) * 16 + li) * 16);
    w_a = 8192; w_j = 2048; w_h = 512; w_kb = 16384;
  } else {
    wp = (const char*)w + (size_t)np * DZ_NPAIR * Kb;
    wl = (unsigned)li * Kb + (unsigned)lg * 16u;
    w_a = 16 * Kb; w_j = 128; w_h = 64; w_kb = 512;
  }
  // slabs of the base weight on their way: a k-block's four, or, where eight token tiles' sums take
  // the registers (and a slab's products take long enough to cover the latency), two
  constexpr int WR = NT > 4 ? 2 : 4;
  h8_t W[WR][2][2];                              // [slab][feature tile][half]
  auto load_w = [&](int kb, int j) {
    const char* b = wp + (size_t)kb * w_kb + j * w_j;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int h = 0; h < 2; ++h) W[j % WR][a][h] = *(const h8_t*)(b + (a * w_a + h * w_h) + wl);
  };

  const char* const mp = (const char*)(P.meta + (size_t)(do_d ? slot : 0) * P.meta_slot_u4) + (size_t)np * P.NKB * 1024;
  const char* const cp = (const char*)(P.codes + (size_t)(do_d ? slot : 0) * P.codes_slot_u4) +
                         (size_t)np * P.NKB * (1024 * Frag<BITS>::NCODE);
  auto load_delta = [&](Frag<BITS>& f, int kb) {
    f.meta = *(const u4_t*)(mp + (size_t)kb * 1024 + lane * 16);
#pragma unroll
    for (int c = 0; c < Frag<BITS>::NCODE; ++c)
      f.code[c] = *(const u4_t*)(cp + (size_t)kb * (1024 * Frag<BITS>::NCODE) + c * 1024 + lane * 16);
  };
  // scales of the four slabs of a k-block (one load for all when a group is at least that long)
  const _Float16* const sp = P.scales + (size_t)(do_d ? slot : 0) * P.scales_slot + np * DZ_NPAIR + li;
  int gi = 0, gleft = P.gslabs;
  auto load_scales = [&](h2_t (&s)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const _Float16* q = sp + (size_t)min(gi, P.G - 1) * P.N;
      s[j] = (h2_t){q[0], q[16]};
      if (--gleft == 0) { gleft = P.gslabs; ++gi; }
    }
  };

  // activations: thread t takes chunk t % 8 of row t / 8 + 32 * i, to LDS chunk (t % 8) ^ (row / 2 % 8)
  unsigned xo[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int pos = min(lo + (tid >> 3) + 32 * i, hi - 1);
    const int row = P.perm ? P.perm[pos] : pos;
    xo[i] = (unsigned)row * Kb + (unsigned)(tid & 7) * 16u;
  }
  const int xw = (tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) << 4);   // (32 rows on: the same swizzle)
  h8_t X[2][NI];
  const int nstage = P.NKB * 2;
  auto load_x = [&](int st) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NI; ++i) X[s][i] = *(const h8_t*)((const char*)P.x + (size_t)st * 256 + s * 128 + xo[i]);
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NI; ++i) *(h8_t*)(smem + buf * STAGE + s * SLAB + i * 4096 + xw) = X[s][i];
  };
  int foff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) foff[h] = li * 128 + (((4 * h + lg) ^ ((li >> 1) & 7)) << 4);

  f4_t acc[2][NT];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = (f4_t){0.f, 0.f, 0.f, 0.f};

  Frag<BITS> cur, nxt;
  h2_t sc[4], scn[4];
  load_x(0);
  if (do_d) {
    load_delta(cur, 0);
    load_scales(sc);
  }
  if (do_w) {
#pragma unroll
    for (int j = 0; j < WR; ++j) load_w(0, j);
  }
  store_x(0);
  load_x(1);
  __builtin_amdgcn_s_waitcnt(0xC07F);            // lgkmcnt(0): this wavefront's part is in LDS
  wg_barrier_nofence();

  for (int kb = 0; kb < P.NKB; ++kb) {
    const int kn = min(kb + 1, P.NKB - 1);       // (the last turn reads its own k-block again)
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      // the next k-block's packed words: a whole k-block ahead, or half of one where registers are short
      if (do_d && st == (NT > 4 ? 1 : 0)) {
        load_delta(nxt, kn);
        if (P.G > 1) load_scales(scn);
      }
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int j = 2 * st + jj;
        const unsigned char* xb = smem + st * STAGE + jj * SLAB;
        h8_t A0, A1;
        int mw = 0;
        if (do_d) {
          mw = (int)cur.meta[j];
          if constexpr (BITS == 2) {
            unpack2(cur.code[0][j], MAGIC, A0, A1);
          } else {
            A0 = unpack4(cur.code[j >> 1][2 * (j & 1)], MAGIC);
            A1 = unpack4(cur.code[j >> 1][2 * (j & 1) + 1], MAGIC);
          }
          A0 *= sc[j][0];
          A1 *= sc[j][1];
        }
        // two or four token tiles' operands at a time (more would not fit beside the prefetched weights)
#pragma unroll
        for (int b0 = 0; b0 < NT; b0 += (NT > 4 ? 2 : 4)) {
          constexpr int GB = NT < 4 ? NT : NT > 4 ? 2 : 4;
          h8_t Bl[GB], Bh[GB];
#pragma unroll
          for (int b = 0; b < GB; ++b)
            if (b0 + b < NT) {
              Bl[b] = *(const h8_t*)(xb + (b0 + b) * 2048 + foff[0]);
              Bh[b] = *(const h8_t*)(xb + (b0 + b) * 2048 + foff[1]);
            }
          if (do_w) {
#pragma unroll
            for (int b = 0; b < GB; ++b)
              if (b0 + b < NT) {
#pragma unroll
                for (int a = 0; a < 2; ++a)
                  acc[a][b0 + b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(W[j % WR][a][0], Bl[b], acc[a][b0 + b], 0, 0, 0);
#pragma unroll
                for (int a = 0; a < 2; ++a)
                  acc[a][b0 + b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(W[j % WR][a][1], Bh[b], acc[a][b0 + b], 0, 0, 0);
              }
          }
          if (do_d) {
#pragma unroll
            for (int b = 0; b < GB; ++b)
              if (b0 + b < NT) {
                const h16_t B = __builtin_shufflevector(Bl[b], Bh[b], 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
                acc[0][b0 + b] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A0, B, acc[0][b0 + b], mw, 0, 0);
                acc[1][b0 + b] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A1, B, acc[1][b0 + b], mw, 0, 1);
              }
          }
          if (NT > 4) __builtin_amdgcn_sched_barrier(0);
        }
        if (do_w) load_w(j + WR < 4 ? kb : kn, (j + WR) & 3);
      }
      // the other buffer was read one stage ago, in front of the last barrier
      store_x(st ^ 1);
      load_x(min(2 * kb + st + 2, nstage - 1));
      __builtin_amdgcn_s_waitcnt(0xC07F);
      wg_barrier_nofence();
    }
    if (do_d) {
      cur = nxt;
      if (P.G > 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[j] = scn[j];
      }
    }
  }

  if (np_own >= P.NP) return;
#pragma unroll
  for (int b = 0; b < NT; ++b) {
    const int pos = lo + b * 16 + li;
    if (pos >= hi) continue;
    const int row = P.perm ? P.perm[pos] : pos;
    _Float16* yrow = P.y + (size_t)row * P.ldy + np_own * DZ_NPAIR + 4 * lg;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      f4_t v = acc[a][b];
      if (P.accumulate) {
        const h4_t old = *(const h4_t*)(yrow + a * 16);
        v += (f4_t){(float)old[0], (float)old[1], (float)old[2], (float)old[3]};
      }
      *(h4_t*)(yrow + a * 16) = (h4_t){(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
    }
  }
}

template <int BITS>
__global__ __launch_bounds__(256, 2) void dz_gemm24_rows_kernel(const RowsParams P) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // The row blocks of one feature tile run next to each other on one XCD: they read the same base
  // weight, which only the first of them fetches from beyond that XCD's L2.
  const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
  // Only the entries in use are counted for that: workgroups of unused ones between the others would
  // each hold a place on a CU until they have read their entry (32000 x 4096, 32 tokens without a
  // delta among 8 slots: 111 -> 57 us).
  int used = 0;
  for (int e = 0; e < P.tiles_m; e += 64) {
    const dz_gemm_tile t = P.tiles[min(e + (int)(threadIdx.x & 63), P.tiles_m - 1)];
    const unsigned long long has = __ballot(t.row_hi > t.row_lo && e + (int)(threadIdx.x & 63) < P.tiles_m);
    if (has) used = e + 64 - __clzll((long long)has);
  }
  if (used == 0) return;
  const int tn = (q / used) * 8 + xcd, tm = q % used;
  if (tn >= P.tiles_n) return;
  const int row_lo = P.tiles[tm].row_lo, row_hi = P.tiles[tm].row_hi, slot = P.tiles[tm].group;
  // (a block of more than RB rows is taken RB rows at a time; the loop's last barrier is behind the
  // last read of either buffer)
  for (int lo = row_lo; lo < row_hi; lo += RB) {
    const int hi = min(lo + RB, row_hi), nt = (hi - lo + 15) >> 4;
    if (nt <= 1) row_block<BITS, 1>(P, smem, lo, hi, slot, tn * BN);
    else if (nt <= 2) row_block<BITS, 2>(P, smem, lo, hi, slot, tn * BN);
    else if (nt <= 3) row_block<BITS, 3>(P, smem, lo, hi, slot, tn * BN);
    else if (nt <= 4) row_block<BITS, 4>(P, smem, lo, hi, slot, tn * BN);
    else if (nt <= 6) row_block<BITS, 6>(P, smem, lo, hi, slot, tn * BN);
    else row_block<BITS, 8>(P, smem, lo, hi, slot, tn * BN);
  }
}

}  // namespace

static int launch(RowsParams P, int bits, int ntiles, hipStream_t st) {
  P.tiles_m = ntiles; P.tiles_n = (P.N + BN - 1) / BN;
  P.NKB = P.K / DZ_KBLOCK; P.NP = P.N / DZ_NPAIR;
  const unsigned long long grid = (unsigned long long)((P.tiles_n + 7) / 8) * 8ull * (unsigned)ntiles;
  if (grid > 0x7fffffffull) return DZ_ESHAPE;
  const int lds = 2 * STAGE;
  static std::atomic<unsigned long long> attr_done[2];
  auto go = [&](auto kern, int which) -> int {
    if (!dz_lds_limit_once(attr_done[which], (const void*)kern, lds)) return DZ_ELAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, st, P);
    return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
  };
  return bits == 2 ? go(dz_gemm24_rows_kernel<2>, 0) : go(dz_gemm24_rows_kernel<4>, 1);
}

extern "C" int dz_multi_delta_gemm_rows(const uint16_t* x, const uint16_t* w_base, int w_tiled, const void* codes_stacked,
                                        const void* meta_stacked, const void* scales_stacked, int S, int bits,
                                        int group_size, const dz_gemm_tile* tiles, int ntiles, const int32_t* perm,
                                        uint16_t* y, int T, int K, int N, int accumulate, int ldy, void* stream) {
  if (!x || !y || !tiles || ntiles < 1 || S < 0) return DZ_EINVAL;
  if (S > 0 && (!codes_stacked || !meta_stacked || !scales_stacked)) return DZ_EINVAL;
  size_t cb, mb, sb;
  int rc = dz_native_sizes(K, N, bits, group_size, &cb, &mb, &sb);
  if (rc) return rc;
  const int gs = (group_size == -1 || group_size == K) ? K : group_size;
  if (T < 1 || ldy < N || ldy % 4) return DZ_ESHAPE;
  if (((uintptr_t)x & 15) || ((uintptr_t)w_base & 15) || ((uintptr_t)y & 7)) return DZ_EALIGN;
  if ((unsigned long long)T * (unsigned)K * 2ull >= (1ull << 31)) return DZ_ESHAPE;   // 32-bit row offsets
  RowsParams P{};
  P.x = (const _Float16*)x; P.w = (const _Float16*)w_base; P.y = (_Float16*)y;
  P.codes = (const u4_t*)codes_stacked; P.meta = (const u4_t*)meta_stacked; P.scales = (const _Float16*)scales_stacked;
  P.codes_slot_u4 = (long long)(cb / 16); P.meta_slot_u4 = (long long)(mb / 16); P.scales_slot = (long long)(sb / 2);
  P.tiles = tiles; P.perm = perm;
  P.K = K; P.N = N; P.S = S; P.G = K / gs; P.gslabs = gs / 64; P.accumulate = accumulate; P.ldy = ldy;
  P.w_tiled = (w_tiled && w_base) ? 1 : 0;
  return launch(P, bits, ntiles, (hipStream_t)stream);
}

extern "C" int dz_gemm_f16_select_rows(const uint16_t* x, const uint16_t* w_base, const uint16_t* w_stack,
                                       long long w_stride, const dz_gemm_tile* tiles, int ntiles, const int32_t* perm,
                                       uint16_t* y, int T, int K, int N, int accumulate, int ldy, void* stream) {
  if (!x || !y || !tiles || ntiles < 1 || !w_base || !w_stack) return DZ_EINVAL;
  if (T < 1 || K < DZ_KBLOCK || K % DZ_KBLOCK || N < DZ_NPAIR || N % DZ_NPAIR || ldy < N || ldy % 4) return DZ_ESHAPE;
  if (((uintptr_t)x & 15) || ((uintptr_t)w_base & 15) || ((uintptr_t)w_stack & 15) || ((uintptr_t)y & 7) || (w_stride & 7))
    return DZ_EALIGN;
  if ((unsigned long long)T * (unsigned)K * 2ull >= (1ull << 31) ||
      (unsigned long long)N * (unsigned)K * 2ull >= (1ull << 31))
    return DZ_ESHAPE;
  RowsParams P{};
  P.x = (const _Float16*)x; P.w = (const _Float16*)w_base; P.y = (_Float16*)y;
  P.w_stack = (const _Float16*)w_stack; P.w_stride = w_stride;
  P.tiles = tiles; P.perm = perm;
  P.K = K; P.N = N; P.G = 1; P.gslabs = K / 64; P.accumulate = accumulate; P.ldy = ldy;   // (S = 0: no deltas)
  return launch(P, 2, ntiles, (hipStream_t)stream);
}
