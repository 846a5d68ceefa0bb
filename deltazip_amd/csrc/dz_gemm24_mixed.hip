// Multi-delta linear layer for more than 128 tokens, and for decode batches of few deltas over large layers, over blocks of
// rows that hold the tokens of several deltas:
//   y[t, :] (+)= x[t, :] @ w_base^T + x[t, :] @ dequant(delta[slot(t)])^T
// A block (dz_tables.h) is up to 8 tiles of 16 tokens, each tile of one delta, up to 4 deltas: base
// weight and activations are read once per block, whatever deltas it holds, and a delta of a few
// tokens costs its words and its tiles instead of a walk over the base weight of its own.
//
// One workgroup (8 wavefronts) computes 256 output features x one block, over all of K or a part of it;
// a wavefront owns one n-pair (32 features) x all tokens of the block.  Base weight and packed words have
// one reader each and go from memory into registers, four slabs (a k-block of 256 columns) and two
// slabs ahead of their use; the activations, which all eight wavefronts read, go straight into LDS a
// k-block ahead (2 x 64 KB, one barrier per k-block).  256 registers per lane: 64 of sums, 64 of base
// weight, 12 per delta of words.  Per slab of 64 columns a tile is 4 dense and 2 sparse products from the
// same operands, read from LDS one tile ahead; a delta's words are unpacked at its first tile, on a branch all
// lanes take together.  Numbers of tiles and deltas are compile-time: with them at run time the
// compiler moved every read next to its use (a slab of 8 tiles and 4 deltas: 2.6 against 1.3 us).
// The products and their order are those of dz_gemm24_rows.hip.
//
// What bounds it, per slab of 8 tiles on an otherwise idle GPU: 0.62 us without a delta, 0.91 with one, 1.01 with
// two, 1.31 with four, of which the matrix cores need 0.43 and (with deltas) 0.64; the rest is the words'
// unpacking, 25 vector instructions a delta, which the wavefront's twin on the SIMD covers in part.  With all
// CUs busy and the base weight of 256 features per CU coming from memory 1.7 us, 4.9 to 5.9 TB/s.  5120 x
// 27648, 2-bit, against one delta per block and against 256 x 256 tiles: 333 tokens of 10 deltas 250 -> 215 us, 1000
// of 32 950 -> 700, 8192 of 16 3460 -> 3020; 13824 x 5120, 333 tokens 160 -> 100 (K in three parts, by the
// number of blocks; in four 129).  A layer of 5120/13824, 333 tokens: 770 -> 521 us (by the card 483 to 557).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/dz_amd.h"
#include "dz_device.h"
#include "dz_tables.h"

namespace {

constexpr int MROWS = DZ_MIXED_ROWS;       // tokens per block
constexpr int MWAVES = 8;
constexpr int MN = 32 * MWAVES;            // features per workgroup
constexpr int MSLAB = MROWS * 64 * 2;      // bytes of 64 columns of activations
constexpr int XSTAGE = 4 * MSLAB;
constexpr int MG = 4;                      // tiles of features that meet a block together

struct MixedParams {
  const _Float16* x;
  const _Float16* w;
  const u4_t* codes;
  const u4_t* meta;
  const _Float16* scales;
  long long meta_slot_u4, scales_slot;
  const int* count;              // blocks in use
  const dz_mixed_block* blocks;
  _Float16* y;
  float* part;                   // partial sums [ksplit][T][N], or nullptr
  int T, K, N, G, accumulate, ldy, tiles_n, NKB, NP, w_tiled;
  int ksplit;                    // slices of K, or 0: by the number of blocks,
  unsigned long long parts_of;   // 4 bits for each of 1 to 16 (more: as for 16)
  unsigned gmagic;               // group of a slab: (slab * gmagic) >> 32
};

__device__ __forceinline__ int slices_for(int used, int ksplit, unsigned long long parts_of) {
  return ksplit ? ksplit : (int)(parts_of >> (4 * (min(used, 16) - 1))) & 15;
}

// f(0), f(1), .. f(N - 1) with constant arguments.  (Arrays that a loop indexes stay in memory until it is
// unrolled, and by then a choice between two of their elements has become a load from a chosen address.)
template <int I = 0, int N, typename F>
__device__ __forceinline__ void each(std::integral_constant<int, N> n, F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<I + 1>(n, f);
  }
}

// Packed words of a delta for one n-pair: the k-block that comes (4 bits: its first half), and what is
// left of the one at hand while its first half is requested again.
template <int BITS>
struct Words;
template <>
struct Words<2> { u4_t meta, code; u2_t meta2, code2; };
template <>
struct Words<4> { u4_t meta, code, code2; u2_t meta2; };

// What every wavefront needs of a block, read before anything that keeps the compiler from scalar loads.
struct BlockHead {
  int nt, nd, slot[DZ_MIXED_DELTAS], tend[DZ_MIXED_DELTAS];
};

// One block of up to NT tiles and ND deltas, columns of k-blocks [kb0, kb1).  GRP: scales change along K.
template <int BITS, bool GRP, int ND, int NT>
__device__ __forceinline__ void mixed_block(const MixedParams& P, unsigned char* smem, const dz_mixed_block* blk,
                                            const BlockHead& head, int n0, int kb0, int kb1, int slice) {   // slice -1: all of K
  constexpr bool HAS_D = ND > 0;
  constexpr int E = HAS_D ? ND : 1;
  constexpr bool AHEAD = ND < (GRP && BITS == 2 ? 3 : 4) || NT < 8;         // a tile's activations are read during the tile before (else: spills)
  constexpr int NI = MSLAB / (64 * MWAVES * 16);   // 1 KiB requests per wavefront and slab
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int np_own = n0 / DZ_NPAIR + wave;
  const int np = min(np_own, P.NP - 1);            // beyond N: the last n-pair again, never stored
  const unsigned Kb = (unsigned)P.K * 2u;
  int held[NI];                                    // rows of x that this lane fetches chunks of
#pragma unroll
  for (int i = 0; i < NI; ++i) held[i] = blk->row[(wave * NI + i) * 8 + (lane >> 3)];

  // base weight: lane (i, g) takes row i of a 16-row tile, columns 32*h + 8*g .. of a slab.  In
  // tiles these sit in fragment g % 2 at position 16 * (2*h + g/2) + i.
  const char* wp;
  int wl, w_a, w_j, w_h, w_kb;
  if (P.w_tiled) {
    wp = (const char*)P.w + (size_t)np * P.NKB * 16384;
    wl = (lg & 1) * 1024 + ((lg >> 1) * 16 + li) * 16;
    w_a = 8192; w_j = 2048; w_h = 512; w_kb = 16384;
  } else {
    wp = (const char*)P.w + (size_t)np * DZ_NPAIR * Kb;
    wl = li * (int)Kb + lg * 16;
    w_a = 16 * (int)Kb; w_j = 128; w_h = 64; w_kb = 512;
  }
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(wp), 0, 0x7fffffff, 0x00020000);
  union W16 { u4_t u; h8_t h; };
  h8_t W[4][2][2];                                 // [slab][feature tile][half]
  auto load_w = [&](int kb, int j) {
    const int at = kb * w_kb + j * w_j;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        W16 v;
        v.u = __builtin_amdgcn_raw_buffer_load_b128(rw, wl, at + a * w_a + h * w_h, 0);
        W[j][a][h] = v.h;
      }
  };

  // ---- deltas of the block
  long long moff[E];                               // bytes to the n-pair's positions (codes: NCODE times as far)
  int tend[E];
  const _Float16* sp[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int slot = HAS_D ? head.slot[e] : 0;
    tend[e] = HAS_D ? head.tend[e] : 0;
    moff[e] = (long long)slot * (P.meta_slot_u4 * 16) + (long long)np * P.NKB * 1024;
    sp[e] = P.scales + (size_t)slot * P.scales_slot + np * DZ_NPAIR;
  }
  Words<BITS> wd[E];
  int raw[2][E];                                   // GRP: lane l holds the scale of row l % 32, slab l / 32 of the half
  h2_t sc[E];                                      // else: rows li and 16 + li
  const unsigned lo16 = (unsigned)lane * 16u;
  auto load_half = [&](int kb, int h) {            // requests of a half of k-block kb, made two slabs ahead
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (h == 0) wd[e].meta = *(const u4_t*)((const char*)P.meta + (moff[e] + kb * 1024) + lo16);
      if constexpr (BITS == 2) {
        if (h == 0) wd[e].code = *(const u4_t*)((const char*)P.codes + (moff[e] + kb * 1024) + lo16);
      } else {
        if (h == 0) wd[e].code = *(const u4_t*)((const char*)P.codes + (2 * moff[e] + kb * 2048) + lo16);
        else wd[e].code2 = *(const u4_t*)((const char*)P.codes + (2 * moff[e] + kb * 2048 + 1024) + lo16);
      }
    }
    if constexpr (GRP) {
      const unsigned s = 4 * kb + 2 * h;
      const int g0 = P.gmagic ? (int)__umulhi(s, P.gmagic) : (int)s, g1 = P.gmagic ? (int)__umulhi(s + 1, P.gmagic) : (int)s + 1;
      const unsigned off = ((unsigned)(lane >> 5 ? g1 : g0) * (unsigned)P.N + (unsigned)(lane & 31)) * 2u;
#pragma unroll
      for (int e = 0; e < E; ++e) raw[h][e] = *(const unsigned short*)((const char*)sp[e] + off);
    }
  };
  auto keep_half = [&]() {                         // the second half's words, out of the registers requested again
#pragma unroll
    for (int e = 0; e < E; ++e) {
      wd[e].meta2 = (u2_t){wd[e].meta[2], wd[e].meta[3]};
      asm volatile("" : "+v"(wd[e].meta2));
      if constexpr (BITS == 2) {
        wd[e].code2 = (u2_t){wd[e].code[2], wd[e].code[3]};
        asm volatile("" : "+v"(wd[e].code2));
      }
    }
  };
  if constexpr (HAS_D && !GRP) {
#pragma unroll
    for (int e = 0; e < E; ++e) sc[e] = (h2_t){sp[e][li], sp[e][16 + li]};
  }

  // ---- activations, from memory into LDS, a k-block ahead of their use: request i of a wavefront and slab is 8
  // rows x 128 bytes, lane l fills chunk l % 8 of row l / 8 with global chunk (l % 8) ^ (row / 2 % 8)
  unsigned xo[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int R = (wave * NI + i) * 8 + (lane >> 3);
    xo[i] = (unsigned)(held[i] < 0 ? ~held[i] : held[i]) * Kb + (unsigned)((lane & 7) ^ ((R >> 1) & 7)) * 16u;
  }
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(P.x), 0, 0x7fffffff, 0x00020000);
  auto load_x = [&](int stage, int kb, int half) {  // two slabs
#pragma unroll
    for (int j = 2 * half; j < 2 * half + 2; ++j)
#pragma unroll
      for (int i = 0; i < NI; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rx, (__attribute__((address_space(3))) void*)(smem + stage * XSTAGE + j * MSLAB + (wave * NI + i) * 1024), 16,
            (int)xo[i], kb * 512 + j * 128, 0, 0);
    __builtin_amdgcn_s_waitcnt(0xC07F);            // lgkmcnt(0): no LDS access is outstanding here, and the compiler knows
    __builtin_amdgcn_sched_barrier(0);
  };
  // A k-block's activations are in: at most the requests that came after them, for three slabs of the next
  // k-block's base weight and for its packed words, are outstanding.  s_waitcnt immediate: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] |
  // vmcnt[5:4] << 14.
  constexpr int AFTER = 12 + (HAS_D ? E * (GRP ? 3 : 2) : 0);
  static_assert(AFTER < 64, "counter of outstanding requests");
  auto wait_x = [&]() { __builtin_amdgcn_s_waitcnt((AFTER & 15) | ((AFTER >> 4) << 14) | 0x0070); };
  int foff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) foff[h] = li * 128 + (((4 * h + lg) ^ ((li >> 1) & 7)) << 4);

  const uint32_t MAGIC = magic_vgpr();
  f4_t acc[2][NT];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = (f4_t){0.f, 0.f, 0.f, 0.f};

  if constexpr (HAS_D) load_half(kb0, 0);
#pragma unroll
  for (int j = 0; j < 4; ++j) load_w(kb0, j);
  __builtin_amdgcn_sched_barrier(0);
  load_x(kb0 & 1, kb0, 0);
  load_x(kb0 & 1, kb0, 1);
  __builtin_amdgcn_s_waitcnt(0x0070);
  wg_barrier_nofence();

  // packed words of slab jc of delta qc
  auto word = [&](auto jc, auto qc, uint32_t& m, uint32_t& c0, uint32_t& c1) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value, q = decltype(qc)::value;
    m = j < 2 ? wd[q].meta[j] : wd[q].meta2[j & 1];
    if constexpr (BITS == 2) {
      c0 = j < 2 ? wd[q].code[j] : wd[q].code2[j & 1];
      c1 = 0;
    } else {
      c0 = j < 2 ? wd[q].code[2 * (j & 1)] : wd[q].code2[2 * (j & 1)];
      c1 = j < 2 ? wd[q].code[2 * (j & 1) + 1] : wd[q].code2[2 * (j & 1) + 1];
    }
  };
  auto spread = [&](auto jc, int r) __attribute__((always_inline)) {   // rows li and 16 + li of the slab's scales
    constexpr int j = decltype(jc)::value;
    const unsigned l16 = (unsigned)__builtin_amdgcn_ds_bpermute((32 * (j & 1) + li) << 2, r) & 0xffffu;
    const unsigned h16 = (unsigned)__builtin_amdgcn_ds_bpermute((32 * (j & 1) + 16 + li) << 2, r);
    H2U u;
    u.u = l16 | (h16 << 16);
    return u.h;
  };
  auto operands = [&](uint32_t c0, uint32_t c1, h2_t s, h8_t& A0, h8_t& A1) __attribute__((always_inline)) {
    if constexpr (BITS == 2) {
      unpack2(c0, MAGIC, A0, A1);
    } else {
      A0 = unpack4(c0, MAGIC);
      A1 = unpack4(c1, MAGIC);
    }
    asm volatile("" : "+v"(s));                    // (one register: no copies of it for packed products)
    A0 *= s[0];
    A1 *= s[1];
  };
  for (int kb = kb0; kb < kb1; ++kb) {
    const int kn = min(kb + 1, kb1 - 1);           // (the last turn requests its own k-block again)
    each(std::integral_constant<int, 4>{}, [&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      if constexpr (HAS_D) {
        if (j == 0 && (BITS == 4 || GRP)) load_half(kb, 1);
        if (j == 2) {
          keep_half();
          load_half(kn, 0);
        }
      }
      if (j < 2) load_x((kb + 1) & 1, kn, j);      // (these were read in the turn before, in front of the barrier)
      const unsigned char* xb = smem + (kb & 1) * XSTAGE + j * MSLAB;
      h8_t A0, A1;
      int mw = 0, e = 0, next = 0;                 // next: the tile at which the next delta, e, starts
      auto unpack = [&]() __attribute__((always_inline)) {   // operands of delta e
        uint32_t m, c0, c1;
        word(jc, std::integral_constant<int, 0>{}, m, c0, c1);
        int r = 0;
        h2_t s;
        if constexpr (GRP) r = raw[j >> 1][0]; else s = sc[0];
        next = tend[0];
        each(std::integral_constant<int, E - 1>{}, [&](auto qc) __attribute__((always_inline)) {
          constexpr int q = decltype(qc)::value + 1;
          const bool is = e == q;
          uint32_t qm, q0, q1;
          word(jc, std::integral_constant<int, q>{}, qm, q0, q1);
          m = is ? qm : m;
          c0 = is ? q0 : c0;
          if constexpr (BITS == 4) c1 = is ? q1 : c1;
          if constexpr (GRP) r = is ? raw[j >> 1][q] : r; else s = is ? sc[q] : s;
          next = is ? tend[q] : next;
        });
        if constexpr (GRP) s = spread(jc, r);
        mw = (int)m;
        operands(c0, c1, s, A0, A1);
        ++e;
      };
      auto read = [&](int b) {
        const h8_t l = *(const h8_t*)(xb + b * 2048 + foff[0]), h = *(const h8_t*)(xb + b * 2048 + foff[1]);
        return __builtin_shufflevector(l, h, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
      };
      h16_t B = read(0);
#pragma unroll
      for (int b = 0; b < NT; ++b) {
        if (HAS_D && (E == 1 ? b == 0 : b == next)) unpack();
        if (!AHEAD && b > 0) B = read(b);
        h16_t Bn = B;
        if (AHEAD && b + 1 < NT) Bn = read(b + 1);
        __builtin_amdgcn_sched_barrier(0);
        const h8_t Bl = __builtin_shufflevector(B, B, 0, 1, 2, 3, 4, 5, 6, 7);
        const h8_t Bh = __builtin_shufflevector(B, B, 8, 9, 10, 11, 12, 13, 14, 15);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int a = 0; a < 2; ++a)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(W[j][a][h], h ? Bh : Bl, acc[a][b], 0, 0, 0);
        if constexpr (HAS_D) {
          acc[0][b] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A0, B, acc[0][b], mw, 0, 0);
          acc[1][b] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(A1, B, acc[1][b], mw, 0, 1);
        }
        B = Bn;
      }
      load_w(kn, j);
      __builtin_amdgcn_sched_barrier(0);
    });
    wait_x();
    wg_barrier_nofence();
  }

  __builtin_amdgcn_s_waitcnt(0x0070);              // the requests behind the last slab write LDS, too
  if (np_own >= P.NP) return;
#pragma unroll
  for (int b = 0; b < NT; ++b) {
    const int row = blk->row[b * 16 + li];
    if (row < 0) continue;
    if (slice >= 0) {
      float* prow = P.part + ((size_t)slice * P.T + row) * P.N + np_own * DZ_NPAIR + 4 * lg;
#pragma unroll
      for (int a = 0; a < 2; ++a) *(f4_t*)(prow + a * 16) = acc[a][b];
      continue;
    }
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

template <int BITS, bool GRP>
__global__ __launch_bounds__(64 * MWAVES, 2) void dz_gemm24_mixed_kernel(const MixedParams P) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int used = *P.count;
  if (used == 0) return;
  // Each XCD takes an eighth of the list of (slice of K, tile of features, block), in which MG tiles
  // at a time meet one block after the other: 32 CUs then share MG tiles' weights and 32 / MG
  // blocks' activations in their L2.  (The grid is for the largest table there could be; workgroups without an
  // item come last and cost nothing that could be measured.)
  const unsigned xcd = blockIdx.x & 7;
  const int ksplit = slices_for(used, P.ksplit, P.parts_of);
  const unsigned per_slice = (unsigned)(P.tiles_n * used), units = per_slice * (unsigned)ksplit;
  const unsigned item = (unsigned)((unsigned long long)units * xcd >> 3) + (blockIdx.x >> 3);
  if (item >= (unsigned)((unsigned long long)units * (xcd + 1) >> 3)) return;
  const int slice = (int)(item / per_slice), at = (int)(item % per_slice);
  const int group = at / (MG * used), wide = min(MG, P.tiles_n - group * MG), r = at - group * MG * used;
  const int tm = r / wide, tn = group * MG + r % wide;
  const dz_mixed_block* blk = P.blocks + tm;
  const int kb0 = P.NKB * slice / ksplit, kb1 = P.NKB * (slice + 1) / ksplit, sums = ksplit > 1 ? slice : -1;
  BlockHead head;
  head.nt = blk->nt;
  head.nd = blk->nd;
#pragma unroll
  for (int e = 0; e < DZ_MIXED_DELTAS; ++e) {
    head.slot[e] = blk->slot[e];
    head.tend[e] = blk->tend[e];
  }
  const int nd = head.nd;
  auto go = [&](auto nt_c) {
    constexpr int NT = decltype(nt_c)::value;
    if (nd == 0) mixed_block<BITS, GRP, 0, NT>(P, smem, blk, head, tn * MN, kb0, kb1, sums);
    else if (nd == 1) mixed_block<BITS, GRP, 1, NT>(P, smem, blk, head, tn * MN, kb0, kb1, sums);
    else if (nd == 2) mixed_block<BITS, GRP, 2, NT>(P, smem, blk, head, tn * MN, kb0, kb1, sums);
    else if (NT == 2) return;                    // (as many tiles as deltas)
    else if (nd == 3 || BITS == 4 || GRP) mixed_block<BITS, GRP, 3, NT>(P, smem, blk, head, tn * MN, kb0, kb1, sums);
    else mixed_block<BITS, GRP, BITS == 4 || GRP ? 3 : 4, NT>(P, smem, blk, head, tn * MN, kb0, kb1, sums);
  };
  switch (head.nt) {
    case 1:
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3:
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    default: go(std::integral_constant<int, 8>{}); break;
  }
}

// y = sum of the K-slices' partial sums, in slice order (nothing to do where there is one slice)
__global__ __launch_bounds__(256) void dz_mixed_sum_kernel(const float* __restrict__ part, _Float16* __restrict__ y, int T, int N, int ksplit,
                                                           int accumulate, int ldy, const int* __restrict__ count,
                                                           unsigned long long parts_of) {
  const int quads = N / 4, used = *count;
  if (used == 0 || (ksplit = slices_for(used, ksplit, parts_of)) == 1) return;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)T * quads) return;
  const int row = (int)(i / quads), c = (int)(i % quads) * 4;
  f4_t v = *(const f4_t*)(part + (size_t)row * N + c);
  for (int s = 1; s < ksplit; ++s) v += *(const f4_t*)(part + ((size_t)s * T + row) * N + c);
  _Float16* yp = y + (size_t)row * ldy + c;
  if (accumulate) {
    const h4_t old = *(const h4_t*)yp;
    v += (f4_t){(float)old[0], (float)old[1], (float)old[2], (float)old[3]};
  }
  *(h4_t*)yp = (h4_t){(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}

__global__ __launch_bounds__(1024) void dz_build_mixed_kernel(const int* __restrict__ seg_off, const int* __restrict__ perm,
                                                              int S, int most, int deltas, int* __restrict__ count,
                                                              dz_mixed_block* __restrict__ blocks, int max_blocks) {
  extern __shared__ int off[];
  for (int k = threadIdx.x; k < S + 2; k += 1024) off[k] = seg_off[k];
  dz_build_mixed_blocks(off, perm, S, most, deltas, count, blocks, max_blocks);
}

// The order and the table in one launch, for a call that has to make its own: on a few hundred tokens two kernels are over
// long before the host has launched them (a call over a small layer 44 -> 37 us, bound by the host's half either way).
__global__ __launch_bounds__(1024) void dz_order_mixed_kernel(const long long* idx, int T, int S, int most, int deltas, int* perm,
                                                              int* count, dz_mixed_block* blocks, int max_blocks, unsigned* status) {
  extern __shared__ int sm[];
  dz_segment_tokens(idx, T, S, perm, status, sm);
  dz_build_mixed_blocks(sm, perm, S, most, deltas, count, blocks, max_blocks);
}

}  // namespace

// Estimated us of a batch in so many blocks and slices of K: 5 for a workgroup's start; a slab of 64 columns 0.9 and
// 0.08 per tile of 16 tokens with all CUs busy, three quarters of it on an idle GPU; up to two waves of workgroups one after the
// other, more of them half a wave longer than their number; the second launch, and its pass over the sums at 4 TB/s.
// Fitted to 307 projections of 129 to 512 tokens, each timed with 1, 2, 3, 4 and 6 slices: the best by it
// takes 0.3 % longer in the mean than the best there is, 14 % at worst (of 700 others 1.3 % and 44 %); with the number of blocks taken to be T / 128 it was
// 6 % and 63 %, for where blocks fill the GPU a little more than once, one more of them is another wave.
// 333 tokens in four blocks, 1 / 2 / 3 / 4 / 6 slices: 13824 x 5120 214 125 100 129 110 us, 5120 x 27648 218 236 245 245 301.
struct MixedCost {
  int T, steps, wide;
  float pass;                                      // over the sums, per slice
  MixedCost(int T_, int K, int N) : T(T_), steps(K / DZ_KBLOCK), wide((N + MN - 1) / MN), pass(2e-6f * (float)T_ * (float)N) {}
  float slab(int blocks) const {
    const int tiles = (T + 24 * blocks - 1) / (16 * blocks), most = MROWS / 16;   // (a segment ends half a tile early)
    return 0.9f + 0.08f * (float)(tiles < most ? tiles : most);
  }
  float us(int blocks, float slab_us, int walk_slabs, int ksplit) const {
    const float full = (float)(wide * blocks) * (float)ksplit / 256.f;
    const float walk = (float)walk_slabs * slab_us * (0.75f + 0.25f * (full < 1.f ? full : 1.f));
    const float all = (5.f + walk) * (full <= 1.f ? 1.f : full <= 2.f ? 2.f : full + 0.5f);
    return ksplit == 1 ? all : all + 4.f + pass * (float)ksplit;
  }
  int walk_slabs(int ksplit) const { return 4 * ((steps + ksplit - 1) / ksplit); }
};

extern "C" float dz_mixed_us(int T, int K, int N, int blocks, int ksplit) {
  if (T < 1 || K < DZ_KBLOCK || N < 1 || blocks < 1 || ksplit < 1 || ksplit > K / DZ_KBLOCK) return 0.f;
  const MixedCost c(T, K, N);
  return c.us(blocks, c.slab(blocks), c.walk_slabs(ksplit), ksplit);
}

// Slices of K for `first` blocks, `first` + 1, .. : `usual`, but where another number is estimated to take a tenth and 3 us
// less.  (Up to 80 estimates, on the host's path: nothing is divided twice.)  One copy of this code, so that whoever asks for
// the parts of the same sizes gets the same.
__attribute__((noinline)) static void parts_for(int T, int K, int N, int first, int count, int usual, int* parts) {
  constexpr int NK = 5;
  const MixedCost c(T, K, N);
  const int ks[NK] = {1, 2, 3, 4, 6};
  int walks[NK];
  for (int i = 0; i < NK; ++i) walks[i] = ks[i] <= c.steps ? c.walk_slabs(ks[i]) : 0;
  const int walk = c.walk_slabs(usual);
  for (int n = 0; n < count; ++n) {
    const int blocks = first + n;
    const float slab = c.slab(blocks), now = c.us(blocks, slab, walk, usual);
    float least = now;
    int best = usual;
    for (int i = 0; i < NK && walks[i]; ++i) {
      const float us = c.us(blocks, slab, walks[i], ks[i]);
      if (us < least) {
        least = us;
        best = ks[i];
      }
    }
    parts[n] = least < 0.9f * now && least < now - 3.f ? best : usual;
  }
}

extern "C" int dz_mixed_parts(int T, int K, int N, int blocks, int usual) {
  if (T < 1 || K < DZ_KBLOCK || N < 1 || blocks < 1 || usual < 1 || usual > K / DZ_KBLOCK) return usual;
  int parts;
  parts_for(T, K, N, blocks, 1, usual, &parts);
  return parts;
}

// Slices of K by the sizes alone: `usual`, but another number (`only` this one, or 0: any) where it is faster for each number of
// blocks from `few` to `many` and a tenth faster in their mean; the one that saves the largest share.
extern "C" int dz_mixed_parts_between(int T, int K, int N, int few, int many, int usual, int only) {
  if (T < 1 || K < DZ_KBLOCK || N < 1 || few < 1 || usual < 1 || usual > K / DZ_KBLOCK) return usual;
  const MixedCost c(T, K, N);
  const int walk = c.walk_slabs(usual);
  int best = usual;
  double share = 0.9;
  for (int ksplit : {1, 2, 3, 4, 6}) {
    if (ksplit > c.steps || ksplit == usual || (only && ksplit != only)) continue;
    const int walk_k = c.walk_slabs(ksplit);
    double sum = 0., sum_usual = 0.;
    bool faster = true;
    for (int b = few; b <= many && faster; ++b) {
      const float slab = c.slab(b), us = c.us(b, slab, walk_k, ksplit), now = c.us(b, slab, walk, usual);
      faster = us < now;
      sum += us;
      sum_usual += now;
    }
    if (faster && sum < share * sum_usual) {
      share = sum / sum_usual;
      best = ksplit;
    }
  }
  return best;
}

// Where the device picks: 4 bits of parts for each of 1 to 16 blocks, and the most of them, which is what the partial sums
// need room for.
struct MixedPick {
  unsigned long long parts_of = 0;
  int most = 1;
  int parts(int blocks) const { return (int)(parts_of >> (4 * (blocks - 1))) & 15; }
};
static MixedPick pick_parts(int T, int K, int N, int usual) {
  MixedPick pick;
  const int fewest = T < 16 * MROWS ? (T + MROWS - 1) / MROWS : 16;
  int each[16];
  parts_for(T, K, N, fewest, 17 - fewest, usual, each + fewest - 1);
  for (int b = 1; b <= 16; ++b) {
    const int parts = each[b < fewest ? fewest - 1 : b - 1];
    pick.parts_of |= (unsigned long long)parts << (4 * (b - 1));
    pick.most = parts > pick.most ? parts : pick.most;
  }
  return pick;
}

extern "C" int dz_mixed_most_parts(int T, int K, int N, int usual) {
  if (T < 1 || K < DZ_KBLOCK || N < 1 || usual < 1 || usual > K / DZ_KBLOCK || usual > 15) return usual;
  return pick_parts(T, K, N, usual).most;
}

// Tiles are at most T / 16 and one more per segment; the blocks that are less than half full are those ended
// by their number of deltas, the last one, and the last one without deltas.
extern "C" int dz_mixed_blocks(int T, int S, int tiles, int deltas) {
  if (T < 1 || S < 0 || tiles < 1 || tiles > MROWS / 16 || deltas < 1 || deltas > DZ_MIXED_DELTAS) return 0;
  const int segments = S + 1 < T ? S + 1 : T, all = T / 16 + segments;
  return (2 * all + tiles - 1) / tiles + segments / deltas + 2;
}

extern "C" int dz_build_mixed(const int32_t* seg_off, const int32_t* perm, int S, int T, int tiles, int deltas, int32_t* table,
                              int max_blocks, void* stream) {
  if (!seg_off || !table) return DZ_EINVAL;
  if (S < 0 || S > DZ_MAX_SLOTS_SEGMENT || T < 1) return DZ_ESHAPE;
  const int need = dz_mixed_blocks(T, S, tiles, deltas);
  if (need < 1 || max_blocks < need) return DZ_ESHAPE;
  hipLaunchKernelGGL(dz_build_mixed_kernel, dim3(1), dim3(1024), (size_t)(S + 2) * 4, (hipStream_t)stream, seg_off,
                     perm, S, tiles, deltas, table, (dz_mixed_block*)(table + DZ_MIXED_HEADER), max_blocks);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

extern "C" int dz_order_mixed(const int64_t* indices, int T, int S, int tiles, int deltas, int32_t* perm, int32_t* table,
                              int max_blocks, uint32_t* status, void* stream) {
  if (!indices || !perm || !table) return DZ_EINVAL;
  if (S < 0 || S > DZ_MAX_SLOTS_SEGMENT || T < 1) return DZ_ESHAPE;
  const int need = dz_mixed_blocks(T, S, tiles, deltas);
  if (need < 1 || max_blocks < need) return DZ_ESHAPE;
  hipLaunchKernelGGL(dz_order_mixed_kernel, dim3(1), dim3(1024), dz_segment_lds(S), (hipStream_t)stream, (const long long*)indices,
                     T, S, tiles, deltas, perm, table, (dz_mixed_block*)(table + DZ_MIXED_HEADER), max_blocks, status);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

extern "C" int dz_multi_delta_gemm_mixed(const uint16_t* x, const uint16_t* w_base, int w_tiled, const void* codes_stacked,
                                         const void* meta_stacked, const void* scales_stacked, int S, int bits,
                                         int group_size, const int32_t* table, int max_blocks, int deltas,
                                         uint16_t* y, int T, int K, int N, int accumulate, int ldy,
                                         int ksplit, float* partials, void* stream) {
  if (!x || !w_base || !y || !table || max_blocks < 1 || S < 1) return DZ_EINVAL;
  if (!codes_stacked || !meta_stacked || !scales_stacked) return DZ_EINVAL;
  size_t cb, mb, sb;
  int rc = dz_native_sizes(K, N, bits, group_size, &cb, &mb, &sb);
  if (rc) return rc;
  const int gs = (group_size == -1 || group_size == K) ? K : group_size;
  if (T < 1 || ldy < N || ldy % 4) return DZ_ESHAPE;
  if (ksplit == 0 || ksplit > K / DZ_KBLOCK || ksplit < -K / DZ_KBLOCK || ksplit < -15) return DZ_ESHAPE;
  if (deltas < 1 || deltas > (bits == 2 && gs == K ? DZ_MIXED_DELTAS : 3)) return DZ_ESHAPE;
  const int tiles_n = (N + MN - 1) / MN;
  int most = ksplit;                               // slices of K
  unsigned long long parts_of = 0, units = (unsigned long long)ksplit * (unsigned)max_blocks;
  if (ksplit < 0) {                                // the device picks: room and workgroups for the most there can be
    const MixedPick pick = pick_parts(T, K, N, -ksplit);
    most = pick.most;
    parts_of = pick.parts_of;
    units = 0;
    for (int used = 1; used <= 16 && used <= max_blocks; ++used) {
      const unsigned long long u = (unsigned long long)pick.parts(used) * (unsigned)(used == 16 ? max_blocks : used);
      units = u > units ? u : units;
    }
    ksplit = 0;
  }
  units *= (unsigned)tiles_n;
  if (most > 1 && !partials) return DZ_EWORKSPACE;
  if (((uintptr_t)x & 15) || ((uintptr_t)w_base & 15) || ((uintptr_t)y & 7) || ((uintptr_t)partials & 15)) return DZ_EALIGN;
  if ((unsigned long long)T * (unsigned)K * 2ull >= (1ull << 31)) return DZ_ESHAPE;   // 32-bit row offsets
  MixedParams P{};
  P.x = (const _Float16*)x; P.w = (const _Float16*)w_base; P.y = (_Float16*)y;
  P.codes = (const u4_t*)codes_stacked; P.meta = (const u4_t*)meta_stacked; P.scales = (const _Float16*)scales_stacked;
  P.meta_slot_u4 = (long long)(mb / 16); P.scales_slot = (long long)(sb / 2);
  P.count = table; P.blocks = (const dz_mixed_block*)(table + DZ_MIXED_HEADER); P.part = partials;
  P.T = T; P.K = K; P.N = N; P.G = K / gs; P.accumulate = accumulate; P.ldy = ldy;
  P.NKB = K / DZ_KBLOCK; P.NP = N / DZ_NPAIR; P.w_tiled = w_tiled ? 1 : 0; P.ksplit = ksplit; P.parts_of = parts_of;
  P.tiles_n = tiles_n;
  const unsigned gslabs = (unsigned)(gs / 64);
  P.gmagic = (unsigned)((0x100000000ull + gslabs - 1) / gslabs);   // (0 where a group is one slab)
  if (units > 0x7ffffff0ull) return DZ_ESHAPE;
  const unsigned grid = (unsigned)(units + 7) / 8 * 8;
  const int lds = 2 * XSTAGE;
  static std::atomic<unsigned long long> attr_done[4];
  auto go = [&](auto kern, int which) -> int {
    if (!dz_lds_limit_once(attr_done[which], (const void*)kern, lds)) return DZ_ELAUNCH;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * MWAVES), lds, (hipStream_t)stream, P);
    return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
  };
  const bool grp = P.G > 1;
  if (bits == 2) rc = grp ? go(dz_gemm24_mixed_kernel<2, true>, 0) : go(dz_gemm24_mixed_kernel<2, false>, 1);
  else rc = grp ? go(dz_gemm24_mixed_kernel<4, true>, 2) : go(dz_gemm24_mixed_kernel<4, false>, 3);
  if (rc || most == 1) return rc;
  const long long quads = (long long)T * (N / 4);
  hipLaunchKernelGGL(dz_mixed_sum_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, (hipStream_t)stream, partials,
                     (_Float16*)y, T, N, ksplit, accumulate, ldy, table, parts_of);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}
