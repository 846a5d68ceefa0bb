// gfx950 kernels of the multi-delta linear layer and their C ABI.
//
//   dz_dequant_kernel / merge   native delta -> fp16 [N, K] (bit-exact with the reference's
//                               QuantLinear.unpack, deltazip/nn_modules/qlinear_cuda.py:246-329)
//   dz_segment_kernel           tokens grouped by delta id
// and the host entry points of the C ABI (the fused layer kernel itself is in dz_mdl32.hip).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/dz_amd.h"
#include "../../include/dz_amd_tuning.h"
#include <atomic>

#include "dz_device.h"
#include "dz_tables.h"

namespace {

// ---------------------------------------------------------------------------------------------
// dequant / merge: one wavefront per (n-pair, k-block) tile, transposed through LDS so that the
// fp16 rows leave as 512-byte runs.
// ---------------------------------------------------------------------------------------------
template <int BITS, bool MERGE>
__global__ __launch_bounds__(64) void dz_dequant_kernel(const uint32_t* __restrict__ codes,
                                                        const uint32_t* __restrict__ meta,
                                                        const _Float16* __restrict__ scales,
                                                        const _Float16* __restrict__ wbase,
                                                        _Float16* __restrict__ out, int K, int N,
                                                        int gs) {
  constexpr int LDT = DZ_KBLOCK + 8;  // padded row of the LDS tile, in halves
  __shared__ __attribute__((aligned(16))) _Float16 tile[DZ_NPAIR * LDT];
  const int nkb = K / DZ_KBLOCK;
  const int np = blockIdx.x / nkb, kb = blockIdx.x % nkb;
  const int la = threadIdx.x, ga = la >> 4, i = la & 15;
  const int zp = 1 << (BITS - 1);
  const u4_t m4 = *(const u4_t*)(meta + dz_meta_word(np, kb, la, 0, nkb));
  u4_t c4[2];
  if (BITS == 2) {
    c4[0] = *(const u4_t*)(codes + dz_code2_word(np, kb, la, 0, nkb));
    c4[1] = c4[0];
  } else {
    c4[0] = *(const u4_t*)(codes + dz_code4_word(np, kb, la, 0, 0, nkb));
    c4[1] = *(const u4_t*)(codes + dz_code4_word(np, kb, la, 2, 0, nkb));
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t mw = m4[j];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int n = np * DZ_NPAIR + 16 * s + i;
      const int g = (kb * DZ_KBLOCK + 64 * j) / gs;
      const float sc = (float)scales[(size_t)g * N + n];
      uint32_t cw;
      if (BITS == 2) cw = c4[0][j];
      else cw = c4[j >> 1][2 * (j & 1) + s];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        h4_t v = {(_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const int e = 2 * p + w;
          const int pos = (mw >> dz_meta_shift(s, e)) & 3;
          int q;
          if (BITS == 2) q = (cw >> dz_code2_shift(s, e)) & 3;
          else q = (cw >> dz_code4_shift(e)) & 15;
          // one exact fp32 product, one round-to-nearest-even to fp16
          const _Float16 val = (_Float16)(sc * (float)(q - zp));
          // a kept column whose code is the zero-point must not hide a value already placed
          // (positions are distinct, so plain selects suffice)
          v[0] = pos == 0 ? val : v[0];
          v[1] = pos == 1 ? val : v[1];
          v[2] = pos == 2 ? val : v[2];
          v[3] = pos == 3 ? val : v[3];
        }
        *(h4_t*)(tile + (16 * s + i) * LDT + 64 * j + dz_group_k0(ga, p)) = v;
      }
    }
  }
  __syncthreads();
  // 32 rows x 512 bytes: lane -> (row half, 16-byte chunk)
#pragma unroll
  for (int it = 0; it < 16; ++it) {
    const int row = it * 2 + (la >> 5), ch = la & 31;
    h8_t v = *(const h8_t*)(tile + row * LDT + ch * 8);
    const size_t o = (size_t)(np * DZ_NPAIR + row) * K + kb * DZ_KBLOCK + ch * 8;
    if (MERGE) {
      h8_t b = *(const h8_t*)(wbase + o);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (_Float16)((float)b[e] + (float)v[e]);
    }
    *(h8_t*)(out + o) = v;
  }
}

// ---------------------------------------------------------------------------------------------
// segment: stable counting sort of tokens by delta id.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void dz_segment_kernel(const long long* __restrict__ idx, int T,
                                                          int S, int* __restrict__ perm,
                                                          int* __restrict__ seg_off, unsigned* status) {
  extern __shared__ int sm[];
  dz_segment_tokens(idx, T, S, perm, status, sm);
  for (int s = threadIdx.x; s < S + 2; s += 1024) seg_off[s] = sm[s];
}

// ---------------------------------------------------------------------------------------------
// delta id -> slot index for every token and every sampled row (the manager's index tensors).
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void dz_map_ids_kernel(const long long* __restrict__ token_ids, int T,
                                                         const long long* __restrict__ prompt_ids, int P,
                                                         const long long* __restrict__ slot_ids, int S,
                                                         long long pad_slot, long long vocab,
                                                         long long extra_vocab,
                                                         long long* __restrict__ base_indices,
                                                         long long* __restrict__ sampler_indices,
                                                         long long* __restrict__ sampler_padded,
                                                         long long* __restrict__ emb_indices, int ld_emb,
                                                         int* __restrict__ n_missing) {
  extern __shared__ long long table[];
  for (int s = threadIdx.x; s < S; s += 256) table[s] = slot_ids[s];
  __syncthreads();
  const int i = blockIdx.x * 256 + threadIdx.x;
  auto find = [&](long long id, bool& missing) -> long long {
    missing = false;
    if (id <= 0) return -1;
    for (int s = 0; s < S; ++s)
      if (table[s] == id) return s;
    missing = true;
    return -1;
  };
  bool miss;
  if (i < T) {
    const long long id = token_ids[i];
    const long long slot = find(id, miss);
    if (miss && n_missing) atomicAdd(n_missing, 1);
    base_indices[i] = slot;
    if (emb_indices) {
      const long long e = id > 0 ? slot : 0;
      long long e0 = e * extra_vocab, e1 = e * (vocab + extra_vocab);
      emb_indices[i] = e0 == -1 ? pad_slot : e0;
      emb_indices[ld_emb + i] = e1 == -1 ? pad_slot : e1;
    }
  }
  if (i < P && sampler_indices) {
    const long long slot = find(prompt_ids[i], miss);
    if (miss && n_missing) atomicAdd(n_missing, 1);
    sampler_indices[i] = slot;
    if (sampler_padded) sampler_padded[i] = (long long)i + (slot == -1 ? pad_slot : slot) * (long long)P;
  }
}

// ---------------------------------------------------------------------------------------------
// embedding rows picked from the base table or from a delta's own table, per token.
// One workgroup per token; 16 bytes per lane and step.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void dz_embedding_select_kernel(const long long* __restrict__ tokens,
                                                                  const long long* __restrict__ idx,
                                                                  const _Float16* __restrict__ base,
                                                                  const _Float16* __restrict__ stack,
                                                                  long long stack_stride, int S, int V,
                                                                  int H, _Float16* __restrict__ out,
                                                                  int ldo) {
  const int t = blockIdx.x;
  const long long tok = tokens[t];
  const long long id = idx[t];
  const _Float16* table = (id >= 0 && id < S) ? stack + id * stack_stride : base;
  u4_t* dst = (u4_t*)(out + (size_t)t * ldo);
  const bool valid = tok >= 0 && tok < V && table != nullptr;
  const u4_t* src = (const u4_t*)(table + (valid ? (size_t)tok * H : 0));
  for (int c = threadIdx.x; c < H / 8; c += 256) {
    u4_t v = {0u, 0u, 0u, 0u};
    if (valid) v = src[c];
    dst[c] = v;
  }
}

// ---------------------------------------------------------------------------------------------
// compressor: fp32 delta [N, K] -> symmetric scales, 2:4 magnitude pruning, codes, native layout
// ---------------------------------------------------------------------------------------------
// Min / max of a scale group, then the symmetric parameters of deltazip/core/quant.py:69-83
// (perchannel, sym): the range is widened to [-m, m] when the group has a negative value, an
// all-zero group gets [-1, 1], scale = (xmax - xmin) / maxq.
__device__ __forceinline__ void minmax4(float& mn, float& mx, f4_t v) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    mn = fminf(mn, v[e]);
    mx = fmaxf(mx, v[e]);
  }
}

__device__ __forceinline__ float symmetric_scale(float mn, float mx, float maxq) {
  float xmin = mn, xmax = fmaxf(fabsf(mn), mx);
  if (xmin < 0.f) xmin = -xmax;
  if (xmin == 0.f && xmax == 0.f) {
    xmin = -1.f;
    xmax = 1.f;
  }
  return (xmax - xmin) / maxq;
}

// Long groups: one wavefront per (row, group), four requests in flight per lane.
__global__ __launch_bounds__(64) void dz_scales_kernel(const float* __restrict__ delta, int K, int N, int gs,
                                                       int G, float maxq, float* __restrict__ scale32,
                                                       _Float16* __restrict__ scale16) {
  const int row = blockIdx.x / G, g = blockIdx.x % G, lane = threadIdx.x;
  const float* p = delta + (size_t)row * K + (size_t)g * gs;
  float mn = 0.f, mx = 0.f;
  int c = lane * 4;
  for (; c + 768 < gs; c += 1024) {
    f4_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *(const f4_t*)(p + c + 256 * u);
#pragma unroll
    for (int u = 0; u < 4; ++u) minmax4(mn, mx, v[u]);
  }
  for (; c < gs; c += 256) minmax4(mn, mx, *(const f4_t*)(p + c));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o));
    mx = fmaxf(mx, __shfl_xor(mx, o));
  }
  if (lane == 0) {
    const float sc = symmetric_scale(mn, mx, maxq);
    scale32[(size_t)g * N + row] = sc;
    scale16[(size_t)g * N + row] = (_Float16)sc;
  }
}

// Groups of 64, 128 or 256 columns: a wavefront takes the groups of 256 columns of a row at once, GS / 4
// lanes each, for up to four such stretches (one wavefront per group leaves half or three quarters
// of its lanes idle, and starts N * G wavefronts).
template <int GS>
__global__ __launch_bounds__(64) void dz_scales_short_kernel(const float* __restrict__ delta, int K, int N, float maxq,
                                                             float* __restrict__ scale32, _Float16* __restrict__ scale16) {
  const int lane = threadIdx.x, nc = K / 256, per_row = (nc + 3) / 4;
  const int row = blockIdx.x / per_row, c0 = (blockIdx.x % per_row) * 4;
  const float* p = delta + (size_t)row * K + lane * 4;
  f4_t v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = *(const f4_t*)(p + min(c0 + u, nc - 1) * 256);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    if (c0 + u >= nc) break;
    float mn = 0.f, mx = 0.f;
    minmax4(mn, mx, v[u]);
#pragma unroll
    for (int o = GS / 8; o > 0; o >>= 1) {
      mn = fminf(mn, __shfl_xor(mn, o));
      mx = fmaxf(mx, __shfl_xor(mx, o));
    }
    if ((lane & (GS / 4 - 1)) == 0) {
      const float sc = symmetric_scale(mn, mx, maxq);
      const size_t at = (size_t)((c0 + u) * (256 / GS) + lane / (GS / 4)) * N + row;
      scale32[at] = sc;
      scale16[at] = (_Float16)sc;
    }
  }
}

void launch_scales(const float* delta, int K, int N, int bits, int gs, float* scale32, uint16_t* scale16, hipStream_t st) {
  const float maxq = (float)((1 << bits) - 1);
  const unsigned grid = (unsigned)N * ((K / 256 + 3) / 4);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(64), 0, st, delta, K, N, maxq, scale32, (_Float16*)scale16); };
  if (gs == 64) go(dz_scales_short_kernel<64>);
  else if (gs == 128) go(dz_scales_short_kernel<128>);
  else if (gs == 256) go(dz_scales_short_kernel<256>);
  else
    hipLaunchKernelGGL(dz_scales_kernel, dim3((unsigned)N * (K / gs)), dim3(64), 0, st, delta, K, N, gs, K / gs, maxq,
                       scale32, (_Float16*)scale16);
}

// The same with the reference's grid search over the clipping range (deltazip/core/quant.py:85-101,
// mse=True, sym): for i = 0 .. int(maxshrink * grid) - 1 the range is shrunk by p = 1 - i / grid,
// the group is rounded to that grid and the candidate with the smallest sum of |q(x) - x|^norm
// wins (the first one on a tie: `err < best`).  One wavefront per (row, scale group); the group
// is re-read from cache for every candidate; sums: fp32 per lane in element order, then a
// butterfly over the lanes.
__global__ __launch_bounds__(64) void dz_scales_mse_kernel(const float* __restrict__ delta, int K, int N, int gs,
                                                           int G, float maxq, float norm, int grid, int ncand,
                                                           float* __restrict__ scale32,
                                                           _Float16* __restrict__ scale16) {
  const int row = blockIdx.x / G, g = blockIdx.x % G, lane = threadIdx.x;
  const float* p = delta + (size_t)row * K + (size_t)g * gs;
  float mn = 0.f, mx = 0.f;
  for (int c = lane * 4; c < gs; c += 256) {
    const f4_t v = *(const f4_t*)(p + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      mn = fminf(mn, v[e]);
      mx = fmaxf(mx, v[e]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o));
    mx = fmaxf(mx, __shfl_xor(mx, o));
  }
  float xmin = mn, xmax = fmaxf(fabsf(mn), mx);
  if (xmin < 0.f) xmin = -xmax;
  if (xmin == 0.f && xmax == 0.f) {
    xmin = -1.f;
    xmax = 1.f;
  }
  const float zero = (maxq + 1.f) * 0.5f;
  float best = INFINITY, best_scale = (xmax - xmin) / maxq;
  for (int i = 0; i < ncand; ++i) {
    const float pf = (float)(1.0 - (double)i / (double)grid);
    const float sc = __fsub_rn(__fmul_rn(pf, xmax), __fmul_rn(pf, xmin)) / maxq;   // every product rounded, as the reference's tensor ops
    float err = 0.f;
    for (int c = lane * 4; c < gs; c += 256) {
      const f4_t v = *(const f4_t*)(p + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float q = fminf(fmaxf(rintf(v[e] / sc) + zero, 0.f), maxq);
        err += powf(fabsf(__fsub_rn(__fmul_rn(sc, q - zero), v[e])), norm);
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) err += __shfl_xor(err, o);
    if (err < best) {
      best = err;
      best_scale = sc;
    }
  }
  if (lane == 0) {
    scale32[(size_t)g * N + row] = best_scale;
    scale16[(size_t)g * N + row] = (_Float16)best_scale;
  }
}

// One workgroup per (n-pair, k-block) tile; the words of lane 16*ga + i of the native arrays hold
// rows i and 16 + i, columns 64*j + 16*ga .. + 15 of the k-block (word j).
//   pruning   in every aligned group of 4 columns the 2 values of largest magnitude stay (ties:
//             the lower column), the others become 0 -- deltazip/core/sparsegpt.py:123-135 with an
//             identity Hessian
//   codes     q = clamp(rint(x / scale) + zero, 0, maxq), fp32, zero = 2^(bits-1) -- quant.py:9-18
//   positions the columns whose code differs from the zero-point, completed with the lowest
//             remaining columns: what the repacker stores for the same codes
// Bound by memory (4096 x 11008, per channel, the pass for the scales included: 96 us with a lane reading
// its own 64 bytes of a row, 64 with the reads below and one wavefront per tile, 60 now), and at a few
// hundred tiles by the chain of one wavefront's rows: with all 32 rows in one, 768 x 640 in groups of 128
// took 33 us, where the separate passes for scales and codes before it took 21; four wavefronts of
// 8 rows 17.
//
// The work of a group of four: six comparisons (a value stays if at least two of its three
// comparisons go its way), four quotients as products with 1 / scale, and two table lookups on
// 4-bit masks.  A quotient's rounding is that of the division unless it lies within 1e-5 of half
// way between two codes (the product is off by 1.5 units in the last place, 1e-6 below 8.5; beyond
// that both are clamped alike); such a group, one with a NaN, or a scale outside [2^-100, 2^100] goes
// the plain way: compress_group_plain.
template <int BITS>
__device__ __forceinline__ void compress_group_plain(const f4_t v, float sc, uint32_t& pos, uint32_t& clo, uint32_t& chi) {
  constexpr int zp = 1 << (BITS - 1);
  constexpr float maxq = (float)((1 << BITS) - 1);
  int c[4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    int rank = 0;   // entries ahead of a: larger magnitude, or equal magnitude at a lower column
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if (b != a) rank += (b > a) ? (fabsf(v[b]) > fabsf(v[a])) : (fabsf(v[b]) >= fabsf(v[a]));
    const float x = rank < 2 ? v[a] : 0.f;
    const float qf = fminf(fmaxf(rintf(x / sc) + (float)zp, 0.f), maxq);
    c[a] = (int)qf;
  }
  int pa = -1, pb = -1;
#pragma unroll
  for (int a = 0; a < 4; ++a)
    if (c[a] != zp) {
      if (pa < 0) pa = a;
      else if (pb < 0) pb = a;
    }
#pragma unroll
  for (int a = 0; a < 4; ++a)
    if (c[a] == zp) {
      if (pa < 0) pa = a;
      else if (pb < 0) pb = a;
    }
  const int lo = min(pa, pb), hi = max(pa, pb);
  pos = (uint32_t)(lo | hi << 2);
  clo = (uint32_t)(lo == 0 ? c[0] : lo == 1 ? c[1] : c[2]);
  chi = (uint32_t)(hi == 1 ? c[1] : hi == 2 ? c[2] : c[3]);
}

// lo | hi << 2 of a mask of at most two columns, completed with the lowest others: entry `mask` of
// a table of 4-bit entries (0, 1, 2, 4, 8: (0,1) (0,1) (0,1) (0,2) (0,3); 3, 5, 9, 6, 10, 12: themselves)
constexpr unsigned long long kept_table() {
  unsigned long long t = 0;
  for (int m = 0; m < 16; ++m) {
    int p[4] = {0, 0, 0, 0}, n = 0;
    for (int a = 0; a < 4; ++a)
      if (m >> a & 1) p[n++] = a;
    if (n > 2) continue;
    for (int a = 0; a < 4 && n < 2; ++a)
      if (!(m >> a & 1)) p[n++] = a;
    const int lo = p[0] < p[1] ? p[0] : p[1], hi = p[0] < p[1] ? p[1] : p[0];
    t |= (unsigned long long)(lo | hi << 2) << (4 * m);
  }
  return t;
}

template <int BITS>
__device__ __forceinline__ void compress_group(const f4_t v, float sc, float rsc, uint32_t& pos, uint32_t& clo, uint32_t& chi) {
  constexpr int zp = 1 << (BITS - 1);
  constexpr float maxq = (float)((1 << BITS) - 1);
  constexpr unsigned long long TABLE = kept_table();
  float r[4], far = 0.f, sum = 0.f;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const float q = v[a] * rsc;
    r[a] = rintf(q);
    far = fmaxf(far, fabsf(q - r[a]));
    sum += fabsf(q);
  }
  if (!(far < 0.49999f && sum == sum)) {
    compress_group_plain<BITS>(v, sc, pos, clo, chi);
    return;
  }
  const float m0 = fabsf(v[0]), m1 = fabsf(v[1]), m2 = fabsf(v[2]), m3 = fabsf(v[3]);
  const bool b01 = m0 >= m1, b02 = m0 >= m2, b03 = m0 >= m3, b12 = m1 >= m2, b13 = m1 >= m3, b23 = m2 >= m3;
  auto two_of = [](bool a, bool b, bool c) { return (a && b) || (c && (a || b)); };
  const bool keep[4] = {two_of(b01, b02, b03), two_of(!b01, b12, b13), two_of(!b02, !b12, b23), two_of(!b03, !b13, !b23)};
  uint32_t mask = 0, c = 0;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const float x = keep[a] ? r[a] : 0.f;
    mask |= x != 0.f ? 1u << a : 0u;
    c |= (uint32_t)fminf(fmaxf(x + (float)zp, 0.f), maxq) << (4 * a);
  }
  const uint32_t half = mask & 8u ? (uint32_t)(TABLE >> 32) : (uint32_t)TABLE;
  pos = (half >> (4 * (mask & 7u))) & 15u;
  clo = (c >> (4 * (pos & 3u))) & 15u;
  chi = (c >> (4 * (pos >> 2))) & 15u;
}

// A lane reads one group of four of a row, the wavefront 1 KiB of a row at a time (with the lane of
// the native layout reading its own 64 bytes of a row, every lane's request falls on a line of its
// own: 4096 x 11008 at 2 bits 76 us at any amount of arithmetic).  The four lanes that share a word
// of the layout or their bits together, and the words meet in LDS.
__device__ __forceinline__ uint32_t or_quad(uint32_t v) {
  v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true);          // lane ^ 1
  return v | (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xf, 0xf, true);    // lane ^ 2
}

//
// GS = 0: scales from memory (groups of another length, and whole rows of more than 16384 columns).  GS = 64, 128, 256: the tile holds whole scale groups, so their scales are
// found here from the values just read (and written out) rather than in a pass of their own
// (4096 x 11008, 4-bit, groups of 128: 90 us with one wavefront per tile, now 75, of 64 88 and 74).
constexpr int COMPRESS_WAVES = 4;   // per tile: rows 4w .. 4w + 3 and 16 + 4w .. of wavefront w

template <int BITS, int GS>
__global__ __launch_bounds__(64 * COMPRESS_WAVES) void dz_compress_kernel(const float* __restrict__ delta,
                                                         float* __restrict__ scale32, _Float16* __restrict__ scale16,
                                                         int K, int N, int gs, uint32_t* __restrict__ codes,
                                                         uint32_t* __restrict__ meta) {
  constexpr int GL = GS ? GS / 4 : 64;             // lanes per scale group
  constexpr int NW = 1 + BITS / 2;                 // words per (lane of the layout, step): positions, codes
  __shared__ __attribute__((aligned(16))) uint32_t words[NW * 256];   // as in memory: meta, then codes
  __shared__ float2 sct[DZ_NPAIR * 4];             // (scale, 1 / scale or NaN) of (row, step)
  const int nkb = K / DZ_KBLOCK;
  const int np = blockIdx.x / nkb, kb = blockIdx.x % nkb;
  const int tid = threadIdx.x, lane = tid & 63, j = lane >> 4, ga = (lane >> 2) & 3, p = lane & 3;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (GS == 0 && tid < 4 * DZ_NPAIR) {
    const int row = tid & 31, step = tid >> 5;      // (a scale group spans whole steps)
    const float sc = scale32[(size_t)((kb * DZ_KBLOCK + step * 64) / gs) * N + np * DZ_NPAIR + row];
    sct[step * DZ_NPAIR + row] = make_float2(sc, sc >= 0x1p-100f && sc <= 0x1p100f ? 1.f / sc : __builtin_nanf(""));
  }
  const float* src = delta + (size_t)np * DZ_NPAIR * K + kb * DZ_KBLOCK + lane * 4;
  // lane p of four stores the positions (0), the codes (1), or the codes of row 16 + i at 4 bits (2)
  const int hold = p == 0 ? j : BITS == 2 ? 256 + j : 256 + (j >> 1) * 256 + 2 * (j & 1) + (p - 1);
  __syncthreads();
  {
    const int i0 = 4 * wave;
    f4_t v[2][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s) v[s][u] = *(const f4_t*)(src + (size_t)(16 * s + i0 + u) * K);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      uint32_t mw = 0, cw[2] = {0, 0};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        float2 sc;
        if constexpr (GS != 0) {
          const f4_t w = v[s][u];
          float top = fmaxf(fmaxf(fabsf(w[0]), fabsf(w[1])), fmaxf(fabsf(w[2]), fabsf(w[3])));
#pragma unroll
          for (int o = GL / 2; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
          const unsigned long long neg = __ballot(w[0] < 0.f || w[1] < 0.f || w[2] < 0.f || w[3] < 0.f);
          const bool any_neg = ((neg >> (lane & ~(GL - 1))) & (~0ull >> (64 - GL))) != 0;
          top = fmaxf(top, 0.f);                   // (all NaN: as a group without a value)
          sc.x = symmetric_scale(any_neg ? -top : 0.f, top, (float)((1 << BITS) - 1));
          sc.y = sc.x >= 0x1p-100f && sc.x <= 0x1p100f ? 1.f / sc.x : __builtin_nanf("");
          if ((lane & (GL - 1)) == 0) sct[lane / GL * DZ_NPAIR + 16 * s + i0 + u].x = sc.x;
        } else {
          sc = sct[j * DZ_NPAIR + 16 * s + i0 + u];
        }
        uint32_t pos, clo, chi;
        compress_group<BITS>(v[s][u], sc.x, sc.y, pos, clo, chi);
        mw |= pos << dz_meta_shift(s, 2 * p);      // elements 2p and 2p + 1 are neighbours
        if (BITS == 2) cw[0] |= (clo << dz_code2_shift(s, 2 * p)) | (chi << dz_code2_shift(s, 2 * p + 1));
        else cw[s] = (clo << dz_code4_shift(2 * p)) | (chi << dz_code4_shift(2 * p + 1));
      }
      mw = or_quad(mw);
      cw[0] = or_quad(cw[0]);
      if (BITS == 4) cw[1] = or_quad(cw[1]);
      if (p < NW) words[hold + (16 * ga + i0 + u) * 4] = p == 0 ? mw : p == 1 ? cw[0] : cw[1];
    }
  }
  __syncthreads();
  if constexpr (GS != 0) {
    constexpr int NG = DZ_KBLOCK / (GS ? GS : 1);
    if (tid < NG * DZ_NPAIR) {
      const size_t o = (size_t)(kb * NG + tid / DZ_NPAIR) * N + np * DZ_NPAIR + (tid & 31);
      scale32[o] = sct[tid].x;
      scale16[o] = (_Float16)sct[tid].x;
    }
  }
  if (wave == 3) *(u4_t*)(meta + dz_meta_word(np, kb, lane, 0, nkb)) = *(const u4_t*)(words + lane * 4);
  if (BITS == 2) {
    if (wave == 2) *(u4_t*)(codes + dz_code2_word(np, kb, lane, 0, nkb)) = *(const u4_t*)(words + 256 + lane * 4);
  } else if (wave == 2) {
    *(u4_t*)(codes + dz_code4_word(np, kb, lane, 0, 0, nkb)) = *(const u4_t*)(words + 256 + lane * 4);
  } else if (wave == 1) {
    *(u4_t*)(codes + dz_code4_word(np, kb, lane, 2, 0, nkb)) = *(const u4_t*)(words + (BITS == 2 ? 256 : 512) + lane * 4);
  }
}

// One scale per row: the values are read once.  A workgroup of eight wavefronts holds R rows of either half
// of an n-pair (rows i0 .. i0 + R - 1 and 16 + i0 ..) whole, in registers, CH k-blocks per wavefront; the
// rows' extremes meet in LDS, and the codes are made from the registers.  The words of R neighbouring rows
// are 16 * R bytes of the native arrays, written from LDS.  Bound by memory: with a pass for the scales and a
// second reading 4096 x 11008, 2 bits, 65 us, now 40 (192 MB, 4.8 TB/s); 5120 x 13824 97 -> 59, 11008 x 4096 69 -> 41,
// 2048 x 2048 18 -> 16.  R is such that a lane holds 32 values (64 where a row has more than 8192): with
// 64 values 4096 x 11008 took 48 us, with 128 5120 x 13824 110: one workgroup per CU then loads, and
// the next computes nothing beside it.
template <int BITS, int CH, int R>
__global__ __launch_bounds__(512, 2) void dz_compress_rows_kernel(const float* __restrict__ delta,
                                                                  float* __restrict__ scale32, _Float16* __restrict__ scale16,
                                                                  int K, int N, uint32_t* __restrict__ codes,
                                                                  uint32_t* __restrict__ meta) {
  constexpr int WAVES = 8, SETS = 1 + BITS / 2;    // 16-byte chunks per (row pair, 16 columns): positions, codes
  __shared__ float tops[WAVES][2 * R];             // largest magnitude; its sign: whether a value is negative
  __shared__ float2 sct[2 * R];                    // scale, 1 / scale or NaN
  __shared__ __attribute__((aligned(16))) uint32_t words[WAVES][SETS * R * 16];
  const int nkb = K / DZ_KBLOCK, per = 16 / R;
  // (the rows of an n-pair on one XCD: their words share the lines of its L2)
  const int np = (int)(blockIdx.x / (8 * per)) * 8 + (int)(blockIdx.x & 7), i0 = (int)(blockIdx.x >> 3) % per * R;
  if (np >= N / DZ_NPAIR) return;
  const int tid = threadIdx.x, lane = tid & 63, j = lane >> 4, ga = (lane >> 2) & 3, p = lane & 3;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* src = delta + ((size_t)np * DZ_NPAIR + i0) * K + lane * 4;
  f4_t v[CH][2 * R];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int r = 0; r < 2 * R; ++r)                // (beyond the row: its last k-block again, not stored)
      v[c][r] = *(const f4_t*)(src + (size_t)(r < R ? r : 16 + r - R) * K + min(wave + WAVES * c, nkb - 1) * DZ_KBLOCK);
#pragma unroll
  for (int r = 0; r < 2 * R; ++r) {
    float top = 0.f;
    bool neg = false;
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        top = fmaxf(top, fabsf(v[c][r][e]));       // (a NaN has no say)
        neg = neg || v[c][r][e] < 0.f;
      }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o));
    const bool any = __ballot(neg) != 0;
    if (lane == 0) tops[wave][r] = any ? -top : top;   // (negative: top > 0)
  }
  __syncthreads();
  if (tid < 2 * R) {
    float top = 0.f;
    bool any = false;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float t = tops[w][tid];
      top = fmaxf(top, fabsf(t));
      any = any || t < 0.f;
    }
    const float sc = symmetric_scale(any ? -top : 0.f, top, (float)((1 << BITS) - 1));
    sct[tid] = make_float2(sc, sc >= 0x1p-100f && sc <= 0x1p100f ? 1.f / sc : __builtin_nanf(""));
    const int row = np * DZ_NPAIR + i0 + (tid < R ? tid : 16 + tid - R);
    scale32[row] = sc;
    scale16[row] = (_Float16)sc;
  }
  __syncthreads();
  uint32_t* const mine = words[wave];
  // lane p of four keeps the positions (0), the codes (1), or the codes of row 16 + i at 4 bits (2)
  const int set = p == 0 ? 0 : BITS == 2 ? 1 : 1 + (j >> 1), at = p == 0 || BITS == 2 ? j : 2 * (j & 1) + (p - 1);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int kb = wave + WAVES * c;
    if (kb >= nkb) break;
#pragma unroll
    for (int u = 0; u < R; ++u) {
      uint32_t mw = 0, cw[2] = {0, 0};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const float2 sc = sct[s * R + u];
        uint32_t pos, clo, chi;
        compress_group<BITS>(v[c][s * R + u], sc.x, sc.y, pos, clo, chi);
        mw |= pos << dz_meta_shift(s, 2 * p);
        if (BITS == 2) cw[0] |= (clo << dz_code2_shift(s, 2 * p)) | (chi << dz_code2_shift(s, 2 * p + 1));
        else cw[s] = (clo << dz_code4_shift(2 * p)) | (chi << dz_code4_shift(2 * p + 1));
      }
      mw = or_quad(mw);
      cw[0] = or_quad(cw[0]);
      if (BITS == 4) cw[1] = or_quad(cw[1]);
      if (p < (BITS == 2 ? 2 : 3)) mine[(set * 4 * R + ga * R + u) * 4 + at] = p == 0 ? mw : p == 1 ? cw[0] : cw[1];
    }
    __builtin_amdgcn_wave_barrier();               // (one wavefront's own words: LDS keeps its order)
    if (lane < SETS * 4 * R) {
      const int which = lane / (4 * R), q = lane % (4 * R), la = 16 * (q / R) + i0 + q % R;
      uint32_t* dst = which == 0 ? meta + dz_meta_word(np, kb, la, 0, nkb)
                                 : codes + (BITS == 2 ? dz_code2_word(np, kb, la, 0, nkb)
                                                      : dz_code4_word(np, kb, la, 2 * (which - 1), 0, nkb));
      *(u4_t*)dst = *(const u4_t*)(mine + lane * 4);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// ---------------------------------------------------------------------------------------------
// 33..128 tokens: the order in which the fused kernel takes the tokens, 32 per chunk.  Tokens of
// one delta stay together, and the chunks are made to meet about the same number of distinct
// deltas (the kernel's time per chunk grows with that number; a plain cut of the id-sorted order
// puts one popular delta alone into a chunk and all the rare ones together into another).
// The segments -- one per delta present -- are ranked by size; counting from the largest, segment
// r goes to group r mod nchunk; the groups are laid out one after the other, each smallest
// segment first, and the chunks are the 32-token cuts of that layout.  Every group holds the same
// number of segments and group g is at least as long as group g + 1, so a cut falls into the tail
// of a group: what spills into the next chunk is part of a popular delta, not several rare ones.
// One workgroup, one thread per token, everything by counting over the (at most 128) tokens: no
// per-slot table, so any number of slots is fine.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(128) void dz_deal_kernel(const long long* __restrict__ idx, int T, int S,
                                                      int* __restrict__ perm_out) {
  __shared__ __attribute__((aligned(16))) int s_key[128], s_size[128], s_dkey[128];
  __shared__ int s_pos[128], s_wcount[2];
  const int tid = threadIdx.x;
  const int nchunk = (T + 31) / 32;
  int key = 0x7fffffff;   // threads beyond T hold no token; their entries never match or count
  if (tid < T) {
    const long long id = idx[tid];
    key = (id < 0 || id >= S) ? 0 : (int)id + 1;
  }
  s_key[tid] = key;
  __syncthreads();
  // Tables are read four entries per LDS read with several reads in flight (a loop that takes one
  // entry per turn waits out the LDS latency every time).
  typedef int i4_t __attribute__((ext_vector_type(4)));
  // my segment: its size, my place in it, its first token (the segment's "leader")
  int size = 0, rin = 0, leader = tid;
#pragma unroll 8
  for (int q = 0; q < 32; ++q) {
    const i4_t v = ((const i4_t*)s_key)[q];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = 4 * q + e;
      const bool same = v[e] == key;
      size += same;
      rin += same && j < tid;
      leader = (same && j < leader) ? j : leader;
    }
  }
  const bool is_leader = tid < T && leader == tid;
  // the segments, compacted (order of their first tokens): size | first token << 8; zero-padded
  const unsigned long long lm = __builtin_amdgcn_ballot_w64(is_leader);
  const int lane = tid & 63, wave = tid >> 6;
  if (lane == 0) s_wcount[wave] = __builtin_popcountll(lm);
  s_size[tid] = 0;
  s_dkey[tid] = 0x7fffffff;
  __syncthreads();
  const int nseg = s_wcount[0] + s_wcount[1];
  const int slot = (wave ? s_wcount[0] : 0) + __builtin_popcountll(lm & ((1ull << lane) - 1ull));
  if (is_leader) s_size[slot] = size | (tid << 8);
  __syncthreads();
  const int nq = (nseg + 3) >> 2;
  // leaders: rank of the segment by (size, first token)
  int rank = 0;
  for (int q = 0; q < nq; ++q) {
    const i4_t v = ((const i4_t*)s_size)[q];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int sj = v[e] & 0xff, fj = v[e] >> 8;
      rank += v[e] != 0 && (sj < size || (sj == size && fj < tid));
    }
  }
  const int dkey = is_leader ? ((((nseg - 1 - rank) % nchunk) << 16) | rank) : 0x7fffffff;
  if (is_leader) s_dkey[slot] = dkey;
  __syncthreads();
  int pos = 0;   // tokens of the segments laid out before mine
  for (int q = 0; q < nq; ++q) {
    const i4_t d = ((const i4_t*)s_dkey)[q];
    const i4_t z = ((const i4_t*)s_size)[q];
#pragma unroll
    for (int e = 0; e < 4; ++e) pos += (d[e] < dkey) ? (z[e] & 0xff) : 0;
  }
  s_pos[tid] = pos;
  __syncthreads();
  if (tid < T) perm_out[s_pos[leader] + rin] = tid;
}

// Base weight, row-major [N, K] -> tiles (dz_layout.h: dz_base_tile_offset / dz_base_frag_offset).
// One thread moves 16 bytes: output chunk c = ((tile * 16 + fragment) * 64 + lane).
__global__ __launch_bounds__(256) void dz_tile_base_kernel(const u4_t* __restrict__ w, u4_t* __restrict__ out,
                                                           int K, int N) {
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c >= (long long)N * K / 8) return;
  const int lane = (int)(c & 63), frag = (int)((c >> 6) & 15);
  const long long tile = c >> 10;
  const int nkb = K / DZ_KBLOCK;
  const int np = (int)(tile / nkb), kb = (int)(tile % nkb);
  const int h = frag & 1, j = (frag >> 1) & 3, s = frag >> 3;
  const int i = lane & 15, g = lane >> 4;
  const long long row = (long long)np * DZ_NPAIR + 16 * s + i;
  const int col = kb * DZ_KBLOCK + 64 * j + 16 * g + 8 * h;
  out[c] = w[(row * K + col) / 8];
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
// K-slice override of the tuning hook (include/dz_amd_tuning.h): per host thread, so that a test
// or a sweep that sets it changes no other caller's launches
thread_local int g_ksplit_override = 0;

inline int check_group(int K, int group_size, int* gs_out) {
  int gs = (group_size == -1 || group_size == K) ? K : group_size;
  if (gs <= 0 || K % gs || (gs != K && gs % 64)) return DZ_EGROUP;
  *gs_out = gs;
  return DZ_OK;
}

constexpr size_t WS_HEADER = 256;  // status word
constexpr int MAX_KSPLIT = 16;
constexpr size_t WS_PERM_BYTES = 4096 + (size_t)DZ_MAX_TOKENS_FUSED * 4;   // reserved + token order

// Workspace of dz_multi_delta_linear_static: device memory that belongs to the library's code
// object (zero bits when the object is loaded; every GPU holds its own copy at its own address).
// Host code must not use the array's name as an address: it asks the runtime for the device
// address once per device (static_scratch_ptr) and passes that on.
constexpr size_t STATIC_SCRATCH_BYTES =
    WS_HEADER + WS_PERM_BYTES + (size_t)MAX_KSPLIT * 32 * (size_t)DZ_STATIC_MAX_N * 4;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::atomic<void*> g_scratch_ptr[MAX_DEVICES];

// Device address of `scratch` on the current device, looked up on the first call per device.
void* static_scratch_ptr() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return nullptr;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p) return p;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
  g_scratch_ptr[dev].store(p, std::memory_order_release);   // two racing threads store the same address
  return p;
}

}  // namespace

extern "C" {

#ifdef DZ_TIMING
void dz_set_timing_buffer(void* p) { hipMemcpyToSymbol(HIP_SYMBOL(g_dz_ts), &p, sizeof(p)); }
#endif

int dz_version(void) { return 100; }

const char* dz_strerror(int code) {
  switch (code) {
    case DZ_OK: return "ok";
    case DZ_EINVAL: return "invalid argument";
    case DZ_ESHAPE: return "unsupported shape (need K % 256 == 0, N % 32 == 0, ldy % 4 == 0, T >= 1)";
    case DZ_EBITS: return "bits must be 2 or 4";
    case DZ_EGROUP: return "group_size must be -1, K, or a multiple of 64 dividing K";
    case DZ_ENOT24: return "delta is not 2:4 sparse";
    case DZ_EZERO: return "zero-point is not 2^(bits-1) (only symmetric quantisation is supported)";
    case DZ_EGIDX: return "g_idx is not k / group_size";
    case DZ_EWORKSPACE: return "workspace missing or too small";
    case DZ_ELAUNCH: return "HIP launch failed";
    case DZ_EALIGN: return "pointer or leading dimension not aligned";
    case DZ_ESTATICMAX: return "N exceeds DZ_STATIC_MAX_N, the largest layer the library's built-in workspace serves";
    default: return "unknown error";
  }
}

void dz_set_ksplit(int nsplit) { g_ksplit_override = nsplit; }

int dz_dequant(const void* codes, const void* meta, const void* scales, int K, int N, int bits,
               int group_size, uint16_t* out, void* stream) {
  if (!codes || !meta || !scales || !out) return DZ_EINVAL;
  int rc = dz_native_sizes(K, N, bits, group_size, nullptr, nullptr, nullptr);
  if (rc) return rc;
  int gs;
  if ((rc = check_group(K, group_size, &gs))) return rc;
  const int grid = (N / DZ_NPAIR) * (K / DZ_KBLOCK);
  hipStream_t st = (hipStream_t)stream;
  if (bits == 2)
    hipLaunchKernelGGL((dz_dequant_kernel<2, false>), dim3(grid), dim3(64), 0, st, (const uint32_t*)codes,
                       (const uint32_t*)meta, (const _Float16*)scales, nullptr, (_Float16*)out, K, N, gs);
  else
    hipLaunchKernelGGL((dz_dequant_kernel<4, false>), dim3(grid), dim3(64), 0, st, (const uint32_t*)codes,
                       (const uint32_t*)meta, (const _Float16*)scales, nullptr, (_Float16*)out, K, N, gs);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_merge(const uint16_t* w_base, const void* codes, const void* meta, const void* scales, int K,
             int N, int bits, int group_size, uint16_t* out, void* stream) {
  if (!w_base || !codes || !meta || !scales || !out) return DZ_EINVAL;
  int rc = dz_native_sizes(K, N, bits, group_size, nullptr, nullptr, nullptr);
  if (rc) return rc;
  int gs;
  if ((rc = check_group(K, group_size, &gs))) return rc;
  const int grid = (N / DZ_NPAIR) * (K / DZ_KBLOCK);
  hipStream_t st = (hipStream_t)stream;
  if (bits == 2)
    hipLaunchKernelGGL((dz_dequant_kernel<2, true>), dim3(grid), dim3(64), 0, st, (const uint32_t*)codes,
                       (const uint32_t*)meta, (const _Float16*)scales, (const _Float16*)w_base,
                       (_Float16*)out, K, N, gs);
  else
    hipLaunchKernelGGL((dz_dequant_kernel<4, true>), dim3(grid), dim3(64), 0, st, (const uint32_t*)codes,
                       (const uint32_t*)meta, (const _Float16*)scales, (const _Float16*)w_base,
                       (_Float16*)out, K, N, gs);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_segment(const int64_t* indices, int T, int S, int32_t* perm, int32_t* seg_off, void* stream) {
  return dz_segment_status(indices, T, S, perm, seg_off, nullptr, stream);
}

int dz_segment_status(const int64_t* indices, int T, int S, int32_t* perm, int32_t* seg_off, uint32_t* status,
                      void* stream) {
  if (!indices || !perm || !seg_off) return DZ_EINVAL;
  if (T < 1 || S < 0 || S > DZ_MAX_SLOTS_SEGMENT) return DZ_ESHAPE;
  const size_t lds = dz_segment_lds(S);   // < 64 KiB
  hipLaunchKernelGGL(dz_segment_kernel, dim3(1), dim3(1024), lds, (hipStream_t)stream,
                     (const long long*)indices, T, S, perm, seg_off, status);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_map_ids(const int64_t* token_ids, int T, const int64_t* prompt_ids, int P,
               const int64_t* slot_ids, int S, int max_deltas, int vocab_size, int extra_vocab_size,
               int64_t* base_indices, int64_t* sampler_indices, int64_t* sampler_indices_padded,
               int64_t* embeddings_indices, int ld_emb, int32_t* n_missing, void* stream) {
  if (!token_ids || !slot_ids || !base_indices) return DZ_EINVAL;
  if (P > 0 && (!prompt_ids || !sampler_indices)) return DZ_EINVAL;
  if (T < 1 || P < 0 || S < 1 || S > DZ_MAX_SLOTS_MAP || max_deltas < 1) return DZ_ESHAPE;
  if (embeddings_indices && ld_emb < T) return DZ_ESHAPE;
  const int n = T > P ? T : P;
  hipLaunchKernelGGL(dz_map_ids_kernel, dim3((n + 255) / 256), dim3(256), (size_t)S * 8,
                     (hipStream_t)stream, (const long long*)token_ids, T, (const long long*)prompt_ids,
                     P, (const long long*)slot_ids, S, (long long)max_deltas - 1, (long long)vocab_size,
                     (long long)extra_vocab_size, (long long*)base_indices, (long long*)sampler_indices,
                     (long long*)sampler_indices_padded, (long long*)embeddings_indices, ld_emb, n_missing);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_embedding_select(const int64_t* tokens, const int64_t* indices, const uint16_t* base_weight,
                        const uint16_t* weight_stack, long long stack_stride, int S, uint16_t* out, int T,
                        int V, int H, int ldo, void* stream) {
  if (!tokens || !indices || !out || (!base_weight && !weight_stack)) return DZ_EINVAL;
  if (T < 1 || V < 1 || H < 8 || H % 8 || ldo < H || ldo % 8 || S < 0 || (S > 0 && !weight_stack)) return DZ_ESHAPE;
  if (((uintptr_t)base_weight & 15) || ((uintptr_t)weight_stack & 15) || ((uintptr_t)out & 15) ||
      (stack_stride & 7))
    return DZ_EALIGN;
  hipLaunchKernelGGL(dz_embedding_select_kernel, dim3(T), dim3(256), 0, (hipStream_t)stream,
                     (const long long*)tokens, (const long long*)indices, (const _Float16*)base_weight,
                     (const _Float16*)weight_stack, stack_stride, S, V, H, (_Float16*)out, ldo);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_compress_2of4(const float* delta, int K, int N, int bits, int group_size, void* out_codes,
                     void* out_meta, uint16_t* out_scales, float* scale_workspace, void* stream) {
  if (!delta || !out_codes || !out_meta || !out_scales || !scale_workspace) return DZ_EINVAL;
  size_t cb, mb, sb;
  int rc = dz_native_sizes(K, N, bits, group_size, &cb, &mb, &sb);
  if (rc) return rc;
  int gs;
  if ((rc = check_group(K, group_size, &gs))) return rc;
  if ((uintptr_t)delta & 15) return DZ_EALIGN;
  hipStream_t st = (hipStream_t)stream;
  const unsigned tiles = (unsigned)(N / DZ_NPAIR) * (K / DZ_KBLOCK);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(tiles), dim3(64 * COMPRESS_WAVES), 0, st, delta, scale_workspace, (_Float16*)out_scales, K, N, gs,
                       (uint32_t*)out_codes, (uint32_t*)out_meta);
  };
  switch (gs) {
    case 64: bits == 2 ? go(dz_compress_kernel<2, 64>) : go(dz_compress_kernel<4, 64>); break;
    case 128: bits == 2 ? go(dz_compress_kernel<2, 128>) : go(dz_compress_kernel<4, 128>); break;
    case 256: bits == 2 ? go(dz_compress_kernel<2, 256>) : go(dz_compress_kernel<4, 256>); break;
    default:
      if (gs == K && K <= 64 * DZ_KBLOCK) {
        // a row's k-blocks over eight wavefronts, at most eight each; the pass for the scales and the tiles are
        // left to longer rows, of which a lane would hold 128 values and more
        const int nkb = K / DZ_KBLOCK;
        auto rows = [&](auto kern, int r) {
          hipLaunchKernelGGL(kern, dim3((unsigned)((N / DZ_NPAIR + 7) / 8 * 8) * (16 / r)), dim3(512), 0, st, delta, scale_workspace,
                             (_Float16*)out_scales, K, N, (uint32_t*)out_codes, (uint32_t*)out_meta);
        };
        if (nkb <= 8) bits == 2 ? rows(dz_compress_rows_kernel<2, 1, 4>, 4) : rows(dz_compress_rows_kernel<4, 1, 4>, 4);
        else if (nkb <= 16) bits == 2 ? rows(dz_compress_rows_kernel<2, 2, 2>, 2) : rows(dz_compress_rows_kernel<4, 2, 2>, 2);
        else if (nkb <= 32) bits == 2 ? rows(dz_compress_rows_kernel<2, 4, 1>, 1) : rows(dz_compress_rows_kernel<4, 4, 1>, 1);
        else bits == 2 ? rows(dz_compress_rows_kernel<2, 8, 1>, 1) : rows(dz_compress_rows_kernel<4, 8, 1>, 1);
        break;
      }
      launch_scales(delta, K, N, bits, gs, scale_workspace, out_scales, st);
      bits == 2 ? go(dz_compress_kernel<2, 0>) : go(dz_compress_kernel<4, 0>);
  }
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_quant_scales(const float* delta, int K, int N, int bits, int group_size, float* scale32,
                    uint16_t* scale16, void* stream) {
  if (!delta || !scale32 || !scale16) return DZ_EINVAL;
  int rc = dz_native_sizes(K, N, bits, group_size, nullptr, nullptr, nullptr);
  if (rc) return rc;
  int gs;
  if ((rc = check_group(K, group_size, &gs))) return rc;
  if ((uintptr_t)delta & 15) return DZ_EALIGN;
  launch_scales(delta, K, N, bits, gs, scale32, scale16, (hipStream_t)stream);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_quant_scales_mse(const float* delta, int K, int N, int bits, int group_size, float norm, int grid,
                        float maxshrink, float* scale32, uint16_t* scale16, void* stream) {
  if (!delta || !scale32 || !scale16) return DZ_EINVAL;
  if (!(norm > 0.f) || grid < 1 || !(maxshrink >= 0.f) || maxshrink > 1.f) return DZ_EINVAL;
  int rc = dz_native_sizes(K, N, bits, group_size, nullptr, nullptr, nullptr);
  if (rc) return rc;
  int gs;
  if ((rc = check_group(K, group_size, &gs))) return rc;
  if ((uintptr_t)delta & 15) return DZ_EALIGN;
  const int G = K / gs;
  const int ncand = (int)((double)maxshrink * (double)grid);   // int(maxshrink * grid), quant.py:87
  hipLaunchKernelGGL(dz_scales_mse_kernel, dim3((unsigned)N * G), dim3(64), 0, (hipStream_t)stream, delta, K, N, gs,
                     G, (float)((1 << bits) - 1), norm, grid, ncand, scale32, (_Float16*)scale16);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_pack_2of4(const float* w, const float* scale32, int K, int N, int bits, int group_size, void* out_codes,
                 void* out_meta, void* stream) {
  if (!w || !scale32 || !out_codes || !out_meta) return DZ_EINVAL;
  int rc = dz_native_sizes(K, N, bits, group_size, nullptr, nullptr, nullptr);
  if (rc) return rc;
  int gs;
  if ((rc = check_group(K, group_size, &gs))) return rc;
  if ((uintptr_t)w & 15) return DZ_EALIGN;
  const unsigned tiles = (unsigned)(N / DZ_NPAIR) * (K / DZ_KBLOCK);
  hipStream_t st = (hipStream_t)stream;
  auto go = [&](auto kern) {                       // (scales are read only)
    hipLaunchKernelGGL(kern, dim3(tiles), dim3(64 * COMPRESS_WAVES), 0, st, w, const_cast<float*>(scale32), (_Float16*)nullptr, K, N, gs,
                       (uint32_t*)out_codes, (uint32_t*)out_meta);
  };
  bits == 2 ? go(dz_compress_kernel<2, 0>) : go(dz_compress_kernel<4, 0>);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

// workspace: [status 256 B][token order][per call: partial sums].  The partial-sum slots are
// their own "ready" marks (all zero bits = empty) and every launch leaves them empty again, so the
// workspace is zero-filled once by its owner and never again.
size_t dz_workspace_bytes(int T, int K, int N) {
  (void)K;
  if (T < 1 || N < 1) return 0;
  return WS_HEADER + WS_PERM_BYTES + (size_t)MAX_KSPLIT * 32 * (size_t)N * 4;
}

static int multi_delta_linear_batch(int ncalls, const uint16_t* const* x, const uint16_t* const* w_base,
                                    const void* const* codes_stacked, const void* const* meta_stacked,
                                    const void* const* scales_stacked, const int64_t* indices,
                                    uint16_t* const* y, const int* N, const int* ldy, int T, int K, int S,
                                    int bits, int group_size, int accumulate, const int32_t* order,
                                    void* workspace, size_t workspace_bytes, void* stream, int base_tiled,
                                    const int32_t* only_if = nullptr) {
  if (ncalls < 1 || ncalls > DZ_MAX_BATCH_CALLS) return DZ_ESHAPE;
  if (!x || !w_base || !indices || !y || !N || !ldy) return DZ_EINVAL;
  if (S > 0 && (!codes_stacked || !meta_stacked || !scales_stacked)) return DZ_EINVAL;
  const void* const none[DZ_MAX_BATCH_CALLS] = {nullptr, nullptr, nullptr, nullptr};
  if (S == 0) codes_stacked = meta_stacked = scales_stacked = none;
  if (S < 0) return DZ_EINVAL;
  if (T < 1 || T > DZ_MAX_TOKENS_FUSED) return DZ_ESHAPE;
  int gs, rc;
  if ((rc = check_group(K, group_size, &gs))) return rc;
  long long n_total = 0;
  for (int j = 0; j < ncalls; ++j) {
    size_t cb, mb, sb;
    if ((rc = dz_native_sizes(K, N[j], bits, group_size, &cb, &mb, &sb))) return rc;
    if (!x[j] || !y[j]) return DZ_EINVAL;
    // S = 0: a plain dense product with the base weight (every id counts as "no delta")
    if (S == 0 ? !w_base[j] : (!codes_stacked[j] || !meta_stacked[j] || !scales_stacked[j])) return DZ_EINVAL;
    if (ldy[j] < N[j] || ldy[j] % 4) return DZ_ESHAPE;
    if (((uintptr_t)x[j] & 15) || ((uintptr_t)y[j] & 7) || (w_base[j] && ((uintptr_t)w_base[j] & 15))) return DZ_EALIGN;
    n_total += N[j];
  }
  if (!workspace || workspace_bytes < dz_workspace_bytes(T, K, (int)n_total)) return DZ_EWORKSPACE;

  hipStream_t st = (hipStream_t)stream;
  int* perm = (int*)((char*)workspace + WS_HEADER) + 1024;
  char* region = (char*)workspace + WS_HEADER + WS_PERM_BYTES;
  MdlParams P[DZ_MAX_BATCH_CALLS];
  for (int j = 0; j < ncalls; ++j) {
    size_t cb, mb, sb;
    dz_native_sizes(K, N[j], bits, group_size, &cb, &mb, &sb);
    MdlParams& Q = P[j];
    Q.x = (const _Float16*)x[j];
    Q.wb = (const _Float16*)w_base[j];
    // The kernel issues a fixed number of requests per round; those of absent deltas re-read 16
    // bytes of slot 0.  Without slots they re-read the base weight instead (offsets stay inside
    // it: a tile index times 1 or 2 KiB is below N*K/4 bytes, the weight has 2*N*K).
    Q.codes = (const u4_t*)(S == 0 ? (const void*)w_base[j] : codes_stacked[j]);
    Q.meta = (const u4_t*)(S == 0 ? (const void*)w_base[j] : meta_stacked[j]);
    Q.scales = (const _Float16*)(S == 0 ? (const void*)w_base[j] : scales_stacked[j]);
    Q.idx = (const long long*)indices;
    Q.y = (_Float16*)y[j];
    Q.status = (unsigned*)workspace;
    Q.partials = (float*)region;
    region += (size_t)MAX_KSPLIT * 32 * (size_t)N[j] * 4;
    Q.codes_slot_u4 = (long long)(cb / 16);
    Q.meta_slot_u4 = (long long)(mb / 16);
    Q.scales_slot = (long long)(sb / 2);
    Q.T = T; Q.K = K; Q.N = N[j]; Q.S = S; Q.gs = gs; Q.G = K / gs;
    Q.accumulate = accumulate; Q.ldy = ldy[j];
    Q.NP = N[j] / DZ_NPAIR; Q.NKB = K / DZ_KBLOCK;
    Q.nsplit = 1; Q.cb = Q.NKB; Q.NPG = 0;
    Q.base_tiled = (base_tiled && w_base[j]) ? 1 : 0;
    Q.only_if = only_if;
    Q.perm = T <= 32 ? nullptr : (order ? order : perm);
    Q.tok0 = 0;
    Q.nchunk = 1;
  }
  // 0: 2-bit, one scale per row (applied to the sums); else scales applied to the operands, with
  // one request (a k-block spans at most two groups) or two (groups of 64) per delta and k-block
  const int pre = (bits == 2 && gs == K) ? 0 : (gs >= 128 ? 1 : 2);
  // 33..128 tokens: group the tokens by delta id on the device (no host round trip) and deal the
  // groups to the chunks of 32; one launch carries all chunks
  if (T > 32 && !order)
    hipLaunchKernelGGL(dz_deal_kernel, dim3(1), dim3(128), 0, st, (const long long*)indices, T, S, perm);
  return dz_launch_mdl32_batch(P, ncalls, bits, pre, st, g_ksplit_override);
}

int dz_multi_delta_linear_batch(int ncalls, const uint16_t* const* x, const uint16_t* const* w_base,
                                const void* const* codes_stacked, const void* const* meta_stacked,
                                const void* const* scales_stacked, const int64_t* indices,
                                uint16_t* const* y, const int* N, const int* ldy, int T, int K, int S,
                                int bits, int group_size, int accumulate, const int32_t* order,
                                void* workspace, size_t workspace_bytes, void* stream) {
  return multi_delta_linear_batch(ncalls, x, w_base, codes_stacked, meta_stacked, scales_stacked, indices, y, N, ldy,
                                  T, K, S, bits, group_size, accumulate, order, workspace, workspace_bytes, stream, 0);
}

int dz_multi_delta_linear_batch_tiled(int ncalls, const uint16_t* const* x, const uint16_t* const* w_base_tiled,
                                      const void* const* codes_stacked, const void* const* meta_stacked,
                                      const void* const* scales_stacked, const int64_t* indices,
                                      uint16_t* const* y, const int* N, const int* ldy, int T, int K, int S,
                                      int bits, int group_size, int accumulate, const int32_t* order,
                                      void* workspace, size_t workspace_bytes, void* stream) {
  return multi_delta_linear_batch(ncalls, x, w_base_tiled, codes_stacked, meta_stacked, scales_stacked, indices, y, N,
                                  ldy, T, K, S, bits, group_size, accumulate, order, workspace, workspace_bytes,
                                  stream, 1);
}

int dz_multi_delta_linear_ordered(const uint16_t* x, const uint16_t* w_base, int w_tiled, const void* codes_stacked,
                                  const void* meta_stacked, const void* scales_stacked, const int64_t* indices, uint16_t* y,
                                  int T, int K, int N, int S, int bits, int group_size, int accumulate, int ldy,
                                  const int32_t* order, void* workspace, size_t workspace_bytes, void* stream) {
  if (!x || !indices || !y) return DZ_EINVAL;
  return multi_delta_linear_batch(1, &x, &w_base, &codes_stacked, &meta_stacked, &scales_stacked, indices, &y, &N, &ldy, T, K, S,
                                  bits, group_size, accumulate, order, workspace, workspace_bytes, stream, w_tiled);
}

int dz_multi_delta_linear_chunks(const uint16_t* x, const uint16_t* w_base, int w_tiled, const void* codes_stacked,
                                 const void* meta_stacked, const void* scales_stacked, const int64_t* indices,
                                 uint16_t* y, int T, int K, int N, int S, int bits, int group_size, int accumulate,
                                 int ldy, const int32_t* only_if, void* workspace, size_t workspace_bytes, void* stream) {
  if (!x || !indices || !y) return DZ_EINVAL;
  if (T < 1) return DZ_ESHAPE;
  // (a first chunk that fails its checks has launched nothing; the others differ in T alone)
  for (int t0 = 0; t0 < T; t0 += DZ_MAX_TOKENS_FUSED) {
    const uint16_t* xc = x + (size_t)t0 * K;
    uint16_t* yc = y + (size_t)t0 * ldy;
    const int t = T - t0 < DZ_MAX_TOKENS_FUSED ? T - t0 : DZ_MAX_TOKENS_FUSED;
    const int rc = multi_delta_linear_batch(1, &xc, &w_base, &codes_stacked, &meta_stacked, &scales_stacked, indices + t0,
                                            &yc, &N, &ldy, t, K, S, bits, group_size, accumulate, nullptr, workspace,
                                            workspace_bytes, stream, w_tiled, only_if);
    if (rc) return rc;
  }
  return DZ_OK;
}

int dz_tile_base(const uint16_t* w, int K, int N, uint16_t* out, void* stream) {
  if (!w || !out) return DZ_EINVAL;
  if (K < DZ_KBLOCK || N < DZ_NPAIR || K % DZ_KBLOCK || N % DZ_NPAIR) return DZ_ESHAPE;
  if (((uintptr_t)w & 15) || ((uintptr_t)out & 15)) return DZ_EALIGN;
  const uintptr_t bytes = (uintptr_t)N * K * 2;
  if ((uintptr_t)w < (uintptr_t)out + bytes && (uintptr_t)out < (uintptr_t)w + bytes) return DZ_EINVAL;   // a permutation: not in place
  const long long chunks = (long long)N * K / 8;   // 16 bytes each
  hipLaunchKernelGGL(dz_tile_base_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const u4_t*)w, (u4_t*)out, K, N);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_token_order(const int64_t* indices, int T, int S, int32_t* order, void* stream) {
  if (!indices || !order) return DZ_EINVAL;
  if (T < 1 || T > DZ_MAX_TOKENS_FUSED || S < 0) return DZ_ESHAPE;
  hipLaunchKernelGGL(dz_deal_kernel, dim3(1), dim3(128), 0, (hipStream_t)stream, (const long long*)indices, T, S, order);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_multi_delta_linear(const uint16_t* x, const uint16_t* w_base, const void* codes_stacked,
                          const void* meta_stacked, const void* scales_stacked,
                          const int64_t* indices, uint16_t* y, int T, int K, int N, int S, int bits,
                          int group_size, int accumulate, int ldy, void* workspace,
                          size_t workspace_bytes, void* stream) {
  if (!x || !indices || !y) return DZ_EINVAL;
  if (S > 0 && (!codes_stacked || !meta_stacked || !scales_stacked)) return DZ_EINVAL;
  if (S == 0 && !w_base) return DZ_EINVAL;
  return dz_multi_delta_linear_batch(1, &x, &w_base, &codes_stacked, &meta_stacked, &scales_stacked, indices, &y,
                                     &N, &ldy, T, K, S, bits, group_size, accumulate, nullptr, workspace,
                                     workspace_bytes, stream);
}

int dz_multi_delta_linear_static(const uint16_t* x, const uint16_t* w_base, const void* codes_stacked,
                                 const void* meta_stacked, const void* scales_stacked,
                                 const int64_t* indices, uint16_t* y, int T, int K, int N, int S, int bits,
                                 int group_size, int accumulate, int ldy, void* stream) {
  if (N > DZ_STATIC_MAX_N) return DZ_ESTATICMAX;
  void* ws = static_scratch_ptr();
  if (!ws) return DZ_ELAUNCH;
  return dz_multi_delta_linear(x, w_base, codes_stacked, meta_stacked, scales_stacked, indices, y, T, K, N, S,
                               bits, group_size, accumulate, ldy, ws, STATIC_SCRATCH_BYTES, stream);
}

}  // extern "C"
