// Hessian-aware compression of a delta: n:m pruning and quantisation, column by column, with the
// error of every column spread over the columns still to come (deltazip/core/sparsegpt.py:25-146).
//
//   dz_hessian_add   H <- H * s0 + (s1 x)^T (s1 x)                         (sparsegpt.py:27-40)
//   dz_obs_sweep     the sweep over blocks of 128 columns                   (sparsegpt.py:92-146)
//
// Every sum runs in ascending index order with one rounding per operation (no fused multiply-add
// in the sums), so that the result is the same bit for bit as a plain fp32 restatement with that
// order: the work is v_mul_f32 / v_add_f32, not matrix instructions, whose order of summation is
// not specified.  In their two-operand form these two run at twice the rate of a three-operand
// instruction once a SIMD has two wavefronts (measured with register-only loops: 62 T lane
// operations per second against 39 T, and 31 T with one wavefront), which is the rate the two
// products below are built for.
#include <type_traits>
#include <utility>

#include "../../include/dz_amd.h"
#include "dz_device.h"

namespace {

constexpr int OBS_BLOCK = 128;
constexpr int OBS_PIECE = 64 + 4;   // floats from an 8 x 8 piece to the next: 16 lanes that read 16 pieces meet 16 times 4 banks
constexpr int OBS_TRI = 136 * OBS_PIECE;   // floats of a block of hinv on and above its diagonal, in such pieces

typedef f4_t f4u_t __attribute__((aligned(4)));   // 16 bytes of an array that is aligned to its elements only

// acc[i][j] += va[i] * vb[j], product and sum rounded separately.  The products of a row are made
// while the row before is summed: an addition that follows its own product at once runs at three
// quarters of the rate.
template <int NI, int NJ>
__device__ __forceinline__ void outer_add(float (&acc)[NI][NJ], const float (&va)[NI], const float (&vb)[NJ]) {
#pragma clang fp contract(off)
  float p[2][NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) p[0][j] = va[0] * vb[j];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (i + 1 < NI) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) p[(i + 1) & 1][j] = va[i + 1] * vb[j];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = acc[i][j] + p[i & 1][j];
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int NV>
struct vec_of {
  typedef float t __attribute__((ext_vector_type(NV)));
  typedef float u __attribute__((ext_vector_type(NV), aligned(4)));   // of an array that is aligned to its elements only
};

// n steps of acc += a b^T over operands staged in LDS: NI values at pa + k * lda, and NJ at pb + k * ldb, or
// for NJ = 8 four of them there and four at pb + k * ldb + second.  The operands of a step are read while the
// step before is summed.  N: a multiple of 8, or 0 for n, which is one.
template <int N, int NI, int NJ>
__device__ __forceinline__ void outer_steps(float (&acc)[NI][NJ], const float* pa, int lda, const float* pb, int ldb,
                                            int second, int n = N) {
  constexpr int NB = NJ == 8 ? 4 : NJ;
  typedef typename vec_of<NI>::t a_t;
  typedef typename vec_of<NB>::t b_t;
  a_t a = *(const a_t*)pa;
  b_t b = *(const b_t*)pb, c;
  if constexpr (NJ == 8) c = *(const b_t*)(pb + second);
  if (N) n = N;
  for (int k0 = 0; k0 < n; k0 += 8) {
#pragma unroll
    for (int k = k0; k < k0 + 8; ++k) {
      // (the read behind the last step repeats the first)
      pa = k + 1 < n ? pa + lda : pa - (n - 1) * lda;
      pb = k + 1 < n ? pb + ldb : pb - (n - 1) * ldb;
      const a_t an = *(const a_t*)pa;
      const b_t bn = *(const b_t*)pb;
      b_t cn;
      if constexpr (NJ == 8) cn = *(const b_t*)(pb + second);
      __builtin_amdgcn_sched_barrier(0);
      float va[NI], vb[NJ];
#pragma unroll
      for (int i = 0; i < NI; ++i) va[i] = a[i];
#pragma unroll
      for (int j = 0; j < NJ; ++j) vb[j] = j < NB ? b[j] : c[j - NB];
      outer_add(acc, va, vb);
      a = an;
      b = bn;
      if constexpr (NJ == 8) c = cn;
    }
  }
}

// ---- H <- H * s0 + sum_t (s1 x[t, a]) * (s1 x[t, b]), t ascending.
// Bound by the multiply-add rate.  The product of columns a and b has the same bits as that of b
// and a, so only the tiles on and above the diagonal are summed and each is written to both places
// (H itself need not be symmetric: either place scales its own old value).  A tile of 64 x 64 is summed
// by four wavefronts, 4 x 4 outputs per thread, 32 tokens of both sides staged at a time and the next 32 on
// their way in registers.  With 4 x 8 per thread there is less to read from LDS (at full occupancy either
// takes 82 us per 2048 tokens and tile of a CU), but two wavefronts per tile leave half the SIMDs
// of a last tile idle and the others at half their rate: 2080 tiles at K = 4096 took 790 us for
// 2048 tokens, now 665, 1128 tiles (K = 3072) 520, now 400.  A tile of 32 x 32 in four wavefronts, 2 x 2 per thread, is
// for the tiles that do not go round the CUs: alone on a CU it takes 76 us where one of 64 x 64 takes 190 (290
// with 4 x 8 per thread), but LDS bounds a CU full of them at 125 us for the outputs of one of 64 x 64.
template <typename XT, int TILE, int NI, int NJ>
__device__ __forceinline__ void hessian_tile(float* __restrict__ H, const XT* __restrict__ x, int T, int K, float s0, float s1,
                                             int ta, int tb, float* sm) {
#pragma clang fp contract(off)
  constexpr int NT = TILE * TILE / (NI * NJ);
  constexpr int STAGE = 2048 / TILE;                    // tokens that 16 KiB hold of both sides
  constexpr int TC = sizeof(XT) == 2 ? STAGE : STAGE / 2;   // tokens per stage
  constexpr int PER = 16 / sizeof(XT);         // elements per 16-byte load
  constexpr int ROWL = TILE / PER;             // loads per (token, TILE columns)
  constexpr int NL = TC * ROWL / NT;           // loads per thread, stage and side
  constexpr int TSTEP = NT / ROWL;             // tokens between a thread's loads
  constexpr int CN = TILE / NJ;
  static_assert(NL >= 1 && TC * ROWL % NT == 0, "");
  typedef typename vec_of<NJ>::t b_t;
  typedef typename vec_of<NJ>::u bu_t;
  typedef typename vec_of<NI>::t a_t;
  float(*st)[STAGE][TILE] = (float(*)[STAGE][TILE])sm;   // [a | b][token][column]; the mirrored tile at the end
  const int a0 = ta * TILE, b0 = tb * TILE;
  const int tid = threadIdx.x, tr = tid / CN, tc = tid % CN;   // rows NI tr .. + NI - 1, columns NJ tc .. + NJ - 1
  float acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = 0.f;

  typedef XT xv_t __attribute__((ext_vector_type(PER), aligned(sizeof(XT))));
  const int lt = tid / ROWL, lc = (tid % ROWL) * PER;
  xv_t next[2][NL];
  // tokens beyond T: the last one again, placed as zeros (adding 0 changes no sum: none is -0)
  auto fetch = [&](int t0) {
    const XT* base = x + (size_t)t0 * K;
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      const unsigned off = (unsigned)min(lt + l * TSTEP, T - 1 - t0) * (unsigned)K + (unsigned)lc;
      next[0][l] = *(const xv_t*)(base + a0 + off);
      next[1][l] = *(const xv_t*)(base + b0 + off);
    }
  };
  auto place = [&](int tokens) {
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      const bool in = lt + l * TSTEP < tokens;
#pragma unroll
      for (int side = 0; side < 2; ++side)
#pragma unroll
        for (int v = 0; v < PER; v += 4) {
          const xv_t& q = next[side][l];
          f4_t f = {(float)q[v], (float)q[v + 1], (float)q[v + 2], (float)q[v + 3]};
#pragma unroll
          for (int e = 0; e < 4; ++e) f[e] = in ? s1 * f[e] : 0.f;
          *(f4_t*)&st[side][lt + l * TSTEP][lc + v] = f;
        }
    }
  };
  const float *pa = &st[0][0][NI * tr], *pb = &st[1][0][NJ * tc];
  fetch(0);
  int t0 = 0;
  for (; t0 + TC <= T; t0 += TC) {
    __syncthreads();
    place(TC);
    __syncthreads();
    if (t0 + TC < T) fetch(t0 + TC);
    outer_steps<TC>(acc, pa, TILE, pb, TILE, 0);
  }
  if (t0 < T) {
    __syncthreads();
    place(T - t0);
    __syncthreads();
    outer_steps<0>(acc, pa, TILE, pb, TILE, 0, (T - t0 + 7) & ~7);
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    bu_t* h = (bu_t*)(H + (size_t)(a0 + NI * tr + i) * K + b0 + NJ * tc);
    const b_t old = *h;
    b_t v;
#pragma unroll
    for (int e = 0; e < NJ; ++e) {
      const float scaled = old[e] * s0;
      v[e] = scaled + acc[i][e];
    }
    *h = v;
  }
  if (ta == tb) return;
  // the mirrored tile, turned in LDS (16-byte chunks of a row rotated by the row: no shared banks)
  float* turn = &st[0][0][0];
  constexpr int NCH = TILE / 4;
  auto chunk = [&](int b, int ch) { return turn + b * TILE + (((ch + b + (b >> 4)) & (NCH - 1)) << 2); };
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    a_t v;
#pragma unroll
    for (int i = 0; i < NI; ++i) v[i] = acc[i][j];
    *(a_t*)(chunk(NJ * tc + j, NI * tr >> 2) + (NI * tr & 3)) = v;
  }
  __syncthreads();
#pragma unroll
  for (int l = 0; l < TILE * NCH / NT; ++l) {
    const int b = (l * NT + tid) / NCH, ch = tid % NCH;
    const f4_t s = *(const f4_t*)chunk(b, ch);
    f4u_t* h = (f4u_t*)(H + (size_t)(b0 + b) * K + a0 + 4 * ch);
    const f4_t old = *h;
    f4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float scaled = old[e] * s0;
      v[e] = scaled + s[e];
    }
    *h = v;
  }
}

// The first `whole` tiles of 64 x 64 as they are, the others in quarters.
template <typename XT>
__global__ __launch_bounds__(256, 4) void dz_hessian_kernel(float* __restrict__ H, const XT* __restrict__ x, int T, int K,
                                                          float s0, float s1, int whole) {
  __shared__ __attribute__((aligned(16))) float sm[4096];
  const int wg = blockIdx.x;
  const bool quarter = wg >= whole;
  // tile number -> (ta <= tb): number = tb (tb + 1) / 2 + ta
  const int n = quarter ? whole + ((wg - whole) >> 2) : wg;
  int tb = (int)((sqrtf(8.f * (float)n + 1.f) - 1.f) * 0.5f);
  while (tb * (tb + 1) / 2 > n) --tb;
  while ((tb + 1) * (tb + 2) / 2 <= n) ++tb;
  const int ta = n - tb * (tb + 1) / 2;
  if (!quarter) return hessian_tile<XT, 64, 4, 4>(H, x, T, K, s0, s1, ta, tb, sm);
  const int qa = 2 * ta + ((wg - whole) & 1), qb = 2 * tb + ((wg - whole) >> 1 & 1);
  if (qa <= qb) hessian_tile<XT, 32, 2, 2>(H, x, T, K, s0, s1, qa, qb, sm);
}

// ---- one block of 128 columns (sparsegpt.py:98-142)
// x / b for b in [2^-40, 2^40], |x| in [2^-80, 2^80], y = 1 / b correctly rounded: two residual steps.
// After the first the quotient is within one unit in the last place, from where the second rounds
// correctly (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000
// processor", IBM J. Res. Dev. 34, 1990); nothing under- or overflows in these ranges.
__device__ __forceinline__ float div_by(float x, float b, float y) {
  const float q0 = x * y;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-b, q0, x), y, q0);
  return __builtin_fmaf(__builtin_fmaf(-b, q1, x), y, q1);
}
constexpr float W_MIN = 0x1p-40f, X_MIN = 0x1p-80f, X_MAX = 0x1p40f, B_MIN = 0x1p-20f, B_MAX = 0x1p20f;
constexpr unsigned T_MAX = 0x5C000000u;   // bits of 2^57: w^2 is below 2^97, whose division is as exact

template <int L>
__device__ __forceinline__ float row_lane(float v) {   // the value of lane L of each row of 16 lanes
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + L, 0xF, 0xF, true));
}
__device__ __forceinline__ float lane_down(float v) {  // each lane of 16 takes the value of the next, the last that of the first
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x12F, 0xF, 0xF, true));
}
template <typename F, int... L>
__device__ __forceinline__ void for_each_lane(F&& f, std::integer_sequence<int, L...>) {
  (f(std::integral_constant<int, L>{}), ...);
}

// Bound by the chain of one column's decision on the one before it.  A row is swept by 16 lanes,
// 8 neighbouring columns each, so the 8 columns of a lane -- whole pruning groups -- are decided in
// that lane's registers and only the column's error travels, by one cross-lane move; a wavefront
// sweeps 4 rows, which gives the 4096 rows of a projection one wavefront per SIMD (with a
// wavefront per row four of them shared a SIMD and each repeated every decision in 64 lanes).
// Sixteen turns of 8 columns: after each the registers move down by one lane, so that the deciding
// lane is always the first of its 16.  The rows of hinv come from LDS.  Divisions by the diagonal
// and by the row's scale use their reciprocals (`div_by`); a turn that meets a value outside the
// range where that is the correctly rounded quotient -- zeros among them -- is run again with
// ordinary divisions.  err_prev: errors of the block before, not yet carried to these columns (they
// are first), or nullptr.
// Where it stands: 49 vector instructions a column, 16 of them the products, one wavefront per SIMD: 23 us per block of 4096
// rows (145 with a wavefront per row).  It was 30 while the 16 lanes, which read one row of 16 pieces of hinv, met the same
// banks (OBS_PIECE; 31 k of the 73 k cycles a CU took were conflicts).  All of 4096 x 4096, us: 2070; columns compared by
// their bits and four workgroups a CU 2057; pieces 68 apart as well 1875; the tail of the products in halves 1800.
template <bool QUANT, int M>   // M: columns per pruning group, 0: no pruning
__device__ __forceinline__ void sweep_rows(float* __restrict__ W, const float* __restrict__ hinv,
                                           const float* __restrict__ scale, int N, int K, int i1, float maxq,
                                           float zero, int prunen, const float* __restrict__ err_prev,
                                           float* __restrict__ err, float* __restrict__ loss, int wg, float* sm) {
#pragma clang fp contract(off)
  float* hs = sm;                                   // 8 x 8 pieces (row group o, column group j >= o), see `piece`
  float* cst = sm + OBS_TRI;                        // [4][128]: d, 1 / d, d^2, 1 / d^2
  const int tid = threadIdx.x, lane = tid & 63, p = lane & 15, rg = tid >> 4;   // rg: row within the workgroup
  const int row = wg * 16 + rg, rowc = min(row, N - 1);
  auto piece = [](int o, int j) { return (((o * (33 - o)) >> 1) + j - o) * OBS_PIECE; };
  // all loads of hinv by a thread are on their way before the first is used
  f4_t hl[16], hh[8];
  auto fetch_tri = [&]() {     // the block's own rows, on and right of the diagonal pieces
#pragma unroll
    for (int l = 0; l < 16; ++l) {
      const int r = l * 8 + (tid >> 5), c = (tid & 31) * 4;
      if ((c >> 3) >= (r >> 3)) hl[l] = *(const f4u_t*)(hinv + (size_t)(i1 + r) * K + i1 + c);
    }
  };
  auto fetch_half = [&](int r0) {   // 64 rows of the block before, all 128 columns
#pragma unroll
    for (int l = 0; l < 8; ++l)
      hh[l] = *(const f4u_t*)(hinv + (size_t)(r0 + l * 8 + (tid >> 5)) * K + i1 + (tid & 31) * 4);
  };
  auto place_half = [&]() {
#pragma unroll
    for (int l = 0; l < 8; ++l) ((f4_t*)hs)[l * 256 + (tid & ~31) + ((tid >> 1) & 15) + 16 * (tid & 1)] = hh[l];   // a lane's two halves of 8 columns 64 floats apart
  };
  if (err_prev) fetch_half(i1 - OBS_BLOCK);
  bool odd = false;   // a divisor outside the range of div_by: every turn takes ordinary divisions
  if (tid < OBS_BLOCK) {
    const float d = hinv[(size_t)(i1 + tid) * K + i1 + tid], dd = d * d;
    cst[tid] = d;
    cst[OBS_BLOCK + tid] = 1.f / d;
    cst[2 * OBS_BLOCK + tid] = dd;
    cst[3 * OBS_BLOCK + tid] = 1.f / dd;
    odd = !(d >= B_MIN && d <= B_MAX);
  }
  float w[8];
  {
    const float* wr = W + (size_t)rowc * K + i1 + 8 * p;
    const f4_t v0 = *(const f4u_t*)wr, v1 = *(const f4u_t*)(wr + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      w[e] = v0[e];
      w[4 + e] = v1[e];
    }
  }
  const float sc = QUANT ? scale[rowc] : 1.f, ysc = 1.f / sc;
  odd = odd || (QUANT && !(sc >= W_MIN && sc <= X_MAX));
  if (err_prev) {
    const float* ep = err_prev + (size_t)rowc * OBS_BLOCK + 8 * p;
    float old[8];                                   // errors of the lane's columns of that block; they move as w does below
    {
      const f4_t v0 = *(const f4u_t*)ep, v1 = *(const f4u_t*)(ep + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        old[e] = v0[e];
        old[4 + e] = v1[e];
      }
    }
    float acc[1][8] = {{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      place_half();
      __syncthreads();
      if (half == 0) fetch_half(i1 - OBS_BLOCK / 2);
      const float* hp = hs + 4 * p;                 // (a row is read while the one before is summed: 10 -> 7 us per block)
      f4_t b = *(const f4_t*)hp, c = *(const f4_t*)(hp + 64);
      for (int k = 0; k < OBS_BLOCK / 2; k += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          hp += u < 7 || k + 8 < OBS_BLOCK / 2 ? OBS_BLOCK : 0;
          const f4_t bn = *(const f4_t*)hp, cn = *(const f4_t*)(hp + 64);
          __builtin_amdgcn_sched_barrier(0);
          const float va[1] = {row_lane<0>(old[u])}, vb[8] = {b[0], b[1], b[2], b[3], c[0], c[1], c[2], c[3]};
          outer_add(acc, va, vb);
          b = bn;
          c = cn;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) old[u] = lane_down(old[u]);
      }
      __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = w[e] - acc[0][e];
  }
  fetch_tri();
#pragma unroll
  for (int l = 0; l < 16; ++l) {
    const int r = l * 8 + (tid >> 5), c = (tid & 31) * 4;
    if ((c >> 3) >= (r >> 3)) *(f4_t*)(hs + piece(r >> 3, c >> 3) + (r & 7) * 8 + (c & 4)) = hl[l];
  }
  odd = __syncthreads_or(odd);

  float left[8];                                    // w - q of the lane's columns
#pragma unroll
  for (int e = 0; e < 8; ++e) left[e] = 0.f;
  for (int o = 0; o < 16; ++o) {
    const float* hp = hs + piece(o, o + min(p, 15 - o));   // (lanes that have wrapped around hold columns that are done)
    // constants of the turn's 8 columns, the same for every lane
    float d[8], y[8], dd[8], ydd[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      d[e] = cst[8 * o + e];
      y[e] = cst[OBS_BLOCK + 8 * o + e];
      dd[e] = cst[2 * OBS_BLOCK + 8 * o + e];
      ydd[e] = cst[3 * OBS_BLOCK + 8 * o + e];
    }
    float q[8], er[8], df[8], ws[8];
    bool bad = false;
    auto turn = [&](auto fast_c) {
      constexpr bool FAST = decltype(fast_c)::value;
      float wmin = 1.f, xmin = 1.f, xmax = 1.f;
      unsigned tmax = 0;     // bits of the largest w^2 / diag^2 (those of a NaN are larger)
      int rank[M > 0 ? M : 1];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        if constexpr (M > 0) {
          if (r % M == 0) {
            // w^2 / diag^2 of the group's columns; the prunen smallest are pruned, ties keep the
            // lower column (sparsegpt.py:123-125)
            float t[M];
#pragma unroll
            for (int c = 0; c < M; ++c) {
              const float ww = w[r + c] * w[r + c];
              t[c] = FAST ? div_by(ww, dd[r + c], ydd[r + c]) : ww / dd[r + c];
              if (FAST) {
                wmin = fminf(wmin, fabsf(w[r + c]));
                tmax = max(tmax, __float_as_uint(t[c]));
              }
            }
            // how many of the group come behind a column
#pragma unroll
            for (int a = 0; a < M; ++a) rank[a] = 0;
#pragma unroll
            for (int a = 0; a < M; ++a)
#pragma unroll
              for (int b = a + 1; b < M; ++b) {
                // (values that are not negative: their bits compare as they do, without a trip through the mask register)
                const int less = FAST ? (int)(((unsigned)__float_as_int(t[a]) - (unsigned)__float_as_int(t[b])) >> 31) : t[b] > t[a];
                rank[a] += less;
                rank[b] += FAST ? 1 - less : t[a] >= t[b];
              }
          }
        }
        const bool pr = M > 0 && rank[r % (M > 0 ? M : 1)] >= M - prunen;
        float qv = pr ? 0.f : w[r];
        if (QUANT) {
          // (a pruned column's code is the zero-point: rint(0 / sc) + zero)
          const float quo = FAST ? div_by(w[r], sc, ysc) : w[r] / sc;
          // clamp(rint + zero, 0, maxq) - zero; the sum makes a zero positive, as that difference does
          qv = sc * (__builtin_amdgcn_fmed3f(rintf(pr ? 0.f : quo), -zero, maxq - zero) + 0.f);
        }
        const float diff = w[r] - qv;
        float e;
        if (FAST) {
          // without rounding a column that stays has no error (diff is 0, and NaN where w is: the range
          // check's minimum and maximum pass over a NaN)
          e = QUANT || pr ? div_by(diff, d[r], y[r]) : diff;
          xmin = fminf(fminf(xmin, fabsf(w[r])), QUANT ? fabsf(diff) : X_MAX);
          xmax = fmaxf(xmax, fabsf(w[r]));
        } else {
          e = diff / d[r];
        }
        q[r] = qv;
        df[r] = diff;
        er[r] = e;
        float eb = row_lane<0>(e);
        asm("" : "+v"(eb));                          // (as an operand of the products the move takes a wait in front of each)
        const f4_t h0 = *(const f4_t*)(hp + 8 * r), h1 = *(const f4_t*)(hp + 8 * r + 4);
        const float h[8] = {h0[0], h0[1], h0[2], h0[3], h1[0], h1[1], h1[2], h1[3]};
        // columns that are done -- the first lane's up to r, and whole lanes that have wrapped around
        // -- are changed too; nothing reads them any more
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const float pp = eb * h[c];
          w[c] = w[c] - pp;
        }
      }
      if (FAST) bad = !(wmin >= W_MIN && xmin >= X_MIN && xmax <= X_MAX && tmax <= T_MAX);
    };
    if (!odd) {
#pragma unroll
      for (int e = 0; e < 8; ++e) ws[e] = w[e];
      turn(std::true_type{});
    }
    if (odd || __builtin_amdgcn_ballot_w64(bad && p == 0) != 0) {
      if (!odd) {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = ws[e];
      }
      turn(std::false_type{});
    }
    if (p == 0) {
      float* wr = W + (size_t)rowc * K + i1 + 8 * o;      // (rows beyond N sweep the last row again: the same values)
      float* ep = err + (size_t)rowc * OBS_BLOCK + 8 * o;
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        *(f4u_t*)(wr + e) = (f4_t){q[e], q[e + 1], q[e + 2], q[e + 3]};
        *(f4u_t*)(ep + e) = (f4_t){er[e], er[e + 1], er[e + 2], er[e + 3]};
      }
    }
    // the next lane's columns move into the deciding lane; what is left of the turn's goes to the lane that loaded them
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float dv = row_lane<0>(df[e]);
      left[e] = p == o ? dv : left[e];
      w[e] = lane_down(w[e]);
    }
  }
  // the row's losses, summed in column order: each lane continues the sum of the lane before it
  float term[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    term[e] = (left[e] * left[e]) / cst[2 * OBS_BLOCK + 8 * p + e];
  }
  float lsum = 0.f;
  auto chain = [&](auto l_c) {
    float s = lsum;
#pragma unroll
    for (int e = 0; e < 8; ++e) s = s + term[e];
    lsum = row_lane<decltype(l_c)::value>(s);
  };
  for_each_lane(chain, std::make_integer_sequence<int, 16>{});
  if (row < N && p == 0) loss[row] = loss[row] + lsum / 2.f;
}

constexpr size_t OBS_LDS = (size_t)(OBS_TRI + 4 * OBS_BLOCK) * 4;   // 38 KiB: four workgroups per CU

// ---- W[:, c0 .. c0 + 127] -= Err @ hinv[i1 .. i1 + 127, c0 ..] for 64 rows, the sum over the block's
// 128 columns in ascending order (sparsegpt.py:146).  Bound by the multiply-add rate: 4 x 8 values
// per thread; the errors are staged with the row index innermost (with the
// column innermost the four rows of a thread fell on one bank) and in stages of 32 columns, so that
// several workgroups fit a CU.  NJ = 4: half a tile,
// 64 columns, for what is left when the others have gone round the CUs (`obs_sweep`).
template <int NJ>
__device__ __forceinline__ void propagate_tile(float* __restrict__ W, const float* __restrict__ err,
                                               const float* __restrict__ hinv, int N, int K, int i1, int r0, int c0,
                                               float* sm) {
#pragma clang fp contract(off)
  constexpr int KC = 32, ELD = 64 + 4, C = 16 * NJ, NH = KC * C / 1024;
  float* es = sm;                   // [KC][ELD]
  float* hs = sm + KC * ELD;        // [KC][C]
  const int tid = threadIdx.x, tr = tid >> 4, tc = tid & 15;   // rows 4 tr .. + 3, columns 4 tc .. + 3 (and 64 + 4 tc .. + 3)
  float acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = 0.f;
  // stage loads: errors as 16 bytes of a row (row tid / 8 and + 32, columns 4 (tid % 8) .. + 3)
  f4_t en[2], hn[NH];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int l = 0; l < 2; ++l)
      en[l] = *(const f4u_t*)(err + (size_t)min(r0 + l * 32 + (tid >> 3), N - 1) * OBS_BLOCK + k0 + 4 * (tid & 7));
#pragma unroll
    for (int l = 0; l < NH; ++l) {
      const int at = l * 256 + tid;
      hn[l] = *(const f4u_t*)(hinv + (size_t)(i1 + k0 + at / (C / 4)) * K + c0 + 4 * (at % (C / 4)));
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < OBS_BLOCK; k0 += KC) {
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
      for (int e = 0; e < 4; ++e) es[(4 * (tid & 7) + e) * ELD + l * 32 + (tid >> 3)] = en[l][e];
#pragma unroll
    for (int l = 0; l < NH; ++l) *(f4_t*)(hs + 4 * (l * 256 + tid)) = hn[l];
    __syncthreads();
    if (k0 + KC < OBS_BLOCK) fetch(k0 + KC);
    outer_steps<KC>(acc, es + 4 * tr, ELD, hs + 4 * tc, C, 64);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + 4 * tr + i;
    if (r >= N) continue;
#pragma unroll
    for (int j = 0; j < NJ; j += 4) {
      f4u_t* wp = (f4u_t*)(W + (size_t)r * K + c0 + 16 * j + 4 * tc);
      f4_t v = *wp;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] - acc[i][j + e];
      *wp = v;
    }
  }
}

// One launch of the sweep: its first `nsweep` workgroups sweep the block at column i1 (after
// carrying the errors of the block before, err_prev, to their own columns), the others carry
// err_prev to the columns `c_lo` and beyond.  The sweep leaves most of the GPU's issue slots free and
// the products fill them, three workgroups of them beside one of the sweep on a CU: at 4096 x 4096, 8.4 -> 2.04 -> 1.80 ms for the
// whole sweep (2.04 with two beside it, conflicts in LDS and no halves; one kernel after the other: 2.6 ms).
template <bool QUANT, int M>
__global__ __launch_bounds__(256, 4) void dz_obs_step_kernel(float* __restrict__ W, const float* __restrict__ hinv,
                                                          const float* __restrict__ scale, int N, int K, int i1,
                                                          float maxq, float zero, int prunen, int nsweep, int whole,
                                                          const float* __restrict__ err_sweep, float* __restrict__ err,
                                                          const float* __restrict__ err_prev, int i_prev, int c_lo,
                                                          float* __restrict__ loss) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int wg = blockIdx.x;
  if (wg < nsweep) {
    sweep_rows<QUANT, M>(W, hinv, scale, N, K, i1, maxq, zero, prunen, err_sweep, err, loss, wg, sm);
  } else {
    const int nr = (N + 63) / 64, at = wg - nsweep;
    const bool half = at >= whole;
    const int t = half ? whole + (at - whole) / 2 : at, r0 = t % nr * 64, c0 = c_lo + t / nr * 128;
    if (half) propagate_tile<4>(W, err_prev, hinv, N, K, i_prev, r0, c0 + ((at - whole) & 1) * 64, sm);
    else propagate_tile<8>(W, err_prev, hinv, N, K, i_prev, r0, c0, sm);
  }
}

}  // namespace

extern "C" {

int dz_hessian_add(float* H, const void* x, int x_is_fp16, int T, int K, float scale_h, float scale_x,
                   void* stream) {
  if (!H || !x) return DZ_EINVAL;
  if (T < 1 || K < 64 || K % 64) return DZ_ESHAPE;
  hipStream_t st = (hipStream_t)stream;
  const int nt = K / 64, n = nt * (nt + 1) / 2;
  // Tiles that do not fill a round of the 256 CUs go in quarters, over all of them (2048 tokens: K = 4096, 32 tiles beyond
  // eight rounds, 731 -> 665 us; K = 2560, 52 beyond three, 350 -> 309; 3968, 161 beyond seven, 660 -> 620), unless
  // they nearly fill it (2816, 222 beyond three, 352 us in quarters and 341 whole).  Below 448 tiles all go in
  // quarters: one round of whole tiles takes as long as two (K = 1600, 325 tiles, 207 us and 169 in
  // quarters; 1856, 435 tiles, 204 and 199; 1984, 496 tiles, 203 and 217).
  const int rest = n % 256, whole = n < 448 ? 0 : rest > 208 ? n : n - rest;
  const dim3 grid((unsigned)(whole + 4 * (n - whole)));
  if (x_is_fp16)
    hipLaunchKernelGGL(dz_hessian_kernel<_Float16>, grid, dim3(256), 0, st, H, (const _Float16*)x, T, K, scale_h,
                       scale_x, whole);
  else
    hipLaunchKernelGGL(dz_hessian_kernel<float>, grid, dim3(256), 0, st, H, (const float*)x, T, K, scale_h,
                       scale_x, whole);
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

// err: errors of two neighbouring blocks (`ahead`), or of one.
static int obs_sweep(float* W, const float* hinv_upper, const float* scale, int N, int K, int bits, int prunen,
                     int prunem, float* err, bool ahead, float* loss, void* stream) {
  if (!W || !hinv_upper || !err || !loss) return DZ_EINVAL;
  if (N < 1 || K < OBS_BLOCK || K % OBS_BLOCK) return DZ_ESHAPE;
  if (scale && bits != 2 && bits != 3 && bits != 4 && bits != 8) return DZ_EBITS;
  if (prunen < 0 || prunem < 0 || (prunen != 0 && (prunem > 8 || prunen >= prunem || 64 % prunem))) return DZ_ESHAPE;
  hipStream_t st = (hipStream_t)stream;
  const float maxq = (float)((1 << bits) - 1), zero = (float)(1 << (bits - 1));
  static std::atomic<unsigned long long> attr_done[8];
  const int which = (scale ? 4 : 0) + (prunen == 0 ? 0 : prunem == 2 ? 1 : prunem == 4 ? 2 : 3);
  const int nsweep = (N + 15) / 16, nr = (N + 63) / 64;
  auto sweep = [&](auto kern) -> int {
    if (!dz_lds_limit_once(attr_done[which], (const void*)kern, (int)OBS_LDS)) return DZ_ELAUNCH;
    auto step = [&](int ns, int i1, const float* err_sweep, float* err_cur, const float* err_prev, int i_prev, int c_lo) {
      // What goes beyond whole tiles, two by two on the 256 CUs, goes in halves: a tile alone on a CU has one wavefront per
      // SIMD, which takes its products at half the rate.  Up to 256 tiles are done before the sweep beside them: launches with 0
      // to 256 take 33 to 35 us, with 320 43.  (us per launch, whole / with halves, 4096 rows: 576 tiles 56 / 48, 768 60 / 57, 1280 82 / 74;
      // whole sweeps with halves beyond 512 tiles / beyond 256: 2560 columns, 1760 rows 639 / 622, 2048 x 2048 477 / 468, 4096
      // columns, 1024 rows 928 / 917, 3072, 1344 rows 729 / 722; 4096 x 4096, none at all / beyond 512 1875 / 1800.)
      const int tiles = err_prev ? nr * ((K - c_lo) / OBS_BLOCK) : 0, over = tiles % 512;
      const int whole = tiles <= 256 ? tiles : tiles - (over > 256 ? over - 256 : over);
      const int grid = ns + whole + 2 * (tiles - whole);
      hipLaunchKernelGGL(kern, dim3(grid), dim3(256), OBS_LDS, st, W, hinv_upper, scale, N, K, i1, maxq, zero, prunen,
                         ns, whole, err_sweep, err_cur, err_prev, i_prev, c_lo, loss);
    };
    for (int i1 = 0, b = 0; i1 < K; i1 += OBS_BLOCK, ++b) {
      const int i2 = i1 + OBS_BLOCK;
      if (ahead) {
        // the next block's columns are brought up to date by its own sweep, one launch later; what
        // lies beyond them by the other workgroups of that launch
        float *cur = err + (size_t)(b & 1) * N * OBS_BLOCK, *prev = err + (size_t)((b & 1) ^ 1) * N * OBS_BLOCK;
        step(nsweep, i1, b ? prev : nullptr, cur, b && i2 < K ? prev : nullptr, i1 - OBS_BLOCK, i2);
      } else {
        step(nsweep, i1, nullptr, err, nullptr, 0, K);
        if (i2 < K) step(0, i1, nullptr, nullptr, err, i1, i2);
      }
    }
    return DZ_OK;
  };
  int rc;
  switch (which) {
    case 0: rc = sweep(dz_obs_step_kernel<false, 0>); break;
    case 1: rc = sweep(dz_obs_step_kernel<false, 2>); break;
    case 2: rc = sweep(dz_obs_step_kernel<false, 4>); break;
    case 3: rc = sweep(dz_obs_step_kernel<false, 8>); break;
    case 4: rc = sweep(dz_obs_step_kernel<true, 0>); break;
    case 5: rc = sweep(dz_obs_step_kernel<true, 2>); break;
    case 6: rc = sweep(dz_obs_step_kernel<true, 4>); break;
    default: rc = sweep(dz_obs_step_kernel<true, 8>); break;
  }
  if (rc) return rc;
  return hipGetLastError() == hipSuccess ? DZ_OK : DZ_ELAUNCH;
}

int dz_obs_sweep(float* W, const float* hinv_upper, const float* scale, int N, int K, int bits, int prunen,
                 int prunem, float* err_workspace, float* loss, void* stream) {
  return obs_sweep(W, hinv_upper, scale, N, K, bits, prunen, prunem, err_workspace, false, loss, stream);
}

int dz_obs_sweep_ahead(float* W, const float* hinv_upper, const float* scale, int N, int K, int bits, int prunen,
                       int prunem, float* err_workspace, float* loss, void* stream) {
  return obs_sweep(W, hinv_upper, scale, N, K, bits, prunen, prunem, err_workspace, true, loss, stream);
}

}  // extern "C"
