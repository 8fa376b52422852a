// The exponential's products of the split mixed form for complex-symmetric matrices (the storage
// idea, split-FP16 planes with one exponent per matrix, is that of ctem_split.hip).
//
// With X = X^T the square C = X X has C(i, j) = sum over k of X(i, k) X(j, k): both operands of a
// step are rows of one strip, the matrix at 32 columns k, and every 32 x 32 output tile (i <= j) takes its
// A operand from the strip's row tile i and its B operand from row tile j, both as 8 consecutive k of
// one row per lane. The polynomial of the exponential is therefore evaluated by squares only
// (ctem_symcoef.h), and a workgroup keeps the whole upper triangle of a product in its accumulators.
//
// Tile image: the 32 x 32 tiles on and above the diagonal, 8 KB each (four planes of 2 KB); a plane
// holds its 32 columns one after the other, each as four 16-byte chunks of 8 rows, chunk ch of
// column c at place ch ^ f((c >> 2) & 3), f = (0, 2, 3, 1). A strip's row tile i <= k is tile (i, k) (rows contiguous:
// LDS transpose reads), a row tile i > k is tile (k, i) (k contiguous: 16-byte reads); the
// exchange of chunks spreads both over the banks.
//
// k_expm_sym (up to 224 beams): one workgroup per matrix does the whole exponential, operands in
// LDS and accumulators in registers. The tile (i, j) is used in strips i and j only, so at strip k the
// live tiles are those with i <= k <= j: at most 16 of the 28 at n = 224, and 19 tiles of LDS
// hold a matrix whose last nine tiles wait in a global buffer until their places are free. A is read in each of the
// polynomial's three steps, B^2 written and read back, and at six and seven tiles a side some registers spill.
// Only the operands are rounded to 22 bits: every other term, 2 X of a squaring included, stays FP32 in the accumulators,
// and B enters the polynomial exactly. Symmetry is used between different tiles only, with the diagonal tiles read as
// rows for one operand and as columns for the other.
//
// Measured on one MI355X, the exponentials of a run against k_sgemm's chain (64 x 64 tiles, three general
// products for a degree-8 polynomial; it moves 2.3 MB to LDS per product at n = 224 and waits for memory):
// bcc Fe, 63,252 directions of 188-250 beams: 142 -> 87 ms, with 9 products per matrix instead of 8; fcc Ni, 1,326 of
// 87-115: 1.03 -> 0.48 ms. Intensities against 64 bits over 140 drawn sets: the 2-norm error is 0.57-0.72 of that chain's
// on average at every size, at most 1.13 of it.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "ctem_ebsd.h"
#include "ctem_internal.h"

namespace ctem {

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef unsigned int u4v __attribute__((ext_vector_type(4)));
#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

constexpr int kTile = 4096;   // halfs of a tile image
constexpr int kPlane = 1024;  // halfs of a plane

// 1 KB from global memory (lane l's 16 bytes at src + 16 l) to LDS (dst + 16 l; src and dst uniform) by
// the load unit, asynchronously: the caller waits with s_waitcnt vmcnt(0) before the barrier ahead of the
// first read. The compiler's builtin makes every later LDS read wait for the load.
__device__ __forceinline__ void to_lds(const _Float16* src, const _Float16* dst, int lane) {
  const unsigned l = (unsigned)(uintptr_t)LDS_PTR(void, dst);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(l), "v"(lane * 16), "s"(src) : "memory", "m0");
}

// halfs offset within a plane of column c's 8-row chunk
__device__ __forceinline__ int chunk_off(int c, int chunk) {
  const int q = (c >> 2) & 3, f = (q >> 1) | (((q ^ (q >> 1)) & 1) << 1);
  return c * 32 + ((chunk ^ f) << 3);
}

// four consecutive rows (half a chunk) of one column, times sc, into the four planes at dst
__device__ __forceinline__ void put_rows(_Float16* dst, const f4v& re, const f4v& im, float sc) {
  h4v o[4];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    o[0][e] = (_Float16)(re[e] * sc);
    o[2][e] = (_Float16)(im[e] * sc);
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    o[1][e] = (_Float16)__builtin_fmaf(re[e], sc, -(float)o[0][e]);
    o[3][e] = (_Float16)__builtin_fmaf(im[e], sc, -(float)o[2][e]);
  }
#pragma unroll
  for (int p = 0; p < 4; p++) *(h4v*)(dst + p * kPlane) = o[p];
}

// Operand reads of this lane: 8 consecutive k of row 16 a + l15 of a strip's row tile, k chunk
// g = lane >> 4, of the four planes. k contiguous: one 16-byte read per plane. Rows contiguous: two
// transpose reads per plane; the 16-lane group g reads rows 16 a .. +15 of columns 8 g .. +3 and
// 8 g + 4 .. +7 (lane 4 e + j points at rows 4 j .. +3 of column e).
struct Reader {
  int k, lo, hi;  // halfs offsets for a = 0
  __device__ __forceinline__ explicit Reader(int lane) {
    const int l15 = lane & 15, g = lane >> 4, e = l15 >> 2, j = l15 & 3;
    k = chunk_off(l15, g);
    lo = chunk_off(8 * g + e, j >> 1) + 4 * (j & 1);
    hi = chunk_off(8 * g + 4 + e, j >> 1) + 4 * (j & 1);
  }
  __device__ __forceinline__ void read(const _Float16* tile, int a, bool rows, h8v (&o)[4]) const {
    if (rows) {
      // chunk 2 a + (j >> 1): bit 1 of the chunk flips with a, under the exchange as well
      const _Float16* pl = tile + (a ? (lo ^ 16) : lo);
      const _Float16* ph = tile + (a ? (hi ^ 16) : hi);
#pragma unroll
      for (int p = 0; p < 4; p++) {
        const s4v x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s4v, pl + p * kPlane));
        const s4v y = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s4v, ph + p * kPlane));
        o[p] = __builtin_bit_cast(h8v, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    } else {
      // column 16 a + l15: the exchange is that of l15
#pragma unroll
      for (int p = 0; p < 4; p++) o[p] = *(const h8v*)(tile + k + a * 512 + p * kPlane);
    }
  }
};

// one tile's accumulators: 16 x 16 subtiles [a][c], lane rows 4 (lane >> 4) + e, column lane & 15
struct Acc {
  f4v re[2][2], im[2][2];
};

// re, im += A B^T over 32 k, for the two row blocks of A and one column block. The twelve products go into fresh sums, added
// to the accumulators by rounded FP32 additions: the matrix cores' own accumulation does not round to nearest, and
// over a whole product its one-sided errors add up (intensities of fcc Ni 9.2e-7 from the 64-bit ones with
// the products accumulated in place). The imaginary planes of B are negated for the last terms,
// -Im A Im B. Smallest terms first.
__device__ __forceinline__ void mma(const h8v (&x)[2][4], h8v (&y)[4], f4v& re0, f4v& re1, f4v& im0, f4v& im1) {
  f4v r[2], i[2];
#define MM(acc, a, u, v) acc[a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[a][u], y[v], acc[a], 0, 0, 0)
#define MM4(u, v, w, z) MM(r, 0, u, v); MM(r, 1, u, v); MM(i, 0, w, z); MM(i, 1, w, z)
  r[0] = r[1] = i[0] = i[1] = (f4v){0, 0, 0, 0};
  MM4(1, 0, 1, 2);
  MM4(0, 1, 0, 3);
  MM(i, 0, 3, 0); MM(i, 1, 3, 0); MM(i, 0, 2, 1); MM(i, 1, 2, 1);
  MM4(0, 0, 0, 2);
#pragma unroll
  for (int p = 2; p < 4; p++) y[p] = __builtin_bit_cast(h8v, __builtin_bit_cast(u4v, y[p]) ^ 0x80008000u);
  MM4(3, 2, 2, 0);
  MM(r, 0, 2, 3); MM(r, 1, 2, 3);
  MM(r, 0, 2, 2); MM(r, 1, 2, 2);
#undef MM4
#undef MM
  re0 += r[0]; im0 += i[0];
  re1 += r[1]; im1 += i[1];
}

// tile t of the upper triangle in row order (row i: (i, i) .. (i, T - 1))
__device__ __forceinline__ int row_tile(int t, int T, int& j) {
  int i = 0;
  while (t >= T - i) { t -= T - i; i++; }
  j = i + t;
  return i;
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(__builtin_fmaf(-a.y, b.y, a.x * b.x), __builtin_fmaf(a.y, b.x, a.x * b.y));
}
__device__ __forceinline__ float2 cmac(float2 s, float2 a, float2 b) {  // s + a b
  return make_float2(__builtin_fmaf(-a.y, b.y, __builtin_fmaf(a.x, b.x, s.x)), __builtin_fmaf(a.y, b.x, __builtin_fmaf(a.x, b.y, s.y)));
}

// Four rows (row ..) of A's column col in tile (i, j), as (re, im) pairs. The table's U(-g) = U(g) holds to about 1e-8
// only; where the assembly's 64 x 64 tiles give both triangles, their mean is taken (the upper one alone costs
// corundum's sets of 33-64 beams half of their precision).
__device__ __forceinline__ void load_a(const float2* A, int n, int i, int j, int row, int col, f4v& m0, f4v& m1) {
  const f4v* p = (const f4v*)(A + (int64_t)col * n + row);
  m0 = p[0];
  m1 = p[1];
  if (j == i + 1 && !(i & 1)) {
    const float2* t = A + (int64_t)row * n + col;
    const float2 t0 = t[0], t1 = t[n], t2 = t[2 * n], t3 = t[3 * n];
    m0 = 0.5f * (m0 + (f4v){t0.x, t0.y, t1.x, t1.y});
    m1 = 0.5f * (m1 + (f4v){t2.x, t2.y, t3.x, t3.y});
  }
}

// exponent of the operand of step ST (1, 2: a bound of the sum) from the exact maximum of the accumulators before it
template <int ST>
__device__ __forceinline__ int operand_exp(const SymCoef& k, float vmax, float bmax) {
  auto mag = [](float2 v) __attribute__((always_inline)) { return fabsf(v.x) + fabsf(v.y); };
  if (ST == 1) vmax = __builtin_fmaf(mag(k.c), bmax, vmax);
  if (ST == 2) vmax = mag(k.r) * __builtin_fmaf(mag(k.d2), bmax, vmax);
  return f16_scale_exp(vmax);
}

// F's tile (i, j): four rows of one column, and mirrored off the diagonal
__device__ __forceinline__ void put_f(float2* F, int n, int i, int j, int row, int col, const f4v& vr, const f4v& vi) {
  f4v* p = (f4v*)(F + (int64_t)col * n + row);
  p[0] = (f4v){vr[0], vi[0], vr[1], vi[1]};
  p[1] = (f4v){vr[2], vi[2], vr[3], vi[3]};
  if (i != j)
#pragma unroll
    for (int e = 0; e < 4; e++) F[(int64_t)(row + e) * n + col] = make_float2(vr[e], vi[e]);
}

// ---- the whole exponential on chip ------------------------------------------------------------

struct ExpmArgs {
  const float2* A;      // [nb][n n] assembled matrices (column-major FP32; tiles on and above the diagonal)
  const int32_t* sq;    // squaring counts, exponents of B = A 2^-s
  const int32_t* bexp;
  const float* bmax;    // max |component| of B
  int32_t nb;
  float2* F;            // [nb][n n] out: exp(A) - I, both triangles
  float* Q;             // [workgroups][N 2048] work: B^2, FP32
  _Float16* spill;      // [workgroups][...] work: tile images that do not fit in LDS; strides of both in bytes: n n 8
  SymCoef c;
};

// T = n / 32; NW waves, at most NS tiles each; NSL LDS tile places
template <int T, int NW, int NS, int NSL, int EU>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(EU, EU))) void k_expm_sym(ExpmArgs g) {
  constexpr int n = 32 * T, N = T * (T + 1) / 2;
  constexpr int64_t per = (int64_t)n * n;
  // strips 2 .. kBring bring in tiles from the global buffer, as columns 0 and 1, 2, 3 become free; each
  // is first used at least one strip later
  constexpr int kOut = N > NSL ? N - NSL : 0, kBring = kOut > 6 ? 4 : kOut > 3 ? 3 : kOut > 0 ? 2 : 0;
  extern __shared__ __attribute__((aligned(16))) _Float16 Ls[];
  float* const red = (float*)(Ls + NSL * kTile);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, g4 = lane >> 4;
  // work space by workgroup, not by matrix: it stays in the caches and their address translations
  float* Q = g.Q + blockIdx.x * per * 2;
  _Float16* spill = g.spill + blockIdx.x * per * 4;

  // equal runs of the tile list; waves w and w + 4 share a SIMD and take neighbouring runs, and
  // with fewer waves than SIMD places the runs rotate over the SIMDs from workgroup to workgroup
  const int u = NW == 8 ? (wave & 3) * 2 + (wave >> 2) : (wave + blockIdx.x) % NW;
  const int t0 = u * N / NW, cnt = (u + 1) * N / NW - t0;
  int si[NS], sj[NS];
#pragma unroll
  for (int q = 0; q < NS; q++) si[q] = row_tile(min(t0 + q, N - 1), T, sj[q]);
  // place of tile (i, j) in LDS: its row order index r, or for r >= NSL the place of the (r - NSL)-th
  // tile in column order, which is free after that tile's column; lane 8 k + i of `tab` holds the
  // offset of strip k's row tile i
  int tab;
  {
    const int k = min(lane >> 3, T - 1), i = min(lane & 7, T - 1), ti = min(i, k), tj = max(i, k);
    int r = ti * T - ti * (ti - 1) / 2 + tj - ti;
    if (N > NSL && r >= NSL) {
      const int m = r - NSL;
      const int jj = m >= 6 ? 3 : m >= 3 ? 2 : m >= 1 ? 1 : 0, ii = m - jj * (jj + 1) / 2;
      r = ii * T - ii * (ii - 1) / 2 + jj - ii;
    }
    tab = r * kTile;
  }
  auto row_at = [&](int k, int i) __attribute__((always_inline)) { return Ls + __builtin_amdgcn_readlane(tab, 8 * k + i); };

#pragma unroll 1
  for (int b = blockIdx.x; b < g.nb; b += gridDim.x) {
  const float2* A = g.A + b * per;
  const int s = g.sq[b];
  const float bscale = ldexpf(1.0f, -s);
  int ex = g.bexp[b];
  const Reader rd(lane);
  Acc acc[NS];
  float un = 1.0f;  // accumulator units 2^(-2 ex)
  // one product on top of the other terms that next_operand left in the accumulators (of a squaring X, of which it
  // takes 2 X). Code of its own for each step, so that nothing but the products decides what becomes of the
  // accumulators.
  auto product = [&](auto st) __attribute__((always_inline)) {
    constexpr int ST = decltype(st)::value;
    const float up = ldexpf(1.0f, 2 * ex), carry = ST == 3 ? 2.0f * un * up : up;
    un = ldexpf(1.0f, -2 * ex);
#pragma unroll
    for (int q = 0; q < NS; q++)
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          acc[q].re[a][c] = ST == 0 ? (f4v){0, 0, 0, 0} : acc[q].re[a][c] * carry;
          acc[q].im[a][c] = ST == 0 ? (f4v){0, 0, 0, 0} : acc[q].im[a][c] * carry;
        }
#pragma unroll 1
    for (int k = 0; k < T; k++) {
      // strip 0: the tiles are in LDS (stores to the global buffer may still be under way); then those
      // stores, and the loads into free places of the strip before
      if (k == 0) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      } else if (k > 1 && k <= kBring + 1) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if (k > 1 && k <= kBring) {
        const int m0 = k == 2 ? 0 : k == 3 ? 3 : 6, m1 = min(kOut, k == 2 ? 3 : k == 3 ? 6 : 10);
#pragma unroll 1
        for (int h = 8 * m0 + wave; h < 8 * m1; h += NW) {
          const int m = h >> 3, pc = (h & 7) * 512;
          const int jj = m >= 6 ? 3 : m >= 3 ? 2 : m >= 1 ? 1 : 0, ii = m - jj * (jj + 1) / 2;
          to_lds(spill + m * kTile + pc, Ls + (ii * T - ii * (ii - 1) / 2 + jj - ii) * kTile + pc, lane);
        }
      }
      h8v x[2][4], y[2][4];
#pragma unroll
      for (int q = 0; q < NS; q++)
        if (q < cnt) {
          if (q == 0 || si[q] != si[q > 0 ? q - 1 : 0]) {
            const _Float16* t = row_at(k, si[q]);
            rd.read(t, 0, si[q] <= k, x[0]);
            rd.read(t, 1, si[q] <= k, x[1]);
          }
          const _Float16* t = row_at(k, sj[q]);
          rd.read(t, 0, sj[q] < k, y[0]);
          mma(x, y[0], acc[q].re[0][0], acc[q].re[1][0], acc[q].im[0][0], acc[q].im[1][0]);
          rd.read(t, 1, sj[q] < k, y[1]);
          mma(x, y[1], acc[q].re[0][1], acc[q].re[1][1], acc[q].im[0][1], acc[q].im[1][1]);
        }
    }
  };
  // the next operand, and in the accumulators the next product's other terms (ctem_symcoef.h). 0: B from memory.
  // 1: B^2 + c B, B^2 to memory. 2: r (W + d2 B), B^2 back. 3: the accumulators. Exponents are from the accumulators'
  // exact maximum over the workgroup, in steps 1 and 2 by a bound of the sum.
  auto next_operand = [&](auto st) __attribute__((always_inline)) {
    constexpr int ST = decltype(st)::value;
    // the lane's place, opaque to the compiler: it would otherwise keep every address in registers
    // through the products
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int l15 = ln & 15, g4 = ln >> 4;
    auto load_b = [&](int q, int a, int c, f4v& m0, f4v& m1) __attribute__((always_inline)) {
      load_a(A, n, si[q], sj[q], 32 * si[q] + 16 * a + 4 * g4, 32 * sj[q] + 16 * c + l15, m0, m1);
    };
    auto z_at = [&](int q, int a, int c) __attribute__((always_inline)) {
      return (f4v*)(Q + (int64_t)min(t0 + q, N - 1) * 2048) + ln * 2 + (2 * a + c) * 128;
    };
    // tile t0 + q's place of rows 4 g4 .. and column l15 of subtile (a, c)
    auto image = [&](int q, int a, int c) __attribute__((always_inline)) {
      const int r = t0 + q;
      _Float16* t = (N > NSL && r >= NSL) ? spill + (r - NSL) * kTile : Ls + r * kTile;
      return t + chunk_off(16 * c + l15, 2 * a + (g4 >> 1)) + 4 * (g4 & 1);
    };
    if constexpr (ST == 0) {
#pragma unroll
      for (int q = 0; q < NS; q++)
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int c = 0; c < 2; c++) load_b(q, a, c, acc[q].re[a][c], acc[q].im[a][c]);
      const float sc = ldexpf(bscale, ex);
#pragma unroll
      for (int q = 0; q < NS; q++) {
        if (q < cnt)
#pragma unroll
          for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
              const f4v m0 = acc[q].re[a][c], m1 = acc[q].im[a][c];
              put_rows(image(q, a, c), (f4v){m0[0], m0[2], m1[0], m1[2]}, (f4v){m0[1], m0[3], m1[1], m1[3]}, sc);
            }
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
    f4v m[2][2][2];
    auto ask = [&](int q) __attribute__((always_inline)) {
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) load_b(q, a, c, m[a][c][0], m[a][c][1]);
    };
    constexpr bool kB = ST == 1 || ST == 2;
    if constexpr (kB && NS < 4) ask(0);
    float vmax = 0.0f;
#pragma unroll
    for (int t = 0; t < 4 * NS; t++) {
      const int q = t >> 2, a = (t >> 1) & 1, c = t & 1;
      if (q < cnt)
#pragma unroll
        for (int e = 0; e < 4; e++) vmax = fmaxf(vmax, fmaxf(fabsf(acc[q].re[a][c][e]), fabsf(acc[q].im[a][c][e])));
    }
    vmax = fmaxf(vmax, dpp_f32<0xB1>(vmax));
    vmax = fmaxf(vmax, dpp_f32<0x4E>(vmax));
    vmax = fmaxf(vmax, dpp_f32<0x124>(vmax));
    vmax = fmaxf(vmax, dpp_f32<0x128>(vmax));
    vmax = fmaxf(vmax, xchg16(vmax));
    vmax = fmaxf(vmax, xchg32(vmax));
    if (lane == 0) red[wave] = vmax;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // and every wave is done with the operand
    asm volatile("" ::: "memory");
    vmax = red[0];
#pragma unroll
    for (int w = 1; w < NW; w++) vmax = fmaxf(vmax, red[w]);
    const float2 f = ST == 1 ? g.c.c : g.c.d2;
    ex = operand_exp<ST>(g.c, vmax * un, kB ? g.bmax[b] : 0.0f);
    const float sc = ldexpf(kB ? 1.0f : un, ex);
#pragma unroll
    for (int q = 0; q < NS; q++) {
      if constexpr (kB && NS >= 4) ask(q);  // (asked for one tile ahead, they spill)
      if (q < cnt) {
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int c = 0; c < 2; c++) {
            f4v& re = acc[q].re[a][c];
            f4v& im = acc[q].im[a][c];
            if constexpr (!kB) {
              put_rows(image(q, a, c), re, im, sc);
            } else {
              f4v* p = z_at(q, a, c);
              f4v zr, zi, xr, xi;
              if constexpr (ST == 2) { zr = p[0]; zi = p[1]; }
#pragma unroll
              for (int e = 0; e < 4; e++) {
                const float2 B = make_float2(m[a][c][e >> 1][2 * (e & 1)] * bscale, m[a][c][e >> 1][2 * (e & 1) + 1] * bscale);
                const float2 v = make_float2(re[e] * un, im[e] * un);
                float2 x = cmac(v, f, B), t;
                if constexpr (ST == 1) {
                  zr[e] = v.x; zi[e] = v.y;
                  t = cmul(g.c.d1, v);
                } else {
                  x = cmul(g.c.r, x);
                  t = cmac(cmac(B, g.c.g, make_float2(zr[e], zi[e])), g.c.e1, v);
                }
                xr[e] = x.x; xi[e] = x.y;
                re[e] = t.x; im[e] = t.y;
              }
              if constexpr (ST == 1) { p[0] = zr; p[1] = zi; }
              put_rows(image(q, a, c), xr, xi, sc);
            }
          }
      }
      if constexpr (kB)
        if (NS < 4 && q + 1 < NS) ask(q + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  next_operand(std::integral_constant<int, 0>{});
  product(std::integral_constant<int, 0>{});
  next_operand(std::integral_constant<int, 1>{});
  product(std::integral_constant<int, 1>{});
  next_operand(std::integral_constant<int, 2>{});
  product(std::integral_constant<int, 2>{});
#pragma unroll 1
  for (int it = 0; it < s; it++) {
    next_operand(std::integral_constant<int, 3>{});
    product(std::integral_constant<int, 3>{});
  }
  // F in FP32, both triangles
  float2* F = g.F + b * per;
#pragma unroll
  for (int q = 0; q < NS; q++)
    if (q < cnt) {
      const int i = si[q], j = sj[q];
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const int row = 32 * i + 16 * a + 4 * g4, col = 32 * j + 16 * c + l15;
          put_f(F, n, i, j, row, col, acc[q].re[a][c] * un, acc[q].im[a][c] * un);
        }
    }
  __syncthreads();  // every wave is done with the last operand
  }
}

// workgroups walk the matrices: as many as fit on the GPU at once (kWg per CU)
template <int T, int NW, int NS, int NSL, int EU, int kWg>
void expm_case(hipStream_t s, int nb, int cus, const ExpmArgs& a) {
  hipLaunchKernelGGL((k_expm_sym<T, NW, NS, NSL, EU>), dim3(std::min(nb, kWg * cus)), dim3(NW * 64),
                     NSL * kTile * sizeof(_Float16) + 64, s, a);
}

// ---- few matrices --------------------------------------------------------------------------------

// The same exponential, bit for bit, a product per launch: a wave takes 32 rows and 16 or 32 columns of a tile, with the
// operands in FP32 from memory (both triangles, split as they are read) and no exchange but the maximum. For a handful of
// matrices of six or seven tiles a side, where k_expm_sym leaves most CUs idle: a direction's result may not depend on
// its batch. Step -1 lays B out (unscaled), 0 to 2 are the polynomial, 3 a squaring. Bound by latency.
struct FewArgs {
  const float2* A;
  const int32_t* sq;
  const int32_t* bexp;
  const float* bmax;
  int32_t n, nb, it;         // it: the squaring's number
  float2* B;                 // [nb][n n]: what step -1 lays out
  const float2* X;           // operand in
  float2* Y;                 // operand out
  float2* F;                 // out: the result of a matrix's last product
  float* Q;                  // [nb][N 2048]: B^2, then the terms of step 2
  const float* max_in;       // [nb]: maximum of the product before, and of this one; `clear` is the next one's
  float* max_out;
  float* clear;
  SymCoef c;
};

// CB: column blocks of 16 per wave, from c0
template <int ST, int CB>
__device__ __forceinline__ void few_step(const FewArgs& g, int b, int t, int c0, int lane) {
  const int n = g.n, T = n >> 5, l15 = lane & 15, g4 = lane >> 4;
  const int64_t per = (int64_t)n * n;
  int j;
  const int i = row_tile(t, T, j), row0 = 32 * i + 4 * g4, col0 = 32 * j + 16 * c0 + l15;
  float2* const B = g.B + b * per;
  if constexpr (ST < 0) {
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int c = 0; c < CB; c++) {
        const int row = row0 + 16 * a, col = col0 + 16 * c;
        f4v m0, m1;
        load_a(g.A + b * per, n, i, j, row, col, m0, m1);
        put_f(B, n, i, j, row, col, (f4v){m0[0], m0[2], m1[0], m1[2]}, (f4v){m0[1], m0[3], m1[1], m1[3]});
      }
    return;
  } else {
    const int s = g.sq[b];
    if (ST == 3 && g.it >= s) return;
    if (t == 0 && c0 == 0 && lane == 0) g.clear[b] = 0.0f;
    const float bscale = ldexpf(1.0f, -s);
    const int ex = ST == 0 ? g.bexp[b] : operand_exp<ST>(g.c, g.max_in[b], g.bmax[b]);
    const float up = ldexpf(1.0f, 2 * ex), un = ldexpf(1.0f, -2 * ex), sc = ldexpf(ST == 0 ? bscale : 1.0f, ex);
    const float2* X = (ST == 0 ? B : g.X + b * per);
    auto z_at = [&](int a, int c) __attribute__((always_inline)) {
      return (f4v*)(g.Q + b * (per * 2)) + ((int64_t)t * 512 + lane * 2 + (2 * a + c0 + c) * 128);
    };
    // (re, im) of four rows of one column of a matrix
    auto load4 = [&](const float2* M, int a, int c, f4v& r, f4v& im) __attribute__((always_inline)) {
      const f4v* p = (const f4v*)(M + (int64_t)(col0 + 16 * c) * n + row0 + 16 * a);
      const f4v m0 = p[0], m1 = p[1];
      r = (f4v){m0[0], m0[2], m1[0], m1[2]};
      im = (f4v){m0[1], m0[3], m1[1], m1[3]};
    };
    f4v re[CB][2], im[CB][2];
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
      for (int a = 0; a < 2; a++) {
        f4v &r = re[c][a], &m = im[c][a];
        r = m = (f4v){0, 0, 0, 0};
        if constexpr (ST == 1 || ST == 2) {
          const f4v* z = z_at(a, c);
          const f4v zr = z[0], zi = z[1];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float2 v = ST == 1 ? cmul(g.c.d1, make_float2(zr[e], zi[e])) : make_float2(zr[e], zi[e]);
            r[e] = v.x * up;
            m[e] = v.y * up;
          }
        }
        if constexpr (ST == 3) {
          load4(X, a, c, r, m);
          r *= 2.0f * up;
          m *= 2.0f * up;
        }
      }
    // eight k of a row or column, split
    auto split8 = [&](const float2 (&v)[8], h8v (&o)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        o[0][e] = (_Float16)(v[e].x * sc);
        o[2][e] = (_Float16)(v[e].y * sc);
        o[1][e] = (_Float16)__builtin_fmaf(v[e].x, sc, -(float)o[0][e]);
        o[3][e] = (_Float16)__builtin_fmaf(v[e].y, sc, -(float)o[2][e]);
      }
    };
    auto column = [&](int q, int k, float2 (&v)[8]) __attribute__((always_inline)) {  // rows k .. of column q
      const f4v* p = (const f4v*)(X + (int64_t)q * n + k);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const f4v u = p[e];
        v[2 * e] = make_float2(u[0], u[1]);
        v[2 * e + 1] = make_float2(u[2], u[3]);
      }
    };
#pragma unroll 1
    for (int k = 0; k < T; k++) {
      const int k0 = 32 * k + 8 * g4;
      float2 vx[2][8], vy[CB][8];
#pragma unroll
      for (int c = 0; c < CB; c++) column(col0 + 16 * c, k0, vy[c]);
#pragma unroll
      for (int a = 0; a < 2; a++) {
        const int r = 32 * i + 16 * a + l15;
        if (i == k) {  // the diagonal tile: row r itself
#pragma unroll
          for (int e = 0; e < 8; e++) vx[a][e] = X[(int64_t)(k0 + e) * n + r];
        } else {
          column(r, k0, vx[a]);
        }
      }
      h8v x[2][4], y[4];
      split8(vx[0], x[0]);
      split8(vx[1], x[1]);
#pragma unroll
      for (int c = 0; c < CB; c++) {
        split8(vy[c], y);
        mma(x, y, re[c][0], re[c][1], im[c][0], im[c][1]);
      }
    }
    float vmax = 0.0f;
    const bool last = (ST == 2 && s == 0) || (ST == 3 && g.it + 1 == s);
    float2* const out = (last ? g.F : g.Y) + b * per;
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
      for (int a = 0; a < 2; a++) {
        const f4v r = re[c][a] * un, m = im[c][a] * un;
        const int row = row0 + 16 * a, col = col0 + 16 * c;
#pragma unroll
        for (int e = 0; e < 4; e++) vmax = fmaxf(vmax, fmaxf(fabsf(r[e]), fabsf(m[e])));
        if constexpr (ST < 2) {
          f4v br, bi, zr, zi, xr, xi;
          load4(B, a, c, br, bi);
          f4v* z = z_at(a, c);
          if constexpr (ST == 1) { zr = z[0]; zi = z[1]; }
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float2 bv = make_float2(br[e] * bscale, bi[e] * bscale), v = make_float2(r[e], m[e]);
            float2 x = cmac(v, ST == 0 ? g.c.c : g.c.d2, bv), w = v;
            if constexpr (ST == 1) {
              x = cmul(g.c.r, x);
              w = cmac(cmac(bv, g.c.g, make_float2(zr[e], zi[e])), g.c.e1, v);
            }
            zr[e] = w.x; zi[e] = w.y;
            xr[e] = x.x; xi[e] = x.y;
          }
          z[0] = zr;
          z[1] = zi;
          put_f(out, n, i, j, row, col, xr, xi);
        } else {
          put_f(out, n, i, j, row, col, r, m);
        }
      }
    if (!last) wave_max_to(vmax, g.max_out + b);
  }
}

template <int ST, int CB>
__global__ __launch_bounds__(64) void k_sym_few(FewArgs g) {
  const int T = g.n >> 5, per = T * (T + 1) / CB;  // waves of a matrix, which keep to one XCD's L2
  const int w = xcd_logical_block(blockIdx.x, gridDim.x), b = w / per, u = w % per;
  few_step<ST, CB>(g, b, CB == 2 ? u : u >> 1, CB == 2 ? 0 : u & 1, threadIdx.x);
}

template <int CB>
void few_steps(hipStream_t s, FewArgs g, float2* const work[4], float* maxima, int smax) {
  const int T = g.n / 32;
  const dim3 grid(g.nb * T * (T + 1) / CB), blk(64);
  g.B = work[0];
  g.Q = (float*)work[1];
  hipLaunchKernelGGL((k_sym_few<-1, CB>), grid, blk, 0, s, g);
  for (int i = 0; i < 3 + smax; i++) {
    g.X = work[2 + (i & 1)];
    g.Y = work[2 + ((i + 1) & 1)];
    g.max_in = maxima + (i % 3) * g.nb;
    g.max_out = maxima + ((i + 1) % 3) * g.nb;
    g.clear = maxima + ((i + 2) % 3) * g.nb;
    g.it = i - 3;
    if (i == 0) hipLaunchKernelGGL((k_sym_few<0, CB>), grid, blk, 0, s, g);
    else if (i == 1) hipLaunchKernelGGL((k_sym_few<1, CB>), grid, blk, 0, s, g);
    else if (i == 2) hipLaunchKernelGGL((k_sym_few<2, CB>), grid, blk, 0, s, g);
    else hipLaunchKernelGGL((k_sym_few<3, CB>), grid, blk, 0, s, g);
  }
}

}  // namespace

// Past 224 the operand and the accumulators do not fit on a CU, and k_sgemm's chain is taken: squares streamed
// through LDS, one product per launch, were up to 7% faster in large batches of 288-352 and 416 beams, up to 9%
// slower at 256 and 448-640, and 1.3-1.9 times slower for a single direction of any size.
bool sym_onchip(int n) { return n <= 224; }

// One, two, three and four-tile matrices: several workgroups per CU share the matrix cores; from
// five tiles on one workgroup of eight waves fills the CU.
void launch_expm_sym(hipStream_t s, int32_t n, int32_t nb, const float2* A, const int32_t* sq, const int32_t* bexp,
                     const float* bmax, float2* F, float2* Q, uint16_t* spill, int32_t cus, const SymCoef& c) {
  if (nb <= 0) return;
  const ExpmArgs a{A, sq, bexp, bmax, nb, F, (float*)Q, (_Float16*)spill, c};
  switch (n / 32) {
    case 1: return expm_case<1, 1, 1, 1, 3, 12>(s, nb, cus, a);
    case 2: return expm_case<2, 1, 3, 3, 2, 6>(s, nb, cus, a);
    case 3: return expm_case<3, 4, 2, 6, 2, 2>(s, nb, cus, a);
    case 4: return expm_case<4, 4, 3, 9, 2, 2>(s, nb, cus, a);
    case 5: return expm_case<5, 8, 2, 15, 2, 1>(s, nb, cus, a);
    case 6: return expm_case<6, 8, 3, 19, 2, 1>(s, nb, cus, a);
    case 7: return expm_case<7, 8, 4, 19, 2, 1>(s, nb, cus, a);
  }
}

// One MI355X, a run of bcc Fe with 20 depths [us], this / k_expm_sym / k_sgemm's chain. 161-187 beams: 1 direction
// 258 / 341 / 322, 48 directions 341 / 351 / 391, 56 365 / 351 / 393. 193-211 beams: 1 direction 292 / 467 / 357, 32 380 / 478 / 429,
// 56 478 / 487 / 472, 64 506 / 488 / 485. Smaller matrices are no slower in one launch than in k_sgemm's chain.
bool sym_few(int n, int nb) { return n > 160 && n <= 224 && nb <= n / 4; }

void launch_sym_few(hipStream_t s, int32_t n, int32_t nb, const float2* A, const int32_t* sq, const int32_t* bexp,
                    const float* bmax, float2* F, float2* const work[4], float* maxima, int32_t smax, const SymCoef& c) {
  const FewArgs g{A, sq, bexp, bmax, n, nb, 0, nullptr, nullptr, nullptr, F, nullptr, nullptr, nullptr, nullptr, c};
  // half as wide while there are fewer waves than SIMDs
  if (nb <= 12) few_steps<1>(s, g, work, maxima, smax);
  else few_steps<2>(s, g, work, maxima, smax);
}

}  // namespace ctem
