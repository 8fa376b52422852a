// The exponential's products of the split mixed form for complex-symmetric matrices (the storage
// idea, split-FP16 planes with one exponent per matrix, is that of ctem_split.hip).
//
// With X = X^T the square C = X X has C(i, j) = sum over k of X(i, k) X(j, k): both operands of a
// step are rows of one strip, the matrix at 32 columns k, and every 32 x 32 output tile (i <= j) takes its
// A operand from the strip's row tile i and its B operand from row tile j, both as 8 consecutive k of
// one row per lane. The polynomial of the exponential is therefore evaluated by squares only
// (sym_coef in ctem_api.hip), and a workgroup keeps the whole upper triangle of a product in its accumulators.
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
// hold a matrix whose last nine tiles wait in a global buffer until their places are free.
//
// Measured on one MI355X, the exponentials of a run against k_sgemm's chain (64 x 64 tiles, three general
// products for a degree-8 polynomial; it moves 2.3 MB to LDS per product at n = 224 and waits for memory):
// bcc Fe, 63,252 directions of 188-250 beams: 141 -> 91 ms, 9 products per matrix instead of 8; fcc Ni, 1,326 of
// 87-115: 1.02 -> 0.51 ms. At n = 224 a strip of a squaring takes
// ~8,100 cycles where its matrix-core work is 5,376 (7 tiles per SIMD); the rest is the wait for LDS after each
// barrier, and ~16,000 cycles per product between products.
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

__device__ __forceinline__ void split2(float s, _Float16& hi, _Float16& lo) {
  hi = (_Float16)s;
  lo = (_Float16)(s - (float)hi);
}

// two FP32 complex entries of one column (re, im, re, im), scaled, into the four planes at dst
__device__ __forceinline__ void put_pair(_Float16* dst, const f4v& r, float f) {
  h2v o[4];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    _Float16 h, l;
    split2(r[2 * t] * f, h, l); o[0][t] = h; o[1][t] = l;
    split2(r[2 * t + 1] * f, h, l); o[2][t] = h; o[3][t] = l;
  }
#pragma unroll
  for (int p = 0; p < 4; p++) *(h2v*)(dst + p * kPlane) = o[p];
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
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int c = 0; c < 2; c++) { re[a][c] = (f4v){0, 0, 0, 0}; im[a][c] = (f4v){0, 0, 0, 0}; }
  }
  // += A B^T over 32 k for column block c. The twelve products go into fresh sums, added to the
  // accumulators by rounded FP32 additions: the matrix cores' own accumulation does not round to nearest, and
  // over a whole product its one-sided errors add up (intensities of fcc Ni 9.2e-7 from the 64-bit ones with
  // the products accumulated in place). The imaginary planes of B are negated for the last terms,
  // -Im A Im B. Smallest terms first.
  __device__ __forceinline__ void mma(const h8v (&x)[2][4], h8v (&y)[4], int c) {
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
#pragma unroll
    for (int a = 0; a < 2; a++) { re[a][c] += r[a]; im[a][c] += i[a]; }
  }
  // += f X for the tile image at t (stored units)
  template <bool REAL>
  __device__ __forceinline__ void add_image(const _Float16* t, float fr, float fi, int l15, int g) {
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const _Float16* o = t + chunk_off(16 * c + l15, 2 * a + (g >> 1)) + 4 * (g & 1);
        const h4v p0 = *(const h4v*)o, p1 = *(const h4v*)(o + kPlane);
        const h4v p2 = *(const h4v*)(o + 2 * kPlane), p3 = *(const h4v*)(o + 3 * kPlane);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          float r = __builtin_fmaf(fr, (float)p1[e], re[a][c][e]), i = __builtin_fmaf(fr, (float)p3[e], im[a][c][e]);
          if (!REAL) {
            r = __builtin_fmaf(-fi, (float)p3[e], r);
            i = __builtin_fmaf(fi, (float)p1[e], i);
          }
          r = __builtin_fmaf(fr, (float)p0[e], r);
          i = __builtin_fmaf(fr, (float)p2[e], i);
          if (!REAL) {
            r = __builtin_fmaf(-fi, (float)p2[e], r);
            i = __builtin_fmaf(fi, (float)p0[e], i);
          }
          re[a][c][e] = r;
          im[a][c][e] = i;
        }
        __builtin_amdgcn_sched_barrier(0);  // one subtile's planes in registers at a time
      }
  }
};

// tile t of the upper triangle in row order (row i: (i, i) .. (i, T - 1))
__device__ __forceinline__ int row_tile(int t, int T, int& j) {
  int i = 0;
  while (t >= T - i) { t -= T - i; i++; }
  j = i + t;
  return i;
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b) { return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }

// ---- the whole exponential on chip ------------------------------------------------------------

struct ExpmArgs {
  const float2* A;      // [nb][n n] assembled matrices (column-major FP32; tiles on and above the diagonal)
  const int32_t* sq;    // squaring counts, exponents of B = A 2^-s
  const int32_t* bexp;
  int32_t nb;
  float2* F;            // [nb][n n] out: exp(A) - I, both triangles
  float* Q;             // [workgroups][N 2048] work: the terms of step 2 in B and Q1, FP32
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
  // B into tile images: two rows of one column per lane, an eighth of a tile (four columns) per wave and
  // turn, the loads of several turns in flight
  {
    constexpr int HT = 8 * N / NW, AT = HT < 14 ? HT : 14;
    const float f = ldexpf(bscale, ex);
    const int lr = 2 * l15;
#pragma unroll 1
    for (int m0 = 0; m0 < HT; m0 += AT) {
      f4v v[AT];
#pragma unroll
      for (int m = 0; m < AT; m++) {
        const int h = min(wave + (m0 + m) * NW, 8 * N - 1);
        int j;
        const int i = row_tile(h >> 3, T, j);
        v[m] = *(const f4v*)(A + (int64_t)(32 * j + 4 * (h & 7) + g4) * n + 32 * i + lr);
      }
#pragma unroll
      for (int m = 0; m < AT; m++) {
        const int h = wave + (m0 + m) * NW, r = h >> 3;
        if (h >= 8 * N) break;
        _Float16* dst = (N > NSL && r >= NSL) ? spill + (r - NSL) * kTile : Ls + r * kTile;
        put_pair(dst + chunk_off(4 * (h & 7) + g4, lr >> 3) + (lr & 7), v[m], f);
      }
    }
  }

  const Reader rd(lane);
  Acc acc[NS];
  float un = 1.0f;  // accumulator units 2^(-2 ex)
  // one product, v = alpha (X X + bx X + bb B + bq Q1): steps 0 to 2 of the polynomial, 3 a squaring. Code of
  // its own for each, so that nothing but the products decides what becomes of the accumulators.
  auto product = [&](auto st) __attribute__((always_inline)) {
    constexpr int ST = decltype(st)::value;
    const float up = ldexpf(1.0f, 2 * ex);
    un = ldexpf(1.0f, -2 * ex);
    float2 fx = ST < 3 ? g.c.bx[ST < 3 ? ST : 0] : make_float2(2.0f, 0.0f);
    fx.x = ldexpf(fx.x, ex);
    fx.y = ldexpf(fx.y, ex);
    if constexpr (ST == 1 || ST == 2) {
      // the accumulators hold the terms in B and Q1 (in flight: next_operand asked for them)
      const float f = ST == 1 ? bscale * up : up;
#pragma unroll
      for (int t = 0; t < 4 * NS; t++) {
        const int q = t >> 2, a = (t >> 1) & 1, c = t & 1;
        const f4v m0 = acc[q].re[a][c], m1 = acc[q].im[a][c];
        if constexpr (ST == 2) {
          acc[q].re[a][c] = m0 * f;
          acc[q].im[a][c] = m1 * f;
        } else {
          const float2 bb = make_float2(g.c.bb[1].x * f, g.c.bb[1].y * f);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float2 y = cmul(bb, e < 2 ? make_float2(m0[2 * e], m0[2 * e + 1]) : make_float2(m1[2 * e - 4], m1[2 * e - 3]));
            acc[q].re[a][c][e] = y.x;
            acc[q].im[a][c][e] = y.y;
          }
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < NS; q++) acc[q].zero();
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
          rd.read(t, 0, sj[q] <= k, y[0]);
          acc[q].mma(x, y[0], 0);
          rd.read(t, 1, sj[q] <= k, y[1]);
          acc[q].mma(x, y[1], 1);
          if (sj[q] == k) {
            const _Float16* t = row_at(k, si[q]);
            acc[q].template add_image<ST == 3>(t, fx.x, fx.y, l15, g4);
          }
        }
    }
    if constexpr (ST == 2) {  // the other steps have alpha = 1
#pragma unroll
      for (int t = 0; t < 4 * NS; t++) {
        const int q = t >> 2, a = (t >> 1) & 1, c = t & 1;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float2 z = cmul(g.c.alpha[2], make_float2(acc[q].re[a][c][e], acc[q].im[a][c][e]));
          acc[q].re[a][c][e] = z.x;
          acc[q].im[a][c][e] = z.y;
        }
      }
    }
  };
  // the accumulators become the next operand, with the exponent from their exact maximum over the
  // workgroup. Ahead of step 1 the terms of step 2 in B and Q1 go to memory; ahead of steps 1 and 2 the
  // freed accumulators receive the step's terms.
  auto next_operand = [&](auto st) __attribute__((always_inline)) {
    constexpr int ST = decltype(st)::value;
    // the lane's place, opaque to the compiler: it would otherwise keep every address in registers
    // through the products
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int l15 = ln & 15, g4 = ln >> 4;
    auto b_at = [&](int q, int a, int c) __attribute__((always_inline)) {
      return (const f4v*)(A + (int64_t)(32 * sj[q] + 16 * c + l15) * n + 32 * si[q] + 16 * a + 4 * g4);
    };
    auto z_at = [&](int q, int a, int c) __attribute__((always_inline)) {
      return (f4v*)(Q + (int64_t)min(t0 + q, N - 1) * 2048) + ln * 2 + (2 * a + c) * 128;
    };
    f4v m[2][2][2];
    auto ask = [&](int q) __attribute__((always_inline)) {
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const f4v* p = b_at(q, a, c);
          m[a][c][0] = p[0];
          m[a][c][1] = p[1];
        }
    };
    if constexpr (ST == 1 && NS < 4) ask(0);
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
    ex = f16_scale_exp(vmax * un);
    const float sc = ldexpf(un, ex);
    const float2 bb = make_float2(g.c.bb[2].x * bscale, g.c.bb[2].y * bscale);
    const float2 bq = make_float2(g.c.bq[2].x * un, g.c.bq[2].y * un);
#pragma unroll
    for (int q = 0; q < NS; q++) {
      if constexpr (ST == 1 && NS >= 4) ask(q);  // (asked for one tile ahead, they spill)
      if (q < cnt) {
        const int r = t0 + q;
        _Float16* dst = (N > NSL && r >= NSL) ? spill + (r - NSL) * kTile : Ls + r * kTile;
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int c = 0; c < 2; c++) {
            put_rows(dst + chunk_off(16 * c + l15, 2 * a + (g4 >> 1)) + 4 * (g4 & 1), acc[q].re[a][c], acc[q].im[a][c], sc);
            if constexpr (ST == 1) {
              f4v zr, zi;
#pragma unroll
              for (int e = 0; e < 4; e++) {
                const float2 y = cmul(bb, make_float2(m[a][c][e >> 1][2 * (e & 1)], m[a][c][e >> 1][2 * (e & 1) + 1]));
                const float2 z = cmul(bq, make_float2(acc[q].re[a][c][e], acc[q].im[a][c][e]));
                zr[e] = y.x + z.x;
                zi[e] = y.y + z.y;
              }
              f4v* p = z_at(q, a, c);
              p[0] = zr;
              p[1] = zi;
            }
          }
      }
      if constexpr (ST == 1) {
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int c = 0; c < 2; c++) { acc[q].re[a][c] = m[a][c][0]; acc[q].im[a][c] = m[a][c][1]; }
        if (NS < 4 && q + 1 < NS) ask(q + 1);
      }
      if constexpr (ST == 2)
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int c = 0; c < 2; c++) {
            const f4v* p = z_at(q, a, c);
            acc[q].re[a][c] = p[0];
            acc[q].im[a][c] = p[1];
          }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
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
          const f4v vr = acc[q].re[a][c] * un, vi = acc[q].im[a][c] * un;
          f4v* p = (f4v*)(F + (int64_t)col * n + row);
          p[0] = (f4v){vr[0], vi[0], vr[1], vi[1]};
          p[1] = (f4v){vr[2], vi[2], vr[3], vi[3]};
          if (i != j)
#pragma unroll
            for (int e = 0; e < 4; e++) F[(int64_t)(row + e) * n + col] = make_float2(vr[e], vi[e]);
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

}  // namespace

// Past 224 the operand and the accumulators do not fit on a CU, and k_sgemm's chain is taken: squares streamed
// through LDS, one product per launch, were up to 7% faster in large batches of 288-352 and 416 beams, up to 9%
// slower at 256 and 448-640, and 1.3-1.9 times slower for a single direction of any size.
bool sym_onchip(int n) { return n <= 224; }

// One, two, three and four-tile matrices: several workgroups per CU share the matrix cores; from
// five tiles on one workgroup of eight waves fills the CU.
void launch_expm_sym(hipStream_t s, int32_t n, int32_t nb, const float2* A, const int32_t* sq, const int32_t* bexp,
                     float2* F, float2* Q, uint16_t* spill, int32_t cus, const SymCoef& c) {
  if (nb <= 0) return;
  const ExpmArgs a{A, sq, bexp, nb, F, (float*)Q, (_Float16*)spill, c};
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

}  // namespace ctem
