// Channeling patterns, up to 64 strong beams (include/ctem_ecp.h; larger sets take the batched
// products of ctem_api.hip): one workgroup per direction does everything after the dynamical matrix, with its
// matrices in LDS and registers. The batched form moves every product through memory (48 KB per
// 32 x 32 product of 0.26 MFLOP) and fills a quarter of its 64 x 64 tiles at 32 beams.
//
//   k_ecp_bloch_small   Blochwv: psi(t) = e^{At} e_1 and the thickness integral of psi^H S psi. With
//                       M(h) = int_0^h e^{A^H s} S e^{As} ds (Hermitian), the integral grows by
//                       psi^H M(h) psi per step h, and M(2h) = M(h) + E(h)^H M(h) E(h), E(2h) = E(h)^2:
//                       three products of the beams' size per doubling, where the exponential of the
//                       block matrix [[A, 0], [S, -A^H]] takes eight
//   k_ecp_scat_small    ScatMat: the program's Pade approximant (math.f90:187-315), the depth recursion
//                       and the per-depth contraction with S (CTEMECP.f90:559-618)
//
// 256 threads (1024 in Blochwv past 32 beams); products on v_mfma_f64_16x16x4_f64, each wave one part of the matrix. LDS
// matrices are column-major with one spare row, which keeps both operands' reads free of bank conflicts.
// Bound: FP64 matrix cores in Blochwv; in ScatMat half the time is the elimination, on the FP64 vector unit.
// Four workgroups per CU at 32 beams (35 KB of LDS, 128 registers), one at 64: with four waves there a single direction of
// 45 beams at 200-650 nm took 940 us, more than the batched form's 876, with sixteen 801. One MI355X, fcc Ni [001] at 30 kV,
// 16-32 beams, a pass against the batched form: Blochwv, 12,853 directions and 10 thicknesses, 19.9 -> 2.2 ms;
// ScatMat, 51,400 directions and 20 steps, 25.6 -> 5.2 ms. 40-57 beams (15 kV), 1,256 directions: Blochwv 12.7 -> 2.0,
// ScatMat 3.5 -> 1.2 ms. At 96 two matrices don't fit in LDS.
#include <hip/hip_runtime.h>

#include "ctem_ebsd.h"
#include "ctem_internal.h"

#pragma clang fp contract(off)

namespace ctem {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ void cmac(double2& s, double2 a, double2 b) {  // s += a b
  s.x = fma(-a.y, b.y, fma(a.x, b.x, s.x));
  s.y = fma(a.y, b.x, fma(a.x, b.y, s.y));
}
__device__ __forceinline__ double lane_of(double v, int l) {  // lane l's v, in scalar registers
  const uint64_t u = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, l), hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
  return __longlong_as_double(((uint64_t)hi << 32) | lo);
}

// max over the workgroup of NW waves, the same in every thread (a NaN wins); red: NW doubles of LDS
template <int NW>
__device__ __forceinline__ double block_max(double v, double* red) {
  auto mx = [](double a, double b) { return (a != a) ? a : ((b != b) ? b : fmax(a, b)); };
  for (int o = 32; o >= 1; o >>= 1) v = mx(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
#pragma unroll
  for (int w = 1; w < NW; w++) v = mx(v, red[w]);
  return v;
}

// The workgroup's view of NP x NP matrices (NP = 32 NT; four waves, each a quadrant, or sixteen): thread-owned
// entries (i, j, e) are row row(i, e), column col(j) of the wave's part, the accumulator layout of the products.
template <int NT, int NW = 4>
struct Wg {
  static constexpr int NP = 32 * NT, LD = NP + 1, WS = NW == 16 ? 4 : 2, TW = 2 * NT / WS, NTH = 64 * NW;
  typedef d4 Acc[TW][TW];
  int l16, l4, wr, wc, n, kn;
  // n: the matrix's own size; rows and columns from there on are those of the zero or the unit matrix,
  // and no sum over k goes past kn
  __device__ __forceinline__ explicit Wg(int n_) : n(n_), kn((n_ + 7) & ~7) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    l16 = lane & 15; l4 = lane >> 4;
    wr = (wave / WS) * 16 * TW; wc = (wave % WS) * 16 * TW;
  }
  __device__ __forceinline__ int row(int i, int e) const { return wr + 16 * i + l4 + 4 * e; }
  __device__ __forceinline__ int col(int j) const { return wc + 16 * j + l16; }
  template <class F>
  __device__ __forceinline__ void each(F f) const {
#pragma unroll
    for (int i = 0; i < TW; i++)
#pragma unroll
      for (int j = 0; j < TW; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) f(i, j, e, row(i, e), col(j));
  }
  // c = X Y, or X^H Y
  template <bool HERM>
  __device__ __forceinline__ void mul(const double2* X, const double2* Y, Acc& cr, Acc& ci) const {
#pragma unroll
    for (int i = 0; i < TW; i++)
#pragma unroll
      for (int j = 0; j < TW; j++) { cr[i][j] = (d4){0, 0, 0, 0}; ci[i][j] = (d4){0, 0, 0, 0}; }
    for (int k0 = 0; k0 < kn; k0 += 8)
#pragma unroll
    for (int k = k0; k < k0 + 8; k += 4) {
      double2 a[TW], b[TW];
#pragma unroll
      for (int i = 0; i < TW; i++) {
        const int r = wr + 16 * i + l16;
        a[i] = HERM ? X[r * LD + k + l4] : X[(k + l4) * LD + r];
        if (HERM) a[i].y = -a[i].y;
        b[i] = Y[(wc + 16 * i + l16) * LD + k + l4];
      }
#pragma unroll
      for (int i = 0; i < TW; i++)
#pragma unroll
        for (int j = 0; j < TW; j++) {
          cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].x, cr[i][j], 0, 0, 0);
          ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].y, ci[i][j], 0, 0, 0);
          cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[i].y, b[j].y, cr[i][j], 0, 0, 0);
          ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b[j].x, ci[i][j], 0, 0, 0);
        }
    }
  }
  __device__ __forceinline__ void put(double2* M, const Acc& r, const Acc& im) const {
    each([&](int i, int j, int e, int rr, int cc) { M[cc * LD + rr] = make_double2(r[i][j][e], im[i][j][e]); });
  }
  // x = X u, the sum of row tid / G in each of its G threads; y = this thread's part of row tid / G of
  // Y u (or Y conj(u))
  static constexpr int G = NTH / NP;
  template <bool CONJ>
  __device__ __forceinline__ void matvec2(const double2* X, const double2* Y, const double2* u, double2& x, double2& y) const {
    const int r = threadIdx.x / G, g = threadIdx.x % G;
    x = y = make_double2(0, 0);
#pragma unroll 4
    for (int c = g; c < kn; c += G) {
      const double2 v = u[c];
      cmac(x, X[c * LD + r], v);
      cmac(y, Y[c * LD + r], CONJ ? make_double2(v.x, -v.y) : v);
    }
    x.x += dpp_f64<0xb1>(x.x); x.y += dpp_f64<0xb1>(x.y);  // quad_perm [1,0,3,2]
    x.x += dpp_f64<0x4e>(x.x); x.y += dpp_f64<0x4e>(x.y);  // quad_perm [2,3,0,1]
    if (G >= 8) { x.x += dpp_f64<0x141>(x.x); x.y += dpp_f64<0x141>(x.y); }  // row_half_mirror
    if (G == 16) { x.x += dpp_f64<0x140>(x.x); x.y += dpp_f64<0x140>(x.y); }  // row_mirror
  }
  static constexpr size_t lds() { return (size_t)(2 * NP * LD + 2 * NP) * sizeof(double2) + 64 * sizeof(double); }
};

__device__ __forceinline__ double2 sgh_at(const DevRefl& R, const DevLut& L, int a, int b) {  // Sgh(hkl_a - hkl_b)
  const int32_t* x = R.hkl + 3 * a;
  const int32_t* y = R.hkl + 3 * b;
  return L.slut[(int64_t)(x[0] - y[0] - L.slo[0]) +
                (int64_t)L.sdim[0] * ((x[1] - y[1] - L.slo[1]) + (int64_t)L.sdim[1] * (x[2] - y[2] - L.slo[2]))];
}

// The launch's time, from its first workgroups' start to its last ones' end, without events around it (those cost
// 10 us a launch, of 60-150 for a hundred directions)
__device__ __forceinline__ void stat_begin(const EcpStat& s) {
  if (threadIdx.x == 0 && blockIdx.x < 64) atomicMax(s.clock, ~(unsigned long long)wall_clock64());
}
__device__ __forceinline__ void stat_end(const EcpStat& s) {
  if (threadIdx.x == 0 && blockIdx.x + 2048 >= gridDim.x) atomicMax(s.clock + 1, (unsigned long long)wall_clock64());
}

// Taylor at ||A h|| <= 1/8 (1-norms of A h and its conjugate transpose): E to degree 12 (five products), M to
// the term of degree 11 in the map X -> X A + (X A)^H (a product each); the first terms left out are
// below 1e-21 and 1e-17. A larger bound saves three products per doubling and costs as many here
constexpr double kThetaSmall = 0.125;
constexpr int kDegM = 11, kSmaxSmall = 51;  // 2^51 kThetaSmall is beyond the range of the larger sets' 48 squarings

template <int NT, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_ecp_bloch_small(Bucket B, BeamView V, DevRefl R, DevLut L, const double2* __restrict__ A1, double t0, double dt,
                       int nt, const float* __restrict__ thick, double nat, int numk, int32_t* __restrict__ err,
                       float* __restrict__ sr, EcpStat stat) {
  typedef Wg<NT, NW> W;
  constexpr int NP = W::NP, LD = W::LD;
  extern __shared__ double2 lds[];
  double2* const P0 = lds;
  double2* const P1 = lds + NP * LD;
  double2* const psi = P1 + NP * LD;
  double* const red = (double*)(psi + 2 * NP);
  const int b = blockIdx.x, dir = B.dirs[b], n = V.nns[dir], tid = threadIdx.x;
  stat_begin(stat);
  const W w(n);
  const int32_t* sidx = V.sidx + V.soff[dir];
  const double2* A = A1 + (int64_t)b * NP * NP;
  // the norms of A
  for (int e = tid; e < NP * NP; e += W::NTH) P0[(e / NP) * LD + e % NP] = A[e];
  __syncthreads();
  double nrm = 0.0;
  if (tid < 2 * NP) {
    const int q = tid % NP;
    for (int m = 0; m < NP; m++) {
      const double2 v = tid < NP ? P0[q * LD + m] : P0[m * LD + q];
      nrm += hypot(v.x, v.y);
    }
  }
  nrm = block_max<NW>(nrm, red);
  double2 sp[W::TW][W::TW][4];  // S^T: Sgh(hkl_c - hkl_r)
  w.each([&](int i, int j, int e, int r, int c) {
    sp[i][j][e] = (r < n && c < n) ? sgh_at(R, L, sidx[c], sidx[r]) : make_double2(0.0, 0.0);
  });

  // E(t) into P0 and M(t) into P1
  int products = 0;
  auto propagators = [&](double t) __attribute__((always_inline)) {
    int s = 0;
    double x = nrm * t;
    if (!isfinite(x)) {
      if (tid == 0) atomicOr(err, 2);
    } else {
      while (x > kThetaSmall && s < kSmaxSmall) { x *= 0.5; s++; }
      if (x > kThetaSmall && tid == 0) atomicOr(err, 4);
    }
    const double h = ldexp(t, -s);
    products += kDegM + 5 + 3 * s;
    typename W::Acc er, ei, mr, mi, cr, ci;
    __syncthreads();
    for (int e = tid; e < NP * NP; e += W::NTH) {
      const double2 v = A[e];
      P0[(e / NP) * LD + e % NP] = make_double2(v.x * h, v.y * h);
    }
    // M / h = S + L(S + L(S + ..) / 3) / 2
    w.each([&](int i, int j, int e, int r, int c) { P1[c * LD + r] = sp[i][j][e]; });
    __syncthreads();
    for (int k = kDegM + 1; k >= 2; k--) {
      w.template mul<false>(P1, P0, cr, ci);
      __syncthreads();
      w.put(P1, cr, ci);
      __syncthreads();
      const double f = 1.0 / k;
      w.each([&](int i, int j, int e, int r, int c) {
        const double2 v = P1[r * LD + c];  // the transposed entry
        mr[i][j][e] = sp[i][j][e].x + (cr[i][j][e] + v.x) * f;
        mi[i][j][e] = sp[i][j][e].y + (ci[i][j][e] - v.y) * f;
      });
      __syncthreads();
      if (k > 2) {
        w.put(P1, mr, mi);
        __syncthreads();
      }
    }
    // E = sum B^k / k!, in powers of B^3
    {
      typename W::Acc br, bi;
      w.each([&](int i, int j, int e, int r, int c) {
        const double2 v = P0[c * LD + r];
        br[i][j][e] = v.x;
        bi[i][j][e] = v.y;
        mr[i][j][e] *= h;
        mi[i][j][e] *= h;
      });
      w.template mul<false>(P0, P0, cr, ci);
      w.put(P1, cr, ci);
      __syncthreads();
      w.template mul<false>(P0, P1, er, ei);
      __syncthreads();
      w.put(P0, er, ei);
      w.each([&](int i, int j, int e, int r, int c) {
        constexpr double f9 = 1.0 / 362880, f10 = 1.0 / 3628800, f11 = 1.0 / 39916800, f12 = 1.0 / 479001600;
        P1[c * LD + r] = make_double2(
            (r == c ? f9 : 0.0) + (f10 * br[i][j][e] + (f11 * cr[i][j][e] + f12 * er[i][j][e])),
            f10 * bi[i][j][e] + (f11 * ci[i][j][e] + f12 * ei[i][j][e]));
      });
      __syncthreads();
      double f = 1.0 / 362880;
#pragma unroll
      for (int k = 6; k >= 0; k -= 3) {
        const double f2 = f * (k + 3), f1 = f2 * (k + 2);
        f = f1 * (k + 1);  // 1 / (k + 2)!, 1 / (k + 1)!, 1 / k!
        w.template mul<false>(P1, P0, er, ei);
        w.each([&](int i, int j, int e, int r, int c) {
          er[i][j][e] = (r == c ? f : 0.0) + (f1 * br[i][j][e] + (f2 * cr[i][j][e] + er[i][j][e]));
          ei[i][j][e] = f1 * bi[i][j][e] + (f2 * ci[i][j][e] + ei[i][j][e]);
        });
        __syncthreads();
        if (k > 0) {
          w.put(P1, er, ei);
          __syncthreads();
        }
      }
    }
    w.put(P0, er, ei);
    w.put(P1, mr, mi);
    __syncthreads();
    for (int q = 0; q < s; q++) {
      w.template mul<false>(P1, P0, cr, ci);  // M E
      __syncthreads();
      w.put(P1, cr, ci);
      __syncthreads();
      w.template mul<true>(P0, P1, cr, ci);  // E^H (M E)
      w.each([&](int i, int j, int e, int, int) { mr[i][j][e] += cr[i][j][e]; mi[i][j][e] += ci[i][j][e]; });
      w.template mul<false>(P0, P0, er, ei);
      __syncthreads();
      w.put(P0, er, ei);
      w.put(P1, mr, mi);
      __syncthreads();
    }
  };

  propagators(t0);
  double run = P1[0].x;
  if (tid < NP) psi[tid] = P0[tid];
  if (tid == 0) sr[dir] = (float)(run / (double)thick[0] / nat);
  if (nt >= 2 && dt != t0) propagators(dt);
  if (tid == 0) stat.nprod[dir] = products;
  __syncthreads();
  for (int it = 1; it < nt; it++) {
    const double2* u = psi + ((it - 1) & 1) * NP;
    double2 x, y;
    w.template matvec2<false>(P0, P1, u, x, y);
    const int r = tid / W::G;
    if (tid % W::G == 0) psi[(it & 1) * NP + r] = x;
    const double v = wave_sum(u[r].x * y.x + u[r].y * y.y);
    if ((tid & 63) == 0) red[NW * (it & 1) + (tid >> 6)] = v;
    __syncthreads();
    if (tid == 0) {
      const double* q = red + NW * (it & 1);
#pragma unroll
      for (int g = 0; g < NW; g += 4) run += (q[g] + q[g + 1]) + (q[g + 2] + q[g + 3]);
      sr[(int64_t)it * numk + dir] = (float)(run / (double)thick[it] / nat);
    }
  }
  stat_end(stat);
}

template <int NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, NT == 1 ? 4 : 1)))
void k_ecp_scat_small(Bucket B, BeamView V, DevRefl R, DevLut L, const double2* __restrict__ A1, int nz,
                      const int32_t* __restrict__ store, double nat, int numk, int32_t* __restrict__ err,
                      float* __restrict__ sr, EcpStat stat) {
  typedef Wg<NT> W;
  constexpr int NP = W::NP, LD = W::LD;
  extern __shared__ double2 lds[];
  double2* const P0 = lds;
  double2* const P1 = lds + NP * LD;
  double2* const psi = P1 + NP * LD;
  double* const red = (double*)(psi + 2 * NP);
  const int b = blockIdx.x, dir = B.dirs[b], n = V.nns[dir], tid = threadIdx.x;
  stat_begin(stat);
  const W w(n);
  const int32_t* sidx = V.sidx + V.soff[dir];
  const double2* A = A1 + (int64_t)b * NP * NP;
  typename W::Acc nr, ni, dr, di, cr, ci;
  // q and j from max |a_ij| (math.f90:208-219)
  double m = 0.0;
  for (int e = tid; e < NP * NP; e += 256) {
    const double2 v = A[e];
    const double a = hypot(v.x, v.y);
    m = (a > m || a != a) ? a : m;
    P0[(e / NP) * LD + e % NP] = v;
  }
  m = block_max<4>(m, red);
  int ilev = 1;
  if (!(m == m) || m > 1000.0) {
    if (tid == 0) atomicOr(err, 4);
  } else if (m > 0.0) {
    ilev = (int)round(log10(m)) + 3;
    ilev = ilev < 1 ? 1 : ilev > 6 ? 6 : ilev;
  }
  const int q = ilev == 1 ? 2 : ilev == 2 ? 3 : 4;
  const int j2 = ilev <= 2 ? 0 : ilev == 3 ? 1 : ilev == 4 ? 5 : ilev == 5 ? 8 : 11;
  const double sc = ldexp(1.0, -j2);
  if (tid == 0) stat.nprod[dir] = q - 1 + j2;
  // N = sum pref_i B^i, D = sum (-1)^i pref_i B^i with the reference's running product pref
  w.each([&](int i, int j, int e, int r, int c) {
    double2 v = P0[c * LD + r];
    v.x *= sc; v.y *= sc;
    P0[c * LD + r] = v;
    P1[c * LD + r] = v;
    cr[i][j][e] = v.x; ci[i][j][e] = v.y;
    nr[i][j][e] = dr[i][j][e] = r == c ? 1.0 : 0.0;
    ni[i][j][e] = di[i][j][e] = 0.0;
  });
  __syncthreads();
  double pref = 1.0;
  for (int t = 1; t <= q; t++) {
    if (t > 1) {
      w.template mul<false>(P1, P0, cr, ci);
      __syncthreads();
      if (t < q) {
        w.put(P1, cr, ci);
        __syncthreads();
      }
    }
    pref = pref * (double)(q - t + 1) / (double)t / (double)(2 * q - t + 1);
    const double sp = (t & 1) ? -pref : pref;
    w.each([&](int i, int j, int e, int, int) {
      nr[i][j][e] += pref * cr[i][j][e]; ni[i][j][e] += pref * ci[i][j][e];
      dr[i][j][e] += sp * cr[i][j][e]; di[i][j][e] += sp * ci[i][j][e];
    });
  }
  __syncthreads();
  w.put(P0, dr, di);
  w.put(P1, nr, ni);
  __syncthreads();
  // E = D^-1 N by Gauss-Jordan elimination on [D | N] in registers: a wave holds NP / 4 rows, a lane one column
  // of them (two at 64 beams), so a column's multipliers are another lane's registers. One barrier a step:
  // every wave offers the row of its largest |re| + |im| in the column, with that value, in LDS; the
  // largest of the four is the pivot. Rows are not moved (iperm: the row of the solution a row holds) and are
  // divided by their pivots at the end. Column k >= n of D is a unit vector.
  {
    constexpr int NC = 2 * NP, Q = NC / 64, RW = NP / 4;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r0 = wave * RW;
    double2 v[Q][RW];
#pragma unroll
    for (int x = 0; x < Q; x++) {
      const int c = lane + 64 * x;
      const double2* src = c < NP ? P0 + c * LD : P1 + (c - NP) * LD;
#pragma unroll
      for (int t = 0; t < RW; t++) v[x][t] = src[r0 + t];
    }
    __syncthreads();
    double2* crow = P1;                       // [2][4][NC]: the offered rows, two sets in turn
    uint64_t* ckey = (uint64_t*)red;          // [2][4]: their values, the row's number in the lowest bits
    double2* dinv = psi;                      // [NP]: 1 / pivot of a row
    int* iperm = (int*)(red + 16);            // [NP]
    if (tid < NP) { dinv[tid] = make_double2(1.0, 0.0); iperm[tid] = tid; }
    unsigned used = 0;
    for (int k = 0; k < n; k++) {
      const int z = k & 1;
      double best = 0.0;
#pragma unroll
      for (int t = 0; t < RW; t++) {
        const uint64_t u = __double_as_longlong(fabs(v[0][t].x) + fabs(v[0][t].y));
        const double a = __longlong_as_double((u & ~(uint64_t)63) | (uint64_t)(r0 + t));
        best = fmax(best, (used >> t & 1u) ? 0.0 : a);
      }
      best = lane_of(best, k);
      const int mine = (int)(__double_as_longlong(best) & 63) - r0;
#pragma unroll
      for (int t = 0; t < RW; t++)
        if (t == mine || (t == 0 && mine < 0))
#pragma unroll
          for (int x = 0; x < Q; x++) crow[(z * 4 + wave) * NC + lane + 64 * x] = v[x][t];
      if (lane == 0) ckey[z * 4 + wave] = __double_as_longlong(best);
      __syncthreads();
      uint64_t key = ckey[z * 4];
#pragma unroll
      for (int g = 1; g < 4; g++) key = max(key, ckey[z * 4 + g]);
      const int p = __builtin_amdgcn_readfirstlane((int)(key & 63));
      const double2* pr = crow + (z * 4 + p / RW) * NC;
      const double2 d = pr[k];
      const double den = d.x * d.x + d.y * d.y, ri = 1.0 / den;
      const double2 inv = key < 64 || !(den > 0.0) ? make_double2(1.0, 0.0) : make_double2(d.x * ri, -(d.y * ri));
      if (tid == 0) {
        if (key < 64) atomicOr(err, 2);
        dinv[p] = inv;
        iperm[p] = k;
      }
      double2 mt[RW];
#pragma unroll
      for (int t = 0; t < RW; t++) {
        mt[t].x = lane_of(v[0][t].x, k);
        mt[t].y = lane_of(v[0][t].y, k);
        if (r0 + t == p) mt[t] = make_double2(0.0, 0.0);
      }
      if ((unsigned)(p - r0) < (unsigned)RW) used |= 1u << (p - r0);
#pragma unroll
      for (int x = 0; x < Q; x++) {
        const double2 g = pr[lane + 64 * x];
        const double2 u = cmul(make_double2(-g.x, -g.y), inv);
#pragma unroll
        for (int t = 0; t < RW; t++) cmac(v[x][t], mt[t], u);
      }
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < Q; x++) {
      const int c = lane + 64 * x;
      if (c >= NP)
#pragma unroll
        for (int t = 0; t < RW; t++) P0[(c - NP) * LD + iperm[r0 + t]] = cmul(v[x][t], dinv[r0 + t]);
    }
    __syncthreads();
  }
  for (int t = 0; t < j2; t++) {
    w.template mul<false>(P0, P0, cr, ci);
    __syncthreads();
    w.put(P0, cr, ci);
    __syncthreads();
  }
  // psi_z = E^z e_1 and d_z = Re psi_z^T Sgh conj(psi_z), summed over the depths
  w.each([&](int i, int j, int e, int r, int c) {
    P1[c * LD + r] = (r < n && c < n) ? sgh_at(R, L, sidx[r], sidx[c]) : make_double2(0.0, 0.0);
  });
  if (tid < NP) psi[tid] = P0[tid];
  __syncthreads();
  double run = 0.0;
  for (int z = 0; z < nz; z++) {
    const double2* u = psi + (z & 1) * NP;
    double2 x, y;
    w.template matvec2<true>(P0, P1, u, x, y);
    const int r = tid / W::G, t = store[z];
    if (tid % W::G == 0) psi[((z + 1) & 1) * NP + r] = x;
    run += u[r].x * y.x - u[r].y * y.y;  // this thread's part of the sum over the depths
    if (t >= 0) {
      const double v = wave_sum(run);
      if ((tid & 63) == 0) red[4 * (z & 1) + (tid >> 6)] = v;
    }
    __syncthreads();
    if (t >= 0 && tid == 0) {
      const double* q = red + 4 * (z & 1);
      sr[(int64_t)t * numk + dir] = (float)(((q[0] + q[1]) + (q[2] + q[3])) / nat);
    }
  }
  stat_end(stat);
}

}  // namespace

// two matrices and the exchange buffers in LDS: 35 KB at 32 beams, 136 KB at 64
bool ecp_small(int npad) { return npad <= 64; }

void launch_ecp_bloch_small(hipStream_t s, const Bucket& B, const BeamView& V, const DevRefl& R, const DevLut& L,
                            const double2* A1, double t0, double dt, int32_t nt, const float* thick, double nat,
                            int32_t numk, int32_t* err, float* sr, const EcpStat& stat) {
  if (B.npad == 32)
    hipLaunchKernelGGL((k_ecp_bloch_small<1, 4>), dim3(B.nb), dim3(256), Wg<1>::lds(), s, B, V, R, L, A1, t0, dt, nt, thick,
                       nat, numk, err, sr, stat);
  else
    hipLaunchKernelGGL((k_ecp_bloch_small<2, 16>), dim3(B.nb), dim3(1024), Wg<2>::lds(), s, B, V, R, L, A1, t0, dt, nt, thick,
                       nat, numk, err, sr, stat);
}

void launch_ecp_scat_small(hipStream_t s, const Bucket& B, const BeamView& V, const DevRefl& R, const DevLut& L,
                           const double2* A1, int32_t nz, const int32_t* store, double nat, int32_t numk, int32_t* err,
                           float* sr, const EcpStat& stat) {
  if (B.npad == 32)
    hipLaunchKernelGGL(k_ecp_scat_small<1>, dim3(B.nb), dim3(256), Wg<1>::lds(), s, B, V, R, L, A1, nz, store, nat, numk,
                       err, sr, stat);
  else
    hipLaunchKernelGGL(k_ecp_scat_small<2>, dim3(B.nb), dim3(256), Wg<2>::lds(), s, B, V, R, L, A1, nz, store, nat, numk,
                       err, sr, stat);
}

}  // namespace ctem
