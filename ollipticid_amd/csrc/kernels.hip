// CDNA4 (gfx950) kernels of the FAS puncture solver.
//
// All stencils are axis stars of radius R = order/2, so the points split
// into R+1 colours (i+j+k) mod (R+1) with no same-colour neighbours: one
// launch updates one colour of every listed box.  A launch works on a
// device-resident item list whose boxes may belong to many hierarchies
// (requests); arithmetic is float64 throughout.
//
// Reference counterparts (WuShichao/OllipticID):
//   k_smooth            elliptic.cc:1126-1242 Smooth, elliptic.h:405-445 ops
//   k_residual          elliptic.cc:944-991 App_Ell_Operator
//   k_robin_*           boundary.cc:447-1101 App_Bound, :1118-1710 operator
//   k_restrict_u        elliptic.cc:1543-1546 (Transferir INSIDE LAGRANGE 3)
//   k_restrict_defect   elliptic.cc:1625-1747 (W = S - R, restrict, S = W + R)
//   k_prolong           elliptic.cc:1827-1902 (V = u - ww, LINEAR, u += V)
//   k_ghost_fill, k_ghost_tiles  elliptic.cc:1905-1908 (BOUNDARY LAGRANGE order+1)
//   k_coarse_solve      elliptic.cc:1782-1816 (coarsest-level loop)
//   k_coefficients      operator.cc:752-868, 2193-2380 (b, c, d, e)
//   k_adm_sphere        elliptic.cc:2447-2611 Compute_ADM_Mass
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdio>

#include "kernels.hpp"

// No implicit contraction: every kernel's rounding is fixed by its source,
// whatever the launch shape or unrolling (a request solves to the same bits
// alone and in a batch).  Hot expressions use explicit fma.
#pragma clang fp contract(off)

namespace oll {

namespace {

constexpr double kEps = DBL_EPSILON;

// ------------------------------------------------------------------
// point operators
// ------------------------------------------------------------------

// axis-star second differences (explicit fma; shared by all stencil kernels)
template <int ORD, typename T>
__device__ __forceinline__ T star(T u0, T s1, T s2, T s3, T s4) {
  if constexpr (ORD == 2) {
    return fma(T(-2), u0, s1);
  } else if constexpr (ORD == 4) {
    return fma(T(-30), u0, fma(T(16), s1, -s2));
  } else if constexpr (ORD == 6) {
    return fma(T(-490), u0, fma(T(270), s1, fma(T(-27), s2, T(2) * s3)));
  } else {
    return fma(T(-14350), u0, fma(T(8064), s1, fma(T(-1008), s2, fma(T(128), s3, T(-9) * s4))));
  }
}
template <int ORD, typename T>
__device__ __forceinline__ T star_sum(T ax, T ay, T az, T ix2, T iy2, T iz2) {
  const T s = fma(ax, ix2, fma(ay, iy2, az * iz2));
  if constexpr (ORD == 2) return s;
  else if constexpr (ORD == 4) return s * (T(1) / T(12));
  else if constexpr (ORD == 6) return s * (T(1) / T(180));
  else return s * (T(1) / T(5040));
}

// axis-star Laplacian at element index p of an array (LDS); neighbour
// element offsets from stencil_offs<NC, 1>
template <int ORD, typename T = double, int NC = ORD / 2 + 1>
__device__ __forceinline__ T lap(const T *__restrict__ u, int p, const Nbr<NC> &n, T ix2,
                                 T iy2, T iz2) {
  constexpr int R = ORD / 2;
  T sx[4] = {0, 0, 0, 0}, syv[4] = {0, 0, 0, 0}, szv[4] = {0, 0, 0, 0};
#pragma unroll
  for (int m = 1; m <= R; ++m) {
    sx[m - 1] = u[p + int(n.xp[m - 1])] + u[p + int(n.xm[m - 1])];
    syv[m - 1] = u[p + int(n.yp[m - 1])] + u[p + int(n.ym[m - 1])];
    szv[m - 1] = u[p + int(n.zp[m - 1])] + u[p + int(n.zm[m - 1])];
  }
  const T u0 = u[p];
  return star_sum<ORD, T>(star<ORD, T>(u0, sx[0], sx[1], sx[2], sx[3]),
                          star<ORD, T>(u0, syv[0], syv[1], syv[2], syv[3]),
                          star<ORD, T>(u0, szv[0], szv[1], szv[2], szv[3]), ix2, iy2, iz2);
}

// N(u) and dN/du_p: EQ 0 Lap u + b (c+u)^-7, EQ 1 + d (c+u) + e (c+u)^5,
// EQ 2 Lap u + u^2, EQ 3 Lap u + b u (c = 0 for EQ 2, 3, so cu = u)
// (NEWTON: 1 / cu by div_newton)
__device__ __forceinline__ double div_newton(double a, double b);
template <int EQ, bool NEWTON = false>
__device__ __forceinline__ void nonlinear(double lapu, double dulap, double b, double cu,
                                          double dd, double ee, double &N, double &dN) {
  if constexpr (EQ == 2) {
    N = lapu + cu * cu;
    dN = dulap + 2.0 * cu;
    return;
  } else if constexpr (EQ == 3) {
    N = lapu + b * cu;
    dN = dulap + b;
    return;
  }
  const double inv = NEWTON ? div_newton(1.0, cu) : 1.0 / cu;
  const double inv2 = inv * inv;
  const double inv4 = inv2 * inv2;
  const double inv7 = inv4 * inv2 * inv;
  const double inv8 = inv4 * inv4;
  N = fma(b, inv7, lapu);
  dN = fma(-7.0 * b, inv8, dulap);
  if constexpr (EQ == 1) {
    const double c2 = cu * cu;
    const double c4 = c2 * c2;
    N = fma(ee, c4 * cu, fma(dd, cu, N));
    dN = fma(5.0 * ee, c4, dN + dd);
  }
}

// Punctures_EM (elliptic.h:510-626) at an interior point: u, its gradient g
// (du: each derivative's coefficient of u_p) and, from the mass and charge
// potentials eta, phi and their gradients ge, gf, the thirteen coefficients
// (elliptic.h:1458-1530)
//   N  = Lap u + num / den,
//   num = B |g|^2 + (B1 u + B2).g + C u^2 + D u + E,
//   den = u^3 + A1 u^2 + A2 u + A3,
// and dN/du_p
__device__ __forceinline__ void em_nonlinear(double lapu, double dulap, double u, const double g[3],
                                             const double du[3], double eta, double phi,
                                             const double ge[3], const double gf[3], double &N,
                                             double &dN) {
  const double f2 = gf[0] * gf[0] + gf[1] * gf[1] + gf[2] * gf[2];
  const double fe = gf[0] * ge[0] + gf[1] * ge[1] + gf[2] * ge[2];
  const double e2 = ge[0] * ge[0] + ge[1] * ge[1] + ge[2] * ge[2];
  const double a1 = 3 * eta;
  const double a2 = 3 * (eta * eta) - 0.25 * (phi * phi);
  const double a3 = eta * eta * eta - 0.25 * eta * phi * phi;
  const double bb = -0.25 * (phi * phi);
  const double cc = -0.25 * f2;
  const double dd = 0.5 * phi * fe - 0.5 * eta * f2;
  const double ee = -0.25 * phi * phi * e2 + 0.5 * phi * eta * fe + 0.25 * (1 - eta * eta) * f2;
  double b1[3], b2[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    b1[a] = 0.5 * phi * gf[a];
    b2[a] = 0.5 * phi * (eta * gf[a] - phi * ge[a]);
  }
  const double u2 = u * u;
  const double num = bb * (g[0] * g[0] + g[1] * g[1] + g[2] * g[2]) + (b1[0] * u + b2[0]) * g[0] +
                     (b1[1] * u + b2[1]) * g[1] + (b1[2] * u + b2[2]) * g[2] + cc * u2 + dd * u + ee;
  const double den = u2 * u + a1 * u2 + a2 * u + a3;
  const double dnum = 2 * bb * (g[0] * du[0] + g[1] * du[1] + g[2] * du[2]) + (b1[0] * u + b2[0]) * du[0] +
                      b1[0] * g[0] + (b1[1] * u + b2[1]) * du[1] + b1[1] * g[1] +
                      (b1[2] * u + b2[2]) * du[2] + b1[2] * g[2] + 2 * cc * u + dd;
  N = lapu + num / den;
  dN = dulap + (dnum * den - num * (3 * u2 + 2 * a1 * u + a2)) / (den * den);
}


// Norm slots: non-negative doubles order like their bit patterns, so a max
// is an unsigned atomic max.  The atomic returns nothing, so the issuing
// wave does not wait for it.
__device__ __forceinline__ void norm_update(unsigned long long *slot, double v) {
  unsigned long long *s = slot + (blockIdx.x & (kNormSubSlots - 1)) * kNormStride;
  atomicMax(s, (unsigned long long)__double_as_longlong(v));
}

// exact g / d for g < 2^24 via a float reciprocal and one correction step
__device__ __forceinline__ unsigned fast_div(unsigned g, unsigned d, float inv_d) {
  unsigned q = unsigned(float(g) * inv_d);
  if (q * d > g) --q;
  else if ((q + 1) * d <= g) ++q;
  return q;
}

// coordinate of index i, lo + i d rounded twice as on the host (the file's
// contract(off) keeps the two operations apart; the __dmul_rn/__dadd_rn
// helpers are compiled under the headers' own contraction setting and fuse)
__device__ __forceinline__ double coord(const DevBox &B, int a, int i) {
  return B.lo[a] + (double)i * B.d[a];
}

__device__ __forceinline__ bool interior(const DevBox &B, int i, int j, int k) {
  const int R = B.R;
  return i >= R && i < B.n[0] - R && j >= R && j < B.n[1] - R && k >= R && k < B.n[2] - R;
}

__device__ __forceinline__ void point_ijk(const DevBox &B, long long q, int &i, int &j, int &k) {
  const unsigned n0 = unsigned(B.n[0]), n1 = unsigned(B.n[1]);
  const unsigned qq = unsigned(q);
  const unsigned plane = n0 * n1;
  k = int(qq / plane);
  const unsigned r = qq - unsigned(k) * plane;
  j = int(r / n0);
  i = int(r - unsigned(j) * n0);
}

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own
// L2.  Remapping so that XCD x runs one contiguous run of logical blocks
// keeps the rows and planes a stencil shares inside one L2.
constexpr unsigned kXcds = 8;
__device__ __forceinline__ unsigned xcd_block() {
  const unsigned b = blockIdx.x, nb = gridDim.x;
  const unsigned q = nb / kXcds, rem = nb % kXcds;
  const unsigned x = b % kXcds, idx = b / kXcds;
  return x * q + (x < rem ? x : rem) + idx;
}

// Row kernels read their box descriptor through the constant address space
// (scalar loads: kernels never write descriptors) and address fields with
// 32-bit byte offsets from a uniform global base.
typedef const __attribute__((address_space(4))) DevBox ConstBox;
typedef __attribute__((address_space(1))) char gchar;

__device__ __forceinline__ ConstBox &cbox(const DevBox *b) { return *(ConstBox *)b; }
// brings every cache line of a box descriptor into the scalar cache with
// loads issued together (one dword per 64 bytes, and the last), and waits
// once for them
__device__ __forceinline__ void fetch_box(const DevBox *b) {
  typedef const __attribute__((address_space(4))) unsigned CWord;
  CWord *w = (CWord *)b;
  constexpr int kWords = int(sizeof(DevBox) / 4);
  unsigned acc = w[kWords - 1];
#pragma unroll
  for (int q = 0; q < kWords; q += 16) acc ^= w[q];
  asm volatile("" ::"s"(acc));
}
// the generic helpers (robin_op_at) take a generic reference
__device__ __forceinline__ const DevBox &cbox_plain(ConstBox &b) { return *(const DevBox *)&b; }
// x / nc and the colour of (i, j, k) from a constant-space box (kernels.hpp
// split_div, colour_of)
__device__ __forceinline__ unsigned divc(ConstBox &B, unsigned x) { return (x * B.ncm) >> 16; }
__device__ __forceinline__ unsigned colourc(ConstBox &B, int i, int j, int k) {
  const unsigned s = unsigned(i + j + k);
  return s - divc(B, s) * unsigned(B.nc);
}

template <typename T>
__device__ __forceinline__ T ld(const void *base, unsigned off) {
  return *(const __attribute__((address_space(1))) T *)((const gchar *)base + off);
}
template <typename T>
__device__ __forceinline__ void st(void *base, unsigned off, T v) {
  *(__attribute__((address_space(1))) T *)((gchar *)base + off) = v;
}
// rho at byte offset o of point (i, j, k): +0 outside B's rho box without
// a load.  Callers take it before the stencil so that the load, when there
// is one, is in flight with the stencil's
__device__ __forceinline__ double rho_at(ConstBox &B, unsigned o, int i, int j, int k) {
  const bool in = (unsigned(i - B.rlo[0]) < unsigned(B.rhi[0] - B.rlo[0])) &
                  (unsigned(j - B.rlo[1]) < unsigned(B.rhi[1] - B.rlo[1])) &
                  (unsigned(k - B.rlo[2]) < unsigned(B.rhi[2] - B.rlo[2]));
  double r = 0.0;
  if (in) r = ld<double>(B.f[F_RHO], o);
  return r;
}

// axis-star Laplacian at byte offset o of a field; neighbour byte offsets
// from stencil_offs<NC, sizeof(T)>
template <int ORD, typename T, int NC = ORD / 2 + 1>
__device__ __forceinline__ T lapb(const void *u, unsigned o, const Nbr<NC> &n, T ix2, T iy2,
                                  T iz2) {
  constexpr int R = ORD / 2;
  T sx[4] = {0, 0, 0, 0}, syv[4] = {0, 0, 0, 0}, szv[4] = {0, 0, 0, 0};
#pragma unroll
  for (int m = 1; m <= R; ++m) {
    sx[m - 1] = ld<T>(u, o + n.xp[m - 1]) + ld<T>(u, o + n.xm[m - 1]);
    syv[m - 1] = ld<T>(u, o + n.yp[m - 1]) + ld<T>(u, o + n.ym[m - 1]);
    szv[m - 1] = ld<T>(u, o + n.zp[m - 1]) + ld<T>(u, o + n.zm[m - 1]);
  }
  const T u0 = ld<T>(u, o);
  return star_sum<ORD, T>(star<ORD, T>(u0, sx[0], sx[1], sx[2], sx[3]),
                          star<ORD, T>(u0, syv[0], syv[1], syv[2], syv[3]),
                          star<ORD, T>(u0, szv[0], szv[1], szv[2], szv[3]), ix2, iy2, iz2);
}

// Punctures_EM's first derivative along one axis at an interior point, as
// the reference's solver evaluates it: dx2 (centred, diff_2nd.cc:238-300) at
// order 2; at orders 4-8 the one-sided five-point stencil, forward on the
// lower half of the axis (index <= n/2, rounded down) and backward above,
// with du its coefficient of the point itself.  p, m: the +1..+4 and
// -1..-4 neighbour byte offsets; ia, na: index and points along the axis
template <int ORD>
__device__ __forceinline__ double em_deriv(const void *u, unsigned o, double u0, const unsigned *pp,
                                           const unsigned *mm, int ia, int na, double id, double &du) {
  if constexpr (ORD == 2) {
    du = 0.0;
    return (ld<double>(u, o + pp[0]) - ld<double>(u, o + mm[0])) * 0.5 * id;
  } else {
    const int nm = na % 2 == 0 ? na / 2 : (na - 1) / 2;
    if (ia <= nm) {
      du = -25 * id / 12.0;
      return -(25 * u0 - 48 * ld<double>(u, o + pp[0]) + 36 * ld<double>(u, o + pp[1]) -
               16 * ld<double>(u, o + pp[2]) + 3 * ld<double>(u, o + pp[3])) *
             id / 12.0;
    }
    du = 25 * id / 12.0;
    return (25 * u0 - 48 * ld<double>(u, o + mm[0]) + 36 * ld<double>(u, o + mm[1]) -
            16 * ld<double>(u, o + mm[2]) + 3 * ld<double>(u, o + mm[3])) *
           id / 12.0;
  }
}

// N(u) and dN/du at byte offset o of box B (u0 = u there, (i, j, k) its
// indices): Lap u from the neighbour offsets nb, the other terms from the
// coefficient fields
template <int ORD, int EQ, class BoxT>
__device__ __forceinline__ void point_op(BoxT &B, const void *u, unsigned o,
                                         const Nbr<colours_of(ORD, EQ)> &nb, double u0, int i, int j,
                                         int k, double &N, double &dN) {
  constexpr int NC = colours_of(ORD, EQ);
  const double lu = lapb<ORD, double, NC>(u, o, nb, B.idx2[0], B.idx2[1], B.idx2[2]);
  if constexpr (EQ == kEqPuncturesEm) {
    double g[3], du[3];
    g[0] = em_deriv<ORD>(u, o, u0, nb.xp, nb.xm, i, B.n[0], B.idx[0], du[0]);
    g[1] = em_deriv<ORD>(u, o, u0, nb.yp, nb.ym, j, B.n[1], B.idx[1], du[1]);
    g[2] = em_deriv<ORD>(u, o, u0, nb.zp, nb.zm, k, B.n[2], B.idx[2], du[2]);
    const double ge[3] = {ld<double>(B.f[F_X0], o), ld<double>(B.f[F_X1], o), ld<double>(B.f[F_X2], o)};
    const double gf[3] = {ld<double>(B.f[F_X3], o), ld<double>(B.f[F_X4], o), ld<double>(B.f[F_X5], o)};
    em_nonlinear(lu, B.dulap, u0, g, du, ld<double>(B.f[F_B], o), ld<double>(B.f[F_D], o), ge, gf, N, dN);
  } else {
    (void)i;
    (void)j;
    (void)k;
    nonlinear<EQ>(lu, B.dulap, ld<double>(B.f[F_B], o), ld<double>(B.f[F_C], o) + u0,
                  EQ == 1 ? ld<double>(B.f[F_D], o) : 0.0, EQ == 1 ? ld<double>(B.f[F_E], o) : 0.0, N, dN);
  }
}

// one DPP step on a double: lanes of rows in ROW_MASK read lane CTRL's value
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = int(b), hi = int(b >> 32);
  const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xF, false);
  const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)h2 << 32) | (unsigned)l2));
}

// Max of doubles none of which is negative or NaN, which order as their bits
// do: of the upper words first, then of the lower words beside the largest
// upper one: 14 instructions over a wave where the maxima of doubles take
// 36.  All lanes of the wave must be active.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ unsigned dpp_max_u32(unsigned v) {
  const unsigned w = unsigned(__builtin_amdgcn_update_dpp(0, int(v), CTRL, ROW_MASK, 0xF, false));
  return v > w ? v : w;
}
// over N = 8 or 16 lanes of a row that hold the same in every row
template <int N>
__device__ __forceinline__ unsigned row_max_u32(unsigned v) {
  v = dpp_max_u32<0xB1, 0xF>(v);
  v = dpp_max_u32<0x4E, 0xF>(v);
  v = dpp_max_u32<0x141, 0xF>(v);
  if constexpr (N == 16) v = dpp_max_u32<0x140, 0xF>(v);
  return v;
}
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
  v = row_max_u32<16>(v);
  v = dpp_max_u32<0x142, 0xA>(v);
  v = dpp_max_u32<0x143, 0xC>(v);
  return unsigned(__builtin_amdgcn_readlane(int(v), 63));
}
__device__ __forceinline__ double wave_max_pos(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned hi = wave_max_u32(unsigned(b >> 32));
  const unsigned lo = wave_max_u32(unsigned(b >> 32) == hi ? unsigned(b) : 0u);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int N>
__device__ __forceinline__ double row_max_pos(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned hi = row_max_u32<N>(unsigned(b >> 32));
  const unsigned lo = row_max_u32<N>(unsigned(b >> 32) == hi ? unsigned(b) : 0u);
  const int h = __builtin_amdgcn_readfirstlane(int(hi)), l = __builtin_amdgcn_readfirstlane(int(lo));
  return __longlong_as_double((long long)(((unsigned long long)unsigned(h) << 32) | unsigned(l)));
}

// what the block's norm slot holds as the block starts (thread 0; 0 without
// a slot).  The slot only grows, so wave_norm leaves the atomic out when the
// block's maximum is no larger: after a phase's first sweep that is nearly
// every block.  An atomic per block on 16 lines cost a colour pass of one
// N=65 box 0.5 us of 4.4.  Only launches of small workgroups (sweep_rule)
// read it: in longer launches the atomics overlap the passes, and the load
// would cost 2%.  Nor is it read in a phase's first pass, where every block
// has its atomic and the load would wait for those before it (one sweep of a
// 129^3 box, 2nd order: 78.5 us a call with the load, 70.2 without; 4th order
// 86 and 74; unread in the whole first sweep 72 and 76).
__device__ __forceinline__ double norm_seen(const unsigned long long *slot, bool first = false) {
  if (first || blockDim.x > kFewRowThreads || threadIdx.x != 0 || !slot) return 0.0;
  return ld<double>(slot, (blockIdx.x & (kNormSubSlots - 1)) * (kNormStride * 8u));
}

// block max of v (every thread must call; blockDim.x a multiple of 64, at
// most kMaxRowThreads), at most one norm update per block: none when the
// slot already held `seen` >= the maximum
__device__ __forceinline__ void wave_norm(unsigned long long *slot, double v, double seen) {
  __shared__ double sh[kMaxRowThreads / 64];
  const double m = wave_max_pos(v);
  if (blockDim.x == 64) {
    if (threadIdx.x == 0 && slot && m > seen) norm_update(slot, m);
    return;
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0 && slot) {
    double b = sh[0];
    const int nw = int(blockDim.x >> 6);
    for (int w = 1; w < nw; ++w) b = fmax(b, sh[w]);
    if (b > seen) norm_update(slot, b);
  }
}

// the block's interior row r -> (j, k)
template <int R>
__device__ __forceinline__ void row_jk(ConstBox &B, unsigned r, int &j, int &k) {
  const unsigned nyi = unsigned(B.n[1] - 2 * R);
  const unsigned kq = fast_div(r, nyi, B.inyi);
  k = R + int(kq);
  j = R + int(r - kq * nyi);
}

// colour passes (NC colours): the thread's slot t of local row lr: element
// index p of its point (i, j, k) of colour `colour` and that point's i mod
// NC; false when the row is past the block or the slot past the row's
// interior colour points
template <int R, int NC = R + 1>
__device__ __forceinline__ bool colour_slot(const RowBlock &Bk, ConstBox &B, unsigned lr, int t,
                                            unsigned per_row, int colour, unsigned &p, int &s,
                                            int &i, int &j, int &k) {
  if (lr >= unsigned(Bk.rows)) return false;
  unsigned row = unsigned(Bk.row0) + lr;
  if (Bk.nseg > 1) {  // segment `seg` of the row: colour points seg * per_row on
    const unsigned seg = row % unsigned(Bk.nseg);
    row /= unsigned(Bk.nseg);
    t += int(seg * per_row);
  }
  row_jk<R>(B, row, j, k);
  // i of the row's first interior point of this colour
  const int first = R + int(unsigned(colour + NC * 3 * kMaxAxisPoints - j - k - R) % NC);
  i = first + t * NC;
  if (i >= B.n[0] - R) return false;
  s = first % NC;
  p = unsigned(colour) * unsigned(B.cs) + unsigned(k) * unsigned(B.ps) + unsigned(j) * unsigned(B.rs) +
      unsigned(first / NC + t);
  return true;
}

// whole-row kernels: sub-row sr = NC * row + c is colour c of interior row
// `row` (with segments, sr * nseg + segment); the thread owns slot t of it
// (of the segment).  Element index p, colour c and i mod NC; false for
// ghost and padding slots
template <int R, int NC = R + 1>
__device__ __forceinline__ bool row_slot(const RowBlock &Bk, ConstBox &B, unsigned per_row,
                                         float inv_per_row, unsigned rpb, unsigned lr0, unsigned &p,
                                         int &c, int &s, int &i, int &j, int &k) {
  const unsigned lrl = fast_div(threadIdx.x, per_row, inv_per_row);
  int t = int(threadIdx.x - lrl * per_row);
  // threads past the chunk's whole rows idle (the next chunk has them)
  const unsigned lr = lr0 + lrl;
  if (lrl >= rpb || lr >= unsigned(Bk.rows)) return false;
  unsigned sr = unsigned(Bk.row0) + lr;
  if (Bk.nseg > 1) {  // segment `seg` of the colour row: slots seg * per_row on
    const unsigned seg = sr % unsigned(Bk.nseg);
    sr /= unsigned(Bk.nseg);
    t += int(seg * per_row);
  }
  const unsigned row = sr / NC;
  c = int(sr - row * NC);
  row_jk<R>(B, row, j, k);
  s = int(unsigned(c + NC * 3 * kMaxAxisPoints - j - k) % NC);
  i = s + t * NC;
  if (i < R || i >= B.n[0] - R) return false;
  p = unsigned(c) * unsigned(B.cs) + unsigned(k) * unsigned(B.ps) + unsigned(j) * unsigned(B.rs) +
      unsigned(t);
  return true;
}

// a whole-row block's rows, rpb = blockDim / per_row at a time: f(rpb,
// lr0) for the first local row lr0 of each chunk (blocks of one launch
// over many requests hold several chunks)
template <class F>
__device__ __forceinline__ void for_rows(const RowBlock &Bk, unsigned per_row, float inv_per_row,
                                         F &&f) {
  const unsigned rpb = fast_div(blockDim.x, per_row, inv_per_row);
#pragma unroll 1
  for (unsigned lr0 = 0; lr0 < unsigned(Bk.rows); lr0 += rpb) f(rpb, lr0);
}

// neighbour byte offsets (ES bytes per element) of a point of colour c
// with i mod NC = s in box B
template <int NC, int ES>
__device__ __forceinline__ Nbr<NC> box_offs(ConstBox &B, int c, int s) {
  return stencil_offs<NC, ES>(c, s, unsigned(B.cs), unsigned(B.rs), unsigned(B.ps));
}

// ------------------------------------------------------------------
// smoother: one colour of one Newton-Gauss-Seidel sweep on the rows of
// every listed block; thread (lr, t) owns colour point t of local row lr
// (smooth_rows, Punctures_EM) or points 2t and 2t + 1 (smooth_pairs)
// ------------------------------------------------------------------
template <int ORD, int EQ>
__device__ __forceinline__ void smooth_rows(const RowBlock &Bk, ConstBox &B, unsigned per_row,
                                            float inv_per_row, int pass) {
  const int colour = pass & (kFirstPass - 1);
  constexpr int R = ORD / 2;
  constexpr int NC = colours_of(ORD, EQ);
  const unsigned lr = fast_div(threadIdx.x, per_row, inv_per_row);
  const int t = int(threadIdx.x - lr * per_row);
  const double seen = norm_seen(Bk.norm, pass >= kFirstPass);
  double rmax = 0.0;
  unsigned p;
  int s, i, j, k;
  const int col = B.flip ? NC - 1 - colour : colour;
  if (colour_slot<R, NC>(Bk, B, lr, t, per_row, col, p, s, i, j, k)) {
    const Nbr<NC> nb = box_offs<NC, 8>(B, col, s);
    const unsigned o = p * 8u;
    double *u = B.f[F_U];
    const double rho = rho_at(B, o, i, j, k);
    const double u0 = ld<double>(u, o);
    double N, dN;
    point_op<ORD, EQ>(B, u, o, nb, u0, i, j, k, N, dN);
    const double res = N - rho;
    const double un = u0 - res / dN;
    st<double>(u, o, un);
    rmax = fabs(res);
    if (!(un == un)) rmax = __longlong_as_double(0x7ff0000000000000LL);  // inf flags NaN
  }
  wave_norm(Bk.norm, rmax, seen);
}

// Two colour points a thread: slots t and t + 1 of a colour row (i and
// i + NC), every field read 16 bytes a lane.  A wave's 8-byte load occupies
// the vector memory unit for as long as its 16-byte load (16.4 cycles each,
// measured on L1- and L2-resident data, aligned or not), and one point a
// thread kept that unit 77% busy (N=161, 6th order: 22 loads a wave).
// k_smooth<6,1> over the N=161 workload's launches 58.8 -> 51.4 us, <8,0>
// at N=129 11.8 -> 10.1 us, <4,0> in a batch of 16 at N=65 21.7 -> 19.5 us.
// The x neighbours of colour c + m of both points are three consecutive slots
// (x + m - NC, x + m, x + m + NC).  Each point's arithmetic is smooth_rows',
// operation for operation.
__device__ __forceinline__ void ld_pair(const void *base, unsigned off, double &a, double &b) {
  typedef double V2 __attribute__((ext_vector_type(2), aligned(8)));
  const V2 v = *(const __attribute__((address_space(1))) V2 *)((const gchar *)base + off);
  a = v.x;
  b = v.y;
}
__device__ __forceinline__ void st_pair(void *base, unsigned off, double a, double b) {
  typedef double V2 __attribute__((ext_vector_type(2), aligned(8)));
  V2 v;
  v.x = a;
  v.y = b;
  *(__attribute__((address_space(1))) V2 *)((gchar *)base + off) = v;
}

// Laplacian terms of the points at byte offsets o and o + 8 (u00, u01 their
// u), NC = ORD / 2 + 1 colours
template <int ORD>
__device__ __forceinline__ void lap_pair(const void *u, unsigned o, const Nbr<ORD / 2 + 1> &n,
                                         double u00, double u01, double ix2, double iy2, double iz2,
                                         double l[2]) {
  constexpr int R = ORD / 2, NC = R + 1;
  double sx[2][4] = {}, sy[2][4] = {}, sz[2][4] = {};
  double xv[R][3];  // [m - 1]: u at x + m - NC, x + m, x + m + NC
#pragma unroll
  for (int m = 1; m <= R; ++m) {
    ld_pair(u, o + n.xm[NC - m - 1], xv[m - 1][0], xv[m - 1][1]);
    xv[m - 1][2] = ld<double>(u, o + n.xp[m - 1] + 8u);
    double p0, p1, m0, m1;
    ld_pair(u, o + n.yp[m - 1], p0, p1);
    ld_pair(u, o + n.ym[m - 1], m0, m1);
    sy[0][m - 1] = p0 + m0;
    sy[1][m - 1] = p1 + m1;
    ld_pair(u, o + n.zp[m - 1], p0, p1);
    ld_pair(u, o + n.zm[m - 1], m0, m1);
    sz[0][m - 1] = p0 + m0;
    sz[1][m - 1] = p1 + m1;
  }
#pragma unroll
  for (int m = 1; m <= R; ++m)
#pragma unroll
    for (int q = 0; q < 2; ++q) sx[q][m - 1] = xv[m - 1][q + 1] + xv[NC - m - 1][q];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const double u0 = q ? u01 : u00;
    l[q] = star_sum<ORD, double>(star<ORD, double>(u0, sx[q][0], sx[q][1], sx[q][2], sx[q][3]),
                                 star<ORD, double>(u0, sy[q][0], sy[q][1], sy[q][2], sy[q][3]),
                                 star<ORD, double>(u0, sz[q][0], sz[q][1], sz[q][2], sz[q][3]), ix2,
                                 iy2, iz2);
  }
}

// What a pass by pairs reads of a box descriptor, in scalar registers.
// load() issues every scalar load at once and waits for them together, with
// the workgroup's record when the box is known before it (read as they were
// used, the fields took eight scalar waits in turn).
struct SweepBox {
  double *u, *b, *c, *d, *e, *rho;
  double ix2, iy2, iz2, dulap;
  unsigned cs, rs, ps;
  int n0, n1, flip;
  float inyi;
  int rlo0, rlo1, rlo2, rhi0, rhi1, rhi2;
  __device__ __forceinline__ void load(ConstBox &B) {
    u = B.f[F_U];
    b = B.f[F_B];
    c = B.f[F_C];
    d = B.f[F_D];
    e = B.f[F_E];
    rho = B.f[F_RHO];
    ix2 = B.idx2[0];
    iy2 = B.idx2[1];
    iz2 = B.idx2[2];
    dulap = B.dulap;
    cs = unsigned(B.cs);
    rs = unsigned(B.rs);
    ps = unsigned(B.ps);
    n0 = B.n[0];
    n1 = B.n[1];
    flip = B.flip;
    inyi = B.inyi;
    rlo0 = B.rlo[0];
    rlo1 = B.rlo[1];
    rlo2 = B.rlo[2];
    rhi0 = B.rhi[0];
    rhi1 = B.rhi[1];
    rhi2 = B.rhi[2];
  }
  __device__ __forceinline__ void wait() const {
    asm volatile("" ::"s"(u), "s"(b), "s"(c), "s"(d), "s"(e), "s"(rho), "s"(ix2), "s"(iy2), "s"(iz2),
                 "s"(dulap), "s"(cs), "s"(rs), "s"(ps), "s"(n0), "s"(n1), "s"(flip), "s"(inyi),
                 "s"(rlo0), "s"(rlo1), "s"(rlo2), "s"(rhi0), "s"(rhi1), "s"(rhi2));
  }
  // rho of the pair of points (i, j, k), (i + nc, j, k): +0 outside the rho
  // box, a pair that reaches into it read whole
  __device__ __forceinline__ void rho_pair(unsigned o, int i, int nc, int j, int k, double r[2]) const {
    r[0] = r[1] = 0.0;
    if ((unsigned(j - rlo1) < unsigned(rhi1 - rlo1)) & (unsigned(k - rlo2) < unsigned(rhi2 - rlo2)) &
        (i + nc >= rlo0) & (i < rhi0))
      ld_pair(rho, o, r[0], r[1]);
  }
};

// N(u) and dN/du of the pair at byte offset o (EQ without first derivatives)
template <int ORD, int EQ>
__device__ __forceinline__ void point_op_pair(const SweepBox &B, unsigned o,
                                              const Nbr<ORD / 2 + 1> &nb, const double u0[2],
                                              double N[2], double dN[2]) {
  double lu[2], b[2], c[2], d[2] = {0.0, 0.0}, e[2] = {0.0, 0.0};
  ld_pair(B.b, o, b[0], b[1]);
  ld_pair(B.c, o, c[0], c[1]);
  if constexpr (EQ == 1) {
    ld_pair(B.d, o, d[0], d[1]);
    ld_pair(B.e, o, e[0], e[1]);
  }
  lap_pair<ORD>(B.u, o, nb, u0[0], u0[1], B.ix2, B.iy2, B.iz2, lu);
#pragma unroll
  for (int q = 0; q < 2; ++q)
    nonlinear<EQ>(lu[q], B.dulap, b[q], c[q] + u0[q], d[q], e[q], N[q], dN[q]);
}

template <int ORD, int EQ>
__device__ __forceinline__ void smooth_pairs(const RowBlock &Bk, const SweepBox &B, unsigned per_row,
                                             float inv_per_row, int pass) {
  const int colour = pass & (kFirstPass - 1);
  constexpr int R = ORD / 2, NC = R + 1;
  const unsigned lr = fast_div(threadIdx.x, per_row, inv_per_row);
  unsigned t = threadIdx.x - lr * per_row;
  const int col = B.flip ? NC - 1 - colour : colour;
  const double seen = norm_seen(Bk.norm, pass >= kFirstPass);
  double rmax = 0.0;
  unsigned row = unsigned(Bk.row0) + lr;
  if (lr < unsigned(Bk.rows)) {
    if (Bk.nseg > 1) {
      const unsigned seg = row % unsigned(Bk.nseg);
      row /= unsigned(Bk.nseg);
      t += seg * per_row;
    }
    const unsigned nyi = unsigned(B.n1 - 2 * R);
    const unsigned kq = fast_div(row, nyi, B.inyi);
    const int k = R + int(kq), j = R + int(row - kq * nyi);
    const int first = R + int(unsigned(col + NC * 3 * kMaxAxisPoints - j - k - R) % NC);
    const int i = first + int(2 * t) * NC;
    if (i < B.n0 - R) {
      // the second point may be a ghost or padding slot: its loads stay
      // inside the field (rows and planes follow every interior row), and
      // it is neither written nor counted
      const bool two = i + NC < B.n0 - R;
      const unsigned p = unsigned(col) * B.cs + unsigned(k) * B.ps + unsigned(j) * B.rs +
                         unsigned(first / NC) + 2 * t;
      const Nbr<NC> nb = stencil_offs<NC, 8>(col, first % NC, B.cs, B.rs, B.ps);
      const unsigned o = p * 8u;
      double rho[2], u0[2], N[2], dN[2], un[2];
      B.rho_pair(o, i, NC, j, k, rho);
      ld_pair(B.u, o, u0[0], u0[1]);
      point_op_pair<ORD, EQ>(B, o, nb, u0, N, dN);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const double res = N[q] - rho[q];
        un[q] = u0[q] - res / dN[q];
        if (q == 0 || two) {
          rmax = fmax(rmax, fabs(res));
          if (!(un[q] == un[q])) rmax = __longlong_as_double(0x7ff0000000000000LL);
        }
      }
      if (two)
        st_pair(B.u, o, un[0], un[1]);
      else
        st<double>(B.u, o, un[0]);
    }
  }
  wave_norm(Bk.norm, rmax, seen);
}

// box1: the one box of every listed block, when the launch covers a single
// box (else null); its descriptor is then fetched without waiting for the
// block's.
// By pairs, four waves per SIMD leave a wave the registers to issue its loads
// (17 at 4th, 25 at 6th, 29 at 8th order) before it waits for the first;
// compiled for more waves it issued 11 to 14 and waited.  With the scalar
// loads together (SweepBox): N=161 smoother 94.2 -> 90.3 ms per two V-cycles,
// 16 x N=65 23.8 -> 23.1, N=129 8th order 21.3 -> 20.4, one 33^3 solve 6.40 ->
// 6.28.  Poisson and Brill waves the same way, N=129, a pass before the pairs
// and now: 2nd order 8.2 -> 6.6 and 6.8 us, 8th 8.5 -> 6.0.  One point a
// thread (Punctures_EM) has few loads to issue and needs the waves: four a
// SIMD instead of five to eight took 24.6 us instead of 20.3 (N=129 2nd
// order), 17.7 instead of 15.4 (4th).
template <int ORD, int EQ>
__global__ __launch_bounds__(kMaxRowThreads)
__attribute__((amdgpu_waves_per_eu(sweep_points(EQ) == 2 ? 4 : 1, sweep_points(EQ) == 2 ? 4 : 8)))
void k_smooth(const RowBlock *__restrict__ blocks,
                                                        unsigned per_row, float inv_per_row,
                                                        int pass, const DevBox *box1) {
  if constexpr (sweep_points(EQ) == 2) {
    RowBlock Bk;
    SweepBox B;
    if (box1) {
      B.load(cbox(box1));
      Bk = blocks[xcd_block()];
      B.wait();
    } else {
      Bk = blocks[xcd_block()];
      B.load(cbox(Bk.box));
      B.wait();
    }
    smooth_pairs<ORD, EQ>(Bk, B, per_row, inv_per_row, pass);
  } else {
    const RowBlock Bk = blocks[xcd_block()];
    const DevBox *box = box1 ? box1 : Bk.box;
    fetch_box(box);
    smooth_rows<ORD, EQ>(Bk, cbox(box), per_row, inv_per_row, pass);
  }
}

// ------------------------------------------------------------------
// fused colour passes.  A sweep reads u from field X and writes every
// updated point to field Y (X and Y are u and r, swapped from sweep to
// sweep; the ghost shell is copied into r first, k_copy_shell): within a
// sweep, a point's neighbours of colours already updated are read from Y,
// the others and the point itself from X, which no launch of the sweep
// writes.  One launch does two consecutive colour passes (pass indices Q
// and Q + 1) on a tile of interior rows: the first pass also on the rows
// the second pass reads (one row and plane below the tile, R above), the
// second on the tile alone.  Every launch that computes a first-pass point
// computes it from the same X and Y values, so tiles that overlap write
// identical values, and each workgroup reads back only what it wrote itself
// (after a barrier).  Each point's arithmetic is k_smooth's: the sweeps
// give the same bits as the colour passes one launch at a time.
// ------------------------------------------------------------------

template <int ORD, int NC, int PI, int M>
__device__ __forceinline__ void star_terms(const void *X, const void *Y, unsigned o,
                                           const Nbr<NC> &n, double *sx, double *sy, double *sz) {
  if constexpr (M <= ORD / 2) {
    const void *bp = nbr_in_y(NC, PI, M) ? Y : X;
    const void *bm = nbr_in_y(NC, PI, -M) ? Y : X;
    sx[M - 1] = ld<double>(bp, o + n.xp[M - 1]) + ld<double>(bm, o + n.xm[M - 1]);
    sy[M - 1] = ld<double>(bp, o + n.yp[M - 1]) + ld<double>(bm, o + n.ym[M - 1]);
    sz[M - 1] = ld<double>(bp, o + n.zp[M - 1]) + ld<double>(bm, o + n.zm[M - 1]);
    star_terms<ORD, NC, PI, M + 1>(X, Y, o, n, sx, sy, sz);
  }
}

// one point of pass PI: reads X and Y as above, writes the new u to Y;
// the arithmetic of k_smooth / point_op / lapb, operation for operation
template <int ORD, int EQ, int PI>
__device__ __forceinline__ double fused_point(ConstBox &B, const void *X, void *Y, int c, int i,
                                              int j, int k) {
  constexpr int R = ORD / 2;
  constexpr int NC = R + 1;
  const int s = i - (i / NC) * NC;
  const unsigned p = unsigned(c) * unsigned(B.cs) + unsigned(k) * unsigned(B.ps) +
                     unsigned(j) * unsigned(B.rs) + unsigned(i / NC);
  const unsigned o = p * 8u;
  const Nbr<NC> nb = box_offs<NC, 8>(B, c, s);
  const double u0 = ld<double>(X, o);
  double sx[4] = {0, 0, 0, 0}, sy[4] = {0, 0, 0, 0}, sz[4] = {0, 0, 0, 0};
  star_terms<ORD, NC, PI, 1>(X, Y, o, nb, sx, sy, sz);
  const double lu = star_sum<ORD, double>(star<ORD, double>(u0, sx[0], sx[1], sx[2], sx[3]),
                                          star<ORD, double>(u0, sy[0], sy[1], sy[2], sy[3]),
                                          star<ORD, double>(u0, sz[0], sz[1], sz[2], sz[3]),
                                          B.idx2[0], B.idx2[1], B.idx2[2]);
  double N, dN;
  nonlinear<EQ>(lu, B.dulap, ld<double>(B.f[F_B], o), ld<double>(B.f[F_C], o) + u0,
                EQ == 1 ? ld<double>(B.f[F_D], o) : 0.0, EQ == 1 ? ld<double>(B.f[F_E], o) : 0.0,
                N, dN);
  const double res = N - ld<double>(B.f[F_RHO], o);
  const double un = u0 - res / dN;
  st<double>(Y, o, un);
  double r = fabs(res);
  if (!(un == un)) r = __longlong_as_double(0x7ff0000000000000LL);  // inf flags NaN
  return r;
}

// pass PI over the first nrows rows of the tile's row list, the flattened
// (row, colour point) index strided over the workgroup; returns the max
// |residual| over the tile's own rows
template <int ORD, int EQ, int PI>
__device__ __forceinline__ double fused_pass(const TileBlock &T, ConstBox &B, const void *X, void *Y,
                                             int nrows, int yb, int ya, int zb) {
  constexpr int R = ORD / 2;
  constexpr int NC = R + 1;
  const int P = (B.n[0] - 2 * R + NC - 1) / NC;  // colour points per interior row, at most
  const int nt = T.ty * T.tz;
  const int c = B.flip ? NC - 1 - PI : PI;
  double rmax = 0.0;
  for (int f = int(threadIdx.x); f < nrows * P; f += int(blockDim.x)) {
    const int r = f / P, t = f - r * P;
    int j, k;
    tile_row(T, r, yb, ya, zb, j, k);
    const int i = colour_first(c, j, k, R, NC) + t * NC;
    if (i >= B.n[0] - R) continue;
    const double res = fused_point<ORD, EQ, PI>(B, X, Y, c, i, j, k);
    if (r < nt) rmax = fmax(rmax, res);
  }
  return rmax;
}

// passes Q and Q + 1 (PAIR) or pass Q alone of one sweep on every listed
// tile; parity 0 reads X = u and writes Y = r, parity 1 the reverse
template <int ORD, int EQ, int Q, int PAIR>
__global__ __launch_bounds__(kFusedThreads) void k_smooth_fused(const TileBlock *__restrict__ blocks,
                                                              int parity) {
  constexpr int R = ORD / 2;
  const TileBlock T = blocks[xcd_block()];
  ConstBox &B = cbox(T.box);
  const void *X = parity ? B.f[F_R] : B.f[F_U];
  void *Y = parity ? B.f[F_U] : B.f[F_R];
  const int nt = T.ty * T.tz;
  const double seen = norm_seen(T.norm);
  double rmax;
  if constexpr (PAIR) {
    int yb, ya, zb, za;
    const int nn[3] = {B.n[0], B.n[1], B.n[2]};
    tile_halo(T, nn, R, yb, ya, zb, za);
    const int nrows = nt + (yb + ya) * T.tz + (zb + za) * T.ty;
    rmax = fused_pass<ORD, EQ, Q>(T, B, X, Y, nrows, yb, ya, zb);
    // the second pass reads the first pass's values this workgroup wrote
    __syncthreads();
    rmax = fmax(rmax, fused_pass<ORD, EQ, Q + 1>(T, B, X, Y, nt, 0, 0, 0));
  } else {
    rmax = fused_pass<ORD, EQ, Q>(T, B, X, Y, nt, 0, 0, 0);
  }
  wave_norm(T.norm, rmax, seen);
}

// whole-row kernels, two slots a thread: slots 2t and 2t + 1 of sub-row sr
// (row_slot); ok[q]: the slot holds an interior point.  Loads of the other
// slot stay inside the field (rows precede and follow every interior row)
template <int R, int NC = R + 1>
__device__ __forceinline__ bool row_pair(const RowBlock &Bk, ConstBox &B, unsigned per_row,
                                         float inv_per_row, unsigned rpb, unsigned lr0, unsigned &p,
                                         int &c, int &s, int &i, int &j, int &k, bool ok[2]) {
  const unsigned lrl = fast_div(threadIdx.x, per_row, inv_per_row);
  unsigned t = threadIdx.x - lrl * per_row;
  const unsigned lr = lr0 + lrl;
  if (lrl >= rpb || lr >= unsigned(Bk.rows)) return false;
  unsigned sr = unsigned(Bk.row0) + lr;
  if (Bk.nseg > 1) {
    const unsigned seg = sr % unsigned(Bk.nseg);
    sr /= unsigned(Bk.nseg);
    t += seg * per_row;
  }
  const unsigned row = sr / NC;
  c = int(sr - row * NC);
  row_jk<R>(B, row, j, k);
  s = int(unsigned(c + NC * 3 * kMaxAxisPoints - j - k) % NC);
  i = s + int(2 * t) * NC;
  ok[0] = i >= R && i < B.n[0] - R;
  ok[1] = i + NC >= R && i + NC < B.n[0] - R;
  p = unsigned(c) * unsigned(B.cs) + unsigned(k) * unsigned(B.ps) + unsigned(j) * unsigned(B.rs) + 2 * t;
  return ok[0] || ok[1];
}

// operator on the interior: mode RES_OPERATOR r = N(u), RES_DEFECT
// w = rho - N(u), RES_DERIVATIVE r = dN/du_p; the norm is max |N(u)| over
// the points where N(u) is a number (fmax drops a NaN, which must not reach
// wave_norm: as a bit pattern it would outrank its wave's other points)
template <int ORD, int EQ>
__global__ __launch_bounds__(kRowThreads) void k_residual(const RowBlock *__restrict__ blocks,
                                                          unsigned per_row, float inv_per_row,
                                                          int mode) {
  constexpr int R = ORD / 2;
  constexpr int NC = colours_of(ORD, EQ);
  const RowBlock Bk = blocks[xcd_block()];
  ConstBox &B = cbox(Bk.box);
  const double seen = norm_seen(Bk.norm);
  double rmax = 0.0;
  if constexpr (sweep_points(EQ) == 2) {
    // two slots a thread, as the colour passes (one: N=161 6th order 234 us a
    // launch, 16 x N=65 4th order 67; two: 188 and 53)
    SweepBox P;
    P.load(B);
    double *out = mode == RES_DEFECT ? B.f[F_W] : B.f[F_R];
    for_rows(Bk, per_row, inv_per_row, [&](unsigned rpb, unsigned lr0) {
      unsigned p;
      int c, s, i, j, k;
      bool ok[2];
      if (!row_pair<R>(Bk, B, per_row, inv_per_row, rpb, lr0, p, c, s, i, j, k, ok)) return;
      const Nbr<R + 1> nb = box_offs<R + 1, 8>(B, c, s);
      const unsigned o = p * 8u;
      double rho[2] = {0.0, 0.0}, u0[2], N[2], dN[2], v[2];
      if (mode == RES_DEFECT) P.rho_pair(o, i, R + 1, j, k, rho);
      ld_pair(P.u, o, u0[0], u0[1]);
      point_op_pair<ORD, EQ>(P, o, nb, u0, N, dN);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        v[q] = mode == RES_DEFECT ? rho[q] - N[q] : (mode == RES_DERIVATIVE ? dN[q] : N[q]);
        if (ok[q]) rmax = fmax(rmax, fabs(N[q]));
      }
      if (ok[0] && ok[1])
        st_pair(out, o, v[0], v[1]);
      else
        st<double>(out, ok[0] ? o : o + 8u, ok[0] ? v[0] : v[1]);
    });
    wave_norm(Bk.norm, rmax, seen);
    return;
  }
  for_rows(Bk, per_row, inv_per_row, [&](unsigned rpb, unsigned lr0) {
    unsigned p;
    int c, s, i, j, k;
    if (!row_slot<R, NC>(Bk, B, per_row, inv_per_row, rpb, lr0, p, c, s, i, j, k)) return;
    const Nbr<NC> nb = box_offs<NC, 8>(B, c, s);
    const unsigned o = p * 8u;
    const double *u = B.f[F_U];
    const double rho = mode == RES_DEFECT ? rho_at(B, o, i, j, k) : 0.0;
    double N, dN;
    point_op<ORD, EQ>(B, u, o, nb, ld<double>(u, o), i, j, k, N, dN);
    if (mode == RES_DEFECT)
      st<double>(B.f[F_W], o, rho - N);
    else
      st<double>(B.f[F_R], o, mode == RES_DERIVATIVE ? dN : N);
    rmax = fmax(rmax, fabs(N));
  });
  wave_norm(Bk.norm, rmax, seen);
}

// ------------------------------------------------------------------
// mixed precision.  One smoothing block of nu sweeps becomes: the FP64
// defect r = rho - N(u) and the linearised diagonal q = dN/du - dulap of
// the current u (k_defect32, also the block's norm), nu multi-colour
// Gauss-Seidel sweeps in FP32 on the correction equation
//   Lap e + q e = r,   e = 0 on the ghost shell          (k_smooth32)
// and the FP64 update u += e (k_update32).  At a converged u the defect is
// zero, e stays zero and u is unchanged: the fixed point is the FP64 one.
// ------------------------------------------------------------------
template <int ORD, int EQ>
__global__ __launch_bounds__(kRowThreads) void k_defect32(const RowBlock *__restrict__ blocks,
                                                          unsigned per_row, float inv_per_row) {
  constexpr int R = ORD / 2;
  constexpr int NC = R + 1;
  const RowBlock Bk = blocks[xcd_block()];
  ConstBox &B = cbox(Bk.box);
  const double seen = norm_seen(Bk.norm);
  SweepBox P;
  P.load(B);
  double rmax = 0.0;
  for_rows(Bk, per_row, inv_per_row, [&](unsigned rpb, unsigned lr0) {
    unsigned p;
    int c, s, i, j, k;
    bool ok[2];
    if (!row_pair<R>(Bk, B, per_row, inv_per_row, rpb, lr0, p, c, s, i, j, k, ok)) return;
    const Nbr<NC> nb = box_offs<NC, 8>(B, c, s);
    const unsigned o = p * 8u;
    double rho[2], u0[2], N[2], dN[2];
    P.rho_pair(o, i, NC, j, k, rho);
    ld_pair(P.u, o, u0[0], u0[1]);
    point_op_pair<ORD, EQ>(P, o, nb, u0, N, dN);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (!ok[q]) continue;
      const unsigned o4 = (p + unsigned(q)) * 4u;
      const double res = rho[q] - N[q];
      st<float>(B.g[G_R], o4, float(res));
      st<float>(B.g[G_Q], o4, float(dN[q] - B.dulap));
      st<float>(B.g[G_E], o4, 0.0f);
      rmax = fmax(rmax, fabs(res));
      if (!(res == res)) rmax = __longlong_as_double(0x7ff0000000000000LL);
    }
  });
  wave_norm(Bk.norm, rmax, seen);
}

template <int ORD>
__global__ __launch_bounds__(kMaxRowThreads) void k_smooth32(const RowBlock *__restrict__ blocks,
                                                          unsigned per_row, float inv_per_row,
                                                          int colour) {
  constexpr int R = ORD / 2;
  constexpr int NC = R + 1;
  const RowBlock Bk = blocks[xcd_block()];
  ConstBox &B = cbox(Bk.box);
  const unsigned lr = fast_div(threadIdx.x, per_row, inv_per_row);
  const int t = int(threadIdx.x - lr * per_row);
  unsigned p;
  int s, i, j, k;
  const int col = B.flip ? NC - 1 - colour : colour;
  if (!colour_slot<R>(Bk, B, lr, t, per_row, col, p, s, i, j, k)) return;
  const Nbr<NC> nb = box_offs<NC, 4>(B, col, s);
  const unsigned o = p * 4u;
  float *e = B.g[G_E];
  const float le = lapb<ORD, float>(e, o, nb, float(B.idx2[0]), float(B.idx2[1]), float(B.idx2[2]));
  const float q = ld<float>(B.g[G_Q], o);
  const float ep = ld<float>(e, o);
  const float res = fmaf(q, ep, le) - ld<float>(B.g[G_R], o);
  // float32 relaxation of a correction: the hardware reciprocal suffices
  st<float>(e, o, fmaf(-res, __builtin_amdgcn_rcpf(float(B.dulap) + q), ep));
}

template <int ORD>
__global__ __launch_bounds__(kRowThreads) void k_update32(const RowBlock *__restrict__ blocks,
                                                          unsigned per_row, float inv_per_row) {
  constexpr int R = ORD / 2;
  const RowBlock Bk = blocks[xcd_block()];
  ConstBox &B = cbox(Bk.box);
  for_rows(Bk, per_row, inv_per_row, [&](unsigned rpb, unsigned lr0) {
    unsigned p;
    int c, s, i, j, k;
    bool ok[2];
    if (!row_pair<R>(Bk, B, per_row, inv_per_row, rpb, lr0, p, c, s, i, j, k, ok)) return;
    double *u = B.f[F_U];
    const unsigned o = p * 8u;
    double u0, u1;
    ld_pair(u, o, u0, u1);
    u0 += double(ld<float>(B.g[G_E], p * 4u));
    u1 += double(ld<float>(B.g[G_E], p * 4u + 4u));
    if (ok[0] && ok[1])
      st_pair(u, o, u0, u1);
    else
      st<double>(u, ok[0] ? o : o + 8u, ok[0] ? u0 : u1);
  });
}

// ------------------------------------------------------------------
// Robin boundary r^2/n sum_d (1/x_d) d_d u + u = S on the ghost shell
// ------------------------------------------------------------------

// value of u at offset m (any sign, |m| <= 4) along axis a from the point
// at storage index p with colour c and i mod nc = s
__device__ __forceinline__ double axis_at(const DevBox &B, const double *__restrict__ u, long long p,
                                          int c, int s, int a, int m) {
  return u[p + axis_offset(B, c, s, a, m)];
}

// first derivative along axis a at (i, j, k), storage index p:
// dx2 (diff_2nd.cc:237-335) for order 2, dx4 (diff_4th.cc:6-89) otherwise.
// coef = coefficient of u at the point itself.
__device__ __forceinline__ double deriv(const DevBox &B, const double *__restrict__ u, long long p,
                                        int a, int i, int j, int k, double &coef) {
  const int n = B.n[a];
  const int ia = a == 0 ? i : (a == 1 ? j : k);
  const double id = B.idx[a];
  const int c = colour_of(B, i, j, k), s = i - split_div(B, i) * B.nc;
#define UA(m) axis_at(B, u, p, c, s, a, (m))
  if (B.order == 2) {
    if (ia == 0) {
      coef = -3.0 * 0.5 * id;
      return (-3.0 * u[p] + 4.0 * UA(1) - UA(2)) * 0.5 * id;
    } else if (ia == n - 1) {
      coef = 3.0 * 0.5 * id;
      return (3.0 * u[p] - 4.0 * UA(-1) + UA(-2)) * 0.5 * id;
    }
    coef = 0.0;
    return (UA(1) - UA(-1)) * 0.5 * id;
  }
  const int nm = (n % 2 == 0) ? n / 2 : (n - 1) / 2;
  if (ia <= nm) {
    coef = -25.0 * id / 12.0;
    return -(25.0 * u[p] - 48.0 * UA(1) + 36.0 * UA(2) - 16.0 * UA(3) + 3.0 * UA(4)) * id / 12.0;
  }
  coef = 25.0 * id / 12.0;
  return (25.0 * u[p] - 48.0 * UA(-1) + 36.0 * UA(-2) - 16.0 * UA(-3) + 3.0 * UA(-4)) * id / 12.0;
#undef UA
}

// box-local views of the fields a Robin stage touches; u may be in LDS
struct BoxData {
  double *u;
  const double *rho;
  double *r;
  double *w;
};

__device__ __forceinline__ BoxData box_data(const DevBox &B) {
  BoxData D;
  D.u = B.f[F_U];
  D.rho = B.f[F_RHO];
  D.r = B.f[F_R];
  D.w = B.f[F_W];
  return D;
}

// Robin update / operator at one shell point; `mask` has bit a set for
// each axis a whose index lies in the ghost shell.
__device__ __forceinline__ void robin_point(const DevBox &B, BoxData D, int i, int j, int k,
                                            int mask, int mode) {
  const long long p = pidx(B, i, j, k);
  double *u = D.u;
  const int ijk[3] = {i, j, k};
  double X[3];
  for (int a = 0; a < 3; ++a) X[a] = coord(B, a, ijk[a]);
  const double r2 = X[0] * X[0] + X[1] * X[1] + X[2] * X[2];
  double sF = 0.0, sdF = 0.0;
  for (int a = 0; a < 3; ++a) {
    if (!(mask & (1 << a))) continue;
    double cf;
    const double dv = deriv(B, u, p, a, i, j, k, cf);
    sF += dv / X[a];
    sdF += cf / X[a];
  }
  const double op = r2 * B.ipn * sF + u[p];
  if (mode == ROBIN_UPDATE) {
    const double Fv = op - D.rho[p];
    const double dF = r2 * B.ipn * sdF + 1.0;
    u[p] = u[p] - Fv / dF;
  } else if (mode == ROBIN_OPERATOR_R) {
    D.r[p] = op;
  } else {
    D.w[p] = D.rho[p] - op;
  }
}

// face column t of a box: all R layers, inner -> outer
__device__ __forceinline__ void robin_face_column(const DevBox &B, BoxData D, int t, int mode) {
  const int R = B.R;
  const int ni = B.n[0] - 2 * R, nj = B.n[1] - 2 * R, nk = B.n[2] - 2 * R;
  const int fx = nj * nk, fy = ni * nk, fz = ni * nj;
  int face, a0, a1;
  if (t < 2 * fx) {
    face = t / fx; t %= fx; a0 = t % nj; a1 = t / nj;  // j, k
  } else if ((t -= 2 * fx) < 2 * fy) {
    face = 2 + t / fy; t %= fy; a0 = t % ni; a1 = t / ni;  // i, k
  } else if ((t -= 2 * fy) < 2 * fz) {
    face = 4 + t / fz; t %= fz; a0 = t % ni; a1 = t / ni;  // i, j
  } else {
    return;
  }
  const int axis = face >> 1, hi = face & 1;
  for (int l = 0; l < R; ++l) {
    const int g = hi ? B.n[axis] - R + l : R - 1 - l;
    int i, j, k;
    if (axis == 0) {
      i = g; j = R + a0; k = R + a1;
    } else if (axis == 1) {
      i = R + a0; j = g; k = R + a1;
    } else {
      i = R + a0; j = R + a1; k = g;
    }
    robin_point(B, D, i, j, k, 1 << axis, mode);
  }
}

// ghost index of position q (0..R-1) on side `hi` of an axis, in the
// reference's iteration order (domain.cc:575-1388): low sides run R-1 -> 0,
// high sides n-R -> n-1
__device__ __forceinline__ int shell_index(int q, int hi, int n, int R) {
  return hi ? n - R + q : R - 1 - q;
}

// Edges and corners: a point's one-sided derivatives read points further
// inwards on its axes, so in the reference's order (inwards points first) a
// point reads exactly the updated values of those shell points, and points
// whose distances inwards have the same sum are independent of each other.
// One lane takes a point and the sums go from the innermost outwards: 2R - 1
// steps for an edge's cross-section instead of R^2, 3R - 2 for a corner
// instead of R^3, from values staged in LDS, with what does not depend on u
// formed before the first step.  The chains of dependent divisions, and a
// staging whose loads waited for each other, bounded both: N=129 8th order
// edges 24 -> 6.2 us, corners 17 -> 8.6; N=161 6th order 14.2 -> 5.9, 11.0 ->
// 7.0; one N=65 request 10.6 -> 5.9, 7.8 -> 6.6.
//
// A corner's cube has kCornerW^3 points (R <= 4 shell layers plus the 4
// inward points the derivatives read).
constexpr int kCornerR = 4;
constexpr int kCornerW = kCornerR + 4;
constexpr int kCornerCube = kCornerW * kCornerW * kCornerW;
constexpr int kCornerR3 = kCornerR * kCornerR * kCornerR;

// box index of local coordinate l (counted inwards from side h) along an axis
__device__ __forceinline__ int corner_index(int l, int h, int n) { return h ? n - 1 - l : l; }

// deriv()'s one-sided derivative at side h from the staged point w[0] and the
// points w[m], w[2 m].. inwards: dx2 at the box faces for order 2, dx4
// otherwise; cf: the coefficient of the point itself
__device__ __forceinline__ double inward_deriv(const double *w, int m, int order, int h, double id) {
  const double u0 = w[0];
  if (order == 2)
    return h ? (3.0 * u0 - 4.0 * w[m] + w[2 * m]) * 0.5 * id : (-3.0 * u0 + 4.0 * w[m] - w[2 * m]) * 0.5 * id;
  const double d = 25.0 * u0 - 48.0 * w[m] + 36.0 * w[2 * m] - 16.0 * w[3 * m] + 3.0 * w[4 * m];
  return h ? d * id / 12.0 : -d * id / 12.0;
}
__device__ __forceinline__ double inward_coef(int order, int h, double id) {
  const double cf = order == 2 ? 3.0 * 0.5 * id : 25.0 * id / 12.0;
  return h ? cf : -cf;
}

// Edge cross-section t of a box (faces must be done): its R x R shell points
// by the section's kEdgeLanes lanes, lane q its own.  Edges XY(4) run along
// z, XZ(4) along y, YZ(4) along x; axis A is x, x, z and B is y, z, y, as
// Fix_Points orders them.  win: the section's kCornerW^2 staged points.
constexpr int kEdgeLanes = 16;
__device__ void robin_edge_section(const DevBox &B, BoxData D, int mode, int t, int q, double *win) {
  const int R = B.R;
  const int nint[3] = {B.n[0] - 2 * R, B.n[1] - 2 * R, B.n[2] - 2 * R};
  int grp, e, s;
  if (t < 4 * nint[2]) {
    grp = 0; e = t / nint[2]; s = t % nint[2];
  } else if (t < 4 * (nint[2] + nint[1])) {
    grp = 1; e = (t - 4 * nint[2]) / nint[1]; s = (t - 4 * nint[2]) % nint[1];
  } else {
    grp = 2;
    e = (t - 4 * (nint[2] + nint[1])) / nint[0];
    s = (t - 4 * (nint[2] + nint[1])) % nint[0];
  }
  const int axa = grp == 2 ? 2 : 0, axb = grp == 1 ? 2 : 1;
  const int h1 = (e >> 1) & 1, h2 = e & 1;
  const int ha = grp == 2 ? h2 : h1, hb = grp == 2 ? h1 : h2;
  const int na = B.n[axa], nb = B.n[axb];
  // box indices of local point (la, lb), counted inwards from the sides
  auto index = [&](int la, int lb, int &i, int &j, int &k) {
    const int pa = corner_index(la, ha, na), pb = corner_index(lb, hb, nb);
    i = axa == 0 ? pa : R + s;
    j = axb == 1 ? pb : R + s;
    k = axa == 2 ? pa : (axb == 2 ? pb : R + s);
  };
  const bool mine = q < R * R;
  const int la = mine ? q / R : 0, lb = mine ? q - la * R : 0;
  int i, j, k;
  index(la, lb, i, j, k);
  if (mode != ROBIN_UPDATE) {  // u stays: every point at once
    if (mine) robin_point(B, D, i, j, k, (1 << axa) | (1 << axb), mode);
    return;
  }
  // all of the square, so that no load waits for a test (what lies beyond the
  // derivatives' reach is not read)
#pragma unroll
  for (int m = 0; m < kCornerW * kCornerW / kEdgeLanes; ++m) {
    const int l = q + m * kEdgeLanes, wa = l / kCornerW, wb = l % kCornerW;
    int wi, wj, wk;
    index(min(wa, na - 1), min(wb, nb - 1), wi, wj, wk);
    win[l] = D.u[pidx(B, wi, wj, wk)];
  }
  const long long p = pidx(B, i, j, k);
  const double rho = D.rho[p];
  const double X[3] = {coord(B, 0, i), coord(B, 1, j), coord(B, 2, k)};
  const double r2n = (X[0] * X[0] + X[1] * X[1] + X[2] * X[2]) * B.ipn;
  // the two axes in ascending order, as robin_point takes them
  const bool a_first = axa < axb;
  const int ax1 = a_first ? axa : axb, ax2 = a_first ? axb : axa;
  const int s1 = a_first ? ha : hb, s2 = a_first ? hb : ha;
  const int m1 = a_first ? kCornerW : 1, m2 = a_first ? 1 : kCornerW;
  const double id1 = B.idx[ax1], id2 = B.idx[ax2];
  const double x1 = ax1 == 0 ? X[0] : X[1], x2 = ax2 == 1 ? X[1] : X[2];
  const double dF = r2n * (inward_coef(B.order, s1, id1) / x1 + inward_coef(B.order, s2, id2) / x2) + 1.0;
  double *w = win + la * kCornerW + lb;
#pragma unroll 1
  for (int sum = 2 * (kCornerR - 1); sum >= 0; --sum) {
    // the section's lanes lie in one wave, whose LDS accesses keep their
    // order: only the compiler has to
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    if (!mine || la + lb != sum) continue;
    const double u0 = w[0];
    const double sF =
        0.0 + inward_deriv(w, m1, B.order, s1, id1) / x1 + inward_deriv(w, m2, B.order, s2, id2) / x2;
    const double un = u0 - (r2n * sF + u0 - rho) / dF;
    w[0] = un;
    D.u[p] = un;
  }
}

// corners of one box, by one block (edges must be done): k outer, j, i
// inner (domain.cc:592-695); corner c has hz = bit 0, hx = bit 1, hy = bit
// 2.  cube: 8 kCornerCube doubles of LDS; corner c is wave c's, a lane a point
__device__ void robin_corners(const DevBox &B, BoxData D, int mode, double *cube) {
  const int R = B.R;
  if (mode != ROBIN_UPDATE) {
    // the operator modes leave u alone: every corner point at once
    const int R3 = R * R * R;
    for (int t = threadIdx.x; t < 8 * R3; t += blockDim.x) {
      const int c = t / R3, q = t - c * R3;
      const int hz = c & 1, hx = (c >> 1) & 1, hy = (c >> 2) & 1;
      const int qk = q / (R * R), qj = (q / R) % R, qi = q % R;
      robin_point(B, D, shell_index(qi, hx, B.n[0], R), shell_index(qj, hy, B.n[1], R),
                  shell_index(qk, hz, B.n[2], R), 7, mode);
    }
    return;
  }
  const int c = int(threadIdx.x) / kCornerR3, q = int(threadIdx.x) % kCornerR3;
  const bool mine = q < R * R * R;
  const int lk = mine ? q / (R * R) : 0, lj = mine ? (q / R) % R : 0, li = mine ? q % R : 0;
  const int l[3] = {li, lj, lk}, h[3] = {(c >> 1) & 1, (c >> 2) & 1, c & 1};
  const int ijk[3] = {corner_index(li, h[0], B.n[0]), corner_index(lj, h[1], B.n[1]),
                      corner_index(lk, h[2], B.n[2])};
  double X[3];
  for (int a = 0; a < 3; ++a) X[a] = coord(B, a, ijk[a]);
  const double r2n = (X[0] * X[0] + X[1] * X[1] + X[2] * X[2]) * B.ipn;
  double sdF = 0.0;
  for (int a = 0; a < 3; ++a) sdF += inward_coef(B.order, h[a], B.idx[a]) / X[a];
  const double dF = r2n * sdF + 1.0;
  double *w = cube + c * kCornerCube + (lk * kCornerW + lj) * kCornerW + li;
  const int st[3] = {1, kCornerW, kCornerW * kCornerW};
  // a point stages itself and, if it is the shell's innermost on an axis, the
  // points inwards of it; every lane loads them (within the box) at once
  const long long p = pidx(B, ijk[0], ijk[1], ijk[2]);
  const double rho = D.rho[p], own = D.u[p];
  const int reach = B.order == 2 ? 2 : 4;
  double in[3][4];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int m = 1; m <= 4; ++m) {
      int at[3] = {ijk[0], ijk[1], ijk[2]};
      at[a] = corner_index(min(l[a] + m, B.n[a] - 1), h[a], B.n[a]);
      in[a][m - 1] = D.u[pidx(B, at[0], at[1], at[2])];
    }
  if (mine) {
    w[0] = own;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int m = 1; m <= 4; ++m)
        if (l[a] == R - 1 && m <= reach) w[m * st[a]] = in[a][m - 1];
  }
#pragma unroll 1
  for (int sum = 3 * (R - 1); sum >= 0; --sum) {
    // one wave, as for the edges
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    if (!mine || l[0] + l[1] + l[2] != sum) continue;
    double sF = 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a) sF += inward_deriv(w, st[a], B.order, h[a], B.idx[a]) / X[a];
    const double u0 = w[0];
    const double un = u0 - (r2n * sF + u0 - rho) / dF;
    w[0] = un;
    D.u[p] = un;
  }
}

// faces: one thread per (box, face column)
__global__ __launch_bounds__(256) void k_robin_faces(const RobinItem *__restrict__ items, int n,
                                                      int total, int mode) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (items[mid].col0 <= g) lo = mid; else hi = mid - 1;
  }
  const DevBox &B = *items[lo].box;
  robin_face_column(B, box_data(B), g - items[lo].col0, mode);
}

// edges: kEdgeLanes lanes per (box, edge cross-section)
constexpr int kRobinEdgeThreads = 256, kEdgeSections = kRobinEdgeThreads / kEdgeLanes;
__global__ __launch_bounds__(kRobinEdgeThreads) void k_robin_edges(const RobinItem *__restrict__ items,
                                                                   int n, int total, int mode) {
  __shared__ double win[kEdgeSections][kCornerW * kCornerW + 2];
  const int sec = int(threadIdx.x) / kEdgeLanes, q = int(threadIdx.x) % kEdgeLanes;
  const int g = int(blockIdx.x) * kEdgeSections + sec;
  if (g >= total) return;
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (items[mid].ecol0 <= g) lo = mid; else hi = mid - 1;
  }
  const DevBox &B = *items[lo].box;
  robin_edge_section(B, box_data(B), mode, g - items[lo].ecol0, q, win[sec]);
}

// corners: one block per box
__global__ __launch_bounds__(8 * kCornerR3) void k_robin_corners(const RobinItem *__restrict__ items,
                                                       int mode) {
  __shared__ double cube[8 * kCornerCube];
  const DevBox &B = *items[blockIdx.x].box;
  robin_corners(B, box_data(B), mode, cube);
}

// Robin operator value at a shell point (no update)
__device__ __forceinline__ double robin_op_at(const DevBox &B, int i, int j, int k) {
  const int R = B.R;
  int mask = 0;
  if (i < R || i >= B.n[0] - R) mask |= 1;
  if (j < R || j >= B.n[1] - R) mask |= 2;
  if (k < R || k >= B.n[2] - R) mask |= 4;
  const long long p = pidx(B, i, j, k);
  const double *__restrict__ u = B.f[F_U];
  const int ijk[3] = {i, j, k};
  double X[3];
  for (int a = 0; a < 3; ++a) X[a] = coord(B, a, ijk[a]);
  const double r2 = X[0] * X[0] + X[1] * X[1] + X[2] * X[2];
  double sF = 0.0;
  for (int a = 0; a < 3; ++a) {
    if (!(mask & (1 << a))) continue;
    double cf;
    sF += deriv(B, u, p, a, i, j, k, cf) / X[a];
  }
  return r2 * B.ipn * sF + u[p];
}

// ------------------------------------------------------------------
// transfers.  Descriptors (target box, transfer, source box) are read
// through the constant address space; fields through 32-bit byte offsets.
// ------------------------------------------------------------------
typedef const __attribute__((address_space(4))) DevXfer ConstXfer;
typedef const __attribute__((address_space(4))) PtBlock ConstPtBlock;

// byte offset of point (i, j, k) of a float64 field
__device__ __forceinline__ unsigned boff(ConstBox &S, int i, int j, int k) {
  return (colourc(S, i, j, k) * unsigned(S.cs) + unsigned(k) * unsigned(S.ps) +
          unsigned(j) * unsigned(S.rs) + divc(S, unsigned(i))) *
         8u;
}

// Walks a float64 field of box S one step at a time from a boff: every step
// of +1 along an axis moves to the next colour block (wrapping after the
// last), plus one row (y), one plane (z), or, along x, one slot when the
// point's x leaves the last residue mod nc.
struct Walk {
  unsigned nc, cs8, wrap8, rs8, ps8;
  __device__ __forceinline__ Walk(ConstBox &S)
      : nc(unsigned(S.nc)), cs8(unsigned(S.cs) * 8u), wrap8((unsigned(S.nc) - 1u) * unsigned(S.cs) * 8u),
        rs8(unsigned(S.rs) * 8u), ps8(unsigned(S.ps) * 8u) {}
  // byte delta of the colour step from colour c; advances c
  __device__ __forceinline__ unsigned colour(unsigned &c) const {
    const bool last = c + 1u == nc;
    c = last ? 0u : c + 1u;
    return last ? 0u - wrap8 : cs8;
  }
  // x of residue r (mod nc) -> x + 1; advances c and r
  __device__ __forceinline__ unsigned x(unsigned &c, unsigned &r) const {
    const bool slot = r + 1u == nc;
    r = slot ? 0u : r + 1u;
    return colour(c) + (slot ? 8u : 0u);
  }
  __device__ __forceinline__ unsigned y(unsigned &c) const { return colour(c) + rs8; }
  __device__ __forceinline__ unsigned z(unsigned &c) const { return colour(c) + ps8; }
};

// point q0 + off of a block in lexicographic order, stepped from the
// block's first point (i0, j0, k0) so that only offsets below 2^24 are
// divided; or point off of a block's patch of rows
__device__ __forceinline__ void pt_lex(const PtBlock &Bk, ConstBox &T, unsigned off, int &i, int &j,
                                       int &k) {
  if (Bk.w > 0) {  // a patch of rows
    const unsigned r = fast_div(off, unsigned(Bk.w), Bk.inw);
    i = Bk.i0 + int(off - r * unsigned(Bk.w));
    j = Bk.j0 + int(r);
    k = Bk.k0;
    return;
  }
  const unsigned n0 = unsigned(T.n[0]), n1 = unsigned(T.n[1]);
  const unsigned x = unsigned(Bk.i0) + off;
  const unsigned dj = fast_div(x, n0, T.in0);
  unsigned jj = unsigned(Bk.j0) + dj, kk = unsigned(Bk.k0);
  if (jj >= n1) {
    const unsigned dk = fast_div(jj, n1, 1.0f / float(n1));
    jj -= dk * n1;
    kk += dk;
  }
  i = int(x - dj * n0);
  j = int(jj);
  k = int(kk);
}

// f(off) for the offsets off < nq of a block's points that fall to this
// thread (kPtThreads threads step through blocks of any length)
template <class F>
__device__ __forceinline__ void for_points(const PtBlock &Bk, F &&f) {
#pragma unroll 1
  for (unsigned off = threadIdx.x; off < Bk.nq; off += kPtThreads) f(off);
}

__device__ __forceinline__ bool is_interior(ConstBox &B, int i, int j, int k) {
  const int R = B.R;
  return i >= R && i < B.n[0] - R && j >= R && j < B.n[1] - R && k >= R && k < B.n[2] - R;
}

__device__ __forceinline__ unsigned axis_flags(ConstXfer &X, const int t[3], unsigned fl[3]) {
  fl[0] = X.ax[0].flags[t[0]];
  fl[1] = X.ax[1].flags[t[1]];
  fl[2] = X.ax[2].flags[t[2]];
  return fl[0] & fl[1] & fl[2];
}

// tensor Lagrange interpolation of field f of box S with KP nodes per axis
// (reference accumulation order, interpolation.cc:257-296); the nodes of
// coincident axes are skipped, their weights being exactly one unit vector
template <int KP>
__device__ __forceinline__ double tinterp(ConstBox &S, const void *f, ConstXfer &X, const int t[3],
                                          const unsigned fl[3]) {
  int s0[3], kk[3];
  const double *w[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (fl[a] & 4) {
      s0[a] = X.ax[a].coinc[t[a]];
      kk[a] = 1;
      w[a] = nullptr;
    } else {
      s0[a] = X.ax[a].start[t[a]];
      kk[a] = KP;
      w[a] = X.ax[a].w + t[a] * KP;
    }
  }
  double wz[KP], wy[KP];
#pragma unroll
  for (int K = 0; K < KP; ++K) {
    wz[K] = w[2] ? w[2][K] : 1.0;
    wy[K] = w[1] ? w[1][K] : 1.0;
  }
  const Walk wk(S);
  unsigned oI = boff(S, s0[0], s0[1], s0[2]);
  unsigned cI = colourc(S, s0[0], s0[1], s0[2]);
  unsigned rI = unsigned(s0[0]) - divc(S, unsigned(s0[0])) * wk.nc;
  double acc = 0.0;
  for (int I = 0; I < kk[0]; ++I) {
    double uj = 0.0;
    unsigned oJ = oI, cJ = cI;
    if constexpr (KP <= 6) {
      // the (J, K) plane of nodes: every load of it issued before the sums
      double v[KP][KP];
#pragma unroll
      for (int J = 0; J < KP; ++J) {
        unsigned off = oJ, c = cJ;
#pragma unroll
        for (int K = 0; K < KP; ++K) {
          v[J][K] = (J < kk[1] && K < kk[2]) ? ld<double>(f, off) : 0.0;
          off += wk.z(c);
        }
        oJ += wk.y(cJ);
      }
#pragma unroll
      for (int J = 0; J < KP; ++J)
        if (J < kk[1]) {
          double uk = 0.0;
#pragma unroll
          for (int K = 0; K < KP; ++K)
            if (K < kk[2]) uk += v[J][K] * wz[K];
          uj += uk * wy[J];
        }
    } else {
      // wider stencils: CJ rows of nodes at a time, every load of them
      // issued before their sums (register budget); the sums keep the
      // order of the row-by-row form
      constexpr int CJ = KP / 2;
      for (int J0 = 0; J0 < kk[1]; J0 += CJ) {
        double v[CJ][KP];
#pragma unroll
        for (int J = 0; J < CJ; ++J) {
          unsigned off = oJ, c = cJ;
#pragma unroll
          for (int K = 0; K < KP; ++K) {
            v[J][K] = (J0 + J < kk[1] && K < kk[2]) ? ld<double>(f, off) : 0.0;
            off += wk.z(c);
          }
          if (J0 + J < kk[1]) oJ += wk.y(cJ);
        }
#pragma unroll
        for (int J = 0; J < CJ; ++J)
          if (J0 + J < kk[1]) {
            double uk = 0.0;
#pragma unroll
            for (int K = 0; K < KP; ++K)
              if (K < kk[2]) uk += v[J][K] * wz[K];
            uj += uk * wy[J0 + J];
          }
      }
    }
    acc += uj * (w[0] ? w[0][I] : 1.0);
    oI += wk.x(cI, rI);
  }
  return acc;
}

// trilinear interpolation of the coarse correction v = u - ww of box S
// (interpolation.cc:125-182; k_corr_v forms v)
__device__ __forceinline__ double trilinear_corr(ConstBox &S, ConstXfer &X, const int t[3]) {
  const void *v = S.f[F_V];
  const int x0 = X.ax[0].start[t[0]], y0 = X.ax[1].start[t[1]], z0 = X.ax[2].start[t[2]];
  const double *wx = X.ax[0].w + 2 * t[0];
  const double *wy = X.ax[1].w + 2 * t[1];
  const double *wzp = X.ax[2].w + 2 * t[2];
  const double dxi = wx[0], dxf = wx[1], dyi = wy[0], dyf = wy[1], dzi = wzp[0], dzf = wzp[1];
  // the eight corners, walked from (x0, y0, z0)
  const Walk wk(S);
  const unsigned c0 = colourc(S, x0, y0, z0);
  unsigned r = unsigned(x0) - divc(S, unsigned(x0)) * wk.nc;
  const unsigned o000 = boff(S, x0, y0, z0);
  unsigned c = c0;
  const unsigned o100 = o000 + wk.x(c, r);  // c = c0 + 1
  unsigned c1 = c;
  const unsigned o110 = o100 + wk.y(c1);     // c1 = c0 + 2
  unsigned c2 = c1;
  const unsigned o111 = o110 + wk.z(c2);
  unsigned cb = c;
  const unsigned o101 = o100 + wk.z(cb);
  unsigned cy = c0;
  const unsigned o010 = o000 + wk.y(cy);    // cy = c0 + 1
  unsigned cz = cy;
  const unsigned o011 = o010 + wk.z(cz);
  unsigned cw = c0;
  const unsigned o001 = o000 + wk.z(cw);
#define V(o) ld<double>(v, o)
  return ((V(o000) * dxi + V(o100) * dxf) * dyi + (V(o010) * dxi + V(o110) * dxf) * dyf) * dzi +
         ((V(o001) * dxi + V(o101) * dxf) * dyi + (V(o011) * dxi + V(o111) * dxf) * dyf) * dzf;
#undef V
}

// the same for a 2:1 nested source (DevXfer::affine): corner nodes and
// weights (1, 0 at a coincident axis; 1/2, 1/2 at a midpoint) from the index
// map instead of the tables, the eight corners walked as above
__device__ __forceinline__ double trilinear_nested(ConstBox &S, ConstXfer &X, const int t[3]) {
  const void *v = S.f[F_V];
  int c[3];
  double wi[3], wf[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int q = t[a] + X.aff[a];
    c[a] = q >> 1;
    const bool mid = (q & 1) != 0;
    wi[a] = mid ? 0.5 : 1.0;
    wf[a] = mid ? 0.5 : 0.0;
    // a coincident axis reads node c twice (weight 0 on the second): keep
    // the second node in range at the source's last node
    if (!mid && c[a] + 1 >= S.n[a]) c[a] = S.n[a] - 2, wi[a] = 0.0, wf[a] = 1.0;
  }
  const Walk wk(S);
  const unsigned c0 = colourc(S, c[0], c[1], c[2]);
  unsigned r = unsigned(c[0]) - divc(S, unsigned(c[0])) * wk.nc;
  const unsigned o000 = boff(S, c[0], c[1], c[2]);
  unsigned cc = c0;
  const unsigned o100 = o000 + wk.x(cc, r);
  unsigned c1 = cc;
  const unsigned o110 = o100 + wk.y(c1);
  unsigned c2 = c1;
  const unsigned o111 = o110 + wk.z(c2);
  unsigned cb = cc;
  const unsigned o101 = o100 + wk.z(cb);
  unsigned cy = c0;
  const unsigned o010 = o000 + wk.y(cy);
  unsigned cz = cy;
  const unsigned o011 = o010 + wk.z(cz);
  unsigned cw = c0;
  const unsigned o001 = o000 + wk.z(cw);
#define V(o) ld<double>(v, o)
  return ((V(o000) * wi[0] + V(o100) * wf[0]) * wi[1] + (V(o010) * wi[0] + V(o110) * wf[0]) * wf[1]) * wi[2] +
         ((V(o001) * wi[0] + V(o101) * wf[0]) * wi[1] + (V(o011) * wi[0] + V(o111) * wf[0]) * wf[1]) * wf[2];
#undef V
}

// trilinear interpolation of field f of box S (interpolation.cc:125-182),
// the corners walked as in trilinear_corr
__device__ __forceinline__ double trilinear_field(ConstBox &S, const void *f, ConstXfer &X,
                                                  const int t[3]) {
  const int x0 = X.ax[0].start[t[0]], y0 = X.ax[1].start[t[1]], z0 = X.ax[2].start[t[2]];
  const double *wx = X.ax[0].w + 2 * t[0];
  const double *wy = X.ax[1].w + 2 * t[1];
  const double *wzp = X.ax[2].w + 2 * t[2];
  const double dxi = wx[0], dxf = wx[1], dyi = wy[0], dyf = wy[1], dzi = wzp[0], dzf = wzp[1];
  const Walk wk(S);
  const unsigned c0 = colourc(S, x0, y0, z0);
  unsigned r = unsigned(x0) - divc(S, unsigned(x0)) * wk.nc;
  const unsigned o000 = boff(S, x0, y0, z0);
  unsigned c = c0;
  const unsigned o100 = o000 + wk.x(c, r);
  unsigned c1 = c;
  const unsigned o110 = o100 + wk.y(c1);
  unsigned c2 = c1;
  const unsigned o111 = o110 + wk.z(c2);
  unsigned cb = c;
  const unsigned o101 = o100 + wk.z(cb);
  unsigned cy = c0;
  const unsigned o010 = o000 + wk.y(cy);
  unsigned cz = cy;
  const unsigned o011 = o010 + wk.z(cz);
  unsigned cw = c0;
  const unsigned o001 = o000 + wk.z(cw);
#define V(o) ld<double>(f, o)
  return ((V(o000) * dxi + V(o100) * dxf) * dyi + (V(o010) * dxi + V(o110) * dxf) * dyf) * dzi +
         ((V(o001) * dxi + V(o101) * dxf) * dyi + (V(o011) * dxi + V(o111) * dxf) * dyf) * dzf;
#undef V
}

// ------------------------------------------------------------------
// Lagrange interpolation of a block of target points as one tensor product.
// The targets nt[0] x nt[1] x nt[2] from t0 take one source box; per axis
// each has its first node, node count (1 on a node) and weights (the
// transfer tables).  The source nodes they read (their bounding box) are
// staged in LDS; then the sums over z are formed for every (x, y) node and z
// target, from these the sums over y for every (x node, y target, z target),
// then those over x: tinterp's sums for every target, in its order and with
// its roundings (the same bits), each formed once instead of by every target
// that shares it: 3 KP instead of KP^3 products per target, times the few
// extra nodes at a tile's edge.  Bound by the LDS reads of the products.
// ------------------------------------------------------------------
template <int KP>
struct TileLds {
  // node extents of 16 targets refined by two (16 / 2 + KP + 1) and of the
  // ghost width along a face's normal (KP + 3); larger regions (targets
  // coarser than the source) take the point-by-point path
  static constexpr int S = 9 + KP, U = KP + 3;
  static constexpr int kNodes = S * S * U > 256 * U ? S * S * U : 256 * U;
  static constexpr int kZ = 16 * S * U;
  double a[kNodes];  // nodes [z][y][x]; then sums over y [z target][y target][x]
  double z[kZ];      // sums over z [z target][y][x]
  double w[3][16 * KP];
  int first[3][16];  // from the region's low corner
  int cnt[3][16];
  int lo[3], ext[3];
};

// writes field tf at every target for which want(i, j, k) holds and some
// source holds the point: `bits` are the flags that make a source eligible
// (bit 0 its non-ghost part, bit 1 its extent), the last eligible source
// counts; to_zero: the last source alone decides, 0 where it is not eligible
template <int KP, class W>
__device__ __forceinline__ void tile_transfer(TileLds<KP> &L, const PtBlock &Bk, ConstBox &T,
                                              const int t0[3], const int nt[3], unsigned bits, int ff,
                                              int tf, bool to_zero, W &&want) {
  ConstXfer *xs = (ConstXfer *)Bk.src;
  // the tile's source: lanes 0-15, 16-31, 32-47 of every wave hold the
  // targets of axes x, y, z
  const int lane = int(threadIdx.x & 63u), la = lane >> 4, li = lane & 15;
  const int lt0 = la == 0 ? t0[0] : (la == 1 ? t0[1] : t0[2]);
  const int lnt = la == 0 ? nt[0] : (la == 1 ? nt[1] : (la == 2 ? nt[2] : 0));
  const bool lv = li < lnt;
  const unsigned long long vm = __ballot(lv);
  int src = -1;
  bool mixed = false;
  unsigned lf = 0;
  for (int x = Bk.nsrc - 1; x >= 0; --x) {
    const unsigned char *fp = la == 0 ? xs[x].ax[0].flags : (la == 1 ? xs[x].ax[1].flags : xs[x].ax[2].flags);
    lf = lv ? fp[lt0 + li] : 0u;
    bool every = false, some = false;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (!(bits & (1u << q))) continue;
      const unsigned long long m = __ballot((lf >> q) & 1u);
      every = every || m == vm;
      some = some || ((m & 0xffffull) && (m & 0xffff0000ull) && (m & 0xffff00000000ull));
    }
    if (every) {
      src = x;
      break;
    }
    mixed = some;
    if (mixed || to_zero) break;
  }
  const int total = nt[0] * nt[1] * nt[2];
  const float in0 = 1.0f / float(nt[0]), in1 = 1.0f / float(nt[1]);
  if (!mixed && src < 0 && !to_zero) return;
  bool fits = !mixed && src >= 0;
  if (fits) {
    ConstXfer &X = xs[src];
    if (threadIdx.x < 64) {
      int first = 1 << 28, cnt = 1;
      if (lv) {
        const bool on = (lf & 4u) != 0;
        const int *p = la == 0 ? (on ? X.ax[0].coinc : X.ax[0].start)
                               : (la == 1 ? (on ? X.ax[1].coinc : X.ax[1].start)
                                          : (on ? X.ax[2].coinc : X.ax[2].start));
        first = p[lt0 + li];
        cnt = on ? 1 : KP;
        const double *w = (la == 0 ? X.ax[0].w : (la == 1 ? X.ax[1].w : X.ax[2].w)) + (lt0 + li) * KP;
#pragma unroll
        for (int m = 0; m < KP; ++m) L.w[la][li * KP + m] = on ? 1.0 : w[m];
      }
      int lo = first, hi = lv ? first + cnt : 0;
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) {
        lo = min(lo, __shfl_xor(lo, d, 16));
        hi = max(hi, __shfl_xor(hi, d, 16));
      }
      if (la < 3) {
        L.first[la][li] = first - lo;
        L.cnt[la][li] = cnt;
        if (li == 0) {
          L.lo[la] = lo;
          L.ext[la] = hi - lo;
        }
      }
    }
    __syncthreads();
    const int ex = L.ext[0], ey = L.ext[1], ez = L.ext[2];
    fits = ex * ey * ez <= TileLds<KP>::kNodes && nt[2] * ey * ex <= TileLds<KP>::kZ &&
           nt[2] * nt[1] * ex <= TileLds<KP>::kNodes;
    if (fits) {
      ConstBox &S = cbox(X.src);
      const void *f = S.f[ff];
      const int lx = L.lo[0], ly = L.lo[1], lz = L.lo[2];
      const float ix = 1.0f / float(ex), iy = 1.0f / float(ey);
      for (int q = threadIdx.x; q < ex * ey * ez; q += kPtThreads) {
        const int r = int(fast_div(unsigned(q), unsigned(ex), ix)), x = q - r * ex;
        const int z = int(fast_div(unsigned(r), unsigned(ey), iy)), y = r - z * ey;
        L.a[q] = ld<double>(f, boff(S, lx + x, ly + y, lz + z));
      }
      __syncthreads();
      const int exy = ex * ey;
      for (int q = threadIdx.x; q < nt[2] * exy; q += kPtThreads) {
        const int zt = int(fast_div(unsigned(q), unsigned(exy), ix * iy)), r = q - zt * exy;
        const double *v = L.a + L.first[2][zt] * exy + r, *w = L.w[2] + zt * KP;
        const int n = L.cnt[2][zt];
        double uk = 0.0;
        if (n == 1) {
          uk += v[0] * w[0];
        } else {
#pragma unroll
          for (int K = 0; K < KP; ++K) uk += v[K * exy] * w[K];
        }
        L.z[q] = uk;
      }
      __syncthreads();
      for (int q = threadIdx.x; q < nt[2] * nt[1] * ex; q += kPtThreads) {
        const int r = int(fast_div(unsigned(q), unsigned(ex), ix)), x = q - r * ex;
        const int zt = int(fast_div(unsigned(r), unsigned(nt[1]), in1)), yt = r - zt * nt[1];
        const double *v = L.z + zt * exy + L.first[1][yt] * ex + x, *w = L.w[1] + yt * KP;
        const int n = L.cnt[1][yt];
        double uj = 0.0;
        if (n == 1) {
          uj += v[0] * w[0];
        } else {
#pragma unroll
          for (int J = 0; J < KP; ++J) uj += v[J * ex] * w[J];
        }
        L.a[q] = uj;
      }
      __syncthreads();
      for (int q = threadIdx.x; q < total; q += kPtThreads) {
        const int r = int(fast_div(unsigned(q), unsigned(nt[0]), in0)), xt = q - r * nt[0];
        const int zt = int(fast_div(unsigned(r), unsigned(nt[1]), in1)), yt = r - zt * nt[1];
        const int i = t0[0] + xt, j = t0[1] + yt, k = t0[2] + zt;
        if (!want(i, j, k)) continue;
        const double *v = L.a + r * ex + L.first[0][xt], *w = L.w[0] + xt * KP;
        const int n = L.cnt[0][xt];
        double acc = 0.0;
        if (n == 1) {
          acc += v[0] * w[0];
        } else {
#pragma unroll
          for (int I = 0; I < KP; ++I) acc += v[I] * w[I];
        }
        st<double>(T.f[tf], boff(T, i, j, k), acc);
      }
      return;
    }
  }
  // sources that differ over the tile, or a region beyond the LDS: point by
  // point
#pragma unroll 1
  for (int q = threadIdx.x; q < total; q += kPtThreads) {
    const int r = int(fast_div(unsigned(q), unsigned(nt[0]), in0)), xt = q - r * nt[0];
    const int zt = int(fast_div(unsigned(r), unsigned(nt[1]), in1)), yt = r - zt * nt[1];
    const int t[3] = {t0[0] + xt, t0[1] + yt, t0[2] + zt};
    if (!want(t[0], t[1], t[2])) continue;
    const unsigned o = boff(T, t[0], t[1], t[2]);
    for (int x = Bk.nsrc - 1; x >= 0; --x) {
      ConstXfer &X = xs[x];
      unsigned fl[3];
      if (axis_flags(X, t, fl) & bits) {
        ConstBox &S = cbox(X.src);
        st<double>(T.f[tf], o, tinterp<KP>(S, S.f[ff], X, t, fl));
        break;
      }
      if (to_zero) {
        st<double>(T.f[tf], o, 0.0);
        break;
      }
    }
  }
}

// multigrid::Transferir (multigrid.cc:122-141, ffunction.cc:2436-2475):
// every point of the region (PtBlock::mg bits 0-1: 0 all, 1 interior, 2
// ghost shell) of the listed target boxes takes field ff of the source
// boxes interpolated at its coordinates, linear (KP = 2) or Lagrange with
// KP nodes per axis: the last source whose non-ghost part holds the point
// (or, with `all` (bit 2), whose extent does); with `to_zero` (bit 3) the
// last source alone decides and a point it does not hold is set to 0 (the
// reference's source loop overwrites every point on each pass)
// Linear transfers, and most onto a coarser level, go point by point; other
// Lagrange ones by tiles of kXferTile targets (tile_transfer): N=129 8th order,
// one 135^3 box from its parent, 1175 -> 78 us.  (transfer_fields has the rule.)
template <int KP>
__global__ __launch_bounds__(kPtThreads) void k_transfer_points(const PtBlock *__restrict__ blocks,
                                                                int ff, int tf) {
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &T = cbox(Bk.box);
  for_points(Bk, [&](unsigned off) {
    int i, j, k;
    pt_lex(Bk, T, off, i, j, k);
    const int region = Bk.mg & 3, all = (Bk.mg >> 2) & 1, to_zero = (Bk.mg >> 3) & 1;
    const bool inside = is_interior(T, i, j, k);
    if ((region == 1 && !inside) || (region == 2 && inside)) return;
    const int t[3] = {i, j, k};
    const unsigned o = boff(T, i, j, k);
    ConstXfer *xs = (ConstXfer *)Bk.src;
    for (int x = Bk.nsrc - 1; x >= 0; --x) {
      ConstXfer &X = xs[x];
      unsigned fl[3];
      const unsigned f = axis_flags(X, t, fl);
      if ((f & 1) || (all && (f & 2))) {
        ConstBox &S = cbox(X.src);
        double v;
        if constexpr (KP == 2) {
          if (f & 4)  // a source node: its value (interpolation.cc:140-147)
            v = ld<double>(S.f[ff], boff(S, X.ax[0].coinc[i], X.ax[1].coinc[j], X.ax[2].coinc[k]));
          else
            v = trilinear_field(S, S.f[ff], X, t);
        } else {
          v = tinterp<KP>(S, S.f[ff], X, t, fl);
        }
        st<double>(T.f[tf], o, v);
        return;
      }
      if (to_zero) {
        st<double>(T.f[tf], o, 0.0);
        return;
      }
    }
  });
}

template <int KP>
__global__ __launch_bounds__(kPtThreads) void k_transfer_tiles(const PtBlock *__restrict__ blocks,
                                                               int ff, int tf) {
  __shared__ TileLds<KP> L;
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &T = cbox(Bk.box);
  const int t0[3] = {Bk.i0, Bk.j0, Bk.k0};
  const int nt[3] = {min(kXferTile[0], T.n[0] - t0[0]), min(kXferTile[1], T.n[1] - t0[1]),
                     min(kXferTile[2], T.n[2] - t0[2])};
  const int region = Bk.mg & 3, all = (Bk.mg >> 2) & 1, to_zero = (Bk.mg >> 3) & 1;
  // a tile of interior points has none of the ghost shell
  if (region == 2 && is_interior(T, t0[0], t0[1], t0[2]) &&
      is_interior(T, t0[0] + nt[0] - 1, t0[1] + nt[1] - 1, t0[2] + nt[2] - 1))
    return;
  tile_transfer<KP>(L, Bk, T, t0, nt, all ? 3u : 1u, ff, tf, to_zero, [&](int i, int j, int k) {
    return region == 0 || is_interior(T, i, j, k) == (region == 1);
  });
}

// u restriction: coarse INSIDE points inside a fine box's non-ghost part
// (all = false), injection at coincident points (Lagrange 3 elsewhere)
__global__ __launch_bounds__(kPtThreads) void k_restrict_u(const PtBlock *__restrict__ blocks) {
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &T = cbox(Bk.box);
  for_points(Bk, [&](unsigned off) {
    int i, j, k;
    pt_lex(Bk, T, off, i, j, k);
    if (!is_interior(T, i, j, k)) return;
    const int t[3] = {i, j, k};
    ConstXfer *xs = (ConstXfer *)Bk.src;
    for (int x = Bk.nsrc - 1; x >= 0; --x) {
      ConstXfer &X = xs[x];
      unsigned fl[3];
      if (!(axis_flags(X, t, fl) & 1)) continue;
      ConstBox &S = cbox(X.src);
      st<double>(T.f[F_U], boff(T, i, j, k), tinterp<4>(S, S.f[F_U], X, t, fl));
      return;
    }
  });
}

// full weighting (1/4, 1/2, 1/4)^3 of field w of box S around node
// (ci, cj, ck), whose 3x3x3 neighbourhood must lie in the box
__device__ __forceinline__ double fw27(ConstBox &S, const void *w, int ci, int cj, int ck) {
  // walk the 27 points from (ci-1, cj-1, ck-1)
  const Walk wk(S);
  unsigned oz = boff(S, ci - 1, cj - 1, ck - 1);
  unsigned cz = colourc(S, ci - 1, cj - 1, ck - 1);
  const unsigned r0 = unsigned(ci - 1) - divc(S, unsigned(ci - 1)) * wk.nc;
  double acc = 0.0;
  for (int dz = -1; dz <= 1; ++dz) {
    const double wz = dz == 0 ? 0.5 : 0.25;
    unsigned oy = oz, cy = cz;
    for (int dy = -1; dy <= 1; ++dy) {
      const double wy = dy == 0 ? 0.5 : 0.25;
      unsigned cx = cy, r = r0;
      const unsigned om = oy;
      const unsigned o0 = om + wk.x(cx, r);
      const unsigned op = o0 + wk.x(cx, r);
      const double wm = ld<double>(w, om);
      const double w0 = ld<double>(w, o0);
      const double wp = ld<double>(w, op);
      acc += wz * wy * (0.25 * wm + 0.5 * w0 + 0.25 * wp);
      oy += wk.y(cy);
    }
    oz += wk.z(cz);
  }
  return acc;
}

// Filtered defect of a fine box whose defect is restricted to points of a
// coarser level that do not coincide with its nodes (a merged box off the
// coarser lattice): v = the full weighting of w at every node whose 3x3x3
// neighbourhood is interior, v = w elsewhere.  The restriction then
// interpolates v instead of w: the filter removes the (i+j+k)-parity
// pattern that the multi-colour sweeps leave in the defect, which the
// Lagrange interpolation would otherwise alias into the coarse correction.
// At a converged u the interior defect is zero, so the fixed point is the
// one of the unfiltered restriction.
__global__ __launch_bounds__(kPtThreads) void k_filter_defect(const PtBlock *__restrict__ blocks) {
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &S = cbox(Bk.box);
  for_points(Bk, [&](unsigned off) {
    int i, j, k;
    pt_lex(Bk, S, off, i, j, k);
    const int R = S.R;
    const unsigned o = boff(S, i, j, k);
    const bool in = i - 1 >= R && i + 1 < S.n[0] - R && j - 1 >= R && j + 1 < S.n[1] - R &&
                    k - 1 >= R && k + 1 < S.n[2] - R;
    st<double>(S.f[F_V], o, in ? fw27(S, S.f[F_W], i, j, k) : ld<double>(S.f[F_W], o));
  });
}

// The same filter, one thread per run of kFilterCx points along x of one
// row: the 9 neighbour rows' kFilterCx + 2 values are loaded once for the
// run (the lanes of a wave then read consecutive slots of one colour block
// per load), and each point sums its 27 terms in fw27's order (same bits).
constexpr int kFilterCx = 4;
__global__ __launch_bounds__(kPtThreads) void k_filter_cols(const PtBlock *__restrict__ blocks) {
  constexpr int NX = kFilterCx + 2;
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &S = cbox(Bk.box);
  if (threadIdx.x >= Bk.nq) return;
  const int n0 = S.n[0], n1 = S.n[1], n2 = S.n[2], R = S.R;
  const int nxc = (n0 + kFilterCx - 1) / kFilterCx;
  const int q = int(Bk.q0 + threadIdx.x);
  const int row = q / nxc;
  const int i0 = (q - row * nxc) * kFilterCx;
  const int k = row / n1, j = row - k * n1;
  const void *w = S.f[F_W];
  const bool in_jk = j - 1 >= R && j + 1 < n1 - R && k - 1 >= R && k + 1 < n2 - R;
  bool in[kFilterCx];
  bool any = false;
#pragma unroll
  for (int p = 0; p < kFilterCx; ++p) {
    const int i = i0 + p;
    in[p] = in_jk && i - 1 >= R && i + 1 < n0 - R;
    any = any || in[p];
  }
  double acc[kFilterCx];
#pragma unroll
  for (int p = 0; p < kFilterCx; ++p) acc[p] = 0.0;
  if (any) {
    // x nodes i0 - 1 .. i0 + kFilterCx of rows j - 1 .. j + 1, planes
    // k - 1 .. k + 1 (all inside the box: in_jk); nodes past the box ends
    // along x are not loaded and feed no filtered point
    const Walk wk(S);
    unsigned ox[NX], cx[NX];
    bool okx[NX];
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int xi = i0 - 1 + x;
      okx[x] = xi >= 0 && xi < n0;
      ox[x] = okx[x] ? boff(S, xi, j - 1, k - 1) : 0u;
      cx[x] = okx[x] ? colourc(S, xi, j - 1, k - 1) : 0u;
    }
#pragma unroll
    for (int dz = -1; dz <= 1; ++dz) {
      const double wz = dz == 0 ? 0.5 : 0.25;
      unsigned oy[NX], cy[NX];
#pragma unroll
      for (int x = 0; x < NX; ++x) {
        oy[x] = ox[x];
        cy[x] = cx[x];
      }
#pragma unroll
      for (int dy = -1; dy <= 1; ++dy) {
        const double wy = dy == 0 ? 0.5 : 0.25;
        double val[NX];
#pragma unroll
        for (int x = 0; x < NX; ++x) val[x] = okx[x] ? ld<double>(w, oy[x]) : 0.0;
#pragma unroll
        for (int p = 0; p < kFilterCx; ++p)
          if (in[p]) acc[p] += wz * wy * (0.25 * val[p] + 0.5 * val[p + 1] + 0.25 * val[p + 2]);
#pragma unroll
        for (int x = 0; x < NX; ++x) oy[x] += wk.y(cy[x]);
      }
#pragma unroll
      for (int x = 0; x < NX; ++x) ox[x] += wk.z(cx[x]);
    }
  }
#pragma unroll
  for (int p = 0; p < kFilterCx; ++p) {
    const int i = i0 + p;
    if (i >= n0) continue;
    const unsigned o = boff(S, i, j, k);
    st<double>(S.f[F_V], o, in[p] ? acc[p] : ld<double>(w, o));
  }
}

// Coarse FAS source: W_c = restriction of the fine defect (full weighting
// where the coarse point coincides with a fine point whose 3x3x3
// neighbourhood is fine interior, injection / Lagrange-2 elsewhere, of the
// filtered defect k_filter_defect leaves in v when the source box is off
// the coarse lattice), then
// rho_c = W_c + R_c with R_c = N(u_c) inside, the Robin operator on the
// shell (multigrid levels).  Refinement levels overwrite rho_c only where
// the point is inside both boxes' non-ghost parts (ffunction.cc:2808-2849).
// Also saves ww_c = u_c on every coarse point.
template <int ORD, int EQ>
__global__ __launch_bounds__(kPtThreads) void k_restrict_defect(const PtBlock *__restrict__ blocks) {
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &T = cbox(Bk.box);
  for_points(Bk, [&](unsigned off) {
    int i, j, k;
    pt_lex(Bk, T, off, i, j, k);
    const unsigned o = boff(T, i, j, k);
    const double uc = ld<double>(T.f[F_U], o);
    st<double>(T.f[F_WW], o, uc);
    const bool inside = is_interior(T, i, j, k);
    if (!Bk.mg && !inside) return;
    const int t[3] = {i, j, k};
    bool covered = false;
    double wc = 0.0;
    ConstXfer *xs = (ConstXfer *)Bk.src;
    for (int x = Bk.nsrc - 1; x >= 0; --x) {
      ConstXfer &X = xs[x];
      unsigned fl[3];
      const unsigned f = axis_flags(X, t, fl);
      if (!((f & 1) || (Bk.mg && (f & 2)))) continue;
      ConstBox &S = cbox(X.src);
      if (f & 8) {
        wc = fw27(S, S.f[F_W], X.ax[0].coinc[i], X.ax[1].coinc[j], X.ax[2].coinc[k]);
      } else {
        wc = tinterp<3>(S, X.filt ? S.f[F_V] : S.f[F_W], X, t, fl);
      }
      covered = true;
      break;
    }
    if (!covered && !Bk.mg) return;
    if (covered) st<double>(T.f[F_W], o, wc); else wc = ld<double>(T.f[F_W], o);
    double Rc;
    if (inside) {
      constexpr int NC = colours_of(ORD, EQ);
      const Nbr<NC> nb = box_offs<NC, 8>(T, int(colourc(T, i, j, k)), i % NC);
      double dN;
      point_op<ORD, EQ>(T, T.f[F_U], o, nb, uc, i, j, k, Rc, dN);
    } else {
      Rc = robin_op_at(cbox_plain(T), i, j, k);
    }
    st<double>(T.f[F_RHO], o, wc + Rc);
  });
}

// v = u - ww on the listed points of a coarse box (the nodes the next
// prolongation reads): the coarse correction, formed once per node instead
// of once per fine point that interpolates from it
__global__ __launch_bounds__(kPtThreads) void k_corr_v(const PtBlock *__restrict__ blocks) {
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &S = cbox(Bk.box);
  for_points(Bk, [&](unsigned off) {
    int i, j, k;
    pt_lex(Bk, S, off, i, j, k);
    const unsigned o = boff(S, i, j, k);
    st<double>(S.f[F_V], o, ld<double>(S.f[F_U], o) - ld<double>(S.f[F_WW], o));
  });
}

// prolongation of the coarse correction v (k_corr_v) and u += I v (all
// points on multigrid levels, interior points on refinement levels).  A
// block covers a column of kProTile tiles (nq planes from (i0, j0, k0)); the
// coarse nodes a tile reads are staged in LDS and the interpolation along x
// is formed once per coarse row, so that a fine point costs four LDS reads
// and its own u instead of eight scattered coarse loads: per launch N=161 187
// -> 88 us, 16 x N=65 95 -> 55.  Each value is trilinear_corr's or
// trilinear_nested's to the bit (x first, then y, then z); tiles whose
// points take different sources go point by point.
__global__ __launch_bounds__(kPtThreads) void k_prolong(const PtBlock *__restrict__ blocks) {
  constexpr int TX = kProTile[0], TY = kProTile[1], TZ = kProTile[2];
  static_assert(TX == 64 && TY * TZ * TX == 4 * kPtThreads && TY == 4 && TZ == 4, "thread mapping");
  constexpr int VX = TX / 2 + 4, VY = TY / 2 + 3, VZ = TZ / 2 + 3;
  __shared__ double V[VX * VY * VZ];  // coarse nodes [z][y][x]
  __shared__ double A[VZ * VY * TX];  // interpolated along x [z][y][x target]
  // per target of an axis (x, then y, then z): first node, node of a
  // coincident target (-1: none), weights of the first and second node
  constexpr int NT = TX + TY + TZ;
  __shared__ int first[NT], same[NT];
  __shared__ double wi[NT], wf[NT];
  __shared__ int lo[3], ext[3];
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &T = cbox(Bk.box);
  ConstXfer *xs = (ConstXfer *)Bk.src;
  const int lane = int(threadIdx.x & 63u), wave = int(threadIdx.x >> 6);
  const int g = Bk.mg ? 0 : T.R;  // the points taken: [g, n - g) on every axis
  const int kend = min(Bk.k0 + int(Bk.nq), T.n[2] - g);
  const int nx = min(TX, T.n[0] - g - Bk.i0), ny = min(TY, T.n[1] - g - Bk.j0);
  for (int k0 = Bk.k0; k0 < kend; k0 += TZ) {
    const int nz = min(TZ, kend - k0);
    // the thread's four targets: (lane, wave, q); their u is loaded first
    const int i = Bk.i0 + lane, j = Bk.j0 + wave;
    const bool mine = lane < nx && wave < ny;
    unsigned o[TZ];
    double u0[TZ];
#pragma unroll
    for (int q = 0; q < TZ; ++q) {
      o[q] = 0;
      u0[q] = 0.0;
      if (mine && q < nz) {
        o[q] = boff(T, i, j, k0 + q);
        u0[q] = ld<double>(T.f[F_U], o[q]);
      }
    }
    // the tile's source: lane x of every wave holds x target x; lanes 0-3 y
    // and 4-7 z targets
    const bool vx = lane < nx;
    const bool vyz = lane < 4 ? lane < ny : (lane < 8 && lane - 4 < nz);
    const int tyz = lane < 4 ? Bk.j0 + lane : k0 + (lane - 4);
    const unsigned long long mx = __ballot(vx), myz = __ballot(vyz);
    int src = -1;
    bool mixed = false;
    unsigned fx = 0, fyz = 0;
    for (int x = Bk.nsrc - 1; x >= 0; --x) {
      fx = vx ? xs[x].ax[0].flags[i] : 0u;
      fyz = vyz ? (lane < 4 ? xs[x].ax[1].flags : xs[x].ax[2].flags)[tyz] : 0u;
      bool every = false, some = false;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const unsigned long long bx = __ballot((fx >> q) & 1u), byz = __ballot((fyz >> q) & 1u);
        every = every || (bx == mx && byz == myz);
        some = some || (bx && (byz & 0xfull) && (byz & 0xf0ull));
      }
      if (every) {
        src = x;
        break;
      }
      if ((mixed = some)) break;
    }
    bool fits = !mixed && src >= 0;
    if (fits) {
      ConstXfer &X = xs[src];
      ConstBox &S = cbox(X.src);
      // wave 0: the x targets; wave 1: y and z
      if (wave < 2) {
        const int ax = wave == 0 ? 0 : (lane < 4 ? 1 : 2);
        const bool v = wave == 0 ? vx : vyz;
        const int t = wave == 0 ? i : tyz;
        const unsigned fl = wave == 0 ? fx : fyz;
        const int slot = wave == 0 ? lane : TX + (lane < 4 ? lane : TY + (lane - 4));
        int c = 1 << 28, cc = -1;
        if (v) {
          double a, b;
          if (X.affine) {
            const int q = t + (ax == 0 ? X.aff[0] : (ax == 1 ? X.aff[1] : X.aff[2]));
            const int sn = ax == 0 ? S.n[0] : (ax == 1 ? S.n[1] : S.n[2]);
            const bool mid = (q & 1) != 0;
            c = q >> 1;
            a = mid ? 0.5 : 1.0;
            b = mid ? 0.5 : 0.0;
            if (!mid && c + 1 >= sn) c = sn - 2, a = 0.0, b = 1.0;
          } else {
            c = (ax == 0 ? X.ax[0].start : (ax == 1 ? X.ax[1].start : X.ax[2].start))[t];
            const double *w = (ax == 0 ? X.ax[0].w : (ax == 1 ? X.ax[1].w : X.ax[2].w)) + 2 * t;
            a = w[0];
            b = w[1];
          }
          if (fl & 4u) cc = (ax == 0 ? X.ax[0].coinc : (ax == 1 ? X.ax[1].coinc : X.ax[2].coinc))[t];
          wi[slot] = a;
          wf[slot] = b;
        }
        // the axis' extent: x over the wave, y and z over lanes 0-3, 4-7
        int l = v ? (cc >= 0 ? min(c, cc) : c) : 1 << 28, h = v ? max(c + 1, cc) : -1;
        const int width = wave == 0 ? 64 : 4;
        for (int d = 1; d < width; d <<= 1) {
          l = min(l, __shfl_xor(l, d));
          h = max(h, __shfl_xor(h, d));
        }
        if (v) {
          first[slot] = c - l;
          same[slot] = cc >= 0 ? cc - l : -1;
        }
        if (wave == 0 ? lane == 0 : (lane == 0 || lane == 4)) {
          lo[ax] = l;
          ext[ax] = h - l + 1;
        }
      }
    }
    __syncthreads();
    fits = fits && ext[0] <= VX && ext[1] <= VY && ext[2] <= VZ;
    if (fits) {
      ConstBox &S = cbox(xs[src].src);
      const void *vf = S.f[F_V];
      const int ex = ext[0], ey = ext[1], ez = ext[2];
      // rows of the node block, one a half wave: ex <= 36 nodes
      for (int r = int(threadIdx.x >> 5); r < ey * ez; r += kPtThreads / 32) {
        const int z = r / ey, y = r - z * ey;
        for (int x = int(threadIdx.x & 31u); x < ex; x += 32)
          V[(z * VY + y) * VX + x] = ld<double>(vf, boff(S, lo[0] + x, lo[1] + y, lo[2] + z));
      }
      __syncthreads();
      for (int r = wave; r < ey * ez; r += kPtThreads / 64) {
        const int z = r / ey, y = r - z * ey;
        if (vx) {
          const double *p = V + (z * VY + y) * VX + first[lane];
          A[(z * VY + y) * TX + lane] = p[0] * wi[lane] + p[1] * wf[lane];
        }
      }
      __syncthreads();
      if (mine) {
        const int sy = TX + wave, y0 = first[sy];
        const double dyi = wi[sy], dyf = wf[sy];
#pragma unroll
        for (int q = 0; q < TZ; ++q) {
          if (q >= nz) break;
          const int sz = TX + TY + q, z0 = first[sz];
          double v;
          if (same[lane] >= 0 && same[sy] >= 0 && same[sz] >= 0) {
            v = V[(same[sz] * VY + same[sy]) * VX + same[lane]];
          } else {
            const double *p = A + (z0 * VY + y0) * TX + lane;
            v = (p[0] * dyi + p[TX] * dyf) * wi[sz] + (p[VY * TX] * dyi + p[(VY + 1) * TX] * dyf) * wf[sz];
          }
          st<double>(T.f[F_U], o[q], u0[q] + v);
        }
      }
    } else if (mine && (mixed || src >= 0)) {
      for (int q = 0; q < nz; ++q) {
        const int t[3] = {i, j, k0 + q};
        for (int x = Bk.nsrc - 1; x >= 0; --x) {
          ConstXfer &X = xs[x];
          unsigned fl[3];
          const unsigned f = axis_flags(X, t, fl);
          if (!(f & 3)) continue;  // all = true
          ConstBox &S = cbox(X.src);
          double v;
          if (f & 4)
            v = ld<double>(S.f[F_V], boff(S, X.ax[0].coinc[t[0]], X.ax[1].coinc[t[1]], X.ax[2].coinc[t[2]]));
          else
            v = X.affine ? trilinear_nested(S, X, t) : trilinear_corr(S, X, t);
          const unsigned ot = boff(T, t[0], t[1], t[2]);
          st<double>(T.f[F_U], ot, ld<double>(T.f[F_U], ot) + v);
          break;
        }
      }
    }
    __syncthreads();  // the LDS is reused by the next tile
  }
}

// shell point q of a box: the R-thick z slabs first, then y slabs, then x slabs
__device__ __forceinline__ void shell_point(ConstBox &B, unsigned q, int &i, int &j, int &k) {
  const unsigned R = unsigned(B.R);
  const unsigned n0 = unsigned(B.n[0]), n1 = unsigned(B.n[1]), n2 = unsigned(B.n[2]);
  const unsigned zs = n0 * n1 * R;  // one z slab
  if (q < 2 * zs) {
    const unsigned s = q >= zs, r = q - s * zs;
    const unsigned plane = n0 * n1;
    const unsigned l = fast_div(r, plane, B.in01), rr = r - l * plane;
    j = int(fast_div(rr, n0, B.in0));
    i = int(rr - unsigned(j) * n0);
    k = s ? int(n2 - R + l) : int(l);
    return;
  }
  q -= 2 * zs;
  const unsigned ys = n0 * R * (n2 - 2 * R);
  if (q < 2 * ys) {
    const unsigned s = q >= ys, r = q - s * ys;
    const unsigned row = fast_div(r, n0, B.in0);
    i = int(r - row * n0);
    const unsigned kk = row / R, l = row - kk * R;
    k = int(R + kk);
    j = s ? int(n1 - R + l) : int(l);
    return;
  }
  q -= 2 * ys;
  const unsigned xs = R * (n1 - 2 * R) * (n2 - 2 * R);
  const unsigned s = q >= xs, r = q - s * xs;
  const unsigned col = r / R, l = r - col * R;
  const unsigned kk = fast_div(col, n1 - 2 * R, B.inyi);
  j = int(R + (col - kk * (n1 - 2 * R)));
  k = int(R + kk);
  i = s ? int(n0 - R + l) : int(l);
}

// column slot q of the ghost shell (ghost_column_slots): the R shell
// points that differ along the slab normal `axis` only (z slabs: columns
// (i, j); y slabs: (i, k) with k interior; x slabs: (j, k) with j, k
// interior; low side first, each face in tiles of kColTile^2 columns);
// returns the column's first point, or false for a padding slot
__device__ __forceinline__ bool face_tile_pos(unsigned r, unsigned f0, unsigned f1, unsigned &a0,
                                              unsigned &a1) {
  const unsigned tx = col_tiles(f0);
  const unsigned st = r / unsigned(kColSuper * kColSuper), w = r % unsigned(kColSuper * kColSuper);
  const unsigned sy = fast_div(st, tx, 1.0f / float(tx));
  const unsigned wave = w / unsigned(kColTile * kColTile), lane = w % unsigned(kColTile * kColTile);
  a0 = (st - sy * tx) * kColSuper + (wave & 1u) * kColTile + lane % kColTile;
  a1 = sy * kColSuper + (wave >> 1) * kColTile + lane / kColTile;
  return a0 < f0 && a1 < f1;
}
__device__ __forceinline__ bool shell_column(ConstBox &B, unsigned q, int &i, int &j, int &k,
                                             int &axis) {
  const unsigned R = unsigned(B.R);
  const unsigned n0 = unsigned(B.n[0]), n1 = unsigned(B.n[1]), n2 = unsigned(B.n[2]);
  unsigned a0, a1;
  const unsigned zc = face_slots(n0, n1);
  if (q < 2 * zc) {
    const unsigned s = q >= zc;
    if (!face_tile_pos(q - s * zc, n0, n1, a0, a1)) return false;
    i = int(a0);
    j = int(a1);
    k = s ? int(n2 - R) : 0;
    axis = 2;
    return true;
  }
  q -= 2 * zc;
  const unsigned yc = face_slots(n0, n2 - 2 * R);
  if (q < 2 * yc) {
    const unsigned s = q >= yc;
    if (!face_tile_pos(q - s * yc, n0, n2 - 2 * R, a0, a1)) return false;
    i = int(a0);
    k = int(R + a1);
    j = s ? int(n1 - R) : 0;
    axis = 1;
    return true;
  }
  q -= 2 * yc;
  const unsigned xc = face_slots(n1 - 2 * R, n2 - 2 * R);
  const unsigned s = q >= xc;
  if (!face_tile_pos(q - s * xc, n1 - 2 * R, n2 - 2 * R, a0, a1)) return false;
  j = int(R + a0);
  k = int(R + a1);
  i = s ? int(n0 - R) : 0;
  axis = 0;
  return true;
}

// the targets of the kColSuper^2 column slots from slot q (a multiple of
// them): first point and extent of the tile, R points along the normal
__device__ __forceinline__ void shell_tile(ConstBox &B, unsigned q, int t0[3], int nt[3]) {
  constexpr unsigned kSlots = kColSuper * kColSuper;
  const unsigned R = unsigned(B.R);
  const unsigned n0 = unsigned(B.n[0]), n1 = unsigned(B.n[1]), n2 = unsigned(B.n[2]);
  const unsigned zc = face_slots(n0, n1), yc = face_slots(n0, n2 - 2 * R);
  int axis;
  unsigned f0, f1, side;  // the face's extents, its side
  if (q < 2 * zc) {
    axis = 2; f0 = n0; f1 = n1; side = q >= zc; q -= side * zc;
  } else if ((q -= 2 * zc) < 2 * yc) {
    axis = 1; f0 = n0; f1 = n2 - 2 * R; side = q >= yc; q -= side * yc;
  } else {
    q -= 2 * yc;
    axis = 0; f0 = n1 - 2 * R; f1 = n2 - 2 * R;
    const unsigned xc = face_slots(f0, f1);
    side = q >= xc; q -= side * xc;
  }
  const unsigned tx = col_tiles(f0), tile = q / kSlots;
  const unsigned ty = tile / tx;
  const unsigned a0 = (tile - ty * tx) * kColSuper, a1 = ty * kColSuper;
  const int e0 = int(min(unsigned(kColSuper), f0 - a0)), e1 = int(min(unsigned(kColSuper), f1 - a1));
  const int nn = axis == 0 ? int(n0) : (axis == 1 ? int(n1) : int(n2));
  const int edge = side ? nn - int(R) : 0, r = int(R);
  // z faces (x, y), y faces (x, z), x faces (y, z); interior along the axes
  // whose faces come before
  t0[0] = axis == 0 ? edge : int(a0);
  t0[1] = axis == 1 ? edge : (axis == 2 ? int(a1) : r + int(a0));
  t0[2] = axis == 2 ? edge : r + int(a1);
  nt[0] = axis == 0 ? r : e0;
  nt[1] = axis == 1 ? r : (axis == 2 ? e1 : e0);
  nt[2] = axis == 2 ? r : e1;
}

// ghost shell of refinement boxes from the coarser level (Lagrange
// order+1, KP = order+2 nodes per axis); one thread per shell point,
// point q being layer q mod R of column slot q / R (shell_column), so that
// a wave's points cover a compact patch of a face
template <int KP>
__global__ __launch_bounds__(kPtThreads) void k_ghost_fill(const PtBlock *__restrict__ blocks) {
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &T = cbox(Bk.box);
  const unsigned R = unsigned(T.R);
  for_points(Bk, [&](unsigned off) {
    const unsigned q = Bk.q0 + off, c = q / R;
    int i0, j0, k0, ax;
    if (!shell_column(T, c, i0, j0, k0, ax)) return;
    const int l = int(q - c * R);
    const int i = i0 + (ax == 0 ? l : 0), j = j0 + (ax == 1 ? l : 0), k = k0 + (ax == 2 ? l : 0);
    const int t[3] = {i, j, k};
    ConstXfer *xs = (ConstXfer *)Bk.src;
    for (int x = Bk.nsrc - 1; x >= 0; --x) {
      ConstXfer &X = xs[x];
      unsigned fl[3];
      const unsigned f = axis_flags(X, t, fl);
      if (!(f & 3)) continue;
      ConstBox &S = cbox(X.src);
      st<double>(T.f[F_U], boff(T, i, j, k), tinterp<KP>(S, S.f[F_U], X, t, fl));
      return;
    }
  });
}

// Ghost shell of refinement boxes by tiles: a workgroup takes kColSuper^2
// columns of one face side (one block of slots, shell_column), R points
// each, and interpolates them as one tensor product (tile_transfer).  Point by
// point (or column by column) every target summed its own (order + 2)^3
// nodes.  Measured, per launch: N=129 8th order 400 -> 32 us, N=161 6th
// order 322 -> 48, 16 x N=65 4th order 146 -> 36.
template <int KP>
__global__ __launch_bounds__(kPtThreads) void k_ghost_tiles(const PtBlock *__restrict__ blocks) {
  __shared__ TileLds<KP> L;
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &T = cbox(Bk.box);
  constexpr unsigned kSlots = kColSuper * kColSuper;
  for (unsigned base = 0; base < Bk.nq; base += kSlots) {
    int t0[3], nt[3];
    shell_tile(T, Bk.q0 + base, t0, nt);
    tile_transfer<KP>(L, Bk, T, t0, nt, 3u, F_U, F_U, false, [&](int, int, int) { return true; });
    __syncthreads();  // L is reused by the next tile
  }
}

// r = u on the ghost shell of the listed boxes (the fused sweeps read
// ghost values from either field)
__global__ __launch_bounds__(kPtThreads) void k_copy_shell(const PtBlock *__restrict__ blocks) {
  const PtBlock Bk = blocks[xcd_block()];
  ConstBox &B = cbox(Bk.box);
  for_points(Bk, [&](unsigned off) {
    int i, j, k;
    shell_point(B, Bk.q0 + off, i, j, k);
    const unsigned o = boff(B, i, j, k);
    st<double>(B.f[F_R], o, ld<double>(B.f[F_U], o));
  });
}

// ------------------------------------------------------------------
// coarsest level: {Robin, one multi-colour sweep} until the sweep norm is
// <= eps or stops changing (elliptic.cc:1782-1816); one block per
// hierarchy, u and rho in LDS (the box's colour-block layout) for the whole loop, b,
// c (d, e) of the owned interior points in registers.  Interior updates are
// over-relaxed by omega (omega = 1 is the reference's Gauss-Seidel-Newton);
// the loop's fixed point, the coarse solution, does not depend on omega.
// The coarsest level always has order 2 (R = 1): its Robin shell is one
// layer of faces, then edges, then corners (boundary.cc:447-1101), each
// phase reading only the previous ones; every thread decodes its shell
// points once.
// ------------------------------------------------------------------
struct CoarseGeo {
  int n[3];
  int rl, rs, ps, cs, nc;
  unsigned ncm;
  double lo[3], d[3], idx[3], idx2[3];
  double ipn, dulap;
};

// element index of (i, j, k) in the LDS copy (the box's colour-block layout)
__device__ __forceinline__ int coarse_p(const CoarseGeo &G, int i, int j, int k) {
  const unsigned s = unsigned(i + j + k);
  const int c = int(s - ((s * G.ncm) >> 16) * unsigned(G.nc));
  return c * G.cs + k * G.ps + j * G.rs + int((unsigned(i) * G.ncm) >> 16);
}

// The Robin updates of the shell (one-sided derivative dx2, diff_2nd.cc:237-335).
// The coarsest level is 2nd order, so its layout has two colours: point
// (i, j, k) is slot i / 2 of row (j, k) in block (i + j + k) & 1, and a step
// along an axis moves to the other block.

// face point t of the coarsest box (x faces, then y, then z, low side
// first): (i, j, k) and its side, 2 axis + high
__device__ __forceinline__ int coarse_face(const CoarseGeo &G, int t, float ini, float inj, int &i,
                                           int &j, int &k) {
  const int ni = G.n[0] - 2, nj = G.n[1] - 2, nk = G.n[2] - 2;
  const int fx = nj * nk, fy = ni * nk, fz = ni * nj;
  if (t < 2 * fx) {
    const int hi = t >= fx;
    t -= hi * fx;
    const int q = int(fast_div(unsigned(t), unsigned(nj), inj));
    i = hi ? G.n[0] - 1 : 0; j = 1 + t - q * nj; k = 1 + q;
    return hi;
  }
  if ((t -= 2 * fx) < 2 * fy) {
    const int hi = t >= fy;
    t -= hi * fy;
    const int q = int(fast_div(unsigned(t), unsigned(ni), ini));
    j = hi ? G.n[1] - 1 : 0; i = 1 + t - q * ni; k = 1 + q;
    return 2 + hi;
  }
  t -= 2 * fy;
  const int hi = t >= fz;
  t -= hi * fz;
  const int q = int(fast_div(unsigned(t), unsigned(ni), ini));
  k = hi ? G.n[2] - 1 : 0; i = 1 + t - q * ni; j = 1 + q;
  return 4 + hi;
}

// a / b from y = 1 / b (rounded): the quotient corrected twice by its exact
// remainder.  a y may be two units off, one correction brings it within one,
// and from there the second rounds as the division does (Markstein 1990);
// zeros, infinities and NaN as the division has them
__device__ __forceinline__ double div_by(double a, double b, double y) {
  double q = a * y;
  q = fma(fma(-q, b, a), y, q);
  return __builtin_amdgcn_div_fixup(fma(fma(-q, b, a), y, q), b, a);
}
// a / b by two Newton steps on the hardware reciprocal and one correction;
// zeros, infinities and NaN as the division has them.  The coarsest solve's
// quotients are far from the exponents' limits, so the scaling steps of the
// general division (2 of its 11) are left out; the rest are its own, to the
// bit.
__device__ __forceinline__ double div_newton(double a, double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = fma(fma(-b, y, 1.0), y, y);
  y = fma(fma(-b, y, 1.0), y, y);
  const double q = a * y;
  return __builtin_amdgcn_div_fixup(fma(fma(-q, b, a), y, q), b, a);
}

// edge t of the coarsest box (XY, XZ, YZ edges) or, with CORNER, corner t:
// (i, j, k) and its sides in the order of their axes
template <bool CORNER>
__device__ __forceinline__ void coarse_edge(const CoarseGeo &G, int t, int ijk[3], int sd[3]) {
  const int ni = G.n[0] - 2, nj = G.n[1] - 2, nk = G.n[2] - 2;
  if (CORNER) {
    sd[0] = (t >> 1) & 1;
    sd[1] = 2 + (t >> 2);
    sd[2] = 4 + (t & 1);
  } else if (t < 4 * nk) {
    const int e = (t >= nk) + (t >= 2 * nk) + (t >= 3 * nk);
    sd[0] = e >> 1;
    sd[1] = 2 + (e & 1);
    ijk[2] = 1 + t - e * nk;
  } else if ((t -= 4 * nk) < 4 * nj) {
    const int e = (t >= nj) + (t >= 2 * nj) + (t >= 3 * nj);
    sd[0] = e >> 1;
    sd[1] = 4 + (e & 1);
    ijk[1] = 1 + t - e * nj;
  } else {
    t -= 4 * nj;
    const int e = (t >= ni) + (t >= 2 * ni) + (t >= 3 * ni);
    sd[0] = 2 + (e & 1);
    sd[1] = 4 + (e >> 1);
    ijk[0] = 1 + t - e * ni;
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int m = 0; m < (CORNER ? 3 : 2); ++m)
      if ((sd[m] >> 1) == a) ijk[a] = (sd[m] & 1) ? G.n[a] - 1 : 0;
}

// r^2 / n at (i, j, k)
__device__ __forceinline__ double coarse_r2n(const CoarseGeo &G, int i, int j, int k) {
  const double X0 = G.lo[0] + (double)i * G.d[0], X1 = G.lo[1] + (double)j * G.d[1],
               X2 = G.lo[2] + (double)k * G.d[2];
  return (X0 * X0 + X1 * X1 + X2 * X2) * G.ipn;
}

// index of the point one step inwards from (i, j, k) at side sd
__device__ __forceinline__ int coarse_in(const CoarseGeo &G, int i, int j, int k, int sd) {
  const int dir = (sd & 1) ? -1 : 1, ax = sd >> 1;
  return coarse_p(G, i + (ax == 0 ? dir : 0), j + (ax == 1 ? dir : 0), k + (ax == 2 ? dir : 0));
}

// One side's derivative at the point at index p (p1: one step inwards) over
// X.  Two steps inwards lie in p's own colour block: one slot, two rows or
// two planes on.
__device__ __forceinline__ double coarse_side(const CoarseGeo &G, const double (*side)[4],
                                              const double *su, double u0, int p, int p1, int sd) {
  const int st = sd < 2 ? 1 : 2 * (sd < 4 ? G.rs : G.ps);
  const int p2 = p + ((sd & 1) ? -st : st);
  const double dv = (-3.0 * u0 + 4.0 * su[p1] - su[p2]) * 0.5 * side[sd][2];
  const double q = div_by(dv, side[sd][0], side[sd][1]);
  __builtin_amdgcn_sched_barrier(0);  // one side at a time: fewer registers
  return q;
}

// One workgroup and its CU carry a box's whole loop, so the kernel is bound
// by the double-precision instructions it issues per sweep, not by memory.
// - Each thread keeps what does not change of its face points: the indices,
//   r^2 / n, dF and 1 / dF (a division becomes a product, four fma and the
//   fix-up, and rounds the same).
// - An interior point reads the shell's faces only, never its edges and
//   corners.  The edges are updated beside the first colour pass and the
//   corners beside the second, without barriers of their own, by the last
//   waves, which have an interior point less.  An edge's constants take the
//   place of the last waves' missing face point, the corners' lie in LDS.
// FACES: face points a thread keeps.  The threads hold all face and edge
// points (FACES * NT): loops for points beyond them, though never entered,
// took registers and scalar registers enough to make the kernel spill.
// OWN: interior points per colour per thread (colour c's points are
// numbered row by row, ceil(ni / 2) slots per interior row).  The
// coefficients of a thread's points stay in registers for the whole loop
// where they fit the register file; otherwise each point's are loaded from
// the (cache-resident) fields as the point is updated.
template <int EQ, int OWN, int NT, int FACES>
__global__ __launch_bounds__(NT) void k_coarse_solve(const CoarseItem *__restrict__ items,
                                                                 double eps, int max_iter) {
  extern __shared__ double lds[];
  __shared__ double sh[NT / 64];
  const CoarseItem It = items[blockIdx.x];
  ConstBox &B = cbox(It.box);
  CoarseGeo G;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    G.n[a] = B.n[a];
    G.lo[a] = B.lo[a];
    G.d[a] = B.d[a];
    G.idx[a] = B.idx[a];
    G.idx2[a] = B.idx2[a];
  }
  G.rl = B.rl;
  G.rs = B.rs;
  G.ps = int(B.ps);
  G.cs = int(B.cs);
  G.nc = B.nc;
  G.ncm = B.ncm;
  G.ipn = B.ipn;
  G.dulap = B.dulap;
  const double omega = It.omega;
  const int n0 = G.n[0], n1 = G.n[1], n2 = G.n[2];
  const int np = int(B.size);
  double *su = lds;
  double *srho = lds + np;
  double *ug = B.f[F_U];
  const double *rg = B.f[F_RHO];
  for (int q = threadIdx.x; q < np; q += NT) {
    su[q] = ld<double>(ug, unsigned(q) * 8u);
    srho[q] = ld<double>(rg, unsigned(q) * 8u);
  }
  // owned interior points, colour by colour
  const int ni = n0 - 2, nj = n1 - 2, nk = n2 - 2;
  const int per_row = (ni + 1) / 2;
  const int slots = nj * nk * per_row;
  constexpr bool kLong = EQ == 1 || EQ == kEqPuncturesEm;  // more coefficients a point
  constexpr bool kCached = OWN * NT <= 2048 || EQ == 0;
  constexpr int NCACHE = kCached ? 2 * OWN : 1;
  constexpr bool kKeepAddr = OWN * NT <= 2048 && !kLong;
  int own_p[2 * OWN];
  double own_b[NCACHE], own_cc[NCACHE], own_d[NCACHE], own_e[NCACHE];
  // the coefficients of owned point q (colour col, slot m)
  auto coeffs = [&](int q, double &b, double &cc, double &d, double &e) {
    const unsigned o = unsigned(own_p[q] & 0x3fffffff) * 8u;
    b = ld<double>(B.f[F_B], o);
    cc = ld<double>(B.f[F_C], o);
    d = e = 0.0;
    if (EQ == 1 || EQ == kEqPuncturesEm) {
      d = ld<double>(B.f[F_D], o);
      e = ld<double>(B.f[F_E], o);
    }
  };
#pragma unroll
  for (int col = 0; col < 2; ++col)
#pragma unroll
    for (int m = 0; m < OWN; ++m) {
      const int q = col * OWN + m;
      const int t = threadIdx.x + m * NT;
      own_p[q] = -1;
      if constexpr (kCached) own_b[q] = own_cc[q] = own_d[q] = own_e[q] = 0.0;
      if (t >= slots) continue;
      const int row = t / per_row, tt = t - row * per_row;
      const int j = 1 + row % nj, k = 1 + row / nj;
      const int i = 1 + ((col - j - k - 1) & 1) + 2 * tt;
      if (i >= n0 - 1) continue;
      own_p[q] = coarse_p(G, i, j, k) | ((i & 1) << 30);
      if constexpr (kCached) coeffs(q, own_b[q], own_cc[q], own_d[q], own_e[q]);
    }
  // shell points: faces (x, y, z pairs), edges (XY, XZ, YZ), corners
  const int nface = 2 * (nj * nk + ni * nk + ni * nj), nedge = 4 * (ni + nj + nk);
  const float ini = 1.0f / float(ni), inj = 1.0f / float(nj);
  // per side (2 axis + high): coordinate X, 1 / X, 1 / d signed inwards and
  // the side's term of dF
  __shared__ double side[6][4];
  if (threadIdx.x < 6) {
    const int ax = threadIdx.x >> 1, hi = threadIdx.x & 1;
    const double X = B.lo[ax] + double(hi ? B.n[ax] - 1 : 0) * B.d[ax];
    side[threadIdx.x][0] = X;
    side[threadIdx.x][1] = 1.0 / X;
    side[threadIdx.x][2] = hi ? -B.idx[ax] : B.idx[ax];
    side[threadIdx.x][3] = -3.0 * 0.5 * side[threadIdx.x][2] / X;
  }
  __syncthreads();
  // owned face points: index | side << 16 (-1: none), indices of the two
  // points inwards, r^2 / n, dF and its reciprocal
  int face_p[FACES];
  unsigned face_in[FACES];
  double face_a[FACES], face_df[FACES], face_y[FACES];
#pragma unroll
  for (int m = 0; m < FACES; ++m) {
    face_p[m] = -1;
    face_in[m] = 0;
    face_a[m] = face_df[m] = face_y[m] = 1.0;
    const int t = threadIdx.x + m * NT;
    if (t >= nface) continue;
    int i, j, k;
    const int sd = coarse_face(G, t, ini, inj, i, j, k);
    const int dir = (sd & 1) ? -1 : 1, ax = sd >> 1;
    face_p[m] = coarse_p(G, i, j, k) | (sd << 16);
    const int p2 = coarse_p(G, i + (ax == 0 ? 2 * dir : 0), j + (ax == 1 ? 2 * dir : 0),
                            k + (ax == 2 ? 2 * dir : 0));
    face_in[m] = unsigned(coarse_in(G, i, j, k, sd)) | (unsigned(p2) << 16);
    face_a[m] = coarse_r2n(G, i, j, k);
    face_df[m] = face_a[m] * side[sd][3] + 1.0;
    face_y[m] = 1.0 / face_df[m];
  }
  // edge points: thread NT - 1 - t keeps edge t as its last face point (the
  // host sees to it that no thread that takes an edge has one there); corner
  // points: one of eight threads each
  const int et = NT - 1 - int(threadIdx.x);
  const bool edge = et < nedge;
  if (edge) {
    int ijk[3], sd[3];
    coarse_edge<false>(G, et, ijk, sd);
    face_p[FACES - 1] = coarse_p(G, ijk[0], ijk[1], ijk[2]) | (sd[0] << 16) | (sd[1] << 20);
    face_in[FACES - 1] = unsigned(coarse_in(G, ijk[0], ijk[1], ijk[2], sd[0])) |
                         unsigned(coarse_in(G, ijk[0], ijk[1], ijk[2], sd[1])) << 16;
    face_a[FACES - 1] = coarse_r2n(G, ijk[0], ijk[1], ijk[2]);
    face_df[FACES - 1] = face_a[FACES - 1] * (side[sd[0]][3] + side[sd[1]][3]) + 1.0;
    face_y[FACES - 1] = 1.0 / face_df[FACES - 1];
  }
  __shared__ double corner[8][3];  // r^2 / n, dF, 1 / dF
  __shared__ int corner_p[8][7];   // index, one step inwards per axis, sides
  if (et < 8) {
    int ijk[3], sd[3];
    coarse_edge<true>(G, et, ijk, sd);
    corner_p[et][0] = coarse_p(G, ijk[0], ijk[1], ijk[2]);
    for (int a = 0; a < 3; ++a) {
      corner_p[et][1 + a] = coarse_in(G, ijk[0], ijk[1], ijk[2], sd[a]);
      corner_p[et][4 + a] = sd[a];
    }
    corner[et][0] = coarse_r2n(G, ijk[0], ijk[1], ijk[2]);
    corner[et][1] = corner[et][0] * (side[sd[0]][3] + side[sd[1]][3] + side[sd[2]][3]) + 1.0;
    corner[et][2] = 1.0 / corner[et][1];
  }
  double prev = 1.0, cur = 1.0;
  int it = 0;
  do {
    prev = cur;
#pragma unroll
    for (int m = 0; m < FACES; ++m) {
      if (face_p[m] < 0 || (m == FACES - 1 && edge)) continue;
      const int p = face_p[m] & 0xffff, sd = face_p[m] >> 16;
      const double u0 = su[p];
      const double dv = (-3.0 * u0 + 4.0 * su[face_in[m] & 0xffffu] - su[face_in[m] >> 16]) * 0.5 * side[sd][2];
      const double op = face_a[m] * div_by(dv, side[sd][0], side[sd][1]) + u0;
      su[p] = u0 - div_by(op - srho[p], face_df[m], face_y[m]);
    }
    __syncthreads();
    double mx = 0.0;
#pragma unroll
    for (int col = 0; col < 2; ++col) {
#pragma unroll
      for (int m = 0; m < OWN; ++m) {
        const int q = col * OWN + m;
        if (own_p[q] < 0) continue;
        // uncached: the point's coefficients loaded here (cache-resident)
        double qb, qc, qd, qe;
        if constexpr (kCached) {
          qb = own_b[q];
          qc = own_cc[q];
          qd = own_d[q];
          qe = own_e[q];
        } else {
          coeffs(q, qb, qc, qd, qe);
        }
        // the neighbours' addresses stay in registers over the loop where
        // there are enough (formed each sweep, 17^3 takes 3.4 us a sweep
        // instead of 3.1; spilled, 21^3 with the scalar field takes 8.6
        // instead of 7.2)
        int po = own_p[q];
        if constexpr (!kKeepAddr) asm volatile("" : "+v"(po));
        const int p = po & 0x3fffffff;
        const Nbr<2> nb = stencil_offs<2, 1>(col, po >> 30, unsigned(G.cs), unsigned(G.rs), unsigned(G.ps));
        const double u0 = su[p], xp = su[p + int(nb.xp[0])], xm = su[p + int(nb.xm[0])],
                     yp = su[p + int(nb.yp[0])], ym = su[p + int(nb.ym[0])],
                     zp = su[p + int(nb.zp[0])], zm = su[p + int(nb.zm[0])], rho = srho[p];
        const double lu = star_sum<2, double>(fma(-2.0, u0, xp + xm), fma(-2.0, u0, yp + ym),
                                              fma(-2.0, u0, zp + zm), G.idx2[0], G.idx2[1], G.idx2[2]);
        double N, dN;
        if constexpr (EQ == kEqPuncturesEm) {
          const unsigned o = unsigned(p) * 8u;
          const double g[3] = {(xp - xm) * 0.5 * G.idx[0], (yp - ym) * 0.5 * G.idx[1],
                               (zp - zm) * 0.5 * G.idx[2]};
          const double ge[3] = {ld<double>(B.f[F_X0], o), ld<double>(B.f[F_X1], o), ld<double>(B.f[F_X2], o)};
          const double gf[3] = {ld<double>(B.f[F_X3], o), ld<double>(B.f[F_X4], o), ld<double>(B.f[F_X5], o)};
          const double du[3] = {0.0, 0.0, 0.0};  // order 2: centred derivatives
          em_nonlinear(lu, G.dulap, u0, g, du, qb, qd, ge, gf, N, dN);
        } else {
          nonlinear<EQ, true>(lu, G.dulap, qb, qc + u0, qd, qe, N, dN);
        }
        const double res = N - rho;
        const double un = u0 - omega * div_newton(res, dN);
        su[p] = un;
        mx = fmax(mx, fabs(res));
        if (!(un == un)) mx = __longlong_as_double(0x7ff0000000000000LL);
        // keep each point's live range local (the unrolled bodies would
        // otherwise be interleaved past the register budget)
        __builtin_amdgcn_sched_barrier(0);
      }
      if (col == 0) {
        if (edge) {
          constexpr int m = FACES - 1;
          int fp = face_p[m];
          asm volatile("" : "+v"(fp));
          const int p = fp & 0xffff;
          const double u0 = su[p];
          const double sF =
              coarse_side(G, side, su, u0, p, int(face_in[m] & 0xffffu), (fp >> 16) & 15) +
              coarse_side(G, side, su, u0, p, int(face_in[m] >> 16), fp >> 20);
          su[p] = u0 - div_by(face_a[m] * sF + u0 - srho[p], face_df[m], face_y[m]);
        }
        __syncthreads();
      } else if (et < 8) {
        int tc = NT - 1 - int(threadIdx.x);
        asm volatile("" : "+v"(tc));
        const int *c = corner_p[tc];
        const int p = c[0];
        const double u0 = su[p];
        double sF = coarse_side(G, side, su, u0, p, c[1], c[4]);
        sF += coarse_side(G, side, su, u0, p, c[2], c[5]);
        sF += coarse_side(G, side, su, u0, p, c[3], c[6]);
        su[p] = u0 - div_by(corner[tc][0] * sF + u0 - srho[p], corner[tc][1], corner[tc][2]);
      }
    }
    const double wm = wave_max_pos(mx);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = wm;
    __syncthreads();
    cur = row_max_pos<NT / 64>(sh[threadIdx.x & (NT / 64 - 1)]);
    ++it;
  } while (cur > eps && prev != cur && it < max_iter && !isinf(cur));
  for (int q = threadIdx.x; q < np; q += NT) st<double>(ug, unsigned(q) * 8u, su[q]);
  if (threadIdx.x == 0) {
    *It.norm = (unsigned long long)__double_as_longlong(cur);
    *It.iters = it;
  }
}

// ------------------------------------------------------------------
// setup: coefficients b, c [,d, e]; rho = Robin value on the shell, 0
// inside; u = 0
// ------------------------------------------------------------------
__device__ double punctures_c(const PunctureArgs &pa, double X, double Y, double Z) {
  double cval = 1.0;
  for (int i = 0; i < pa.n; ++i) {
    const double x = X - pa.p[i].x, y = Y - pa.p[i].y, z = Z - pa.p[i].z;
    double r = sqrt(x * x + y * y + z * z);
    if (r < 2 * kEps) r = 2 * kEps;
    cval += 0.5 * pa.p[i].m / r;
  }
  return cval;
}

__device__ double punctures_b(const PunctureArgs &pa, double X, double Y, double Z) {
  double A00 = 0, A11 = 0, A22 = 0, A01 = 0, A02 = 0, A12 = 0;
  for (int i = 0; i < pa.n; ++i) {
    const Puncture &q = pa.p[i];
    const double x = X - q.x, y = Y - q.y, z = Z - q.z;
    const double x2 = x * x, y2 = y * y, z2 = z * z;
    double r2 = x2 + y2 + z2;
    if (r2 < 2 * kEps) r2 = 2 * kEps;
    const double r = sqrt(r2);
    const double f = 1.5 / (r2 * r2 * r);
    A00 += f * (q.px * x * (x2 + r2) + q.py * y * (x2 - r2) + q.pz * z * (x2 - r2) +
                4.0 * x * (q.sy * z - q.sz * y));
    A11 += f * (q.px * x * (y2 - r2) + q.py * y * (y2 + r2) + q.pz * z * (y2 - r2) +
                4.0 * y * (q.sz * x - q.sx * z));
    A22 += f * (q.px * x * (z2 - r2) + q.py * y * (z2 - r2) + q.pz * z * (z2 + r2) +
                4.0 * z * (q.sx * y - q.sy * x));
    A01 += f * (q.px * y * (r2 + x2) + q.py * x * (r2 + y2) + q.pz * x * y * z -
                2.0 * q.sx * x * z + 2.0 * q.sy * y * z + 2.0 * q.sz * (x2 - y2));
    A02 += f * (q.px * z * (r2 + x2) + q.py * x * y * z + q.pz * x * (r2 + z2) +
                2.0 * q.sx * x * y + 2.0 * q.sy * (z2 - x2) - 2.0 * q.sz * y * z);
    A12 += f * (q.px * x * y * z + q.py * z * (r2 + y2) + q.pz * y * (r2 + z2) +
                2.0 * q.sx * (y2 - z2) - 2.0 * q.sy * x * y + 2.0 * q.sz * x * z);
  }
  return 0.125 * (A00 * A00 + A11 * A11 + A22 * A22 + 2.0 * (A01 * A01 + A02 * A02 + A12 * A12));
}

__device__ double sf_phi(const PunctureArgs &pa, double r) {
  switch (pa.ps_case) {
    case 1: return pa.ps_phi0 * tanh((r - pa.ps_r0) * pa.ps_isigma);
    case 2: return pa.ps_phi0 * exp(-(r - pa.ps_r0) * (r - pa.ps_r0) * pa.ps_isigma);
    case 3: {
      const double x = r, l2 = 0.6;
      return (0.0481646 * exp(-0.0581545 * (x - 1.8039e-08) * (x - 1.8039e-08) / l2) +
              0.298408 * exp(-0.111412 * (x + 9.6741e-09) * (x + 9.6741e-09) / l2) +
              0.42755 * exp(-0.207156 * (x - 1.09822e-08) * (x - 1.09822e-08) / l2) +
              0.204229 * exp(-0.37742 * (x + 2.13778e-08) * (x + 2.13778e-08) / l2) +
              0.021649 * exp(-0.68406 * (x - 8.78608e-08) * (x - 8.78608e-08) / l2)) * l2;
    }
    default:
      return pa.ps_phi0 * 0.5 * (tanh((r + pa.ps_r0) * pa.ps_isigma) - tanh((r - pa.ps_r0) * pa.ps_isigma));
  }
}

__device__ double sf_d(const PunctureArgs &pa, double r) {
  switch (pa.ps_case) {
    case 1: {
      const double ch = cosh((r - pa.ps_r0) * pa.ps_isigma);
      const double ch2 = ch * ch;
      return pa.ps_d1 / (ch2 * ch2);
    }
    case 2:
      return pa.ps_de1 * (r - pa.ps_r0) * (r - pa.ps_r0) *
             exp(-2 * pa.ps_isigma * (r - pa.ps_r0) * (r - pa.ps_r0));
    case 3: {
      const double x = r, l2 = 10000;
      const double g = -2 * (0.0581545 * (x - 1.8039e-08) * 0.0481646 * exp(-0.0581545 * (x - 1.8039e-08) * (x - 1.8039e-08) / l2) +
                             0.111412 * (x + 9.6741e-09) * 0.298408 * exp(-0.111412 * (x + 9.6741e-09) * (x + 9.6741e-09) / l2) +
                             0.207156 * (x - 1.09822e-08) * 0.42755 * exp(-0.207156 * (x - 1.09822e-08) * (x - 1.09822e-08) / l2) +
                             0.37742 * (x + 2.13778e-08) * 0.204229 * exp(-0.37742 * (x + 2.13778e-08) * (x + 2.13778e-08) / l2) +
                             0.68406 * (x - 8.78608e-08) * 0.021649 * exp(-0.68406 * (x - 8.78608e-08) * (x - 8.78608e-08) / l2)) /
                       (l2 * l2);
      return M_PI * g * g;
    }
    default: {
      const double a = 1. / cosh((r + pa.ps_r0) * pa.ps_isigma);
      const double b = 1. / cosh((r - pa.ps_r0) * pa.ps_isigma);
      const double t = a * a - b * b;
      return pa.ps_de1 * 0.25 * t * t;
    }
  }
}

__device__ double sf_e(const PunctureArgs &pa, double r) {
  if (pa.ps_case == 2 || pa.ps_case == 3 || pa.ps_case == 4) {
    const double ff = pa.ps_e2 * sf_phi(pa, r);
    const double g = 1 - exp(ff);
    return pa.ps_e1 * g * g * exp(-2 * ff);
  }
  return 0.0;
}

__global__ __launch_bounds__(256) void k_coefficients(DevBox B, PunctureArgs pa, double robin_a) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long np = (long long)B.n[0] * B.n[1] * B.n[2];
  if (q >= np) return;
  int i, j, k;
  point_ijk(B, q, i, j, k);
  const long long p = pidx(B, i, j, k);
  const double x = coord(B, 0, i), y = coord(B, 1, j), z = coord(B, 2, k);
  const bool inner = interior(B, i, j, k);
  if (pa.eq == 2) {
    // operator.cc:640-662: rho = Gaussian_source, u = Gaussian (elliptic.h)
    const double r2 = x * x + y * y + z * z, a = 0.004;
    B.f[F_B][p] = 0.0;
    B.f[F_C][p] = 0.0;
    B.f[F_RHO][p] = inner ? a * exp(-r2) * (a + exp(0.5 * r2) * (r2 - 3.0)) : robin_a;
    B.f[F_U][p] = a * exp(-0.5 * r2);
    return;
  }
  if (pa.eq == kEqPuncturesEm) {
    // operator.cc:1010-1100 and 3043-3310: eta = sum m / (2r) and phi =
    // sum q / r with their gradients (r and r^3 clamped at 2 eps); rho = 0,
    // u = 1
    double e[4] = {0, 0, 0, 0}, g[4] = {0, 0, 0, 0};
    for (int b = 0; b < pa.n; ++b) {
      const Puncture &P = pa.p[b];
      const double X = x - P.x, Y = y - P.y, Z = z - P.z;
      double r = sqrt(X * X + Y * Y + Z * Z);
      if (r < 2 * kEps) r = 2 * kEps;
      double r3 = pow(X * X + Y * Y + Z * Z, 1.5);
      if (r3 < 2 * kEps) r3 = 2 * kEps;
      e[0] += P.m / r;
      e[1] -= P.m * X / r3;
      e[2] -= P.m * Y / r3;
      e[3] -= P.m * Z / r3;
      g[0] += P.q / r;
      g[1] -= P.q * X / r3;
      g[2] -= P.q * Y / r3;
      g[3] -= P.q * Z / r3;
    }
    B.f[F_B][p] = 0.5 * e[0];
    B.f[F_C][p] = 0.0;
    B.f[F_D][p] = g[0];
    B.f[F_E][p] = 0.0;
    B.f[F_X0][p] = 0.5 * e[1];
    B.f[F_X1][p] = 0.5 * e[2];
    B.f[F_X2][p] = 0.5 * e[3];
    B.f[F_X3][p] = g[1];
    B.f[F_X4][p] = g[2];
    B.f[F_X5][p] = g[3];
    B.f[F_RHO][p] = inner ? 0.0 : robin_a;
    B.f[F_U][p] = 1.0;
    return;
  }
  if (pa.eq == 3) {
    // operator.cc:707-725 and brill (operator.cc:1688-1698): b = Lq, rho = 0, u = 1
    const double amp = 1.9, z2 = z * z, rho2 = x * x + y * y;
    const double qrr = 2.0 * amp * exp(-rho2 - z2) * (1.0 - 5.0 * rho2 + 2.0 * rho2 * rho2);
    const double qzz = 2.0 * amp * exp(-rho2 - z2) * rho2 * (2.0 * z2 - 1.0);
    B.f[F_B][p] = 0.25 * (qrr + qzz);
    B.f[F_C][p] = 0.0;
    B.f[F_RHO][p] = inner ? 0.0 : robin_a;
    B.f[F_U][p] = 1.0;
    return;
  }
  B.f[F_B][p] = punctures_b(pa, x, y, z);
  B.f[F_C][p] = punctures_c(pa, x, y, z);
  if (pa.eq == 1) {
    const double r = sqrt(x * x + y * y + z * z);
    B.f[F_D][p] = sf_d(pa, r);
    B.f[F_E][p] = sf_e(pa, r);
  }
  B.f[F_RHO][p] = inner ? 0.0 : robin_a;
  B.f[F_U][p] = 0.0;
}

// elliptic.cc:1977-2222 ApproximateID: the terms of the punctures up to the
// first with zero mass, added in puncture order
__global__ __launch_bounds__(256) void k_approx_u(DevBox B, PunctureArgs pa) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long np = (long long)B.n[0] * B.n[1] * B.n[2];
  if (q >= np) return;
  int i, j, k;
  point_ijk(B, q, i, j, k);
  const double x = coord(B, 0, i), y = coord(B, 1, j), z = coord(B, 2, k);
  double u = 0.0;
  for (int b = 0; b < pa.n && pa.p[b].m != 0.0; ++b) u += approx_puncture_u(pa.p[b], x, y, z);
  B.f[F_U][pidx(B, i, j, k)] = u;
}

// ------------------------------------------------------------------
// ADM mass surface integrand: dU = x_hat . grad(c + u) interpolated
// (trilinear) onto a 101 x 101 sphere of radius 0.375 min L around the box
// centre, times sin(theta)
// ------------------------------------------------------------------
__device__ int cell_of(const DevBox &B, int a, double x) {
  const int np = B.n[a];
  const double lo = B.lo[a], hi = coord(B, a, np - 1);
  if (!(lo < x && x < hi)) return (lo >= x) ? 1 : np - 1;
  int lo_i = 0, hi_i = np;
  int i = (np % 2 == 0) ? np / 2 : (np - 1) / 2;
  do {
    const double xi = coord(B, a, i);
    if (xi > x || fabs(xi - x) <= 3 * kEps)
      hi_i = i;
    else
      lo_i = i;
    const int s = hi_i + lo_i;
    i = (s % 2 == 0) ? s / 2 : (s - 1) / 2;
  } while (lo_i + 1 < hi_i);
  return i + 1;
}

__device__ double dU_at(const DevBox &B, const double ctr[3], int i, int j, int k) {
  const long long p = pidx(B, i, j, k);
  const int ijk[3] = {i, j, k};
  double X[3], g[3];
  for (int a = 0; a < 3; ++a) {
    X[a] = coord(B, a, ijk[a]) - ctr[a];
    double cf;
    g[a] = deriv(B, B.f[F_C], p, a, i, j, k, cf) + deriv(B, B.f[F_U], p, a, i, j, k, cf);
  }
  const double ir = 1.0 / sqrt(X[0] * X[0] + X[1] * X[1] + X[2] * X[2]);
  return ir * (X[0] * g[0] + X[1] * g[1] + X[2] * g[2]);
}

__global__ __launch_bounds__(256) void k_adm_sphere(const DevBox *__restrict__ boxes,
                                                     const double *__restrict__ centres,
                                                     double *__restrict__ sph, int nt) {
  const int box = blockIdx.y;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nt * nt) return;
  const DevBox &B = boxes[box];
  const double ctr[3] = {centres[3 * box], centres[3 * box + 1], centres[3 * box + 2]};
  const double L0 = coord(B, 0, B.n[0] - 1) - B.lo[0];
  const double L1 = coord(B, 1, B.n[1] - 1) - B.lo[1];
  const double L2 = coord(B, 2, B.n[2] - 1) - B.lo[2];
  const double r0 = 0.375 * fmin(L0, fmin(L1, L2));
  const int it = q / nt, ip = q % nt;
  const double dtheta = M_PI / (nt - 1), dphi = 2 * M_PI / (nt - 1);
  const double th = it * dtheta, ph = ip * dphi;
  const double X[3] = {ctr[0] + r0 * cos(ph) * sin(th), ctr[1] + r0 * sin(ph) * sin(th),
                       ctr[2] + r0 * cos(th)};
  int c[3];
  bool coinc = true;
  for (int a = 0; a < 3; ++a) {
    c[a] = cell_of(B, a, X[a]);
    if (!(fabs(X[a] - coord(B, a, c[a])) <= 3 * kEps)) coinc = false;
  }
  double v;
  if (coinc) {
    v = dU_at(B, ctr, c[0], c[1], c[2]);
  } else {
    for (int a = 0; a < 3; ++a) c[a] = c[a] == 0 ? 1 : c[a];
    const double fx = (X[0] - coord(B, 0, c[0] - 1)) * B.idx[0];
    const double fy = (X[1] - coord(B, 1, c[1] - 1)) * B.idx[1];
    const double fz = (X[2] - coord(B, 2, c[2] - 1)) * B.idx[2];
    const double gx = 1 - fx, gy = 1 - fy, gz = 1 - fz;
    const int I = c[0], J = c[1], K = c[2];
    v = ((dU_at(B, ctr, I - 1, J - 1, K - 1) * gx + dU_at(B, ctr, I, J - 1, K - 1) * fx) * gy +
         (dU_at(B, ctr, I - 1, J, K - 1) * gx + dU_at(B, ctr, I, J, K - 1) * fx) * fy) * gz +
        ((dU_at(B, ctr, I - 1, J - 1, K) * gx + dU_at(B, ctr, I, J - 1, K) * fx) * gy +
         (dU_at(B, ctr, I - 1, J, K) * gx + dU_at(B, ctr, I, J, K) * fx) * fy) * fz;
  }
  sph[(long long)box * nt * nt + q] = v * sin(th);
}

// Points q0 .. q0 + n - 1 of one field of a box, lexicographic (i fastest),
// to or from `host` (pinned memory the GPU reaches over PCIe), the colour
// blocks' order undone or made on the way.  Bound by PCIe: a wave's 512
// bytes of `host` are contiguous, its NC runs in the colour blocks 128 bytes
// each.  A host loop over the colour blocks' index map took 14.8 ms for the
// 4.5 M points of one N=161 box, copies included; this way 1.7 ms.
template <bool TO_HOST>
__global__ __launch_bounds__(256) void k_field_host(DevBox B, double *__restrict__ f,
                                                     double *__restrict__ host, unsigned q0,
                                                     unsigned n) {
  const unsigned q = blockIdx.x * 256u + threadIdx.x;
  if (q >= n) return;
  int i, j, k;
  point_ijk(B, (long long)q0 + q, i, j, k);
  const long long p = pidx(B, i, j, k);
  if constexpr (TO_HOST)
    host[q] = f[p];
  else
    f[p] = host[q];
}

// lane N of the caller's row of 16 lanes
template <int N>
__device__ __forceinline__ double row_lane(double v) {
  return dpp_f64<0x150 + N, 0xF>(v);
}
template <int N>
__device__ __forceinline__ int row_lane(int v) {
  return __builtin_amdgcn_update_dpp(v, v, 0x150 + N, 0xF, 0xF, false);
}

// Lagrange interpolation of one field at arbitrary points (one box per
// point), interpolation.cc:189-303.  16 lanes (one DPP row) a point: the
// lanes search the axes' cells and evaluate the weights side by side, then
// each sums the z nodes of its (x, y) column of nodes (NI = 8: x node
// lane % 8 of two y nodes at a time; 16: up to ten x nodes, one y node), and
// the columns are added over y and x in the reference's order through row
// broadcasts.  One point a thread did 168 dependent divisions and 512
// scattered loads in turn: 200,000 points at order 7 took 595 us, now 258.
template <int NI>
__global__ __launch_bounds__(256) void k_interp_points(const DevBox *__restrict__ boxes, int field,
                                                        const int *__restrict__ pbox,
                                                        const double *__restrict__ pxyz, int npts,
                                                        int ord, double *__restrict__ out) {
  constexpr int NMAX = NI == 8 ? 8 : 10;  // nodes per axis, at most
  constexpr int NJ = 16 / NI;             // y nodes at a time
  const int lane = int(threadIdx.x & 15u);
  const int q = int(blockIdx.x * (blockDim.x / 16u) + (threadIdx.x >> 4));
  if (q >= npts) return;
  const DevBox &B = boxes[pbox[q]];
  const double *__restrict__ f = B.f[field];
  const double X[3] = {pxyz[3 * q], pxyz[3 * q + 1], pxyz[3 * q + 2]};
  // lanes 0, 1, 2 of the row search axes x, y, z
  const int ax = lane < 3 ? lane : 0;
  const double xa = ax == 0 ? X[0] : (ax == 1 ? X[1] : X[2]);
  const int ca = cell_of(B, ax, xa);
  const int hit = fabs(xa - coord(B, ax, ca)) <= 3 * kEps;
  const int c[3] = {row_lane<0>(ca), row_lane<1>(ca), row_lane<2>(ca)};
  if (row_lane<0>(hit) & row_lane<1>(hit) & row_lane<2>(hit)) {
    if (lane == 0) out[q] = f[pidx(B, c[0], c[1], c[2])];
    return;
  }
  // a box with fewer than ord + 1 points per axis takes the widest stencil
  // it holds (interpolation.cc:221-250 would read outside the box there)
  ord = min(ord, min(B.n[0], min(B.n[1], B.n[2])) - 1);
  int s[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    int s0 = (ord % 2 == 0) ? c[a] - ord / 2 : c[a] - (ord + 1) / 2;
    if (s0 < 0) s0 = 0;
    else if (s0 + ord >= B.n[a]) s0 = B.n[a] - ord - 1;
    s[a] = s0;
  }
  // weight of node m of axis a at lane m of wt[a]
  auto weight = [&](double x, double lo, double d, int s0, int m) {
    const double xn = lo + (double)(s0 + m) * d;
    double lp = 1.0;
    for (int l = 0; l <= ord; ++l) {
      const double xl = lo + (double)(s0 + l) * d;
      const double t = (x - xl) / (xn - xl);
      if (l != m) lp *= t;
    }
    return lp;
  };
  const int m8 = lane & 7, hi = lane >> 3;
  double wt[3];
  if constexpr (NI == 8) {
    // the lower lanes weight x and then z, the upper ones y
    const double w01 = weight(hi ? X[1] : X[0], hi ? B.lo[1] : B.lo[0], hi ? B.d[1] : B.d[0],
                              hi ? s[1] : s[0], m8);
    wt[0] = w01;
    wt[1] = dpp_f64<0x128, 0xF>(w01);  // row_ror:8
    wt[2] = weight(X[2], B.lo[2], B.d[2], s[2], m8);
  } else {
#pragma unroll
    for (int a = 0; a < 3; ++a) wt[a] = weight(X[a], B.lo[a], B.d[a], s[a], lane);
  }
  double wz[NMAX], wy[NMAX];
#define OLL_ROW8(F) F(0) F(1) F(2) F(3) F(4) F(5) F(6) F(7)
#define OLL_W(m) \
  wz[m] = row_lane<m>(wt[2]); \
  wy[m] = row_lane<m>(wt[1]);
  OLL_ROW8(OLL_W)
  if constexpr (NMAX > 8) {
    OLL_W(8)
    OLL_W(9)
  }
#undef OLL_W
  // the lane's x node (clamped: lanes past the stencil load its last node
  // and their sums are not used)
  const int I = min(NI == 8 ? m8 : lane, ord), Jb = NI == 8 ? hi : 0;
  const int nc = B.nc;
  const int xi = s[0] + I, xslot = split_div(B, xi);
  double uj = 0.0;  // the lane's column sums over y (NI = 8: of the row's lower lanes)
  const double *__restrict__ col0 = f + (long long)s[2] * B.ps + xslot;
  // y nodes J0 (and J0 + 1)
  auto columns = [&](int J0, double w0, double w1) {
    const int yj = s[1] + min(J0 + Jb, ord);
    int col = xi + yj + s[2];
    col -= split_div(B, col) * nc;
    const double *__restrict__ row = col0 + (long long)yj * B.rs;
    double v[NMAX];
#pragma unroll
    for (int K = 0; K < NMAX; ++K) {
      v[K] = 0.0;
      if (K <= ord) v[K] = row[(long long)col * B.cs];
      row += B.ps;
      col = col + 1 == nc ? 0 : col + 1;
    }
    double uk = 0.0;
#pragma unroll
    for (int K = 0; K < NMAX; ++K)
      if (K <= ord) uk += v[K] * wz[K];
    uj += uk * w0;
    if constexpr (NJ == 2) {
      const double up = dpp_f64<0x128, 0xF>(uk);  // the row's other half
      if (J0 + 1 <= ord) uj += up * w1;
    }
  };
#pragma unroll
  for (int J0 = 0; J0 < NMAX; J0 += NJ)
    if (J0 <= ord) columns(J0, wy[J0], NJ == 2 ? wy[J0 + NJ - 1] : 0.0);
  double acc = 0.0;
#define OLL_A(m) \
  if (m <= ord) acc += row_lane<m>(uj) * row_lane<m>(wt[0]);
  OLL_ROW8(OLL_A)
  if constexpr (NMAX > 8) {
    OLL_A(8)
    OLL_A(9)
  }
#undef OLL_A
#undef OLL_ROW8
  if (lane == 0) out[q] = acc;
}

__global__ void k_zero_u64(unsigned long long *p, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

// clear item blockIdx.x: its own word count, never another member's
__global__ void k_zero_lists(const ZeroItem *items) {
  const ZeroItem it = items[blockIdx.x];
  for (long long i = threadIdx.x; i < it.count; i += blockDim.x) it.p[i] = 0ull;
}

inline unsigned ceil_div(long long a, long long b) { return unsigned((a + b - 1) / b); }

template <int ORD, int EQ>
void smooth_impl(hipStream_t s, const RowBlock *blocks, int nb, int per_row, int pass,
                 int threads, hipEvent_t e0, hipEvent_t e1, const DevBox *box1) {
  if (nb == 0) return;
  if (e0)  // timed (never under graph capture): the runtime stamps e0, e1
    hipExtLaunchKernelGGL((k_smooth<ORD, EQ>), dim3(nb), dim3(threads), 0, s, e0, e1, 0, blocks,
                          unsigned(per_row), 1.0f / float(per_row), pass, box1);
  else
    hipLaunchKernelGGL((k_smooth<ORD, EQ>), dim3(nb), dim3(threads), 0, s, blocks,
                       unsigned(per_row), 1.0f / float(per_row), pass, box1);
}

template <int ORD, int EQ>
void residual_impl(hipStream_t s, const RowBlock *blocks, int nb, int per_row, int mode) {
  if (nb == 0) return;
  hipLaunchKernelGGL((k_residual<ORD, EQ>), dim3(nb), dim3(kRowThreads), 0, s, blocks,
                     unsigned(per_row), 1.0f / float(per_row), mode);
}

template <int ORD, int EQ>
void defect32_impl(hipStream_t s, const RowBlock *blocks, int nb, int per_row) {
  if (nb == 0) return;
  hipLaunchKernelGGL((k_defect32<ORD, EQ>), dim3(nb), dim3(kRowThreads), 0, s, blocks,
                     unsigned(per_row), 1.0f / float(per_row));
}

template <int ORD, int EQ>
void smooth32_impl(hipStream_t s, const RowBlock *blocks, int nb, int per_row, int colour,
                   int threads, hipEvent_t e0, hipEvent_t e1) {
  if (nb == 0) return;
  if (e0)
    hipExtLaunchKernelGGL((k_smooth32<ORD>), dim3(nb), dim3(threads), 0, s, e0, e1, 0, blocks,
                          unsigned(per_row), 1.0f / float(per_row), colour);
  else
    hipLaunchKernelGGL((k_smooth32<ORD>), dim3(nb), dim3(threads), 0, s, blocks,
                       unsigned(per_row), 1.0f / float(per_row), colour);
}

template <int ORD, int EQ>
void update32_impl(hipStream_t s, const RowBlock *blocks, int nb, int per_row) {
  if (nb == 0) return;
  hipLaunchKernelGGL((k_update32<ORD>), dim3(nb), dim3(kRowThreads), 0, s, blocks,
                     unsigned(per_row), 1.0f / float(per_row));
}

template <int ORD, int EQ>
void restrict_defect_impl(hipStream_t s, const PtBlock *blocks, int nb) {
  if (nb == 0) return;
  hipLaunchKernelGGL((k_restrict_defect<ORD, EQ>), dim3(nb), dim3(kPtThreads), 0, s, blocks);
}


}  // namespace

// ------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------

#define OLL_DISPATCH_ORDER_EQ(ORDER, E, KERNEL, ...)                  \
  switch (ORDER) {                                                    \
    case 2: KERNEL<2, E>(__VA_ARGS__); break;                         \
    case 4: KERNEL<4, E>(__VA_ARGS__); break;                         \
    case 6: KERNEL<6, E>(__VA_ARGS__); break;                         \
    default: KERNEL<8, E>(__VA_ARGS__); break;                        \
  }
#define OLL_DISPATCH_ORDER(ORDER, EQ, KERNEL, ...)                    \
  do {                                                                \
    switch (EQ) {                                                     \
      case 1: OLL_DISPATCH_ORDER_EQ(ORDER, 1, KERNEL, __VA_ARGS__) break; \
      case 2: OLL_DISPATCH_ORDER_EQ(ORDER, 2, KERNEL, __VA_ARGS__) break; \
      case 3: OLL_DISPATCH_ORDER_EQ(ORDER, 3, KERNEL, __VA_ARGS__) break; \
      case kEqPuncturesEm: OLL_DISPATCH_ORDER_EQ(ORDER, kEqPuncturesEm, KERNEL, __VA_ARGS__) break; \
      default: OLL_DISPATCH_ORDER_EQ(ORDER, 0, KERNEL, __VA_ARGS__) break; \
    }                                                                 \
  } while (0)

void launch_coefficients_box(hipStream_t s, const DevBox &B, const PunctureArgs &pa,
                             double robin_a) {
  const long long np = (long long)B.n[0] * B.n[1] * B.n[2];
  hipLaunchKernelGGL(k_coefficients, dim3(ceil_div(np, 256)), dim3(256), 0, s, B, pa, robin_a);
}

void launch_approx_box(hipStream_t s, const DevBox &B, const PunctureArgs &pa) {
  const long long np = (long long)B.n[0] * B.n[1] * B.n[2];
  hipLaunchKernelGGL(k_approx_u, dim3(ceil_div(np, 256)), dim3(256), 0, s, B, pa);
}

// threads per colour-pass workgroup, [mixed][order / 2 - 1]
static int g_sweep_threads[2][4] = {{256, 256, 256, 256}, {256, 256, 256, 256}};

int sweep_threads(int mixed, int order) {
  return g_sweep_threads[mixed ? 1 : 0][std::min(3, std::max(0, order / 2 - 1))];
}

bool set_sweep_threads(int mixed, int order, int threads) {
  if (!(order == 2 || order == 4 || order == 6 || order == 8)) return false;
  if (threads < 64 || threads > kMaxRowThreads || threads % 64 != 0) return false;
  g_sweep_threads[mixed ? 1 : 0][order / 2 - 1] = threads;
  return true;
}

void launch_smooth(hipStream_t s, const RowBlock *blocks, int nblocks, int per_row, int order,
                   int eq, int pass, int threads, hipEvent_t e0, hipEvent_t e1,
                   const DevBox *box1) {
  OLL_DISPATCH_ORDER(order, eq, smooth_impl, s, blocks, nblocks, per_row, pass, threads, e0, e1,
                     box1);
}

// tile shape of the fused passes, [order / 2 - 1]
static FusedShape g_fused_shape[4] = {{8, 8, 256}, {8, 8, 256}, {8, 8, 256}, {8, 8, 256}};

FusedShape fused_shape(int order) { return g_fused_shape[std::min(3, std::max(0, order / 2 - 1))]; }

bool set_fused_shape(int order, int ty, int tz, int threads) {
  if (!(order == 2 || order == 4 || order == 6 || order == 8)) return false;
  if (ty < 1 || tz < 1 || ty > 64 || tz > 64) return false;
  if (threads < 64 || threads > kFusedThreads || threads % 64 != 0) return false;
  g_fused_shape[order / 2 - 1] = FusedShape{ty, tz, threads};
  return true;
}

template <int ORD, int EQ, int Q, int PAIR>
void fused_impl(hipStream_t s, const TileBlock *blocks, int nb, int parity, int threads,
                hipEvent_t e0, hipEvent_t e1) {
  if (nb == 0) return;
  if (e0)  // timed (never under graph capture): the runtime stamps e0, e1
    hipExtLaunchKernelGGL((k_smooth_fused<ORD, EQ, Q, PAIR>), dim3(nb), dim3(threads), 0, s, e0,
                          e1, 0, blocks, parity);
  else
    hipLaunchKernelGGL((k_smooth_fused<ORD, EQ, Q, PAIR>), dim3(nb), dim3(threads), 0, s, blocks,
                       parity);
}

template <int ORD, int EQ>
void fused_order(hipStream_t s, const TileBlock *blocks, int nb, int q, int pair, int parity,
                 int threads, hipEvent_t e0, hipEvent_t e1) {
  constexpr int NC = ORD / 2 + 1;
  // pairs (0, 1), (2, 3); a single pass for the last colour when NC is odd
  if (pair && q == 0) return fused_impl<ORD, EQ, 0, 1>(s, blocks, nb, parity, threads, e0, e1);
  if constexpr (NC >= 4)
    if (pair && q == 2) return fused_impl<ORD, EQ, 2, 1>(s, blocks, nb, parity, threads, e0, e1);
  if constexpr (NC % 2 == 1)
    if (!pair && q == NC - 1)
      return fused_impl<ORD, EQ, NC - 1, 0>(s, blocks, nb, parity, threads, e0, e1);
}

void launch_smooth_fused(hipStream_t s, const TileBlock *blocks, int nblocks, int order, int eq,
                         int q, int pair, int parity, int threads, hipEvent_t e0, hipEvent_t e1) {
  switch (eq) {
    case 1: OLL_DISPATCH_ORDER_EQ(order, 1, fused_order, s, blocks, nblocks, q, pair, parity, threads, e0, e1) break;
    case 2: OLL_DISPATCH_ORDER_EQ(order, 2, fused_order, s, blocks, nblocks, q, pair, parity, threads, e0, e1) break;
    case 3: OLL_DISPATCH_ORDER_EQ(order, 3, fused_order, s, blocks, nblocks, q, pair, parity, threads, e0, e1) break;
    default: OLL_DISPATCH_ORDER_EQ(order, 0, fused_order, s, blocks, nblocks, q, pair, parity, threads, e0, e1) break;
  }
}

void launch_copy_shell(hipStream_t s, const PtBlock *blocks, int nblocks) {
  if (nblocks == 0) return;
  hipLaunchKernelGGL(k_copy_shell, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
}

void launch_residual(hipStream_t s, const RowBlock *blocks, int nblocks, int per_row, int order,
                     int eq, int mode) {
  OLL_DISPATCH_ORDER(order, eq, residual_impl, s, blocks, nblocks, per_row, mode);
}

void launch_defect32(hipStream_t s, const RowBlock *blocks, int nblocks, int per_row, int order,
                     int eq) {
  OLL_DISPATCH_ORDER(order, eq, defect32_impl, s, blocks, nblocks, per_row);
}

void launch_smooth32(hipStream_t s, const RowBlock *blocks, int nblocks, int per_row, int order,
                     int colour, int threads, hipEvent_t e0, hipEvent_t e1) {
  OLL_DISPATCH_ORDER(order, 0, smooth32_impl, s, blocks, nblocks, per_row, colour, threads, e0, e1);
}

void launch_update32(hipStream_t s, const RowBlock *blocks, int nblocks, int per_row, int order) {
  OLL_DISPATCH_ORDER(order, 0, update32_impl, s, blocks, nblocks, per_row);
}

void launch_robin(hipStream_t s, const RobinItem *items, int n, int total_cols, int total_edges,
                  int mode) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_robin_faces, dim3(ceil_div(total_cols, 256)), dim3(256), 0, s, items, n,
                     total_cols, mode);
  hipLaunchKernelGGL(k_robin_edges, dim3(ceil_div(total_edges, kEdgeSections)),
                     dim3(kRobinEdgeThreads), 0, s, items, n, total_edges, mode);
  hipLaunchKernelGGL(k_robin_corners, dim3(n), dim3(8 * kCornerR3), 0, s, items, mode);
}

void launch_restrict_u(hipStream_t s, const PtBlock *blocks, int nblocks) {
  if (nblocks == 0) return;
  hipLaunchKernelGGL(k_restrict_u, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
}

void launch_restrict_defect(hipStream_t s, const PtBlock *blocks, int nblocks, int order, int eq) {
  OLL_DISPATCH_ORDER(order, eq, restrict_defect_impl, s, blocks, nblocks);
}

void launch_filter_defect(hipStream_t s, const PtBlock *blocks, int nblocks, int runs) {
  if (nblocks == 0) return;
  if (runs)
    hipLaunchKernelGGL(k_filter_cols, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
  else
    hipLaunchKernelGGL(k_filter_defect, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
}

int filter_run_length() { return kFilterCx; }

void launch_corr_v(hipStream_t s, const PtBlock *blocks, int nblocks) {
  if (nblocks == 0) return;
  hipLaunchKernelGGL(k_corr_v, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
}

void launch_prolong(hipStream_t s, const PtBlock *blocks, int nblocks) {
  if (nblocks == 0) return;
  hipLaunchKernelGGL(k_prolong, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
}

template <int KP>
void ghost_impl(hipStream_t s, const PtBlock *blocks, int nblocks, int columns) {
  if (columns)
    hipLaunchKernelGGL(k_ghost_tiles<KP>, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
  else
    hipLaunchKernelGGL(k_ghost_fill<KP>, dim3(nblocks), dim3(kPtThreads), 0, s, blocks);
}

void launch_ghost_fill(hipStream_t s, const PtBlock *blocks, int nblocks, int order, int columns) {
  if (nblocks == 0) return;
  switch (order) {
    case 2: ghost_impl<4>(s, blocks, nblocks, columns); break;
    case 4: ghost_impl<6>(s, blocks, nblocks, columns); break;
    case 6: ghost_impl<8>(s, blocks, nblocks, columns); break;
    default: ghost_impl<10>(s, blocks, nblocks, columns); break;
  }
}

// coarse-solve shape by box size: up to 2048 points of a colour and a shell
// that the threads hold, 1024 threads with 2 points each and their
// coefficients in registers (512 threads with 4 each for EM, whose longer
// update would spill at 1024 threads; the scalar field's 17^3 753 us with 512
// threads, 598 with 1024); up to 4096 (the 21^3 coarsest box of N=161), 1024
// threads with 4 each.  Every cube of up to 4096 points of a colour has a
// shell of at most 3 * 1024 points.
bool launch_coarse_solve(hipStream_t s, const CoarseItem *items, int n, int max_pts, int max_int,
                         int max_shell, int eq, double eps, int max_iter) {
  const size_t lds = 2 * sizeof(double) * size_t(max_pts);  // max_pts: largest B.size
  // max_int: largest number of points of one colour slot list, ceil(ni/2) nj nk
  // max_shell: largest number of face and edge points
  if (lds > size_t(kCoarseMostLds) || max_int > kCoarseMostSlots || max_shell > kCoarseMostShell)
    return false;
  if (n == 0) return true;
  const bool em = eq == kEqPuncturesEm;
  const bool small = max_int <= 2048 && max_shell <= (em ? 3 * 512 : 2 * 1024);
#define OLL_COARSE(E)                                                                              \
  if (small)                                                                                       \
    hipLaunchKernelGGL((k_coarse_solve<E, 2, 1024, 2>), dim3(n), dim3(1024), lds, s, items, eps, max_iter); \
  else                                                                                             \
    hipLaunchKernelGGL((k_coarse_solve<E, 4, 1024, 3>), dim3(n), dim3(1024), lds, s, items, eps, max_iter);
  switch (eq) {
    case 1: OLL_COARSE(1) break;
    case 2: OLL_COARSE(2) break;
    case 3: OLL_COARSE(3) break;
    case kEqPuncturesEm:
      if (small)
        hipLaunchKernelGGL((k_coarse_solve<kEqPuncturesEm, 4, 512, 3>), dim3(n), dim3(512), lds, s, items, eps, max_iter);
      else
        hipLaunchKernelGGL((k_coarse_solve<kEqPuncturesEm, 4, 1024, 3>), dim3(n), dim3(1024), lds, s, items, eps, max_iter);
      break;
    default: OLL_COARSE(0) break;
  }
#undef OLL_COARSE
  return true;
}

bool launch_transfer_fields(hipStream_t s, const PtBlock *blocks, int nblocks, int ff, int tf,
                            int nodes, bool tiles) {
  if (nblocks == 0) return true;
#define OLL_TF(KP)                                                                                     \
  if (tiles)                                                                                           \
    hipLaunchKernelGGL(k_transfer_tiles<KP>, dim3(nblocks), dim3(kPtThreads), 0, s, blocks, ff, tf);   \
  else                                                                                                 \
    hipLaunchKernelGGL(k_transfer_points<KP>, dim3(nblocks), dim3(kPtThreads), 0, s, blocks, ff, tf)
  switch (nodes) {
    case 2:
      hipLaunchKernelGGL(k_transfer_points<2>, dim3(nblocks), dim3(kPtThreads), 0, s, blocks, ff, tf);
      break;
    case 3: OLL_TF(3); break;
    case 4: OLL_TF(4); break;
    case 5: OLL_TF(5); break;
    case 6: OLL_TF(6); break;
    case 7: OLL_TF(7); break;
    case 8: OLL_TF(8); break;
    case 9: OLL_TF(9); break;
    case 10: OLL_TF(10); break;
    default: return false;
  }
#undef OLL_TF
  return true;
}

void launch_zero_lists(hipStream_t s, const ZeroItem *items, int n) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_zero_lists, dim3(n), dim3(256), 0, s, items);
}

void kernels_init() {
  static bool done = false;
  if (done) return;
#define OLL_COARSE_FNS(E)                                               \
  reinterpret_cast<const void *>(&k_coarse_solve<E, 2, 1024, 2>), \
      reinterpret_cast<const void *>(&k_coarse_solve<E, 4, 1024, 3>)
  const void *fns[] = {OLL_COARSE_FNS(0), OLL_COARSE_FNS(1), OLL_COARSE_FNS(2), OLL_COARSE_FNS(3),
                       reinterpret_cast<const void *>(&k_coarse_solve<kEqPuncturesEm, 4, 512, 3>),
                       reinterpret_cast<const void *>(&k_coarse_solve<kEqPuncturesEm, 4, 1024, 3>)};
#undef OLL_COARSE_FNS
  for (const void *f : fns)
    (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kCoarseMostLds);
  done = true;
}

void launch_zero_u64(hipStream_t s, unsigned long long *p, long long n) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_zero_u64, dim3(ceil_div(n, 256)), dim3(256), 0, s, p, n);
}

void launch_adm_sphere(hipStream_t s, const DevBox *boxes, int nbox, const double *centres,
                       double *sph, int nt) {
  hipLaunchKernelGGL(k_adm_sphere, dim3(ceil_div(nt * nt, 256), nbox), dim3(256), 0, s, boxes,
                     centres, sph, nt);
}

void launch_field_host(hipStream_t s, const DevBox &B, int field, double *host, unsigned q0,
                       unsigned n, bool to_host) {
  if (n == 0) return;
  if (to_host)
    hipLaunchKernelGGL(k_field_host<true>, dim3(ceil_div(n, 256)), dim3(256), 0, s, B, B.f[field], host, q0, n);
  else
    hipLaunchKernelGGL(k_field_host<false>, dim3(ceil_div(n, 256)), dim3(256), 0, s, B, B.f[field], host, q0, n);
}

void launch_interp_points(hipStream_t s, const DevBox *boxes, int field, const int *pbox,
                          const double *pxyz, int npts, int ord, double *out) {
  const dim3 grid(ceil_div(npts, 16));
  if (ord <= 7)
    hipLaunchKernelGGL(k_interp_points<8>, grid, dim3(256), 0, s, boxes, field, pbox, pxyz, npts, ord, out);
  else
    hipLaunchKernelGGL(k_interp_points<16>, grid, dim3(256), 0, s, boxes, field, pbox, pxyz, npts, ord, out);
}

}  // namespace oll
