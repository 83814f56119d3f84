// Cartesian (Taylor-series) basis: P2M, M2M, M2L, L2L, L2P and the periodic
// far field, for P = 4, 6, 8 (NTERM = P (P+1) (P+2) / 6 real coefficients).
//
// Reference: kernels/LaplaceCartesianCPU.cxx (Index :3-24, power/derivative/
// scale and the M2M/M2L/L2L/L2P sums :26-252, getCoef/sumM2L :254-588, the
// kernel entry points :590-704).  Conventions:
//   M_k = sum_b q_b (X_c - x_b)^k / k!          (P2M, M2M)
//   C_k = d^k (1/r) at dX = X_i - X_j - X_p     (raw derivatives; MASS: times
//                                                M0_i M0_j)
//   L_a += M_0 C_a + sum_{b} M_b C_{a+b}         (MASS: C_a for the first term)
//   phi(x) = sum_k L_k (x - X_c)^k / k!          (L2L, L2P)
// with k a multi-index, |k| <= P-1.  Coefficients are stored in the real parts
// of the handle's complex M and L arrays (imaginary parts 0), at the index
// order of Index<kx,ky,kz>::I: by degree, then kx descending, then ky
// descending.
//
// The upward pass follows the reference's operation order without FMA
// contraction (multipoles bit-identical to the reference).  M2L takes one
// wave per target cell and one lane per pair, in registers.
#include <algorithm>
#include <utility>

#include "harmonics.h"
#include "internal.h"

namespace exafmm {

template <int P>
struct Cart {
  static constexpr int NT = P * (P + 1) * (P + 2) / 6;
};

// Index of (a, b, c): n(n+1)(n+2)/6 + m(m+1)/2 + (m - b), n = a+b+c, m = b+c.
__host__ __device__ inline int cidx(int a, int b, int c) {
  const int n = a + b + c, m = b + c;
  return n * (n + 1) * (n + 2) / 6 + m * (m + 1) / 2 + (m - b);
}

__host__ __device__ inline void cmi(int t, int &a, int &b, int &c) {
  int n = 0;
  while ((n + 1) * (n + 2) * (n + 3) / 6 <= t) n++;
  const int r = t - n * (n + 1) * (n + 2) / 6;
  int m = 0;
  while ((m + 1) * (m + 2) / 2 <= r) m++;
  b = m - (r - m * (m + 1) / 2);
  c = m - b;
  a = n - m;
}

// v / i correctly rounded for a small whole number i: the quotient by the
// rounded reciprocal, corrected once by its exact remainder.
__device__ inline double div_small(double v, int i) {
  const double y = kInv.v[i], q = v * y;
  return fma(fma(-q, (double)i, v), y, q);
}

// One coefficient of Kernels::power (:183-186,213-216,243-246): the chain
// C_(a,0,0) = C_(a-1,0,0) dx / a, C_(a,b,0) = C_(a,b-1,0) dy / b,
// C_(a,b,c) = C_(a,b,c-1) dz / c, started from v.
__device__ inline double cpow(double v, int a, int b, int c, double dx, double dy, double dz) {
#pragma clang fp contract(off)
  for (int i = 1; i <= a; i++) v = div_small(v * dx, i);
  for (int i = 1; i <= b; i++) v = div_small(v * dy, i);
  for (int i = 1; i <= c; i++) v = div_small(v * dz, i);
  return v;
}

// Derivative tensor C_k = d^k (1/r) of one offset into row[0, NT): the
// Taylor coefficients a_k = ((1-2n) sum_d x_d a_{k-e_d} + (1-n) sum_d
// a_{k-2e_d}) / n / r^2 (Kernels::derivative, :187-191), then k! (scale).
template <int P>
__device__ inline void cart_coef(double *row, double dx, double dy, double dz, double invR2, double invR) {
  constexpr int NT = Cart<P>::NT;
  row[0] = invR;
  int t = 1;
  for (int n = 1; n < P; n++)
    for (int a = n; a >= 0; a--)
      for (int b = n - a; b >= 0; b--, t++) {
        const int c = n - a - b;
        double s1 = 0, s2 = 0;
        if (a >= 1) s1 += dx * row[cidx(a - 1, b, c)];
        if (b >= 1) s1 += dy * row[cidx(a, b - 1, c)];
        if (c >= 1) s1 += dz * row[cidx(a, b, c - 1)];
        if (a >= 2) s2 += row[cidx(a - 2, b, c)];
        if (b >= 2) s2 += row[cidx(a, b - 2, c)];
        if (c >= 2) s2 += row[cidx(a, b, c - 2)];
        row[t] = ((1 - 2 * n) * s1 + (1 - n) * s2) / n * invR2;
      }
  t = 1;
  for (int n = 1; n < P; n++)
    for (int a = n; a >= 0; a--)
      for (int b = n - a; b >= 0; b--, t++) {
        const int c = n - a - b;
        double f = 1;
        for (int i = 2; i <= a; i++) f *= i;
        for (int i = 2; i <= b; i++) f *= i;
        for (int i = 2; i <= c; i++) f *= i;
        row[t] *= f;
      }
  (void)NT;
}

// Terms (a, b) of sumM2L at order P (:373-588): |a| + |b| <= P-1, where the
// reference's unrolled forms for P <= 7 leave out |b| = P-1 at a = 0.
__host__ __device__ inline bool m2l_term(int P, int da, int db) {
  return da + db <= P - 1 && !(P <= 7 && da == 0 && db == P - 1);
}

// Index tables of the packed coefficients.
template <int P>
struct CartTab {
  static constexpr int NT = Cart<P>::NT;
  int x[NT], y[NT], z[NT];
  int prev[NT], dir[NT];  // the factor of power's chain: index less one in direction dir
  constexpr CartTab() : x(), y(), z(), prev(), dir() {
    int t = 0;
    for (int n = 0; n < P; n++)
      for (int a = n; a >= 0; a--)
        for (int b = n - a; b >= 0; b--, t++) {
          const int c = n - a - b;
          x[t] = a;
          y[t] = b;
          z[t] = c;
          dir[t] = c > 0 ? 2 : b > 0 ? 1 : 0;
          prev[t] = n == 0 ? 0 : idx(a - (dir[t] == 0), b - (dir[t] == 1), c - (dir[t] == 2));
        }
  }
  static constexpr int idx(int a, int b, int c) {
    const int n = a + b + c, m = b + c;
    return n * (n + 1) * (n + 2) / 6 + m * (m + 1) / 2 + c;
  }
};

// ---------------------------------------------------------------------------
// Upward pass: P2M (:590-598) at leaves, M2M (:600-612) at parents, then
// setRmax and R /= theta as in the spherical pass (radii = 0: left out, where
// the radii are made beside the multipoles).

__device__ inline void cart_radius(double4 *cX, int c, double rb, double rmax, double theta, int useRmax) {
  double R = rb;
  if (useRmax) R = R < rmax ? R : rmax;
  R /= theta;
  cX[c].w = R;
}

__device__ inline double wave_max(double v) {  // exact in any order
  for (int d = 32; d >= 1; d >>= 1) {
    const double o = __shfl_xor(v, d);
    v = o > v ? o : v;
  }
  return v;
}

// Every leaf among `cells`, one wave each: lanes own bodies and run power's
// chain once for all coefficients, then own coefficients and add the bodies
// in order.  (A lane per coefficient, each with its own chain of up to P - 1
// divisions per body, took 84 us for 4096 leaves of 27 bodies at P = 6;
// this takes 16 us.)
template <int P>
__global__ void __launch_bounds__(64)
    k_p2m_cart(const int *__restrict__ cells, const double4 *__restrict__ body, double4 *__restrict__ cX,
               const double *__restrict__ cRb, const int *__restrict__ cNChild, const int *__restrict__ cBody,
               const int *__restrict__ cNBody, cplx *__restrict__ M, double theta, int useRmax, int radii) {
#pragma clang fp contract(off)
  constexpr int NT = Cart<P>::NT;
  constexpr int NO = (NT + 63) / 64;
  constexpr int CH = P <= 6 ? 64 : 32;  // bodies at a time (29 to 32 KB of LDS)
  constexpr CartTab<P> tab{};
  __shared__ double sR[NT][CH + 1];
  const int c = cells[blockIdx.x];
  if (cNChild[c] != 0) return;
  const int lane = threadIdx.x;
  const double4 Xc = cX[c];
  double acc[NO], rmax = 0;
#pragma unroll
  for (int o = 0; o < NO; o++) acc[o] = 0;
  const int b0 = cBody[c], nb = cNBody[c];
  for (int base = 0; base < nb; base += CH) {
    const int cnt = min(CH, nb - base);
    __syncthreads();
    if (lane < cnt) {
      const double4 v = body[b0 + base + lane];
      const double r = exact_dist(Xc.x, Xc.y, Xc.z, v.x, v.y, v.z);
      rmax = r > rmax ? r : rmax;
      const double d[3] = {Xc.x - v.x, Xc.y - v.y, Xc.z - v.z};
      double C[NT];
      C[0] = v.w;
      sR[0][lane] = v.w;
#pragma unroll
      for (int t = 1; t < NT; t++) {
        const int k = tab.dir[t], i = k == 0 ? tab.x[t] : k == 1 ? tab.y[t] : tab.z[t];
        const double w = C[tab.prev[t]] * d[k];
        C[t] = i == 1 ? w : div_small(w, i);
        sR[t][lane] = C[t];
      }
    }
    __syncthreads();
#pragma unroll
    for (int o = 0; o < NO; o++) {
      const int t = lane + 64 * o;
      if (t < NT)
        for (int k = 0; k < cnt; k++) acc[o] += sR[t][k];
    }
  }
#pragma unroll
  for (int o = 0; o < NO; o++)
    if (lane + 64 * o < NT) M[(size_t)c * NT + lane + 64 * o] = {acc[o], 0.0};
  rmax = wave_max(rmax);
  if (radii && lane == 0) cart_radius(cX, c, cRb[c], rmax, theta, useRmax);
}

// The parents among `cells` (one level), one wave per child; the children's
// two sums per coefficient are then added in child order, as one lane walking
// the children would.  Latency-bound: 21 us per level of up to 512 parents,
// 97 us with one wave for all 8 children.
template <int P>
__global__ void __launch_bounds__(512)
    k_m2m_cart(const int *__restrict__ cells, double4 *__restrict__ cX, const double *__restrict__ cRb,
               const int *__restrict__ cChild, const int *__restrict__ cNChild, cplx *__restrict__ M, double theta,
               int useRmax, int radii) {
#pragma clang fp contract(off)
  constexpr int NT = Cart<P>::NT;
  __shared__ double sC[8][NT], sM[8][NT], s0[8][NT], s1[8][NT];
  __shared__ double sred[8];
  const int c = cells[blockIdx.x];
  const int nchild = cNChild[c];
  if (nchild == 0) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double4 Xc = cX[c];
  double acc = 0, rmax = 0;
  for (int base = 0; base < nchild; base += 8) {  // (an octree cell has 8 at most)
    const int cnt = min(8, nchild - base);
    __syncthreads();
    if (wave < cnt) {
      const int cc = cChild[c] + base + wave;
      const double4 Xj = cX[cc];
      const double dx = Xc.x - Xj.x, dy = Xc.y - Xj.y, dz = Xc.z - Xj.z;
      for (int t = lane; t < NT; t += 64) {
        int a, b, cz;
        cmi(t, a, b, cz);
        sC[wave][t] = cpow(1.0, a, b, cz, dx, dy, dz);
        sM[wave][t] = M[(size_t)cc * NT + t].re;
      }
      if (lane == 0) sred[wave] = exact_dist(Xc.x, Xc.y, Xc.z, Xj.x, Xj.y, Xj.z) + Xj.w;
    }
    __syncthreads();
    if (wave < cnt)
      for (int t = lane; t < NT; t += 64) {
        s0[wave][t] = sC[wave][t] * sM[wave][0];
        int ka, kb, kc;
        cmi(t, ka, kb, kc);
        // MultipoleSum: 0 <= k <= n, k != 0, lexicographic (kx, ky, kz).
        double sum = 0;
        for (int a = 0; a <= ka; a++)
          for (int b = 0; b <= kb; b++)
            for (int cz = 0; cz <= kc; cz++) {
              if (a == 0 && b == 0 && cz == 0) continue;
              sum += sC[wave][cidx(ka - a, kb - b, kc - cz)] * sM[wave][cidx(a, b, cz)];
            }
        s1[wave][t] = sum;
      }
    __syncthreads();
    if ((int)threadIdx.x < NT)
      for (int w = 0; w < cnt; w++) {
        acc += s0[w][threadIdx.x];
        if (threadIdx.x > 0) acc += s1[w][threadIdx.x];
        rmax = sred[w] > rmax ? sred[w] : rmax;
      }
  }
  if ((int)threadIdx.x < NT) M[(size_t)c * NT + threadIdx.x] = {acc, 0.0};
  if (radii && threadIdx.x == 0) cart_radius(cX, c, cRb[c], rmax, theta, useRmax);
}

// ---------------------------------------------------------------------------
// Downward pass: L2L (:631-645) for the cells of one level, then L2P
// (:647-664) at the leaves among them.
template <int P>
__global__ void __launch_bounds__(64)
    k_downward_cart(const int *__restrict__ cells, const double4 *__restrict__ body, const double4 *__restrict__ cX,
                    const int *__restrict__ cParent, const int *__restrict__ cNChild, const int *__restrict__ cBody,
                    const int *__restrict__ cNBody, const cplx *__restrict__ M, cplx *__restrict__ L,
                    double4 *__restrict__ trg, int do_l2l, int mass) {
#pragma clang fp contract(off)
  constexpr int NT = Cart<P>::NT;
  __shared__ double sC[NT];
  __shared__ double sL[NT];
  __shared__ double sLc[NT];
  const int c = cells[blockIdx.x];
  const int lane = threadIdx.x;
  const double4 Xc = cX[c];
  if (do_l2l) {
    const int p = cParent[c];
    const double4 Xp = cX[p];
    const double dx = Xc.x - Xp.x, dy = Xc.y - Xp.y, dz = Xc.z - Xp.z;
    for (int t = lane; t < NT; t += 64) {
      int a, b, cz;
      cmi(t, a, b, cz);
      sC[t] = cpow(1.0, a, b, cz, dx, dy, dz);
      sL[t] = L[(size_t)p * NT + t].re;
    }
    const double m0 = mass ? M[(size_t)c * NT].re : 1.0;
    __syncthreads();
    for (int t = lane; t < NT; t += 64) {
      double own = L[(size_t)c * NT + t].re;
      if (mass) own /= m0;
      own += sL[t];
      if (t == 0) {
        for (int i = 1; i < NT; i++) own += sC[i] * sL[i];
      } else {
        int a, b, cz;
        cmi(t, a, b, cz);
        const int dn = a + b + cz;
        double sum = 0;
        int k = 1;
        for (int n = 1; n <= P - 1 - dn; n++)
          for (int ka = n; ka >= 0; ka--)
            for (int kb = n - ka; kb >= 0; kb--, k++)
              sum += sC[k] * sL[cidx(a + ka, b + kb, cz + n - ka - kb)];
        own += sum;
      }
      L[(size_t)c * NT + t] = {own, 0.0};
      sLc[t] = own;
    }
  } else {
    for (int t = lane; t < NT; t += 64) sLc[t] = L[(size_t)c * NT + t].re;
  }
  if (cNChild[c] != 0) return;
  __syncthreads();
  const int b0 = cBody[c], nb = cNBody[c];
  for (int bi = lane; bi < nb; bi += 64) {
    const double4 v = body[b0 + bi];
    const double dx = v.x - Xc.x, dy = v.y - Xc.y, dz = v.z - Xc.z;
    double4 tv = trg[b0 + bi];
    tv.x += sLc[0];
    tv.y += sLc[1];
    tv.z += sLc[2];
    tv.w += sLc[3];
    double gx = 0, gy = 0, gz = 0;
    int k = 1;
    for (int n = 1; n < P; n++)
      for (int ka = n; ka >= 0; ka--)
        for (int kb = n - ka; kb >= 0; kb--, k++) {
          const int kc = n - ka - kb;
          const double Ck = cpow(1.0, ka, kb, kc, dx, dy, dz);
          tv.x += Ck * sLc[k];
          if (n <= P - 2) {
            gx += Ck * sLc[cidx(ka + 1, kb, kc)];
            gy += Ck * sLc[cidx(ka, kb + 1, kc)];
            gz += Ck * sLc[cidx(ka, kb, kc + 1)];
          }
        }
    tv.y += gx;
    tv.z += gy;
    tv.w += gz;
    trg[b0 + bi] = tv;
  }
}

// ---------------------------------------------------------------------------
// M2L over the CSR interaction list: one wave per target cell and one lane per
// pair, the pair's derivative tensor and the target's sums in registers, every
// index fixed at compile time; the lanes' sums are added in lane order through
// LDS at the end.  At P = 6 a pair is 462 multiply-adds and about 400 operations
// of the recurrence, and 448 bytes of its source's multipole; 2 x 56 doubles
// leave two waves per SIMD, with 26 registers spilled, so latency bounds it: the
// VALU issues 36% of the time, loads hit the L2 to 98%.  1.41 M pairs over 4680
// targets at P = 6: 105 us alone and 302 beside P2P, which takes 283 alone; 2180
// us beside P2P with a batch of tensors in LDS and a term list per lane (62 KB for
// one wave left two waves per CU).
// At P = 8 the 2 x 120 doubles do not fit 512 registers, so two kernels each
// make the tensor and sum a part of the outputs, those up to degree 4 (35
// outputs, 1358 of the 1716 terms) and the others: a cube of 100k bodies
// evaluates in 1045 us (1170 us with all outputs in one kernel, 163 registers
// spilled; 1080 and 1058 us cut after degree 3 and 5; 5150 us with tensors in
// LDS), 5k bodies in 468 us (478, 462, 471; 990).

// Real parts of the multipoles, packed (what k_m2l_cart_reg reads).
constexpr int kPackGrid = 1 << 20;  // workgroups at most
__global__ void k_cart_pack(const cplx *__restrict__ M, int64_t n, double *__restrict__ Mp) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    Mp[i] = M[i].re;
}

// One Taylor coefficient (Kernels::derivative, :187-191) from the lower ones.
template <int P, int T>
__device__ __forceinline__ void cart_taylor(double (&C)[Cart<P>::NT], const double (&d)[3], double invR2) {
  constexpr CartTab<P> tab{};
  constexpr int x = tab.x[T], y = tab.y[T], z = tab.z[T], n = x + y + z;
  double s1 = 0, s2 = 0;
  if constexpr (x >= 1) s1 += d[0] * C[CartTab<P>::idx(x - 1, y, z)];
  if constexpr (x >= 2) s2 += C[CartTab<P>::idx(x - 2, y, z)];
  if constexpr (y >= 1) s1 += d[1] * C[CartTab<P>::idx(x, y - 1, z)];
  if constexpr (y >= 2) s2 += C[CartTab<P>::idx(x, y - 2, z)];
  if constexpr (z >= 1) s1 += d[2] * C[CartTab<P>::idx(x, y, z - 1)];
  if constexpr (z >= 2) s2 += C[CartTab<P>::idx(x, y, z - 2)];
  C[T] = ((1.0 - 2 * n) / n * s1 + (1.0 - n) / n * s2) * invR2;
}


// C[1..] from C[0], times k!.
template <int P, int... T>
__device__ __forceinline__ void cart_tensor(double (&C)[Cart<P>::NT], const double (&d)[3], double invR2,
                                            std::integer_sequence<int, T...>) {
  constexpr CartTab<P> tab{};
  (cart_taylor<P, T + 1>(C, d, invR2), ...);
  ((C[T + 1] *= (int)factorial(tab.x[T + 1]) * (int)factorial(tab.y[T + 1]) * (int)factorial(tab.z[T + 1])), ...);
}

// The terms of the multipole's coefficient B on the outputs [A0, A1).
template <int P, int A0, int A1, int B>
__device__ __forceinline__ void cart_terms(double (&l)[A1 - A0], const double (&C)[Cart<P>::NT], double m) {
  constexpr CartTab<P> tab{};
  constexpr int db = tab.x[B] + tab.y[B] + tab.z[B], da = P - db;  // outputs of a lower degree than da
  constexpr int n = da * (da + 1) * (da + 2) / 6, end = n < A1 ? n : A1;
#pragma unroll
  for (int a = A0; a < end; a++)
    if (m2l_term(P, tab.x[a] + tab.y[a] + tab.z[a], db))
      l[a - A0] += m * C[CartTab<P>::idx(tab.x[a] + tab.x[B], tab.y[a] + tab.y[B], tab.z[a] + tab.z[B])];
}

template <int P, int A0, int A1, int... B2>
__device__ __forceinline__ void cart_contract(double (&l)[A1 - A0], const double (&C)[Cart<P>::NT],
                                              const double2 *__restrict__ mp, int mass,
                                              std::integer_sequence<int, B2...>) {
  (
      [&] {
        const double2 m2 = mp[B2];
        cart_terms<P, A0, A1, 2 * B2>(l, C, mass && B2 == 0 ? 1.0 : m2.x);
        cart_terms<P, A0, A1, 2 * B2 + 1>(l, C, m2.y);
      }(),
      ...);
}

// Outputs [A0, A1).
template <int P, int A0, int A1>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(P <= 6 ? 2 : 1)))
    k_m2l_cart_reg(const int *__restrict__ tgt_list, const int *__restrict__ off, const int *__restrict__ src,
                   const unsigned char *__restrict__ img, const double4 *__restrict__ cX,
                   const double *__restrict__ Mp, cplx *__restrict__ L, double cycle, int mass) {
  constexpr int NT = Cart<P>::NT;
  constexpr CartTab<P> tab{};
  constexpr int kRow = 28;  // outputs reduced at a time
  __shared__ double sh[kRow][65];
  const int c = tgt_list[blockIdx.x], lane = threadIdx.x;
  const double4 Xi = cX[c];
  const double mi0 = mass ? Mp[(size_t)c * NT] : 1.0;
  constexpr int NA = A1 - A0;
  double l[NA];
#pragma unroll
  for (int a = 0; a < NA; a++) l[a] = 0;
  const int e0 = off[c], e1 = off[c + 1];
  for (int e = e0 + lane; e < e1; e += 64) {
    const int s = src[e], im = img[e];
    const double4 Xj = cX[s];
    const double2 *mp = reinterpret_cast<const double2 *>(Mp + (size_t)s * NT);
    const double px = (im / 9 - 1) * cycle, py = ((im / 3) % 3 - 1) * cycle, pz = (im % 3 - 1) * cycle;
    const double d[3] = {Xi.x - Xj.x - px, Xi.y - Xj.y - py, Xi.z - Xj.z - pz};
    const double invR2 = 1 / (d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    // Taylor coefficients (Kernels::derivative, :187-191), then times k!.
    double C[NT];
    C[0] = (mass ? mi0 * Mp[(size_t)s * NT] : 1.0) * sqrt(invR2);
    cart_tensor<P>(C, d, invR2, std::make_integer_sequence<int, NT - 1>{});
    cart_contract<P, A0, A1>(l, C, mp, mass, std::make_integer_sequence<int, NT / 2>{});
  }
#pragma unroll
  for (int a0 = 0; a0 < NA; a0 += kRow) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRow; r++)
      if (a0 + r < NA) sh[r][lane] = l[a0 + r];
    __syncthreads();
    const int r = lane >> 1, half = 32 * (lane & 1);  // two lanes per output
    double v = 0;
    if (r < kRow)
      for (int i = 0; i < 32; i++) v += sh[r][half + i];
    v += __shfl_xor(v, 1);
    if (r < kRow && a0 + r < NA && half == 0) {
      cplx o = L[(size_t)c * NT + A0 + a0 + r];
      o.re += v;
      L[(size_t)c * NT + A0 + a0 + r] = o;
    }
  }
}

template <int P>
static void m2l_cart_reg(Handle &h, const M2LList &lst, const double4 *cX, const cplx *M, int64_t nc, cplx *L) {
  constexpr int NT = Cart<P>::NT;
  if (lst.ntgt == 0) return;
  h.cart_M.resize(nc * NT);
  hipLaunchKernelGGL(k_cart_pack, dim3(std::min(div_up(nc * NT, 256), kPackGrid)), dim3(256), 0, h.stream, M, nc * NT, h.cart_M.p);
  constexpr int A1 = P <= 6 ? NT : 35;
  hipLaunchKernelGGL((k_m2l_cart_reg<P, 0, A1>), dim3(lst.ntgt), dim3(64), 0, h.stream, lst.tgt, lst.off, lst.src,
                     lst.img, cX, h.cart_M.p, L, h.cfg.cycle, h.cfg.mass);
  if constexpr (A1 < NT)
    hipLaunchKernelGGL((k_m2l_cart_reg<P, A1, NT>), dim3(lst.ntgt), dim3(64), 0, h.stream, lst.tgt, lst.off, lst.src,
                       lst.img, cX, h.cart_M.p, L, h.cfg.cycle, h.cfg.mass);
  EXA_HIP(hipGetLastError());
}

// The pairs of `lst` on arrays of nc cells.
static void m2l_cart(Handle &h, const M2LList &lst, const double4 *cX, const cplx *M, int64_t nc, cplx *L) {
  switch (h.cfg.P) {
    case 4: m2l_cart_reg<4>(h, lst, cX, M, nc, L); break;
    case 6: m2l_cart_reg<6>(h, lst, cX, M, nc, L); break;
    case 8: m2l_cart_reg<8>(h, lst, cX, M, nc, L); break;
    default: throw Error(EXAFMM_HIP_EUNSUP, "Cartesian P must be one of 4, 6, 8");
  }
}

// ---------------------------------------------------------------------------
// traversePeriodic (traversal.h:127-185) in the Cartesian basis, by lattice
// sums as in the spherical one (periodic.hip): the derivative tensors of a
// sublevel's 702 offsets are summed once, in units of the cycle, and so are
// the 26 neighbours' powers (6 us at P = 6 and 3 levels; 1.9 ms as single
// translations, whose recurrence ran on one lane).  Both sums vanish unless all three
// indices are even (and, for the derivatives, at degree 2).
template <int P>
__global__ void __launch_bounds__(1024) k_periodic_cart_table(double *__restrict__ tab, double *__restrict__ rows) {
  constexpr int NT = Cart<P>::NT;
  const int tid = threadIdx.x;
  // One offset per lane: its tensor (or powers) in its own row, then lane
  // t adds coefficient t of every row, in offset order.
  const int x = tid / 81 - 4, y = (tid / 9) % 9 - 4, z = tid % 9 - 4;
  const int far = max(max(abs(x), abs(y)), abs(z));
  if (tid < 729 && far >= 2) {
    const double invR2 = 1.0 / (x * x + y * y + z * z);
    cart_coef<P>(rows + (size_t)tid * NT, x, y, z, invR2, sqrt(invR2));
  } else if (tid < 729 && far == 1) {
    for (int t = 0; t < NT; t++) {
      int a, b, c;
      cmi(t, a, b, c);
      rows[(size_t)tid * NT + t] = cpow(1.0, a, b, c, x, y, z);
    }
  }
  __threadfence_block();
  __syncthreads();
  if (tid >= NT) return;
  int a, b, c;
  cmi(tid, a, b, c);
  double s = 0, r = 0;
  for (int v = 0; v < 729; v++) {
    const int m = max(max(abs(v / 81 - 4), abs((v / 9) % 9 - 4)), abs(v % 9 - 4));
    if (m >= 2) s += rows[(size_t)v * NT + tid];
    if (m == 1) r += rows[(size_t)v * NT + tid];
  }
  const bool odd = (a | b | c) & 1;
  tab[tid] = odd || a + b + c == 2 ? 0.0 : s;
  tab[NT + tid] = odd ? 0.0 : r;
}

// The nsub sublevels, 8 lanes per output (they split the terms and add their
// sums in lane order); multipoles in units of the current cycle.
template <int P>
__global__ void __launch_bounds__(1024)
    k_periodic_cart_far(const cplx *__restrict__ M, cplx *__restrict__ L, const double *__restrict__ tab,
                        double cycle, int nsub, int mass) {
  constexpr int NT = Cart<P>::NT;
  static_assert(8 * NT <= 1024, "8 lanes per output");
  __shared__ double sM[NT], sN[NT], sC[NT], sR[NT];
  __shared__ unsigned char sx[NT], sy[NT], sz[NT];
  const int tid = threadIdx.x, o = tid >> 3, part = tid & 7;
  const double icycle = 1 / cycle;
  if (tid < NT) {
    int a, b, c;
    cmi(tid, a, b, c);
    sx[tid] = a;
    sy[tid] = b;
    sz[tid] = c;
    double f = 1;
    for (int i = 0; i < a + b + c; i++) f *= icycle;
    sM[tid] = M[tid].re * f;
    sC[tid] = tab[tid];
    sR[tid] = tab[NT + tid];
  }
  __syncthreads();
  const bool on = o < NT;
  const int xa = on ? sx[o] : 0, ya = on ? sy[o] : 0, za = on ? sz[o] : 0, da = xa + ya + za;
  const double mi0 = M[0].re;
  auto sum8 = [](double v) {  // of the 8 lanes of an output
    v += __shfl_xor(v, 1);
    v += __shfl_xor(v, 2);
    return v + __shfl_xor(v, 4);
  };
  double iu = icycle, l = 0, third = 1;
  for (int i = 0; i < da; i++) third *= 1.0 / 3;
  for (int lev = 0; lev < nsub; lev++, iu /= 3) {
    const double m0 = sM[0];
    double s = 0;
    if (on)
      for (int b = part; b < NT; b += 8) {
        const int xb = sx[b], yb = sy[b], zb = sz[b];
        if (m2l_term(P, da, xb + yb + zb))
          s += (mass && b == 0 ? 1.0 : sM[b]) * sC[cidx(xa + xb, ya + yb, za + zb)];
      }
    double f = mass ? mi0 * m0 * iu : iu;
    for (int i = 0; i < da; i++) f *= iu;
    l += f * sum8(s);
    if (lev == nsub - 1) break;
    // M2M of the 26 copies: sum over k <= a of R_(a - k) M_k.
    s = 0;
    if (on)
      for (int b = part; b <= o; b += 8) {
        const int xb = sx[b], yb = sy[b], zb = sz[b];
        if (xb <= xa && yb <= ya && zb <= za)
          s += (mass && b > 0 ? sM[b] * m0 : sM[b]) * sR[cidx(xa - xb, ya - yb, za - zb)];
      }
    s = sum8(s);
    if (on && part == 0) sN[o] = s;
    __syncthreads();
    const double n0 = sN[0];
    if (on && part == 0) sM[o] = third * (mass && o > 0 ? s / n0 : s);
    __syncthreads();
  }
  if (on && part == 0) {
    cplx v = L[o];
    v.re += l;
    L[o] = v;
  }
}

template <int P>
static void periodic_cart_impl(Handle &h) {
  constexpr int NT = Cart<P>::NT;
  if (h.cfg.images <= 1) return;
  if (!h.per_ready) {
    h.per_tab.resize((2 + 729) * NT);  // the sums, and the rows they are made from
    hipLaunchKernelGGL(k_periodic_cart_table<P>, dim3(1), dim3(1024), 0, h.stream, h.per_tab.p,
                       h.per_tab.p + 2 * NT);
    h.per_ready = true;
  }
  hipLaunchKernelGGL(k_periodic_cart_far<P>, dim3(1), dim3(1024), 0, h.stream, h.M.p, h.L.p, h.per_tab.p, h.cfg.cycle,
                     h.cfg.images - 1, h.cfg.mass);
  EXA_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// All leaves first (they need nothing), then the parents level by level.
template <int P>
static void p2m_cart_impl(Handle &h, hipStream_t st, int radii) {
  const int l0 = h.lvl_off[std::min(h.leaf_level, h.nlevels - 1)];  // the cells that can be leaves
  launch_ranges(h.ncells - l0, 64, [&](int c, int cnt) {
    hipLaunchKernelGGL(k_p2m_cart<P>, dim3(cnt), dim3(64), 0, st, h.lvl_cells.p + l0 + c, h.body4.p, h.cX.p, h.cRb.p,
                       h.cNChild.p, h.cBody.p, h.cNBody.p, h.M.p, h.cfg.theta, h.cfg.useRmax, radii);
  });
}

template <int P>
static void m2m_cart_impl(Handle &h, hipStream_t st, int radii) {
  for (int t = h.nlevels - 2; t >= 0; t--) {
    const int cnt = h.lvl_off[t + 1] - h.lvl_off[t];
    if (cnt == 0) continue;
    launch_ranges(cnt, 512, [&](int c, int n) {
      hipLaunchKernelGGL(k_m2m_cart<P>, dim3(n), dim3(512), 0, st, h.lvl_cells.p + h.lvl_off[t] + c, h.cX.p, h.cRb.p,
                         h.cChild.p, h.cNChild.p, h.M.p, h.cfg.theta, h.cfg.useRmax, radii);
    });
  }
  EXA_HIP(hipGetLastError());
}

template <int P>
static void downward_cart_impl(Handle &h) {
  for (int t = 0; t < h.nlevels; t++) {
    const int cnt = h.lvl_off[t + 1] - h.lvl_off[t];
    if (cnt == 0) continue;
    hipLaunchKernelGGL(k_downward_cart<P>, dim3(cnt), dim3(64), 0, h.stream, h.lvl_cells.p + h.lvl_off[t],
                       h.body4.p, h.cX.p, h.cParent.p, h.cNChild.p, h.cBody.p, h.cNBody.p, h.M.p, h.L.p, h.trg4.p,
                       t > 0 ? 1 : 0, h.cfg.mass);
  }
  EXA_HIP(hipGetLastError());
}

#define EXA_DISPATCH_CART(fn, h)                                                  \
  switch ((h).cfg.P) {                                                            \
    case 4: fn<4>(h); break;                                                      \
    case 6: fn<6>(h); break;                                                      \
    case 8: fn<8>(h); break;                                                      \
    default: throw Error(EXAFMM_HIP_EUNSUP, "Cartesian P must be one of 4, 6, 8"); \
  }

#define EXA_DISPATCH_CART_UP(fn, h, st, radii)                                    \
  switch ((h).cfg.P) {                                                            \
    case 4: fn<4>(h, st, radii); break;                                           \
    case 6: fn<6>(h, st, radii); break;                                           \
    case 8: fn<8>(h, st, radii); break;                                           \
    default: throw Error(EXAFMM_HIP_EUNSUP, "Cartesian P must be one of 4, 6, 8"); \
  }

void run_upward_cart(Handle &h) {
  EXA_DISPATCH_CART_UP(p2m_cart_impl, h, h.stream, 1);
  EXA_DISPATCH_CART_UP(m2m_cart_impl, h, h.stream, 1);
}
void run_p2m_cart(Handle &h, hipStream_t st) { EXA_DISPATCH_CART_UP(p2m_cart_impl, h, st, 0); }
void run_m2m_cart(Handle &h, hipStream_t st) { EXA_DISPATCH_CART_UP(m2m_cart_impl, h, st, 0); }
void run_downward_cart(Handle &h) { EXA_DISPATCH_CART(downward_cart_impl, h); }
void run_m2l_cart(Handle &h) {
  if (h.nm2l_tgt == 0) return;
  m2l_cart(h, M2LList{h.m2l_tgt.p, h.nm2l_tgt, h.m2l_off.p, h.m2l_src.p, h.m2l_img.p, h.nm2l}, h.cX.p, h.M.p,
           h.ncells,
           h.L.p);
}
void run_periodic_cart(Handle &h) {
  if (h.cfg.images <= 0 || h.ncells == 0) return;
  EXA_DISPATCH_CART(periodic_cart_impl, h);
}

// The Cartesian pass kernels on a caller-built cell set (per-cell operators).
template <int P>
static void upward_cart_cells_impl(Handle &h, const CellSetView &v) {
  hipLaunchKernelGGL(k_p2m_cart<P>, dim3(v.ncell), dim3(64), 0, h.stream, v.cells, v.body, v.cX, v.cRb, v.cNChild,
                     v.cBody, v.cNBody, v.M, h.cfg.theta, h.cfg.useRmax, 1);
  hipLaunchKernelGGL(k_m2m_cart<P>, dim3(v.ncell), dim3(512), 0, h.stream, v.cells, v.cX, v.cRb, v.cChild, v.cNChild,
                     v.M, h.cfg.theta, h.cfg.useRmax, 1);
}

template <int P>
static void downward_cart_cells_impl(Handle &h, const CellSetView &v) {
  hipLaunchKernelGGL(k_downward_cart<P>, dim3(v.ncell), dim3(64), 0, h.stream, v.cells, v.body, v.cX, v.cParent,
                     v.cNChild, v.cBody, v.cNBody, v.M, v.L, v.trg, v.do_l2l, h.cfg.mass);
}

#define EXA_DISPATCH_CART2(fn, h, a)                                              \
  switch ((h).cfg.P) {                                                            \
    case 4: fn<4>(h, a); break;                                                   \
    case 6: fn<6>(h, a); break;                                                   \
    case 8: fn<8>(h, a); break;                                                   \
    default: throw Error(EXAFMM_HIP_EUNSUP, "Cartesian P must be one of 4, 6, 8"); \
  }

void launch_upward_cart_cells(Handle &h, const CellSetView &v) {
  EXA_DISPATCH_CART2(upward_cart_cells_impl, h, v);
  EXA_HIP(hipGetLastError());
}
void launch_downward_cart_cells(Handle &h, const CellSetView &v) {
  EXA_DISPATCH_CART2(downward_cart_cells_impl, h, v);
  EXA_HIP(hipGetLastError());
}
void launch_m2l_cart_arrays(Handle &h, const M2LList &lst, const double4 *cX, const cplx *M, int nc, cplx *L) {
  m2l_cart(h, lst, cX, M, nc, L);
}

}  // namespace exafmm
