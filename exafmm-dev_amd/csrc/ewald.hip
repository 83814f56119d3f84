// Ewald summation of the periodic Coulomb potential and gradient (the check
// the periodic FMM is compared with).
//
// Reference: include/ewald.h:25-181 (driven by examples/ewald.cxx:91-112).
//   wave part:  W_k = sum_j q_j e^{i k.x_j s} (s = 2 pi / cycle), scaled by
//               coef exp(-|k|^2 coef2) / |k|^2, then per body
//               phi += Re(W e^{-i k.x s}),  grad -= s k Im(...)
//               over the half-space waves |k| <= ksize (initWaves);
//   real part:  per target leaf, the source tree is walked; a source cell is
//               kept while the wrapped distance of the cell centres is below
//               3 cutoff, and each kept source leaf's bodies interact with
//               the image fixed by that wrap (erfc-screened, R^2 < cutoff^2);
//   self term:  phi_i -= 2 alpha q_i / sqrt(pi).
// The results are already normalised (no q_i factor), like the reference's.
//
// Kernels: the wave sums factorise, e^{i k.x s} = e_x^l e_y^m e_z^n, so both
// transforms run on complex powers instead of one sincos per (body, wave):
// forward, a lane owns the four (+-m, +-n) waves of one (l, m) row and a tile
// of n; back, a lane owns a body and walks the rows.  The real part gives one
// wave to a target leaf (lanes select source leaves, bodies staged in LDS);
// source leaves that cannot hold a pair inside the cut-off (centre distance
// minus both cells' extents) are skipped: they contribute nothing in the
// reference either.  Every kernel writes its own slot of partial results,
// added in slot order at the end.
#include <algorithm>
#include <cmath>
#include <vector>

#include "internal.h"

namespace exafmm {

// ---------------------------------------------------------------------------
// Wave part.
//
// Rows are the pairs (l, m), l, m >= 0, of the half space's projection; for a
// row and n >= 0 the forward transform accumulates, with A = q e_x^l e_y^m,
// B = q e_x^l e_y^-m and c + i s = e_z^n, the eight sums
//   P = sum A_re c, Q = sum A_im s, R = sum A_re s, S = sum A_im c
// for A and for B: W(l, m, +-n) = (P -+ Q) + i (S +- R), so four
// multiply-adds serve two waves.
constexpr int kNT = 6;         // n values per lane (48 sums, 96 VGPRs)
constexpr int kDftBodies = 256;  // a workgroup takes a multiple of this many bodies and writes one partial

// Phase fraction of coordinate x: x / cycle less its nearest integer.
__device__ inline double phase(double x, double icycle) {
  const double f = x * icycle;
  return f - rint(f);
}

// Bodies are staged NB at a time as their powers e_x^l (times q), e_y^m and
// the workgroup's tile of e_z^n; the 4 waves take every fourth body and add
// their sums through LDS in wave order.  Bound by FP64 issue (56 operations
// per lane and body; the powers cost one sincospi per axis and body).  32768
// bodies, ksize 11: 36 us, 236 us with a sincos per (body, wave) and one wave
// vector per workgroup of 256 lanes.
template <int NB>
__global__ void __launch_bounds__(256)
    k_ewald_dft(const double4 *__restrict__ body, int n, const int2 *__restrict__ rows, int nrows, int K,
                double icycle, int per, double *__restrict__ part) {
  extern __shared__ double2 sh[];  // [2 (K + 1) + kNT][NB + 1]
  constexpr int LD = NB + 1;
  double2 *sx = sh, *sy = sh + (K + 1) * LD, *sz = sh + 2 * (K + 1) * LD;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row = blockIdx.y * 64 + lane, n0 = blockIdx.z * kNT;
  const int2 lm = rows[min(row, nrows - 1)];
  double a[8][kNT];
#pragma unroll
  for (int k = 0; k < 8; k++)
#pragma unroll
    for (int j = 0; j < kNT; j++) a[k][j] = 0;
  const int b0 = blockIdx.x * per, b1 = min(n, b0 + per);
  for (int base = b0; base < b1; base += NB) {
    const int cnt = min(NB, b1 - base);
    __syncthreads();
    for (int i = tid; i < 3 * NB; i += 256) {
      const int axis = i / NB, b = i % NB;
      if (b >= cnt) continue;
      const double4 x = body[base + b];
      const double f = phase(axis == 0 ? x.x : axis == 1 ? x.y : x.z, icycle);
      double s1, c1;
      sincospi(2 * f, &s1, &c1);
      double2 *out = (axis == 0 ? sx : axis == 1 ? sy : sz) + b;
      double2 v = make_double2(axis == 0 ? x.w : 1.0, 0);
      int cntp = K + 1;
      if (axis == 2) {
        const double g = n0 * f;
        sincospi(2 * (g - rint(g)), &v.y, &v.x);
        cntp = kNT;
      }
      for (int p = 0; p < cntp; p++) {
        out[p * LD] = v;
        v = make_double2(v.x * c1 - v.y * s1, v.x * s1 + v.y * c1);
      }
    }
    __syncthreads();
    for (int b = wave; b < cnt; b += 4) {
      const double2 ex = sx[lm.x * LD + b], ey = sy[lm.y * LD + b];
      const double rr = ex.x * ey.x, ii = ex.y * ey.y, ri = ex.x * ey.y, ir = ex.y * ey.x;
      const double Ar = rr - ii, Ai = ri + ir, Br = rr + ii, Bi = ir - ri;
#pragma unroll
      for (int j = 0; j < kNT; j++) {
        const double2 z = sz[j * LD + b];
        a[0][j] = fma(Ar, z.x, a[0][j]);
        a[1][j] = fma(Ai, z.y, a[1][j]);
        a[2][j] = fma(Ar, z.y, a[2][j]);
        a[3][j] = fma(Ai, z.x, a[3][j]);
        a[4][j] = fma(Br, z.x, a[4][j]);
        a[5][j] = fma(Bi, z.y, a[5][j]);
        a[6][j] = fma(Br, z.y, a[6][j]);
        a[7][j] = fma(Bi, z.x, a[7][j]);
      }
    }
  }
  // The four waves' sums in wave order: wave 0 starts, the others add.
  double *red = reinterpret_cast<double *>(sh);  // [8 kNT][64]
  for (int w = 0; w < 4; w++) {
    __syncthreads();
    if (wave == w)
#pragma unroll
      for (int k = 0; k < 8; k++)
#pragma unroll
        for (int j = 0; j < kNT; j++) {
          const int i = (k * kNT + j) * 64 + lane;
          red[i] = w ? red[i] + a[k][j] : a[k][j];
        }
  }
  __syncthreads();
  // part[group][z][k][j][row], rows padded to whole tiles of 64.
  const size_t nrp = (size_t)gridDim.y * 64;
  double *pp = part + (((size_t)blockIdx.x * gridDim.z + blockIdx.z) * 8 * kNT) * nrp + blockIdx.y * 64;
  for (int i = tid; i < 8 * kNT * 64; i += 256) pp[(size_t)(i >> 6) * nrp + (i & 63)] = red[i];
}

// Sums the groups' partials and writes what the way back reads: for each
// signed row (l, m) and n >= 0, U = W(n) + W(-n) and V = i (W(-n) - W(n)),
// scaled by coef exp(-K2 coef2) / K2; zero outside the half space or the
// sphere.  idx[row] = the signed rows of (l, m) and (l, -m), -1 for none.
__global__ void __launch_bounds__(256)
    k_ewald_waves(const double *__restrict__ part, int groups, int nz, int nrp, const int2 *__restrict__ rows,
                  int nrows, const int2 *__restrict__ idx, int K, double coef, double coef2, double4 *__restrict__ UV) {
  __shared__ double sw[8][33];
  // 32 (row, n) entries per workgroup, 8 sums each.
  const int e = blockIdx.x * 32 + (threadIdx.x & 31), k = threadIdx.x >> 5;
  const int row = e % nrp, n = e / nrp;
  const bool on = row < nrows && n <= K;
  double v = 0;
  if (on) {
    const double *p = part + ((size_t)(n / kNT) * 8 * kNT + k * kNT + n % kNT) * nrp + row;
#pragma unroll 16
    for (int g = 0; g < groups; g++) v += p[(size_t)g * nz * 8 * kNT * nrp];
  }
  sw[k][threadIdx.x & 31] = v;
  __syncthreads();
  if (!on || k >= 2) return;  // k = 0: (l, m), k = 1: (l, -m)
  const int2 lm = rows[row];
  const int out = k == 0 ? idx[row].x : idx[row].y;
  if (out < 0) return;
  const int i = threadIdx.x & 31, o = 4 * k;
  const double P = sw[o][i], Q = sw[o + 1][i], R = sw[o + 2][i], S = sw[o + 3][i];
  const int k2 = lm.x * lm.x + lm.y * lm.y + n * n;
  const bool in = k2 > 0 && k2 <= K * K;
  const double f = in ? coef * exp(-(double)k2 * coef2) / (double)k2 : 0.0;
  double4 uv;
  if (n == 0)  // the one wave (l, m, 0)
    uv = make_double4(f * P, f * S, 0, 0);
  else if (lm.x == 0 && lm.y == 0)  // only n > 0 of the row (0, 0): W = (P - Q) + i (S + R), W(-n) = 0
    uv = make_double4(f * (P - Q), f * (S + R), f * (S + R), -f * (P - Q));
  else
    uv = make_double4(2 * f * P, 2 * f * S, 2 * f * R, 2 * f * Q);
  UV[(size_t)out * (K + 1) + n] = uv;
}

// Back transform: lane = body, the signed rows split over blockIdx.y.  Per
// row Z = sum_n U c + V s and Y = sum_n n (V c - U s); with E = e_x^l e_y^m,
// phi += Re(Z E*), d_x += l Im(Z E*), d_y += m Im(Z E*), d_z += Re(Y E*).
// The table entries are the same for all lanes (scalar loads); bound by FP64
// issue: 14 operations per row entry (50 us at 32768 bodies, ksize 11; 655 us
// with a sincos per wave).
__global__ void __launch_bounds__(256)
    k_ewald_idft(const double4 *__restrict__ body, int n, const int4 *__restrict__ srows, int nsrows, int K,
                 const double4 *__restrict__ UV, double icycle, double scale, double4 *__restrict__ out) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  const double4 x = b < n ? body[b] : make_double4(0, 0, 0, 0);
  const double fx = phase(x.x, icycle), fy = phase(x.y, icycle), fz = phase(x.z, icycle);
  double c1, s1, cy, sy;
  sincospi(2 * fz, &s1, &c1);
  sincospi(2 * fy, &sy, &cy);
  const int r0 = (int)((int64_t)nsrows * blockIdx.y / gridDim.y);
  const int r1 = (int)((int64_t)nsrows * (blockIdx.y + 1) / gridDim.y);
  double t0 = 0, t1 = 0, t2 = 0, t3 = 0, er = 1, ei = 0;
  int lp = -1, mp = 0;
  for (int r = r0; r < r1; r++) {
    const int4 q = srows[r];  // l, m, largest n
    if (q.x != lp || q.y != mp + 1) {  // a new run of m: E from its phase
      const double gx = q.x * fx, gy = q.y * fy;
      const double g = (gx - rint(gx)) + (gy - rint(gy));
      sincospi(2 * g, &ei, &er);
    } else {
      const double t = er * cy - ei * sy;
      ei = er * sy + ei * cy;
      er = t;
    }
    lp = q.x;
    mp = q.y;
    const double4 *uv = UV + (size_t)r * (K + 1);
    double c = 1, s = 0, Zr = 0, Zi = 0, Yr = 0, Yi = 0;
    for (int k = 0; k <= q.z; k++) {
      const double4 w = uv[k];
      Zr = fma(w.x, c, Zr);
      Zi = fma(w.y, c, Zi);
      Zr = fma(w.z, s, Zr);
      Zi = fma(w.w, s, Zi);
      const double kd = k;
      Yr = fma(kd, fma(w.z, c, -(w.x * s)), Yr);
      Yi = fma(kd, fma(w.w, c, -(w.y * s)), Yi);
      const double t = c * c1 - s * s1;
      s = c * s1 + s * c1;
      c = t;
    }
    const double im = Zi * er - Zr * ei;
    t0 += Zr * er + Zi * ei;
    t1 = fma((double)q.x, im, t1);
    t2 = fma((double)q.y, im, t2);
    t3 += Yr * er + Yi * ei;
  }
  if (b < n) out[(size_t)blockIdx.y * n + b] = make_double4(t0, t1 * scale, t2 * scale, t3 * scale);
}

// ---------------------------------------------------------------------------
// Real part.

__device__ inline double wrap1(double v, double w) {  // vec.h:193-205
  if (v < -w / 2) v += w;
  if (v > w / 2) v -= w;
  return v;
}

// a b + c with c in scalar registers.  The compiler's own choice for a
// polynomial is v_fmac_f64, which overwrites its addend: every step then
// copies its coefficient into vector registers first (34 of 128 instructions
// of a pair, and 36 pairs of VGPRs that hold the coefficients).
__device__ inline double fma_s(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}

// e^-s for s >= 0: 2^k e^r, |r| <= ln 2 / 2, degree-11 interpolation of e^r
// at Chebyshev nodes (4e-18).
__device__ inline double exp_neg(double s) {
  constexpr double c[12] = {
    1.0, 1.0, 0.5000000000000019, 0.1666666666666668, 0.04166666666648795, 0.008333333333319589,
    0.0013888888952352863, 0.00019841269890076403, 2.4801485441561313e-05, 2.755724088722987e-06,
    2.763265472252779e-07, 2.511004920481866e-08};
  s = fmin(s, 1500.0);  // 0 from here on
  const double k = rint(s * -1.4426950408889634);
  double r = fma(k, -0.6931471805599453, -s);
  r = fma(k, -2.3190468138462996e-17, r);
  double p = c[11];
#pragma unroll
  for (int i = 10; i >= 0; i--) p = i < 2 ? fma(p, r, c[i]) : fma_s(p, r, c[i]);  // c[0] = c[1] = 1: inline
  return ldexp(p, (int)k);
}

// e^{x^2} erfc(x) for x >= 0: (x + 3) e^{x^2} erfc(x) is smooth from 3 at 0
// to 1/sqrt(pi) at infinity; degree-23 interpolation at Chebyshev nodes in
// t = (x - 3) / (x + 3) (2e-17; evaluated in FP64 2e-16 rms, 6e-16 at most,
// over [0, 6]).
__device__ inline double erfc_scaled(double x) {
  constexpr double c[24] = {
    1.0740069070883396, -0.8833944531698836, 0.5902283571041085, -0.31046726190056667, 0.11952776128697859,
    -0.026827234624480615, -0.0012124166215147798, 0.0030340620011959822, -0.0005483097452477533,
    -0.0002767778482009659, 0.00010756178250002073, 3.03981905221208e-05, -1.7471605752302332e-05,
    -4.749391032132141e-06, 2.7678112255272805e-06, 9.994379361081014e-07, -4.117597591893759e-07,
    -2.3454670002624263e-07, 5.001320184291237e-08, 5.166814761898455e-08, -3.5913611171610945e-09,
    -8.887844891516949e-09, 1.1159123899250243e-11, 8.447852784322954e-10};
  const double d = x + 3;
  double u = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, u, 1.0);
  u = fma(u, fma(e, e, e), u);
  const double t = fma(-6.0, u, 1.0);
  double p = c[23];
#pragma unroll
  for (int i = 22; i >= 0; i--) p = fma_s(p, t, c[i]);
  return p * u;
}

constexpr int kEwStage = 128;

// One wave per target leaf (blockIdx.x) and share of the source cells
// (blockIdx.y: every gridDim.y-th chunk of 64 cells).  A pass takes T = a
// power of two targets, replicated over 64 / T lane groups that split the
// staged bodies; a leaf whose size leaves more than a quarter of T idle takes
// a second, smaller pass.  Lanes select the source leaves of a chunk; their
// bodies within the cut-off of the targets' box fill the stage in parallel
// through a slot map (without that test 23% of the pairs evaluated were out of
// range, with it 15%; 2.31 ms and 2.28).  A pair is about 65
// FP64 operations (erfc and exp as polynomials with one reciprocal square
// root and one reciprocal, instead of the library's erfc, exp, sqrt and
// divide), which bounds the kernel: about 90 issued with the tests and LDS
// reads.  32768 bodies, cut-off half the box: 2.28 ms (3.0 ms with the
// coefficients in VGPRs), 8.47 ms with the library functions, at least 16
// lanes per leaf and leaves staged one after another.
__global__ void __launch_bounds__(64)
    k_ewald_real(int ncells, const double4 *__restrict__ cX, const double *__restrict__ cRb,
                 const int *__restrict__ cParent, const int *__restrict__ cNChild, const int *__restrict__ cBody,
                 const int *__restrict__ cNBody, const double4 *__restrict__ body, int n, double4 *__restrict__ out,
                 double alpha, double cutoff, double cycle, int walk) {
  __shared__ double4 sb[kEwStage];
  __shared__ double4 sshift[64];  // image shift; w: unused
  __shared__ int sfrom[64];       // first body less the leaf's first slot
  __shared__ unsigned char smap[kEwStage];
  const int c = blockIdx.x;
  if (cNChild[c] != 0 || cNBody[c] == 0) return;
  const int lane = threadIdx.x;
  const int tb0 = cBody[c], tn = cNBody[c];
  const double4 Xi = cX[c];
  const double Rbi = cRb[c];
  const double cut2 = cutoff * cutoff, a3 = alpha * alpha * alpha, a2 = alpha * alpha;
  const double k2sqrtpi = 1.1283791670955126;  // 2 / sqrt(pi)
  out += (size_t)blockIdx.y * n;
  for (int tbase = 0, T; tbase < tn; tbase += T) {
    const int rem = tn - tbase;
    T = 8;
    while (T < rem && T < 64) T *= 2;
    if (T > 8 && 4 * rem <= 3 * T) T /= 2;
    const int G = 64 / T, g = lane / T, ti = lane & (T - 1);
    const bool active = ti < rem;
    const double4 xi = active ? body[tb0 + tbase + ti] : make_double4(0, 0, 0, 0);
    double pot = 0, gx = 0, gy = 0, gz = 0;
    // The targets' box.
    double lo[3], hi[3];
    for (int d = 0; d < 3; d++) {
      const double x = d == 0 ? xi.x : d == 1 ? xi.y : xi.z;
      lo[d] = active ? x : 1e300;
      hi[d] = active ? x : -1e300;
    }
    for (int w = 32; w >= 1; w >>= 1)
      for (int d = 0; d < 3; d++) {
        lo[d] = fmin(lo[d], __shfl_xor(lo[d], w));
        hi[d] = fmax(hi[d], __shfl_xor(hi[d], w));
      }
    for (int base = 64 * blockIdx.y; base < ncells; base += 64 * gridDim.y) {
      // Lanes select the source leaves of this chunk and their images.
      const int cj = base + lane;
      bool keep = false;
      double px = 0, py = 0, pz = 0;
      int sb0 = 0, sn = 0;
      if (cj < ncells && cNChild[cj] == 0 && cNBody[cj] > 0) {
        const double4 Xj = cX[cj];
        const double dx = wrap1(Xi.x - Xj.x, cycle), dy = wrap1(Xi.y - Xj.y, cycle), dz = wrap1(Xi.z - Xj.z, cycle);
        px = Xi.x - Xj.x - dx;
        py = Xi.y - Xj.y - dy;
        pz = Xi.z - Xj.z - dz;
        const double R = sqrt(dx * dx + dy * dy + dz * dz);
        keep = R < 3 * cutoff;
        // Body extents: a body lies within sqrt(3) Rb of its cell centre
        // (1% margin for the rounding of the cell geometry).
        keep = keep && (R - 1.01 * 1.7320508075688772 * (Rbi + cRb[cj]) < cutoff);
        // Every ancestor must pass the 3 cutoff test too (depth-bounded walk).
        for (int a = cj, d = 0; keep && walk && a != 0 && d < 64; d++) {
          a = cParent[a];
          const double4 Xa = cX[a];
          const double ex = wrap1(Xi.x - Xa.x, cycle), ey = wrap1(Xi.y - Xa.y, cycle), ez = wrap1(Xi.z - Xa.z, cycle);
          keep = sqrt(ex * ex + ey * ey + ez * ez) < 3 * cutoff;
        }
        if (keep) {
          sb0 = cBody[cj];
          sn = cNBody[cj];
        }
      }
      if (!__ballot(keep)) continue;
      // Slots of the kept leaves: an inclusive scan over the lanes.
      int end = sn;
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(end, d);
        if (lane >= d) end += o;
      }
      const int first = end - sn, total = __shfl(end, 63);
      __syncthreads();  // the last stage's bodies and maps are done with
      sshift[lane] = make_double4(px, py, pz, 0);
      sfrom[lane] = sb0 - first;
      for (int w0 = 0; w0 < total; w0 += kEwStage) {
        const int cnt = min(kEwStage, total - w0);
        __syncthreads();
        for (int k = max(first, w0); k < min(end, w0 + kEwStage); k++) smap[k - w0] = (unsigned char)lane;
        __syncthreads();
        int nst = 0;  // staged bodies: those within the cut-off of the targets' box
        for (int k0 = 0; k0 < cnt; k0 += 64) {
          const int k = k0 + lane;
          bool in = k < cnt;
          const int l = smap[in ? k : 0];
          double4 v = body[sfrom[l] + w0 + (in ? k : 0)];
          const double4 p = sshift[l];
          v.x += p.x;
          v.y += p.y;
          v.z += p.z;
          const double dx = fmax(fmax(lo[0] - v.x, v.x - hi[0]), 0.0), dy = fmax(fmax(lo[1] - v.y, v.y - hi[1]), 0.0),
                       dz = fmax(fmax(lo[2] - v.z, v.z - hi[2]), 0.0);
          in = in && dx * dx + dy * dy + dz * dz < cut2 * (1 + 1e-9);
          const unsigned long long m = __ballot(in);
          if (in) sb[nst + (int)__popcll(m & ((1ull << lane) - 1))] = v;
          nst += (int)__popcll(m);
        }
        __syncthreads();
        for (int k = g; k < nst; k += G) {
          const double4 xj = sb[k];
          const double dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
          const double R2 = dx * dx + dy * dy + dz * dz;
          if (active && 0 < R2 && R2 < cut2) {
            const double s = R2 * a2;
            double ix = __builtin_amdgcn_rsq(s);  // 1 / (alpha R): estimate and one quadratic Newton step
            const double e = fma(-s * ix, ix, 1.0);
            ix = fma(ix * e, fma(0.375, e, 0.5), ix);
            const double E = exp_neg(s);
            const double ex = E * erfc_scaled(s * ix) * ix;  // erfc(alpha R) / (alpha R)
            const double dtmp = xj.w * a3 * (ix * ix) * fma(k2sqrtpi, E, ex);
            pot = fma(xj.w * alpha, ex, pot);
            gx = fma(-dx, dtmp, gx);
            gy = fma(-dy, dtmp, gy);
            gz = fma(-dz, dtmp, gz);
          }
        }
      }
    }
    // The lane groups' sums, in group order.
    __syncthreads();
    sb[lane] = make_double4(pot, gx, gy, gz);
    __syncthreads();
    if (g == 0 && active) {
      double4 s = sb[ti];
      for (int gg = 1; gg < G; gg++) {
        const double4 o = sb[gg * T + ti];
        s.x += o.x;
        s.y += o.y;
        s.z += o.z;
        s.w += o.w;
      }
      out[tb0 + tbase + ti] = s;
    }
    __syncthreads();
  }
}

// dst (caller order) += the slots of partial results (tree order), in slot
// order, and the self term -2 alpha q / sqrt(pi) if asked for.
__global__ void k_ewald_finish(const double4 *__restrict__ slots, int nslots, const double4 *__restrict__ body,
                               const int *__restrict__ bidx, int n, int self, double alpha,
                               double4 *__restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double4 s = make_double4(0, 0, 0, 0);
  for (int k = 0; k < nslots; k++) {
    const double4 v = slots[(size_t)k * n + i];
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  if (self) s.x -= 1.1283791670955126 * body[i].w * alpha;  // M_2_SQRTPI q alpha
  double4 d = dst[bidx[i]];
  d.x += s.x;
  d.y += s.y;
  d.z += s.z;
  d.w += s.w;
  dst[bidx[i]] = d;
}

// The rows of the half space of initWaves (ewald.h:64-90: l > 0, or l = 0 and
// m > 0, or l = m = 0 and n > 0, with l^2 + m^2 + n^2 <= ksize^2).
struct WaveRows {
  std::vector<int> rows;   // (l, m) with m >= 0
  std::vector<int> idx;    // their signed rows of m and -m (-1: none)
  std::vector<int> srows;  // signed rows (l, m, largest n, 0), m ascending
};

static WaveRows wave_rows(int ksize) {
  WaveRows w;
  const int K = ksize;
  for (int l = 0; l <= K; l++) {
    int mmax = 0;
    while (l * l + (mmax + 1) * (mmax + 1) <= K * K) mmax++;
    const int mlo = l == 0 ? 0 : -mmax;
    const int s0 = (int)w.srows.size() / 4;
    for (int m = mlo; m <= mmax; m++) {
      int nmax = 0;
      while (l * l + m * m + (nmax + 1) * (nmax + 1) <= K * K) nmax++;
      for (int v : {l, m, nmax, 0}) w.srows.push_back(v);
    }
    for (int m = 0; m <= mmax; m++) {
      w.rows.push_back(l);
      w.rows.push_back(m);
      w.idx.push_back(s0 + m - mlo);
      w.idx.push_back(m > 0 && l > 0 ? s0 - m - mlo : -1);
    }
  }
  return w;
}

// Wave part into `nslot` slots of out (n entries each).
static void wave_part(Handle &h, int K, double alpha, double sigma, double cycle, double4 *out, int nslot) {
  const int n = h.n;
  if (h.ew_ksize != K) {
    const WaveRows w = wave_rows(K);
    std::vector<int> blob(w.srows);
    blob.insert(blob.end(), w.rows.begin(), w.rows.end());
    blob.insert(blob.end(), w.idx.begin(), w.idx.end());
    h.ew_ksize = 0;
    h.ew_rows.resize(blob.size());
    EXA_HIP(hipMemcpyAsync(h.ew_rows.p, blob.data(), blob.size() * sizeof(int), hipMemcpyHostToDevice, h.stream));
    EXA_HIP(hipStreamSynchronize(h.stream));  // blob is freed here
    h.ew_ksize = K;
    h.ew_nrows = (int)w.rows.size() / 2;
    h.ew_nsrows = (int)w.srows.size() / 4;
  }
  const int nrows = h.ew_nrows, nsrows = h.ew_nsrows;
  const int4 *srows = reinterpret_cast<const int4 *>(h.ew_rows.p);
  const int2 *rows = reinterpret_cast<const int2 *>(srows + nsrows), *idx = rows + nrows;
  const int ny = div_up(nrows, 64), nz = div_up(K + 1, kNT), nrp = 64 * ny;
  // About 1024 workgroups at most, so that the partials stay small; few bodies
  // and waves take one round of the stage per workgroup, to fill more CUs (wave
  // part of 1728 bodies, ksize 2, 86 -> 69 us; from 64 workgroups on the partials
  // cost what it gains).
  const int least = (int64_t)ny * nz * div_up(n, kDftBodies) < 64 ? kDftBodies / 4 : kDftBodies;
  const int per = least * div_up(n, (int64_t)least * std::max(1, 1024 / (ny * nz)));
  const int groups = div_up(n, per);
  const size_t npart = (size_t)groups * nz * 8 * kNT * nrp;
  h.ew_waves.resize(npart + (size_t)nsrows * (K + 1) * 4);
  double *part = h.ew_waves.p;
  double4 *UV = reinterpret_cast<double4 *>(part + npart);
  const double scale = 2 * M_PI / cycle;
  const double coef = .5 / M_PI / M_PI / sigma / cycle;
  const double coef2 = scale * scale / (4 * alpha * alpha);
  // As many bodies at a time as 64 KB of powers hold (64 up to ksize 27).
  auto lds = [&](int nb) {
    return std::max<size_t>((size_t)(2 * (K + 1) + kNT) * (nb + 1) * sizeof(double2), 8 * kNT * 64 * sizeof(double));
  };
  auto dft = [&](auto kernel, int nb) {
    hipLaunchKernelGGL(kernel, dim3(groups, ny, nz), dim3(256), lds(nb), h.stream, h.body4.p, n, rows, nrows, K,
                       1 / cycle, per, part);
  };
  constexpr size_t kLds = 65536;
  if (lds(64) <= kLds)
    dft(k_ewald_dft<64>, 64);
  else if (lds(16) <= kLds)
    dft(k_ewald_dft<16>, 16);
  else if (lds(4) <= kLds)
    dft(k_ewald_dft<4>, 4);
  else if (lds(1) <= kLds)
    dft(k_ewald_dft<1>, 1);
  else
    throw Error(EXAFMM_HIP_EUNSUP, "ewald: ksize too large");
  hipLaunchKernelGGL(k_ewald_waves, dim3(div_up((int64_t)nrp * nz * kNT, 32)), dim3(256), 0, h.stream, part, groups,
                     nz, nrp, rows, nrows, idx, K, coef, coef2, UV);
  hipLaunchKernelGGL(k_ewald_idft, dim3(div_up(n, 256), nslot), dim3(256), 0, h.stream, h.body4.p, n, srows, nsrows, K,
                     UV, 1 / cycle, scale, out);
}

void run_ewald(Handle &h, int ksize, double alpha, double sigma, double cutoff, double cycle, int parts,
               double *trg) {
  const int n = h.n;
  // Slots: the row splits of the back transform (enough workgroups to fill
  // the chip), then the source splits of the real part.
  int nwave = 0, nreal = 0;
  if ((parts & 1) && ksize > 0) {
    nwave = std::min(16, std::max(1, div_up((int64_t)4096 * 64, n)));
    if (ksize < 4) nwave = std::min(nwave, ksize == 1 ? 3 : ksize == 2 ? 7 : 15);  // no more than rows
  }
  if (parts & 2) {
    const int chunks = div_up(h.ncells, 64);
    nreal = std::max(1, std::min(chunks, std::min(64, 8192 / h.ncells)));
  }
  h.ew_trg.resize((size_t)std::max(1, nwave + nreal) * n);
  if (nwave) wave_part(h, ksize, alpha, sigma, cycle, h.ew_trg.p, nwave);  // wavePart, ewald.h:166-181
  if (parts & 2) {  // realPart, ewald.h:145-156
    // The ancestor walk can be skipped when 3 cutoff exceeds every wrapped
    // centre distance: a wrapped coordinate difference is at most
    // max(cycle / 2, extent - cycle) for bodies spanning `extent`.
    sync_bounds(h);
    double ext = 0;
    for (int d = 0; d < 3; d++) ext = std::max(ext, h.xmax[d] - h.xmin[d]);
    const double bound = std::sqrt(3.0) * std::max(0.5 * cycle, ext - cycle);
    const int walk = 3 * cutoff > bound * 1.000001 ? 0 : 1;
    hipLaunchKernelGGL(k_ewald_real, dim3(h.ncells, nreal), dim3(64), 0, h.stream, h.ncells, h.cX.p, h.cRb.p,
                       h.cParent.p, h.cNChild.p, h.cBody.p, h.cNBody.p, h.body4.p, n,
                       h.ew_trg.p + (size_t)nwave * n, alpha, cutoff, cycle, walk);
  }
  EXA_HIP(hipGetLastError());
  // Accumulate into the caller's array (caller order); selfTerm, ewald.h:159-163.
  h.out4.resize(n);
  EXA_HIP(hipMemcpyAsync(h.out4.p, trg, n * sizeof(double4), hipMemcpyHostToDevice, h.stream));
  hipLaunchKernelGGL(k_ewald_finish, dim3(div_up(n, 256)), dim3(256), 0, h.stream, h.ew_trg.p, nwave + nreal,
                     h.body4.p, h.bidx.p, n, (parts & 4) ? 1 : 0, alpha, h.out4.p);
  EXA_HIP(hipGetLastError());
  EXA_HIP(hipMemcpyAsync(trg, h.out4.p, n * sizeof(double4), hipMemcpyDeviceToHost, h.stream));
  EXA_HIP(hipStreamSynchronize(h.stream));
}

}  // namespace exafmm
