// Periodic far field and the dipole correction.
//
// traversePeriodic (include/traversal.h:127-185): the 27 nearest images of
// the tree are part of the interaction lists; beyond them, for each of
// images-1 sublevels, the root's local expansion receives M2L from the 26 x 27
// images at offsets (3 i + c) cycle, i != 0, of a periodic parent whose
// multipole starts as the root's; the parent's multipole then becomes the M2M
// of its 26 neighbour copies (the centre copy is not a child of the periodic
// parent in the reference, NCHILD = 26), and cycle triples.  MASS mode
// denormalises around the M2M and finally divides the root's L by M0.
//
// Work: every sublevel's 702 translations read one multipole and add into one
// cell, so they are one translation by the lattice sum of the harmonics, and
// the M2M of the 26 copies one translation by their sum.  The offsets are
// integer vectors times the sublevel's cycle and the harmonics homogeneous:
// the two sums over the integer vectors depend on the order alone and are
// kept by the handle, and one workgroup walks the sublevels (10 us at P = 10,
// 3 levels; 750 us as 702 translations per sublevel on 26 workgroups).  By
// the cube's symmetry the sums are real and vanish unless n is even, not 2,
// and m a multiple of 4.
//
// getDipole / dipoleCorrection (include/up_down_pass.h:151-168).
#include <cmath>

#include "harmonics.h"
#include "internal.h"

namespace exafmm {

// Sum of the values that the 64 k lanes of a workgroup hold, in a fixed
// order (sh: blockDim.x doubles; every lane gets it).
__device__ inline double block_sum(double v, double *sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  return sh[0];
}

// Lattice sums of coefficient t = blockIdx.x: tab[t] = sum of S_n^m over the
// integer vectors 3 i + c (i, c in {-1, 0, 1}^3, i != 0), tab[NT + t] = sum of
// R_n^m over the 26 neighbour vectors.
template <int P>
__global__ void __launch_bounds__(256) k_periodic_table(double *__restrict__ tab) {
  constexpr int NT = Expn<P>::NT;
  __shared__ double sh[256];
  int n, m;
  coef_nm(blockIdx.x, n, m);
  double s = 0, r = 0;
  for (int v = threadIdx.x; v < 729; v += 256) {
    const int x = v / 81 - 4, y = (v / 9) % 9 - 4, z = v % 9 - 4;
    const int far = max(max(abs(x), abs(y)), abs(z));
    if (far == 0) continue;
    const Geom g = make_geom(x, y, z);
    double re, im;
    if (far >= 2) {
      singular_nm(n, m, g, re, im);
      s += re;
    } else {
      regular_nm(n, m, g, re, im);
      r += re;
    }
  }
  const bool zero = (n & 1) || (m & 3) || n == 2;
  s = block_sum(s, sh);
  __syncthreads();
  r = block_sum(r, sh);
  if (threadIdx.x == 0) {
    tab[blockIdx.x] = zero ? 0.0 : s;
    tab[NT + blockIdx.x] = zero ? 0.0 : r;
  }
}

// The nsub sublevels.  Multipoles are kept in units of the current cycle
// (M_n cycle^-n), so both sums apply as they are.  Work items are (output
// (j, k), n); an output's items are added in n order.
template <int P>
__global__ void __launch_bounds__(512)
    k_periodic_far(const cplx *__restrict__ M, cplx *__restrict__ L, const double *__restrict__ tab, double cycle,
                   int nsub, int mass) {
  constexpr int NT = Expn<P>::NT;
  __shared__ cplx sM[NT], sL[NT], sp[NT * P];
  __shared__ double sS[NT], sR[NT];
  const int tid = threadIdx.x;
  const double icycle = 1 / cycle;
  for (int t = tid; t < NT; t += 512) {
    int n, m;
    coef_nm(t, n, m);
    double f = 1;
    for (int i = 0; i < n; i++) f *= icycle;
    sM[t] = {M[t].re * f, M[t].im * f};
    sL[t] = {0, 0};
    sS[t] = tab[t];
    sR[t] = tab[NT + t];
  }
  const double mi0 = M[0].re;
  double iu = icycle;  // 1 / cycle of the sublevel
  __syncthreads();
  for (int lev = 0; lev < nsub; lev++, iu /= 3) {
    // M2L (LaplaceSphericalCPU.cxx:149-191; MASS: :157-172, where the source's
    // M_0 counts as 1 and the translation is scaled by both M_0).
    const double m0 = sM[0].re;
    for (int i = tid; i < NT * P; i += 512) {
      const int t = i / P, n = i % P;
      int j, k;
      coef_nm(t, j, k);
      const int a = j + n;
      double lr = 0, li = 0;
      if (a < P && !(a & 1)) {
        for (int m = -n + ((n + k) & 3); m <= n; m += 4) {  // m = k mod 4
          const double y = sS[tri(a) + abs(m - k)];
          cplx v = sM[tri(n) + abs(m)];
          if (mass && n == 0) v = {1, 0};
          if (m < 0) {  // conj(M_n^-m)
            lr += v.re * y;
            li -= v.im * y;
          } else {
            const double f = (((k - m) * (k < m) + m) & 1) ? -y : y;
            lr += f * v.re;
            li += f * v.im;
          }
        }
      }
      sp[i] = {lr, li};
    }
    __syncthreads();
    for (int t = tid; t < NT; t += 512) {
      int j, k;
      coef_nm(t, j, k);
      double f = ((j & 1) ? -iu : iu) * (mass ? mi0 * m0 : 1.0);
      for (int i = 0; i < j; i++) f *= iu;
      double lr = 0, li = 0;
      for (int n = 0; n < P - j; n++) {
        lr += sp[t * P + n].re;
        li += sp[t * P + n].im;
      }
      sL[t].re += f * lr;
      sL[t].im += f * li;
    }
    __syncthreads();
    if (lev == nsub - 1) break;
    if (mass) {  // traversal.h:155-156
      for (int t = tid; t < NT; t += 512)
        if (t > 0) {
          sM[t].re *= m0;
          sM[t].im *= m0;
        }
      __syncthreads();
    }
    // M2M of the 26 copies (LaplaceSphericalCPU.cxx:120-147 with the real,
    // even sums), then the next sublevel's units.
    for (int i = tid; i < NT * P; i += 512) {
      const int t = i / P, n = i % P;
      int j, k;
      coef_nm(t, j, k);
      double lr = 0, li = 0;
      if (n <= j && !(n & 1)) {
        for (int m = -(n & ~3); m <= n; m += 4) {
          const double y = sR[tri(n) + abs(m)];
          if (m < k && m >= -j + k + n) {
            const cplx v = sM[tri(j - n) + k - m];
            lr += v.re * y;
            li += v.im * y;
          } else if (m >= k && m <= j + k - n) {
            const cplx v = sM[tri(j - n) + m - k];
            const double f = (k & 1) ? -y : y;
            lr += f * v.re;
            li -= f * v.im;
          }
        }
      }
      sp[i] = {lr, li};
    }
    __syncthreads();
    const double n0 = sp[0].re;  // of t = 0 (n = 0 alone)
    for (int t = tid; t < NT; t += 512) {
      int j, k;
      coef_nm(t, j, k);
      double f = mass && t > 0 ? 1 / n0 : 1.0;  // traversal.h:176-178
      for (int i = 0; i < j; i++) f *= 1.0 / 3;
      double lr = 0, li = 0;
      for (int n = 0; n <= j; n++) {
        lr += sp[t * P + n].re;
        li += sp[t * P + n].im;
      }
      sM[t] = {f * lr, f * li};
    }
    __syncthreads();
  }
  for (int t = tid; t < NT; t += 512) {
    cplx l = L[t];
    l.re += sL[t].re;
    l.im += sL[t].im;
    L[t] = l;
  }
}

__global__ void k_periodic_mass_L(const cplx *__restrict__ M, cplx *__restrict__ L, int nt) {
  const double m0 = M[0].re;  // traversal.h:181-183
  for (int t = threadIdx.x; t < nt; t += blockDim.x) {
    L[t].re /= m0;
    L[t].im /= m0;
  }
}

template <int P>
static void periodic_impl(Handle &h) {
  constexpr int NT = Expn<P>::NT;
  if (!h.per_ready) {
    h.per_tab.resize(2 * NT);
    hipLaunchKernelGGL(k_periodic_table<P>, dim3(NT), dim3(256), 0, h.stream, h.per_tab.p);
    h.per_ready = true;
  }
  if (h.cfg.images > 1)
    hipLaunchKernelGGL(k_periodic_far<P>, dim3(1), dim3(512), 0, h.stream, h.M.p, h.L.p, h.per_tab.p, h.cfg.cycle,
                       h.cfg.images - 1, h.cfg.mass);
  if (h.cfg.mass) hipLaunchKernelGGL(k_periodic_mass_L, dim3(1), dim3(64), 0, h.stream, h.M.p, h.L.p, NT);
  EXA_HIP(hipGetLastError());
}

void run_periodic(Handle &h) {
  if (h.cfg.images <= 0 || h.ncells == 0) return;
  if (h.cfg.basis == 1) {
    run_periodic_cart(h);
    if (h.cfg.mass) hipLaunchKernelGGL(k_periodic_mass_L, dim3(1), dim3(64), 0, h.stream, h.M.p, h.L.p, h.nterm);
    EXA_HIP(hipGetLastError());
    return;
  }
  switch (h.cfg.P) {
    case 4: periodic_impl<4>(h); break;
    case 6: periodic_impl<6>(h); break;
    case 8: periodic_impl<8>(h); break;
    case 10: periodic_impl<10>(h); break;
    case 12: periodic_impl<12>(h); break;
    default: throw Error(EXAFMM_HIP_EUNSUP, "P must be one of 4, 6, 8, 10, 12");
  }
}

// ---------------------------------------------------------------------------
// Dipole of the bodies about X0 (tree order, up_down_pass.h:151-157):
// per-block partial sums, then one block adds them in block order.
constexpr int kDipBlocks = 256;

__global__ void __launch_bounds__(256)
    k_dipole_partial(const double4 *__restrict__ body, int n, double x0, double y0, double z0,
                     double *__restrict__ part) {
  __shared__ double s[3][256];
  double d[3] = {0, 0, 0};
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const double4 b = body[i];
    d[0] += (b.x - x0) * b.w;
    d[1] += (b.y - y0) * b.w;
    d[2] += (b.z - z0) * b.w;
  }
  for (int k = 0; k < 3; k++) s[k][threadIdx.x] = d[k];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int k = 0; k < 3; k++) s[k][threadIdx.x] += s[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 3) part[blockIdx.x * 3 + threadIdx.x] = s[threadIdx.x][0];
}

__global__ void k_dipole_final(const double *__restrict__ part, int nb, double *__restrict__ out) {
  if (threadIdx.x < 3) {
    double v = 0;
    for (int b = 0; b < nb; b++) v += part[b * 3 + threadIdx.x];
    out[threadIdx.x] = v;
  }
}

void run_get_dipole(Handle &h, const double *X0, double *out) {
  h.red.reserve(3 * kDipBlocks + 3);
  hipLaunchKernelGGL(k_dipole_partial, dim3(kDipBlocks), dim3(256), 0, h.stream, h.body4.p, h.n, X0[0], X0[1],
                     X0[2], h.red.p);
  hipLaunchKernelGGL(k_dipole_final, dim3(1), dim3(64), 0, h.stream, h.red.p, kDipBlocks, h.red.p + 3 * kDipBlocks);
  EXA_HIP(hipGetLastError());
  EXA_HIP(hipMemcpyAsync(out, h.red.p + 3 * kDipBlocks, 3 * sizeof(double), hipMemcpyDeviceToHost, h.stream));
  EXA_HIP(hipStreamSynchronize(h.stream));
}

// dipoleCorrection (up_down_pass.h:160-168) on the tree-order results.
__global__ void k_dipole_correction(const double4 *__restrict__ body, double4 *__restrict__ trg, int n, double coef,
                                    double dx, double dy, double dz, int numBodies) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double nd = (dx * dx + dy * dy) + dz * dz;
  double4 t = trg[i];
  t.x -= coef * nd / numBodies / body[i].w;
  t.y -= coef * dx;
  t.z -= coef * dy;
  t.w -= coef * dz;
  trg[i] = t;
}

void run_dipole_correction(Handle &h, const double *dipole, int numBodies, double cycle) {
  const double coef = 4 * M_PI / (3 * cycle * cycle * cycle);
  if (h.n == 0) return;
  hipLaunchKernelGGL(k_dipole_correction, dim3(div_up(h.n, 256)), dim3(256), 0, h.stream, h.body4.p, h.trg4.p, h.n,
                     coef, dipole[0], dipole[1], dipole[2], numBodies);
  EXA_HIP(hipGetLastError());
}

}  // namespace exafmm
