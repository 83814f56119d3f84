// M2L of lattice pairs as dense contractions on the matrix cores.
//
// Reference: kernels/LaplaceSphericalCPU.cxx:149-191 (non-MASS).  Octree cell
// centres of one level lie on that level's lattice, so the offset between a
// target of width w and a source of the same level or one level up or down
// is X_i - X_j = d u with d an integer vector and u = w / 4.  The singular
// harmonics are homogeneous, S_a(u d) = u^-(a+1) S_a(d), so with
// M~_n = M_n u^-n the translation of every such pair is one fixed real matrix
// per offset d:  L_j = u^-(j+1) T(d) M~.  In real form (rows (j, k, re|im),
// columns (n, m, re|im), m >= 0) the reference's sum over m = -n..n folds
// into 2 x 2 blocks, with M'_n^m = (-1)^m M_n^m, M'_n^-m = conj M_n^m and the
// signed harmonics S' of the spherical kernel:
//   T[(j,k,re),(n,m,re)] = (-1)^j ((-1)^m S1r + [m>0] S2r)
//   T[(j,k,re),(n,m,im)] = (-1)^j (-(-1)^m S1i + [m>0] S2i)
//   T[(j,k,im),(n,m,re)] = (-1)^j ((-1)^m S1i + [m>0] S2i)
//   T[(j,k,im),(n,m,im)] = (-1)^j ((-1)^m S1r - [m>0] S2r)
// S1 = S'_{j+n}^{m-k}(d), S2 = S'_{j+n}^{-m-k}(d), zero unless j + n < P.
//
// Work split: targets are grouped into tiles of 64 cells of one level and
// one octant, ordered by their distances to the domain's faces (cells of one
// octant share most of their interaction offsets, and those of one face
// class also the missing ones, so a tile's columns are mostly busy at every
// offset);
// a tile's local expansions (112 rows x 64 columns) stay in MFMA
// accumulators while the workgroup walks the offsets: per offset the matrix
// T(d) is staged in LDS in MFMA fragment order (only the 16 x 4 blocks that
// are not identically zero: j + n < P), each lane gathers its column's source
// multipole scaled by u^-n, and the 4 waves (16 columns each) run
// v_mfma_f64_16x16x4 (v_mfma_f32_16x16x4 in the mixed form).  Pairs with a
// periodic image across one face of the box, on the finest levels, take part
// with matrices made for their actual offsets in every evaluation.  Pairs that
// are not lattice pairs (levels two or more apart, other periodic images, MASS
// mode, offsets beyond kLatD) go to the per-pair kernel.
#include <algorithm>
#include <climits>
#include <type_traits>
#include <vector>

#include "harmonics.h"
#include "internal.h"

namespace exafmm {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr double kLatUnit = 4;                   // u = w / kLatUnit
constexpr int kLatD = 60;                         // |d_c| <= kLatD (in units of u)
constexpr double kLatFar = (double)((int64_t)1 << 40);  // |centre| (in units of u), 2^12 below what FP64 resolves
constexpr int kLatSide = 2 * kLatD + 1;
constexpr int kLatKeys = kLatSide * kLatSide * kLatSide;

// Image offsets.  The box length is no multiple of a cell width, so a source
// seen across a face is off the targets' lattice; but all pairs of one level,
// face and lattice offset have the same actual offset, and with it the same
// T.  Their keys follow the lattice keys: (level mod 3, face, offset), the
// offset taken to the nearest lattice image, |d_c| <= kImgD, its components
// all 0, all 2 or all odd mod 4 (the three level relations).  Unlike the
// lattice's, their T depends on box and cell sizes and is made anew in every
// evaluation.
//
// Used on the finest kImgLevels levels that are dense, from level 3 on: there
// a T (31 KB at P = 10, 30 ns to make and to read) serves 100 to 1000 pairs of
// 1.8 ns each on the per-pair kernel (a lattice of 64^3 bodies, theta = 0.35).
// Images across an edge of the box share one offset among 40 to 50 pairs, as
// coarser levels and the few cells of a sparse level do, and gain nothing:
// they stay with the per-pair kernel, a tenth of the image pairs.
constexpr int kImgLevels = 3;
constexpr int kImgD = 44;
constexpr int kImgN0 = kImgD / 2 + 1, kImgN2 = kImgD / 2, kImgN1 = kImgD;  // values per component
constexpr int kImgFace = kImgN0 * kImgN0 * kImgN0 + kImgN2 * kImgN2 * kImgN2 + kImgN1 * kImgN1 * kImgN1;
constexpr int kImgLevelKeys = 6 * kImgFace;
static_assert(kImgD % 4 == 0, "the offsets of each level relation fill their range");

struct LatImages {
  int finest = -1;  // finest level of image offsets (-1: none)
  double cycle = 0;
};

template <int P>
struct MfmaShape {
  static constexpr int NT = P * (P + 1) / 2;
  static constexpr int NR = 2 * NT;              // real rows / columns
  static constexpr int RB = (NR + 15) / 16;      // row blocks
  static constexpr int KC = (NR + 3) / 4;        // column chunks
  static constexpr int jmin(int rb) {
    int r = rb * 16 / 2, j = 0;
    while ((j + 1) * (j + 2) / 2 <= r) j++;
    return j;
  }
  static constexpr int kc_end(int rb) {
    const int j = jmin(rb);
    const int cols = 2 * ((P - j) * (P - j + 1) / 2);  // columns with n <= P-1-j
    return (cols + 3) / 4;
  }
  static constexpr int base(int rb) {
    int s = 0;
    for (int i = 0; i < rb; i++) s += kc_end(i);
    return s;
  }
  static constexpr int NBLK = base(RB);
};

// n of packed coefficient t = n(n+1)/2 + m.
template <int P>
struct DegreeTable {
  int n[P * (P + 1) / 2 + 1];
  constexpr DegreeTable() : n() {
    int t = 0;
    for (int a = 0; a < P; a++)
      for (int b = 0; b <= a; b++) n[t++] = a;
    n[t] = P;
  }
};

// Component r of lane l of the 16x16x4 MFMA result holds D[row][l%16] with
// row = (l/16) + 4 r (FP64) or 4 (l/16) + r (FP32); A[l%16][l/16] and
// B[l/16][l%16] are lane l's operands for both.
template <typename R>
__device__ inline int d_row(int lane, int r) {
  return sizeof(R) == 8 ? (lane >> 4) + 4 * r : 4 * (lane >> 4) + r;
}

template <typename R>
struct MfmaAcc;
template <>
struct MfmaAcc<double> {
  typedef v4d type;
  static __device__ inline v4d mac(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
};
template <>
struct MfmaAcc<float> {
  typedef v4f type;
  static __device__ inline v4f mac(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

// ---------------------------------------------------------------------------
// What the set-up kernels leave for the host and for the contraction.
struct LatState {
  int unknown;  // pairs with an offset that the table does not know yet: nothing of this set-up is used
  int nirr;     // irregular pairs
  int nsteps;   // (tile, offset) steps
  int ntiles;   // tiles with steps
  int noffs;    // offsets with steps
  int pad;
};
static_assert(sizeof(LatState) % 8 == 0, "cleared by whole words");

// Face that image im lies across (-x, +x, -y, ... +z), or -1.
__device__ inline int image_face(int im) {
  return im == 4 ? 0 : im == 22 ? 1 : im == 10 ? 2 : im == 16 ? 3 : im == 12 ? 4 : im == 14 ? 5 : -1;
}

__device__ inline bool image_level(const LatImages &li, int l) { return l >= 3 && l <= li.finest && l > li.finest - kImgLevels; }

// Number of the image offset (x, y, z) among those of one level and face, or
// -1, and back.
__device__ inline int image_index(int x, int y, int z) {
  if (abs(x) > kImgD || abs(y) > kImgD || abs(z) > kImgD) return -1;
  const int c = (x & 3) == 2 ? 2 : x & 1 ? 1 : 0;
  if (c == 1 ? !(y & z & 1) : (y & 3) != c || (z & 3) != c) return -1;
  if (c == 0) return ((x + kImgD) / 4 * kImgN0 + (y + kImgD) / 4) * kImgN0 + (z + kImgD) / 4;
  constexpr int b2 = kImgN0 * kImgN0 * kImgN0, b1 = b2 + kImgN2 * kImgN2 * kImgN2;
  if (c == 2) return b2 + ((x + kImgD - 2) / 4 * kImgN2 + (y + kImgD - 2) / 4) * kImgN2 + (z + kImgD - 2) / 4;
  return b1 + ((x + kImgD - 1) / 2 * kImgN1 + (y + kImgD - 1) / 2) * kImgN1 + (z + kImgD - 1) / 2;
}

__device__ inline void image_offset(int i, int &x, int &y, int &z) {
  constexpr int b2 = kImgN0 * kImgN0 * kImgN0, b1 = b2 + kImgN2 * kImgN2 * kImgN2;
  const int n = i < b2 ? kImgN0 : i < b1 ? kImgN2 : kImgN1, step = i < b1 ? 4 : 2;
  const int lo = i < b2 ? -kImgD : i < b1 ? 2 - kImgD : 1 - kImgD;
  i -= i < b2 ? 0 : i < b1 ? b2 : b1;
  x = lo + step * (i / (n * n));
  y = lo + step * (i / n % n);
  z = lo + step * (i % n);
}

// The lattice's whole number of units nearest to the box length.
__device__ inline int image_units(double cycle, double rt) { return 4 * (int)rint(cycle / (2 * rt)); }
static_assert(kLatUnit == 4, "image offsets in units of a quarter cell");

// Key of the offset of target t and source s (image im), or -1.
__device__ inline int lat_key(int t, int s, int im, const double4 *__restrict__ cX, const double *__restrict__ cRb,
                              const int *__restrict__ cLevel, const LatImages &li) {
  // Same level or one level apart: then the offset's residue mod 4 fixes
  // the level relation (0: same, 2: source one up, odd: source one down).
  const double rt = cRb[t], rs = cRb[s];
  if (!(rs == rt || rs == 2 * rt || 2 * rs == rt)) return -1;
  int face = -1, l = 0;
  if (im != 13) {
    if (li.finest < 0 || (face = image_face(im)) < 0 || !image_level(li, l = cLevel[t])) return -1;
  }
  // Offsets in units of u = 2 R_t / kLatUnit; the lattice values are whole
  // numbers to far better than the 1e-6 test below.
  const double iu = kLatUnit / (2 * rt);
  const double4 a = cX[t], b = cX[s];
  // Centres far from the origin are rounded; where that is not far below a unit,
  // cells of one level may have one centre and would share a slot.
  if (!(fmax(fmax(fabs(a.x), fabs(a.y)), fabs(a.z)) * iu < kLatFar)) return -1;
  const double dx = (a.x - b.x) * iu, dy = (a.y - b.y) * iu, dz = (a.z - b.z) * iu;
  const double rx = rint(dx), ry = rint(dy), rz = rint(dz);
  if (!(fabs(dx - rx) < 1e-6 && fabs(dy - ry) < 1e-6 && fabs(dz - rz) < 1e-6)) return -1;
  if (im != 13) {
    if (!(fabs(rx) < 1e6 && fabs(ry) < 1e6 && fabs(rz) < 1e6 && li.cycle < 1e6 * rt)) return -1;
    const int pc = image_units(li.cycle, rt) * (face & 1 ? 1 : -1);
    const int i = image_index((int)rx - (face / 2 == 0 ? pc : 0), (int)ry - (face / 2 == 1 ? pc : 0),
                              (int)rz - (face / 2 == 2 ? pc : 0));
    return i < 0 ? -1 : kLatKeys + (l % kImgLevels * 6 + face) * kImgFace + i;
  }
  if (fabs(rx) <= kLatD && fabs(ry) <= kLatD && fabs(rz) <= kLatD)
    return (((int)rx + kLatD) * kLatSide + ((int)ry + kLatD)) * kLatSide + ((int)rz + kLatD);
  return -1;
}

// Every M2L pair's step, tile * noff + o (o: number of its offset among the
// noff known ones), into pstep, -1 for a pair that is not on the lattice (or
// whose target is in no tile); act flags the steps in use, used the image
// offsets (the others by k_lat_count).  A pair with an
// unknown offset flags it in hist and makes the set-up unusable.  (A fixed grid
// and one atomic per workgroup for the irregular count: one per wave took 500 us
// in a periodic list of 11 M pairs, a fifth of them irregular.)
__global__ void k_lat_classify(const int *__restrict__ ptgt, const int *__restrict__ src,
                               const unsigned char *__restrict__ img, int64_t np, const double4 *__restrict__ cX,
                               const double *__restrict__ cRb, const int *__restrict__ o_of_key,
                               const int *__restrict__ tile_of, const int *__restrict__ cLevel, LatImages li, int nreg,
                               int noff, unsigned char *__restrict__ act, unsigned char *__restrict__ used,
                               int *__restrict__ pstep, unsigned char *__restrict__ hist, LatState *__restrict__ st) {
  __shared__ int sn;
  if (threadIdx.x == 0) sn = 0;
  __syncthreads();
  int nirr = 0;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < np; e += (int64_t)gridDim.x * blockDim.x) {
    const int t = ptgt[e];
    const int key = lat_key(t, src[e], img[e], cX, cRb, cLevel, li);
    const int tile = tile_of[t];
    int v = -1;
    if (key >= 0 && tile >= 0) {
      const int o = o_of_key[key];
      if (o < 0) {
        // A read first, so that the many pairs of one offset do not all store.
        if (!hist[key]) hist[key] = 1;
        if (!st->unknown) st->unknown = 1;
      } else {
        v = tile * noff + o;
        act[v] = 1;
        if (o >= nreg && !used[o]) used[o] = 1;
      }
    }
    pstep[e] = v;
    nirr += v < 0;
  }
  if (nirr) atomicAdd(&sn, nirr);
  __syncthreads();
  if (threadIdx.x == 0 && sn) atomicAdd(&st->nirr, sn);
}

// T(d) rows in memory and LDS: TE entries padded to whole 1 KiB chunks (one
// chunk = one wave-wide 16-byte-per-lane LDS DMA).
template <int P, typename R>
struct TPad {
  static constexpr int TE = MfmaShape<P>::NBLK * 64;
  static constexpr int CH = 1024 / (int)sizeof(R);
  static constexpr int NCH = (TE + CH - 1) / CH;
  static constexpr int TEP = NCH * CH;
};

// Source multipole rows for the contraction: lane (column n, kq) of a wave
// needs entries 4 kc + kq (kc = 0 .. KC-1) of its column's row.  A row keeps
// them in groups of VL = 16 bytes / sizeof(R) consecutive kc per kq, the four
// kq groups of one run of kc side by side: every 16-byte vector load of a
// lane is one group, and the 4 lanes of a column read 64 contiguous bytes.
// KC is padded to KCP (a multiple of VL) with zeros.
template <int P, typename R>
struct MsRow {
  static constexpr int VL = 16 / (int)sizeof(R);
  static constexpr int KCP = (MfmaShape<P>::KC + VL - 1) / VL * VL;
  static constexpr int NKP = KCP * 4;  // entries per row
};

// T(d) of offset key okey[o] into row o of T, in fragment order: block
// (rb, kc) holds T[rb*16 + l%16][kc*4 + l/16] at lane l.  T depends on the
// key alone (offset in units of u and, through its residue, the level
// relation), so rows are kept across evaluations.
template <int P, typename R>
__global__ void __launch_bounds__(64) k_lat_tmat(const int *__restrict__ okey, R *__restrict__ T) {
  using S = MfmaShape<P>;
  constexpr int NT = S::NT;
  __shared__ cplx sS[P * P];
  const int o = blockIdx.x, lane = threadIdx.x;
  const int key = okey[o];
  const double dx = key / (kLatSide * kLatSide) - kLatD, dy = (key / kLatSide) % kLatSide - kLatD,
               dz = key % kLatSide - kLatD;
  const Geom g = make_geom(dx, dy, dz);
  // Source multipoles arrive scaled by their own cell's u^-n; u_s = 2^D u_t
  // with D = 0, +1, -1 for offsets = 0, 2, odd mod 4, so column (n, m) of T
  // takes the exact factor 2^(D n).
  const int rx = ((key / (kLatSide * kLatSide)) - kLatD) & 3;
  const int dlev = rx == 0 ? 0 : (rx == 2 ? 1 : -1);
  for (int t = lane; t < NT; t += 64) {
    int a, b;
    coef_nm(t, a, b);
    double re, im;
    singular_nm(a, b, g, re, im);
    const double sg = (b & 1) ? -1.0 : 1.0;  // S'_a^b = (-1)^b S_a^b (b > 0)
    sS[a * a + a + b] = {sg * re, sg * im};
    if (b > 0) sS[a * a + a - b] = {re, -im};  // S'_a^-b = S_a^-b = conj S_a^b
  }
  __syncthreads();
  for (int rb = 0; rb < S::RB; rb++)
    for (int kc = 0; kc < S::kc_end(rb); kc++) {
      const int row = rb * 16 + (lane & 15), col = kc * 4 + (lane >> 4);
      double v = 0;
      if (row < S::NR && col < S::NR) {
        int j, k, n, m;
        coef_nm(row >> 1, j, k);
        coef_nm(col >> 1, n, m);
        if (j + n < P) {
          const int a = j + n;
          const cplx S1 = sS[a * a + a + m - k];
          const cplx S2 = m > 0 ? sS[a * a + a - m - k] : cplx{0, 0};
          const double sm = (m & 1) ? -1.0 : 1.0, sj = (j & 1) ? -1.0 : 1.0;
          const int pr = row & 1, pc = col & 1;
          if (pr == 0 && pc == 0) v = sm * S1.re + S2.re;
          if (pr == 0 && pc == 1) v = -sm * S1.im + S2.im;
          if (pr == 1 && pc == 0) v = sm * S1.im + S2.im;
          if (pr == 1 && pc == 1) v = sm * S1.re - S2.re;
          v = ldexp(v * sj, dlev * n);
        }
      }
      T[(size_t)o * TPad<P, R>::TEP + (S::base(rb) + kc) * 64 + lane] = (R)v;
    }
  for (int i = S::NBLK * 64 + lane; i < TPad<P, R>::TEP; i += 64) T[(size_t)o * TPad<P, R>::TEP + i] = 0;
}

// T of the image offsets in use (numbers from nreg on), as k_lat_tmat for
// the actual offset of their level and face.  A workgroup makes kImgT of them
// together, so that the entries' index arithmetic is done once for all; bound
// by the stores: 6800 offsets at P = 10 are 212 MB, 0.32 ms alone with one
// workgroup per kImgT and 0.45 ms beside P2P and the step lists, which hide it.
// lvl: for each level mod 3 the first of its cells in lvl_cells.
constexpr int kImgT = 16, kImgTParts = 4;  // (each in kImgTParts workgroups, for balance)
struct ImgLevels {
  int cell[kImgLevels];
};

template <int P, typename R>
__global__ void __launch_bounds__(256)
    k_lat_tmat_image(int nreg, int noff, const int *__restrict__ okey, const int *__restrict__ orow,
                     const unsigned char *__restrict__ used, ImgLevels lvl, const int *__restrict__ lvl_cells,
                     const double *__restrict__ cRb, double cycle, R *__restrict__ T, const LatState *__restrict__ st) {
  using S = MfmaShape<P>;
  constexpr int NT = S::NT, TEP = TPad<P, R>::TEP;
  __shared__ double sS[kImgT][2 * P * P];
  __shared__ int srow[kImgT], sdlev[kImgT];
  __shared__ Geom sg[kImgT];
  if (st->unknown) return;
  const int o0 = nreg + blockIdx.x * kImgT;
  if (threadIdx.x < kImgT) {
    const int o = o0 + threadIdx.x;
    srow[threadIdx.x] = -1;
    if (o < noff && used[o]) {
      const int k = okey[o] - kLatKeys, face = k / kImgFace % 6;
      int x, y, z;
      image_offset(k % kImgFace, x, y, z);
      const double rt = cRb[lvl_cells[lvl.cell[k / kImgLevelKeys]]];
      // The offset to the nearest lattice image, and what the image is off it.
      const double p = (face & 1 ? 1 : -1) * (image_units(cycle, rt) - cycle * (kLatUnit / (2 * rt)));
      sg[threadIdx.x] = make_geom(x + (face / 2 == 0 ? p : 0), y + (face / 2 == 1 ? p : 0), z + (face / 2 == 2 ? p : 0));
      srow[threadIdx.x] = orow[o];
      sdlev[threadIdx.x] = (x & 3) == 0 ? 0 : (x & 3) == 2 ? 1 : -1;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kImgT * NT; i += 256) {
    const int q = i % kImgT, t = i / kImgT;
    if (srow[q] < 0) continue;
    int a, b;
    coef_nm(t, a, b);
    double re, im;
    singular_nm(a, b, sg[q], re, im);
    const double s = (b & 1) ? -1.0 : 1.0;
    sS[q][2 * (a * a + a + b)] = s * re;
    sS[q][2 * (a * a + a + b) + 1] = s * im;
    if (b > 0) {
      sS[q][2 * (a * a + a - b)] = re;
      sS[q][2 * (a * a + a - b) + 1] = -im;
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, part = 4 * blockIdx.y + wave;
  int blk = 0;
  for (int rb = 0; rb < S::RB; rb++)
    for (int kc = 0; kc < S::kc_end(rb); kc++, blk++) {
      if (blk % (4 * kImgTParts) != part) continue;
      // Entry = c1 S1 + c2 S2, each a component of a harmonic.
      const int row = rb * 16 + (lane & 15), col = kc * 4 + (lane >> 4);
      int i1 = 0, i2 = 0, n = 0;
      double c1 = 0, c2 = 0;
      if (row < S::NR && col < S::NR) {
        int j, k, m;
        coef_nm(row >> 1, j, k);
        coef_nm(col >> 1, n, m);
        if (j + n < P) {
          const int a = j + n, pr = row & 1, pc = col & 1;
          const double sm = (m & 1) ? -1.0 : 1.0, sj = (j & 1) ? -1.0 : 1.0;
          i1 = 2 * (a * a + a + m - k) + (pr ^ pc);
          c1 = sj * (pc & ~pr ? -sm : sm);
          if (m > 0) {
            i2 = 2 * (a * a + a - m - k) + (pr ^ pc);
            c2 = pr & pc ? -sj : sj;
          }
        }
      }
      const double up = ldexp(1.0, n), down = ldexp(1.0, -n);
      for (int q = 0; q < kImgT; q++) {
        const int to = __builtin_amdgcn_readfirstlane(srow[q]), dlev = __builtin_amdgcn_readfirstlane(sdlev[q]);
        if (to < 0) continue;
        const double v = c1 * sS[q][i1] + c2 * sS[q][i2];
        T[(size_t)to * TEP + blk * 64 + lane] = (R)(dlev == 0 ? v : v * (dlev > 0 ? up : down));
      }
    }
  for (int q = part; q < kImgT; q += 4 * kImgTParts)
    for (int i = S::NBLK * 64 + lane; srow[q] >= 0 && i < TEP; i += 64) T[(size_t)srow[q] * TEP + i] = 0;
}

// Target tiles: cells grouped by (level, octant), and inside a group ordered
// by face class, then cell order.  The face class is the six distances of the cell
// to the faces of its level's grid, each clipped at kTileK: cells near the
// domain boundary lack the offsets that point outside it, and cells of one
// class lack the same ones, so tiles cut from class-ordered cells have
// fewer steps with idle columns.  The class only orders work: any order
// gives the same pairs.
constexpr int kTileK = 4;
constexpr int kTileClassBits = 14;  // (kTileK + 1)^6 = 15625 classes
static_assert((kTileK + 1) * (kTileK + 1) * (kTileK + 1) * (kTileK + 1) * (kTileK + 1) * (kTileK + 1) <=
                  (1 << kTileClassBits),
              "face classes fit their key bits");
constexpr int kTileNoGroup = 255 << kTileClassBits;  // cells in no group sort last

// Face class of the cell whose Morton index on its level's grid is kk
// (coordinate bits interleaved x, y, z from bit 0).
__device__ inline int face_class(uint64_t kk, int l) {
  int g[3] = {0, 0, 0};
  for (int i = 0; i < l && i < 21; i++)
    for (int a = 0; a < 3; a++) g[a] |= (int)((kk >> (3 * i + a)) & 1) << i;
  const int64_t side = (int64_t)1 << (l < 21 ? l : 21);
  int cls = 0;
  for (int a = 0; a < 3; a++) {
    const int lo = (int)min<int64_t>(g[a], kTileK), hi = (int)min<int64_t>(side - 1 - g[a], kTileK);
    cls = (cls * (kTileK + 1) + lo) * (kTileK + 1) + hi;
  }
  return cls;
}

// Tile slots are laid out by what the tree can hold, so that no count has to
// reach the host: a level's octant group has at most one cell per parent (the
// builders leave their number), and level l gets 8 ceil(parents / 64) slots
// from base[l] on, chunk q of octant o at base[l] + 8 q + o (consecutive
// tiles cover one region of space).  Slots without cells are skipped later.
// Each costs its partial results (0.13 MB at P = 4, 0.46 at P = 10) and its row
// of step flags all the same, and parents have half as many children on surfaces
// as they could, a third with a body to a leaf: from kTilesUnread slots on the
// host waits for the octants' counts (3.1 M bodies, ncrit = 1, P = 4: 63.4 ms and
// 67 GB with the bound, 52.9 ms and 39 GB with the counts; 1 M: 15.0 and 14.5 ms).
constexpr int kTilesUnread = 1 << 14;
constexpr int kTileLevels = 32;  // deeper cells are in no tile (their pairs go per pair)
struct TileLevels {
  int nlevels;
  int off[kTileLevels + 1];   // cells of level l: lvl_cells[off[l] .. off[l + 1])
  int cap[kTileLevels + 1];   // most cells of one octant
  int base[kTileLevels + 1];  // first tile slot of level l
};

// What cKey adds to the Morton index of a level's cells.
__device__ inline uint64_t level_offset(int l, bool key_lvloff) {
  return key_lvloff ? ((1ull << (3 * l)) - 1) / 7 : 0;
}

// Cells of each (level, octant), 8 l + o.
__global__ void __launch_bounds__(256)
    k_tile_octants(int nc, const int *__restrict__ lvl, const uint64_t *__restrict__ ckey, bool key_lvloff,
                   int *__restrict__ cnt) {
  __shared__ int s[8 * kTileLevels];
  static_assert(8 * kTileLevels == 256, "one count a thread");
  s[threadIdx.x] = 0;
  __syncthreads();
  for (int c = blockIdx.x * 256 + threadIdx.x; c < nc; c += gridDim.x * 256) {
    const int l = lvl[c];
    if (l < kTileLevels) atomicAdd(&s[8 * l + (int)((ckey[c] - level_offset(l, key_lvloff)) & 7)], 1);
  }
  __syncthreads();
  if (s[threadIdx.x]) atomicAdd(&cnt[threadIdx.x], s[threadIdx.x]);
}

// One workgroup per (octant, level): its cells in cell order, sorted by class
// in LDS.  For groups of up to kTileSort cells; the class and the cell's place
// in its level share a word.  (One launch for all levels, beside the
// traversal; the radix sort of all cells, about 10 launches and 60 us of the
// main stream at 4700 cells, stays for larger levels.)
constexpr int kTileSort = 4096;
constexpr int kTilePosBits = 15;  // 8 kTileSort places
static_assert(kTileClassBits + kTilePosBits < 32 && 8 * kTileSort <= (1 << kTilePosBits), "sort words");
__global__ void __launch_bounds__(1024)
    k_tiles(TileLevels tl, const int *__restrict__ lvl_cells, const uint64_t *__restrict__ ckey, bool key_lvloff,
            int *__restrict__ tile_tgt, int *__restrict__ tile_of, int *__restrict__ col_of) {
  extern __shared__ unsigned skey[];
  __shared__ int swave[17];
  const int oct = blockIdx.x, l = blockIdx.y + 1, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int *cells = lvl_cells + tl.off[l];
  const uint64_t lvloff = level_offset(l, key_lvloff);
  const int nl = tl.off[l + 1] - tl.off[l], cap = tl.cap[l];
  if (blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = tid; i < tl.off[1]; i += 1024) tile_of[lvl_cells[i]] = -1;  // roots
  int m = 0;
  for (int b = 0; b < nl; b += 1024) {
    const int i = b + tid;
    uint64_t kk = 0;
    if (i < nl) kk = ckey[cells[i]] - lvloff;
    const int o = i < nl ? (int)(kk & 7) : -1;
    const unsigned long long in = __ballot(o == oct);
    __syncthreads();
    if (lane == 0) swave[wave] = (int)__popcll(in);
    __syncthreads();
    int before = m;
    for (int w = 0; w < 16; w++) {
      if (w < wave) before += swave[w];
      m += swave[w];
    }
    before += (int)__popcll(in & ((1ull << lane) - 1));
    if (o == oct && before < cap)
      skey[before] = ((unsigned)face_class(kk, l) << kTilePosBits) | (unsigned)i;
    else if (o == oct)
      tile_of[cells[i]] = -1;
  }
  m = min(m, cap);
  int p2 = 1;
  while (p2 < m) p2 *= 2;
  for (int i = m + tid; i < p2; i += 1024) skey[i] = ~0u;
  __syncthreads();
  for (int k = 2; k <= p2; k *= 2)
    for (int j = k / 2; j > 0; j /= 2) {
      for (int i = tid; i < p2; i += 1024) {
        const int x = i ^ j;
        if (x > i) {
          const unsigned u = skey[i], v = skey[x];
          if ((u > v) == ((i & k) == 0)) {
            skey[i] = v;
            skey[x] = u;
          }
        }
      }
      __syncthreads();
    }
  const int nslot = 8 * (tl.base[l + 1] - tl.base[l]);  // columns of this octant's slots
  for (int r = tid; r < nslot; r += 1024) {
    const int t = tl.base[l] + (r / 64) * 8 + oct, col = r % 64;
    int c = -1;
    if (r < m) {
      c = cells[skey[r] & ((1u << kTilePosBits) - 1)];
      tile_of[c] = t;
      col_of[c] = col;
    }
    tile_tgt[t * 64 + col] = c;
  }
}

// The same by a radix sort over all cells, keys (level, octant, class).
__global__ void k_tile_key(int nc, const int *__restrict__ lvl, const uint64_t *__restrict__ ckey, bool key_lvloff,
                           int *__restrict__ key, int *__restrict__ val) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  int k = kTileNoGroup;
  const int l = lvl[c];
  if (l > 0 && l < kTileLevels - 1) {
    const uint64_t kk = ckey[c] - level_offset(l, key_lvloff);
    k = ((l * 8 + (int)(kk & 7)) << kTileClassBits) | face_class(kk, l);
  }
  key[c] = k;
  val[c] = c;
}

__global__ void k_tile_assign(int nc, TileLevels tl, const int *__restrict__ skey, const int *__restrict__ sval,
                              int *__restrict__ tile_tgt, int *__restrict__ tile_of, int *__restrict__ col_of) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nc) return;
  const int g = skey[p] >> kTileClassBits, c = sval[p];
  if (g >= (kTileNoGroup >> kTileClassBits)) {
    tile_of[c] = -1;
    return;
  }
  int lo = 0, hi = p;  // first entry of the group
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((skey[mid] >> kTileClassBits) < g)
      lo = mid + 1;
    else
      hi = mid;
  }
  const int r = p - lo, t = tl.base[g >> 3] + (r / 64) * 8 + (g & 7), col = r % 64;
  if (r >= tl.cap[g >> 3]) {  // beyond the group's slots, as in k_tiles
    tile_of[c] = -1;
    return;
  }
  tile_tgt[t * 64 + col] = c;
  tile_of[c] = t;
  col_of[c] = col;
}

// The offsets a tile can use: the lattice's, and the image offsets of its level.
struct LatRanges {
  int nreg;                           // lattice offsets
  int nlv;                            // levels with image offsets
  int tile0[kImgLevels], tile1[kImgLevels];  // tiles of the level
  int lo[kImgLevels], hi[kImgLevels];        // numbers of its image offsets
};

__device__ inline void tile_images(const LatRanges &lr, int tile, int &lo, int &hi) {
  lo = hi = 0;
  for (int i = 0; i < kImgLevels; i++)
    if (i < lr.nlv && tile >= lr.tile0[i] && tile < lr.tile1[i]) {
      lo = lr.lo[i];
      hi = lr.hi[i];
    }
}

// Steps per tile: the flags of its row of act.  Flags the lattice offsets in use.
__global__ void __launch_bounds__(256)
    k_lat_count(const unsigned char *__restrict__ act, int noff, LatRanges lr, int *__restrict__ cnt,
                unsigned char *__restrict__ used) {
  __shared__ int sw[4];
  const unsigned char *a = act + (size_t)blockIdx.x * noff;
  int n = 0, lo, hi;
  tile_images(lr, blockIdx.x, lo, hi);
  for (int o = threadIdx.x; o < lr.nreg; o += 256)
    if (a[o]) {
      n++;
      if (!used[o]) used[o] = 1;
    }
  for (int o = lo + threadIdx.x; o < hi; o += 256) n += a[o];
  for (int d = 32; d >= 1; d >>= 1) n += __shfl_xor(n, d);
  if ((threadIdx.x & 63) == 0) sw[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) cnt[blockIdx.x] = sw[0] + sw[1] + sw[2] + sw[3];
}

// The tile's steps, in offset order, from step0[tile] = the counts of the
// tiles before it: aidx[tile * noff + o] = step, alist[step] = the offset's T
// row; their slots are emptied.
__global__ void __launch_bounds__(256)
    k_lat_steps(const unsigned char *__restrict__ act, const int *__restrict__ cnt, int noff, LatRanges lr,
                const unsigned char *__restrict__ used, const int *__restrict__ orow, int *__restrict__ aidx, int *__restrict__ step0,
                int *__restrict__ alist, int4 *__restrict__ slot, LatState *__restrict__ st,
                LatState *__restrict__ host) {
  __shared__ int sw[4], sn[4], su[4];
  const int tile = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int base = 0, full = 0;
  for (int t = tid; t < tile; t += 256) {
    const int c = cnt[t];
    base += c;
    full += c > 0;
  }
  int offs = 0;
  for (int o = tid; tile == (int)gridDim.x - 1 && o < noff; o += 256) offs += used[o];
  for (int d = 32; d >= 1; d >>= 1) {
    base += __shfl_xor(base, d);
    full += __shfl_xor(full, d);
    offs += __shfl_xor(offs, d);
  }
  if (lane == 0) {
    sw[wave] = base;
    sn[wave] = full;
    su[wave] = offs;
  }
  __syncthreads();
  base = sw[0] + sw[1] + sw[2] + sw[3];
  const int mine = cnt[tile];
  if (tid == 0) {
    step0[tile] = base;
    if (tile == (int)gridDim.x - 1) {
      step0[tile + 1] = base + mine;
      st->nsteps = base + mine;
      st->ntiles = sn[0] + sn[1] + sn[2] + sn[3] + (mine > 0);
      st->noffs = su[0] + su[1] + su[2] + su[3];
      *host = *st;  // (pinned)
    }
  }
  if (mine == 0) return;
  for (int i = tid; i < mine * 16; i += 256) slot[(size_t)base * 16 + i] = make_int4(-1, -1, -1, -1);
  int lo, hi;
  tile_images(lr, tile, lo, hi);
  const int nuse = lr.nreg + hi - lo;
  for (int b = 0; b < nuse; b += 256) {
    const int u = b + tid, o = u < lr.nreg ? u : lo + u - lr.nreg;
    const bool in = u < nuse && act[(size_t)tile * noff + o];
    const unsigned long long m = __ballot(in);
    __syncthreads();
    if (lane == 0) sw[wave] = (int)__popcll(m);
    __syncthreads();
    int k = base + (int)__popcll(m & ((1ull << lane) - 1));
    for (int w = 0; w < 4; w++) {
      if (w < wave) k += sw[w];
      base += sw[w];
    }
    if (in) {
      aidx[(size_t)tile * noff + o] = k;
      alist[k] = orow[o];
    }
  }
}

// Every lattice pair's source cell s into its (step, column) slot, as -2 - s.
// No two pairs share a slot: the traversal visits a pair of cells once, the
// key fixes the source's level and position, and cells of one level differ in
// position.  That holds for bounds that enclose the bodies; with bounds from
// the caller (CHECK) a taken slot makes the later pair irregular.  (The
// exchange costs more than the store: 250 against 95 us for 6.7 M pairs.)
template <bool CHECK>
__global__ void k_lat_slots(const int *__restrict__ ptgt, const int *__restrict__ src, int64_t np,
                            const int *__restrict__ col_of, const int *__restrict__ aidx, int *__restrict__ pstep,
                            int *__restrict__ slot, LatState *__restrict__ st) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= np || st->unknown) return;
  const int v = pstep[e];
  if (v < 0) return;
  int *p = &slot[aidx[v] * 64 + col_of[ptgt[e]]];
  const int w = -2 - src[e];
  if (!CHECK) {
    *p = w;
  } else if (atomicCAS(p, -1, w) != -1) {
    pstep[e] = -1;
    atomicAdd(&st->nirr, 1);
  }
}

// Offsets known after this set-up (the known ones and those hist flags, to
// be numbered in key order), and those of them with no row in the T table.
__global__ void k_lat_flag(const unsigned char *__restrict__ hist, const int *__restrict__ o_of_key,
                           const int *__restrict__ row_of_key, int n, int *__restrict__ flag,
                           int *__restrict__ nflag) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k > n) return;
  const bool used = k < n && (hist[k] || o_of_key[k] >= 0);
  flag[k] = used ? 1 : 0;
  nflag[k] = used && row_of_key[k] < 0 ? 1 : 0;
}

// Numbers the flagged offsets (o_of_key, orow: number -> T row), gives the
// new ones the rows from `base` on and clears hist.
__global__ void k_lat_number(const int *__restrict__ flag, const int *__restrict__ scan,
                             const int *__restrict__ nflag, const int *__restrict__ nscan, int n, int base,
                             int *__restrict__ row_of_key, int *__restrict__ keys, int *__restrict__ o_of_key,
                             int *__restrict__ okey, int *__restrict__ orow, unsigned char *__restrict__ hist) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  hist[k] = 0;
  if (!flag[k]) return;
  int row = row_of_key[k];
  if (nflag[k]) {
    row = base + nscan[k];
    row_of_key[k] = row;
    keys[nscan[k]] = k;
  }
  o_of_key[k] = scan[k];
  okey[scan[k]] = k;
  orow[scan[k]] = row;
}

// What the host needs of the two scans over n keys: known and new offsets, the
// new ones of the lattice, and the known ones below each level's image keys.
__global__ void k_lat_marks(const int *__restrict__ kscan, const int *__restrict__ nscan, int n,
                            int *__restrict__ host) {
  const int i = threadIdx.x;
  if (i == 0) host[0] = kscan[n];
  if (i == 1) host[1] = nscan[n];
  if (i == 2) host[2] = nscan[kLatKeys];
  if (i <= kImgLevels) host[3 + i] = kscan[min(n, kLatKeys + i * kImgLevelKeys)];
}

__global__ void k_fill_int(int *__restrict__ p, int64_t n, int v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// Source multipoles scaled by their own cell's u^-n (u = w / kLatUnit), in
// the precision of the contraction, as MsRow rows (zero padded); row nc is
// all zero and stands for an empty column.
template <int P, typename R>
__global__ void __launch_bounds__(256)
    k_lat_mscale(int b0, int nc, const double *__restrict__ cRb, const cplx *__restrict__ M, R *__restrict__ Ms) {
  using S = MfmaShape<P>;
  using MR = MsRow<P, R>;
  constexpr int NR = S::NR, NKP = MR::NKP, VL = MR::VL;
  constexpr DegreeTable<P> deg{};
  const int64_t i = (int64_t)(b0 + blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= (int64_t)(nc + 1) * NKP) return;
  const int c = (int)(i / NKP), p = (int)(i % NKP);
  const int r = p % (4 * VL), kq = r / VL, kc = (p / (4 * VL)) * VL + r % VL;
  const int k = 4 * kc + kq;  // real row of the packed expansion (re, im interleaved)
  double v = 0;
  if (c < nc && k < NR) {
    const double iu = kLatUnit / (2 * cRb[c]);
    double f = 1;
    for (int q = 0; q < deg.n[k >> 1]; q++) f *= iu;
    v = reinterpret_cast<const double *>(M)[(size_t)c * NR + k] * f;
  }
  Ms[i] = (R)v;
}

// Steps of a tile are split into kLatSeg segments; segment s runs on XCD s
// (work item 8 tile + s is taken by workgroups w = item mod gridDim.x, the
// grid is a multiple of 8, and workgroups are dealt round-robin over the
// 8 XCDs), so an XCD only ever needs the T(d) of one eighth of the offsets
// and keeps them in its L2.
constexpr int kLatSeg = 8;
// Words of Handle::hpin the lattice set-up reads back (LatState; registration counts).
constexpr int kPinLat = 64, kPinMarks = kPinLat + 8;
static_assert(sizeof(LatState) <= 8 * sizeof(int), "pinned words");

typedef __attribute__((address_space(3))) void lds_void;
// s_waitcnt immediate for vmcnt(0) with expcnt and lgkmcnt left alone.
constexpr int kVmcnt0 = 0x0F70;
typedef __attribute__((address_space(1))) void glb_void;

// One workgroup (4 waves) per (tile of 64 target cells, segment of the
// tile's steps).  R = double: FP64 MFMA.  R = float (mixed form): FP32
// tables, multipoles and MFMA, the FP32 accumulators flushed into FP64 after
// every step (a step's K-sum is the only FP32 accumulation).  Software
// pipeline: while step i runs on the matrix cores, T of step i + 1 streams
// into the other LDS buffer by LDS DMA (global_load_lds_dwordx4), the
// multipole columns of step i + 1 stream into the other register set and the
// slot indices of step i + 2 are read; one barrier per step.  The two LDS
// buffers are separate arrays, the two column sets separate register arrays,
// and the step loop is unrolled by two, so every access names its buffer
// statically (no register copy between steps).  The segment's partial
// expansions (unscaled) go to part[] for k_lat_reduce.
//
// A wave without a pair in its 16 columns sits the step out: in adaptive trees
// half the columns of a step and more are empty (250k clustered bodies, P = 12,
// FP32: 1.66 ms, 1.55 without them).  Up to P = 8 in FP64 and P = 10 in FP32 the
// registers allow three or four workgroups per CU: 4.2 M clustered bodies, P =
// 8, took 8.5 ms with two and 7.5 with three; 1 M bodies, P = 10, FP32, 0.69
// and 0.64.
template <int P, typename R>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(P <= 10 ? 2 : 1, 4)))
    k_m2l_mfma(int nc, int nitems, const int *__restrict__ step0, const int *__restrict__ alist,
               const int *__restrict__ slot, const R *__restrict__ T, const R *__restrict__ Ms,
               double *__restrict__ part, const LatState *__restrict__ st) {
  using S = MfmaShape<P>;
  using A = MfmaAcc<R>;
  using TP = TPad<P, R>;
  constexpr bool F32 = sizeof(R) == 4;
  using MR = MsRow<P, R>;
  typedef R vec __attribute__((ext_vector_type(16 / sizeof(R))));
  constexpr int RB = S::RB, KCP = MR::KCP, NKP = MR::NKP;
  constexpr int TEP = TP::TEP, CH = TP::CH, NCH = TP::NCH, VL = MR::VL;
  __shared__ __attribute__((aligned(16))) R sT0[TEP];
  __shared__ __attribute__((aligned(16))) R sT1[TEP];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (st->unknown) return;  // the set-up is redone
  // Items (tile, segment) = (item / 8, item % 8); a grid that is a multiple
  // of 8 keeps every item of a segment on one XCD.
  for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
    const int tile = item / kLatSeg, seg = item % kLatSeg;
    const int col = wave * 16 + (lane & 15);
    const int kq = lane >> 4;
    const int a0 = step0[tile], a1 = step0[tile + 1];
    if (a0 == a1) continue;  // a tile without steps
    const int i0 = a0 + (a1 - a0) * seg / kLatSeg, i1 = a0 + (a1 - a0) * (seg + 1) / kLatSeg;
    typename A::type acc[RB];
    v4d acc64[F32 ? RB : 1];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) acc[rb] = typename A::type{0, 0, 0, 0};
#pragma unroll
    for (int rb = 0; rb < (F32 ? RB : 1); rb++) acc64[rb] = v4d{0, 0, 0, 0};
    // T(d) of step i into an LDS buffer: chunk ch by wave ch % 4.
    auto fetch_T = [&](R *dst, int i) {
      const R *Tn = T + (size_t)alist[i] * TEP + lane * VL;
      for (int ch = wave; ch < NCH; ch += 4)
        __builtin_amdgcn_global_load_lds((glb_void *)(Tn + ch * CH), (lds_void *)(dst + ch * CH), 16, 0, 0);
    };
    R b0[KCP], b1[KCP];
    int sn = -1;
    // Column of slot value sl (-2 - source cell, or -1: row nc of zeros)
    // into v[0 .. KCP): one 16-byte load per VL entries (its kq group of the
    // MsRow row).
    auto load_col = [&](R *v, int sl) {
      const int cell = sl <= -2 ? -2 - sl : nc;
      const vec *src = reinterpret_cast<const vec *>(Ms + (size_t)cell * NKP) + kq;
#pragma unroll
      for (int j = 0; j < KCP / VL; j++) {
        const vec x = src[j * 4];
#pragma unroll
        for (int u = 0; u < VL; u++) v[j * VL + u] = x[u];
      }
    };
    // Step i from buffers CUR = (i - i0) & 1 while step i + 1 is fetched
    // into the other ones.
    bool busy = false;
    auto step = [&](auto curc, int i) {
      constexpr int CUR = decltype(curc)::value;
      const R *sTc = CUR ? sT1 : sT0;
      R *sTn = CUR ? sT0 : sT1;
      const R *b = CUR ? b1 : b0;
      R *bn = CUR ? b0 : b1;
      const bool more = i + 1 < i1, busy_next = more && __any(sn <= -2);
      int snn = -1;
      if (more) {
        if (busy_next) load_col(bn, sn);
        fetch_T(sTn, i + 1);
        if (i + 2 < i1) snn = slot[(size_t)(i + 2) * 64 + col];
      }
      if (busy) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
#pragma unroll
          for (int kc = 0; kc < S::kc_end(rb); kc++)
            acc[rb] = A::mac(sTc[(S::base(rb) + kc) * 64 + lane], b[kc], acc[rb]);
        }
        if (F32) {
#pragma unroll
          for (int rb = 0; rb < (F32 ? RB : 1); rb++)
            for (int r = 0; r < 4; r++) {
              acc64[rb][r] += (double)acc[rb][r];
              acc[rb][r] = 0;
            }
        }
      }
      if (more) sn = snn;
      busy = busy_next;
      __builtin_amdgcn_s_waitcnt(kVmcnt0);  // this wave's DMA and loads have landed
      __syncthreads();
    };
    // Prologue: step i0's T and columns.
    if (i0 < i1) {
      fetch_T(sT0, i0);
      sn = slot[(size_t)i0 * 64 + col];
      busy = __any(sn <= -2);
      load_col(b0, sn);
      sn = i0 + 1 < i1 ? slot[(size_t)(i0 + 1) * 64 + col] : -1;
    }
    __builtin_amdgcn_s_waitcnt(kVmcnt0);
    __syncthreads();
    for (int i = i0; i < i1; i += 2) {
      step(std::integral_constant<int, 0>{}, i);
      if (i + 1 < i1) step(std::integral_constant<int, 1>{}, i + 1);
    }
    double *pp = part + (size_t)item * (RB * 16) * 64;
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = rb * 16 + d_row<R>(lane, r);
        const double v = F32 ? acc64[F32 ? rb : 0][r] : (double)acc[rb][r];
        pp[(size_t)row * 64 + col] = v;
      }
  }
}

// L of each tile column += u^-(j+1) * (sum of the segments' partials, in
// segment order), u = w / kLatUnit of the column's own target cell (the cells
// of a tile share a level, not necessarily a size: batched systems).
template <int P>
__global__ void __launch_bounds__(256)
    k_lat_reduce(const int *__restrict__ tile_tgt, const int *__restrict__ step0, const double *__restrict__ cRb,
                 const double *__restrict__ part, cplx *__restrict__ L, const LatState *__restrict__ st) {
  using S = MfmaShape<P>;
  constexpr int NR = S::NR, NRP = S::RB * 16;
  constexpr DegreeTable<P> deg{};
  const int tile = blockIdx.x;
  if (st->unknown || step0[tile] == step0[tile + 1]) return;
  double *Lr = reinterpret_cast<double *>(L);
  // Rows r0 .. r0 + 15 of the tile: the segment sums read column-fastest
  // (as the partials lie), then written row-fastest through LDS (the 16 rows
  // of one target are 128 contiguous bytes of L).
  __shared__ double sv[16][65];
  const int r0 = 16 * blockIdx.y, nrow = min(NR, r0 + 16) - r0;
  const int col = threadIdx.x & 63, rq = threadIdx.x >> 6;
  double v[4] = {0, 0, 0, 0};
  const double *pp = part + ((size_t)tile * kLatSeg * NRP + r0) * 64 + col;
  for (int sg = 0; sg < kLatSeg; sg++)
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (rq + 4 * k < nrow) v[k] += pp[((size_t)sg * NRP + rq + 4 * k) * 64];
#pragma unroll
  for (int k = 0; k < 4; k++) sv[rq + 4 * k][col] = v[k];
  __syncthreads();
  const int row = threadIdx.x & 15;
  if (row >= nrow) return;
  for (int c = threadIdx.x >> 4; c < 64; c += 16) {
    const int tgt = tile_tgt[tile * 64 + c];
    if (tgt < 0) continue;
    const double iw = 1.0 / (2 * cRb[tgt] / kLatUnit);
    double f = iw;
    for (int q = 0; q < deg.n[(r0 + row) >> 1]; q++) f *= iw;
    // Rounded before it is added: the sum with the per-pair kernel's part is
    // then the same whichever of the two comes first.
    {
#pragma clang fp contract(off)
      const double v = sv[row][c] * f;
      Lr[(size_t)tgt * NR + r0 + row] += v;
    }
  }
}

// ---------------------------------------------------------------------------
template <int P>
static void mscale_impl(Handle &h, hipStream_t st) {
  using S = MfmaShape<P>;
  const int nc = h.ncells;
  const int64_t nms = (int64_t)(nc + 1) * MsRow<P, float>::NKP;
  const int64_t nmd = (int64_t)(nc + 1) * MsRow<P, double>::NKP;
  if (h.cfg.precision == 1) {
    h.lat_Msf.resize(nms);
    launch_ranges(div_up(nms, 256), 256, [&](int b0, int nb) {
      hipLaunchKernelGGL((k_lat_mscale<P, float>), dim3(nb), dim3(256), 0, st, b0, nc, h.cRb.p, h.M.p, h.lat_Msf.p);
    });
  } else {
    h.lat_Ms.resize(nmd);
    launch_ranges(div_up(nmd, 256), 256, [&](int b0, int nb) {
      hipLaunchKernelGGL((k_lat_mscale<P, double>), dim3(nb), dim3(256), 0, st, b0, nc, h.cRb.p, h.M.p, h.lat_Ms.p);
    });
  }
}

// Largest slot array sized by the all-steps-active bound (512 MB of int).
constexpr int64_t kSlotBound = (int64_t)1 << 27;

// Levels of the current tree whose image pairs take part.
static LatImages lat_images(const Handle &h) {
  LatImages li;
  if (h.cfg.images == 0 || h.lat_img_off) return li;
  for (int l = 3; l < std::min(h.nlevels, kTileLevels - 1) && l <= 20; l++)
    if (2 * (int64_t)(h.lvl_off[l + 1] - h.lvl_off[l]) >= (int64_t)1 << (3 * l)) li.finest = l;
  li.cycle = h.cfg.cycle;
  return li;
}

// Offset keys: the lattice's, and the image offsets' in a periodic box.
static int lat_keys(const Handle &h) { return kLatKeys + (h.cfg.images > 0 ? kImgLevels * kImgLevelKeys : 0); }

// An empty T table for expansion order P in FP32 or FP64, no offset known.
static void tc_reset(Handle &h, int P, bool f32) {
  const int nk = lat_keys(h);
  h.lat_tc_map.resize(nk + 1);
  h.lat_ookey.resize(nk + 1);
  h.lat_hist.resize(nk + 8);
  for (int *p : {h.lat_tc_map.p, h.lat_ookey.p})
    hipLaunchKernelGGL(k_fill_int, dim3(div_up(nk + 1, 256)), dim3(256), 0, h.stream, p, (int64_t)nk + 1, -1);
  zero_device(h.lat_hist.p, nk + 7, h.stream);
  h.lat_tc_rows = h.lat_noff = h.lat_nreg = 0;
  for (int &i : h.lat_img0) i = 0;
  h.lat_tc_keyn = nk;
  h.lat_tc_P = P;
  h.lat_tc_f32 = f32;
}

// Grow a buffer to `want` elements, keeping its first `keep`.
template <typename R>
static void grow_keep_rows(Handle &h, DBuf<R> &b, size_t want, size_t keep) {
  if (want <= b.cap) return;
  DBuf<R> nb;
  nb.reserve(std::max(want, 2 * b.cap));
  if (keep) EXA_HIP(hipMemcpyAsync(nb.p, b.p, keep * sizeof(R), hipMemcpyDeviceToDevice, h.stream));
  EXA_HIP(hipStreamSynchronize(h.stream));
  b.release();
  b.p = nb.p;
  b.cap = nb.cap;
  b.n = want;
  nb.p = nullptr;
  nb.cap = 0;
}

static LatState *lat_state(Handle &h) { return reinterpret_cast<LatState *>(h.lat_act.p); }

// The contraction and the reduction of the last lattice set-up (its step
// lists, slots and tiles), on the main stream.
template <int P>
static void lattice_contract(Handle &h) {
  const int nitems = h.lat_run_ntiles * kLatSeg;
  if (h.cfg.precision == 1)
    hipLaunchKernelGGL((k_m2l_mfma<P, float>), dim3(h.lat_run_ngrid), dim3(256), 0, h.stream, h.ncells, nitems,
                       h.lat_step0.p, h.lat_alist.p, h.lat_slot.p, h.lat_Tf.p, h.lat_Msf.p, h.lat_part.p, lat_state(h));
  else
    hipLaunchKernelGGL((k_m2l_mfma<P, double>), dim3(h.lat_run_ngrid), dim3(256), 0, h.stream, h.ncells, nitems,
                       h.lat_step0.p, h.lat_alist.p, h.lat_slot.p, h.lat_T.p, h.lat_Ms.p, h.lat_part.p, lat_state(h));
  EXA_HIP(hipGetLastError());
}

template <int P>
static void lattice_reduce(Handle &h) {
  hipLaunchKernelGGL(k_lat_reduce<P>, dim3(h.lat_run_ntiles, MfmaShape<P>::RB), dim3(256), 0, h.stream,
                     h.lat_tile_tgt.p, h.lat_step0.p, h.cRb.p, h.lat_part.p, h.L.p, lat_state(h));
  EXA_HIP(hipGetLastError());
}

// Target tiles of the current tree, on stream st (its own scratch: this runs
// beside the traversal).
void run_lattice_tiles(Handle &h, hipStream_t st) {
  if (!lattice_applies(h)) return;
  const int nc = h.ncells, TPB = 256;
  TileLevels tl{};
  int base = 0, most = 0;
  tl.nlevels = std::min(h.nlevels, kTileLevels - 1);
  auto layout = [&](const int *octants) {
    base = most = 0;
    for (int l = 0; l <= kTileLevels; l++) {
      tl.off[l] = h.lvl_off[std::min(l, h.nlevels)];
      tl.base[l] = base;
      if (l == 0 || l >= tl.nlevels) continue;
      int group = std::min(h.lvl_par[l - 1], h.lvl_off[l + 1] - h.lvl_off[l]);
      if (octants) group = std::min(group, *std::max_element(octants + 8 * l, octants + 8 * l + 8));
      tl.cap[l] = group;
      most = std::max(most, group);
      base += 8 * div_up(group, 64);
    }
  };
  layout(nullptr);
  if (base > kTilesUnread) {
    int octants[8 * kTileLevels];
    h.lat_tcnt.resize(8 * kTileLevels);
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(256), 0, st, h.lat_tcnt.p, (int64_t)(8 * kTileLevels), 0);
    hipLaunchKernelGGL(k_tile_octants, dim3(std::min(1024, div_up(nc, 256))), dim3(256), 0, st, nc, h.cLevel.p,
                       h.cKey.p, h.key_lvloff, h.lat_tcnt.p);
    EXA_HIP(hipGetLastError());
    EXA_HIP(hipMemcpyAsync(octants, h.lat_tcnt.p, sizeof(octants), hipMemcpyDeviceToHost, st));
    EXA_HIP(hipStreamSynchronize(st));
    layout(octants);
  }
  h.lat_ntiles = base;
  h.lat_tbase.assign(tl.base, tl.base + kTileLevels + 1);
  h.lat_tile_of.resize(nc);
  h.lat_col_of.resize(nc);
  h.lat_tile_tgt.resize((size_t)std::max(1, base) * 64);
  if (base == 0) {
    hipLaunchKernelGGL(k_fill_int, dim3(div_up(nc, TPB)), dim3(TPB), 0, st, h.lat_tile_of.p, (int64_t)nc, -1);
  } else if (most <= kTileSort && h.nlevels < kTileLevels) {
    int p2 = 1;
    while (p2 < most) p2 *= 2;
    hipLaunchKernelGGL(k_tiles, dim3(8, tl.nlevels - 1), dim3(1024), p2 * sizeof(unsigned), st, tl, h.lvl_cells.p,
                       h.cKey.p, h.key_lvloff, h.lat_tile_tgt.p, h.lat_tile_of.p, h.lat_col_of.p);
  } else {
    h.lat_tkey.resize(2 * (size_t)nc);
    h.lat_tval.resize(2 * (size_t)nc);
    int *tk = h.lat_tkey.p, *tv = h.lat_tval.p;
    hipLaunchKernelGGL(k_tile_key, dim3(div_up(nc, TPB)), dim3(TPB), 0, st, nc, h.cLevel.p, h.cKey.p, h.key_lvloff, tk,
                       tv);
    bool alt = false;
    sort_pairs_int_int(tk, tk + nc, tv, tv + nc, nc, 8 + kTileClassBits, alt, st, h.tmp3);
    hipLaunchKernelGGL(k_fill_int, dim3(div_up((int64_t)base * 64, TPB)), dim3(TPB), 0, st, h.lat_tile_tgt.p,
                       (int64_t)base * 64, -1);
    hipLaunchKernelGGL(k_tile_assign, dim3(div_up(nc, TPB)), dim3(TPB), 0, st, nc, tl, alt ? tk + nc : tk,
                       alt ? tv + nc : tv, h.lat_tile_tgt.p, h.lat_tile_of.p, h.lat_col_of.p);
  }
  EXA_HIP(hipGetLastError());
}

// Steps and slots of the current M2L list with the offsets known so far, and
// the matrices of its image offsets.  Nothing waits for the device; whether
// every offset was known, and how many pairs are irregular, is read back
// behind it (ev_cnt).
template <int P>
static void lattice_steps(Handle &h) {
  const int64_t np = h.nm2l, nall = (int64_t)h.lat_ntiles * h.lat_noff;
  const int TPB = 256, gp = div_up(np, TPB);
  const int *ptgt = h.raw_mi.p, *psrc = h.raw_mj.p;
  LatState *const host = reinterpret_cast<LatState *>(h.hpin + kPinLat);
  if (nall > INT_MAX) throw Error(EXAFMM_HIP_EUNSUP, "lattice M2L: too many (tile, offset) steps");
  const LatImages li = lat_images(h);
  const int nimg = h.lat_noff - h.lat_nreg;
  LatRanges lr{};
  ImgLevels lvl{};
  lr.nreg = h.lat_nreg;
  int64_t nbound = (int64_t)h.lat_ntiles * h.lat_nreg;  // most steps
  for (int l = std::max(3, li.finest - kImgLevels + 1); l <= li.finest; l++) {
    const int i = lr.nlv++, slot = l % kImgLevels;
    lvl.cell[slot] = h.lvl_off[l];
    lr.tile0[i] = h.lat_tbase[l];
    lr.tile1[i] = h.lat_tbase[l + 1];
    lr.lo[i] = h.lat_img0[slot];
    lr.hi[i] = h.lat_img0[slot + 1];
    nbound += (int64_t)(lr.tile1[i] - lr.tile0[i]) * (lr.hi[i] - lr.lo[i]);
  }
  h.lat_act.resize(sizeof(LatState) + nall + h.lat_noff + 8);
  h.lat_aidx.resize(nall + 1);
  h.lat_pslot.resize(np);
  h.lat_tcnt.resize(h.lat_ntiles + 1);
  h.lat_step0.resize(h.lat_ntiles + 1);
  unsigned char *act = h.lat_act.p + sizeof(LatState), *used = act + nall;
  zero_device(h.lat_act.p, sizeof(LatState) + (nall + h.lat_noff + 7) / 8 * 8, h.stream);
  hipLaunchKernelGGL(k_lat_classify, dim3(std::min(gp, 4096)), dim3(TPB), 0, h.stream, ptgt, psrc, h.raw_mimg.p, np,
                     h.cX.p, h.cRb.p, h.lat_ookey.p, h.lat_tile_of.p, h.cLevel.p, li, h.lat_nreg, h.lat_noff, act,
                     used, h.lat_pslot.p, h.lat_hist.p, lat_state(h));
  // The image offsets' matrices beside the step lists (third stream).
  const bool image = nimg > 0 && li.finest >= 0;
  if (image) {
    const dim3 grid(div_up(nimg, kImgT), kImgTParts);
    EXA_HIP(hipEventRecord(h.ev_used, h.stream));
    EXA_HIP(hipStreamWaitEvent(h.stream3, h.ev_used, 0));
    if (h.lat_tc_f32)
      hipLaunchKernelGGL((k_lat_tmat_image<P, float>), grid, dim3(256), 0, h.stream3, h.lat_nreg, h.lat_noff,
                         h.lat_okey.p, h.lat_orow.p, used, lvl, h.lvl_cells.p, h.cRb.p, li.cycle, h.lat_Tf.p,
                         lat_state(h));
    else
      hipLaunchKernelGGL((k_lat_tmat_image<P, double>), grid, dim3(256), 0, h.stream3, h.lat_nreg, h.lat_noff,
                         h.lat_okey.p, h.lat_orow.p, used, lvl, h.lvl_cells.p, h.cRb.p, li.cycle, h.lat_T.p,
                         lat_state(h));
    EXA_HIP(hipEventRecord(h.ev_image, h.stream3));
  }
  if (nall > 0) {
    hipLaunchKernelGGL(k_lat_count, dim3(h.lat_ntiles), dim3(256), 0, h.stream, act, h.lat_noff, lr, h.lat_tcnt.p,
                       used);
    // Step lists sized for every (tile, offset) being in use, so that the
    // host need not wait for the count, unless that bound is large.
    int64_t nact = nbound;
    if (nbound * 64 > kSlotBound) {
      std::vector<int> cnt(h.lat_ntiles);
      EXA_HIP(hipMemcpyAsync(cnt.data(), h.lat_tcnt.p, h.lat_ntiles * sizeof(int), hipMemcpyDeviceToHost, h.stream));
      EXA_HIP(hipStreamSynchronize(h.stream));
      nact = 0;
      for (int c : cnt) nact += c;
    }
    if (nact * 64 > INT_MAX) throw Error(EXAFMM_HIP_EUNSUP, "lattice M2L: too many (tile, offset) steps");
    h.lat_alist.resize(nact > 0 ? nact : 1);
    h.lat_slot.resize(nact > 0 ? nact * 64 : 4);
    hipLaunchKernelGGL(k_lat_steps, dim3(h.lat_ntiles), dim3(256), 0, h.stream, act, h.lat_tcnt.p, h.lat_noff, lr,
                       used, h.lat_orow.p, h.lat_aidx.p, h.lat_step0.p, h.lat_alist.p,
                       reinterpret_cast<int4 *>(h.lat_slot.p), lat_state(h), host);
    if (!h.tree_given) EXA_HIP(hipEventRecord(h.ev_cnt, h.stream));
    hipLaunchKernelGGL(h.tree_given ? k_lat_slots<true> : k_lat_slots<false>, dim3(gp), dim3(TPB), 0, h.stream, ptgt,
                       psrc, np, h.lat_col_of.p, h.lat_aidx.p, h.lat_pslot.p, h.lat_slot.p, lat_state(h));
  }
  if (nall == 0 || h.tree_given) {  // (k_lat_slots may add irregular pairs)
    EXA_HIP(hipMemcpyAsync(host, lat_state(h), sizeof(LatState), hipMemcpyDeviceToHost, h.stream));
    EXA_HIP(hipEventRecord(h.ev_cnt, h.stream));
  }
  if (image) EXA_HIP(hipStreamWaitEvent(h.stream, h.ev_image, 0));
  EXA_HIP(hipGetLastError());
}

// The offsets that the last lattice_steps flagged as unknown: numbers for
// them (and new numbers for the others: in key order, so that a tile's steps
// come in the same order whatever the table held before) and rows of T(d).
template <int P>
static void lattice_register(Handle &h) {
  const int TPB = 256, nk = h.lat_tc_keyn, gk = div_up(nk + 1, TPB);
  const bool f32 = h.lat_tc_f32;
  const int *marks = h.hpin + kPinMarks;
  h.lat_flag.resize(nk + 1);
  h.lat_kscan.resize(nk + 1);
  h.lat_tc_flag.resize(nk + 1);
  h.lat_tc_scan.resize(nk + 1);
  for (int again = 0;; again++) {
    hipLaunchKernelGGL(k_lat_flag, dim3(gk), dim3(TPB), 0, h.stream, h.lat_hist.p, h.lat_ookey.p, h.lat_tc_map.p, nk,
                       h.lat_flag.p, h.lat_tc_flag.p);
    exclusive_scan_int(h, h.lat_flag.p, h.lat_kscan.p, nk + 1);
    exclusive_scan_int(h, h.lat_tc_flag.p, h.lat_tc_scan.p, nk + 1);
    hipLaunchKernelGGL(k_lat_marks, dim3(1), dim3(64), 0, h.stream, h.lat_kscan.p, h.lat_tc_scan.p, nk,
                       h.hpin + kPinMarks);
    EXA_HIP(hipStreamSynchronize(h.stream));
    // Image offsets that would make too many steps: none from here on.
    const bool drop = (int64_t)h.lat_ntiles * marks[0] > INT_MAX && marks[0] > marks[3] && !h.lat_img_off;
    if (drop) h.lat_img_off = true;
    if (!drop && (again || h.lat_tc_rows == 0 || h.lat_tc_rows + marks[1] <= h.lat_tc_max)) break;
    tc_reset(h, P, f32);  // start the table afresh with this list's offsets alone
    lattice_steps<P>(h);
  }
  const int noff = marks[0], nnew = marks[1], nlat = marks[2];
  for (int i = 0; i <= kImgLevels; i++) h.lat_img0[i] = marks[3 + i];
  h.lat_nreg = marks[3];
  h.lat_okey.resize(std::max(1, noff));
  h.lat_tc_keys.resize(std::max(1, nnew));
  h.lat_orow.resize(std::max(1, noff));
  hipLaunchKernelGGL(k_lat_number, dim3(gk), dim3(TPB), 0, h.stream, h.lat_flag.p, h.lat_kscan.p, h.lat_tc_flag.p,
                     h.lat_tc_scan.p, nk, h.lat_tc_rows, h.lat_tc_map.p, h.lat_tc_keys.p, h.lat_ookey.p, h.lat_okey.p,
                     h.lat_orow.p, h.lat_hist.p);
  h.lat_noff = noff;
  if (nnew > 0) {
    if (f32) {
      constexpr size_t TEP = TPad<P, float>::TEP;
      grow_keep_rows(h, h.lat_Tf, (size_t)(h.lat_tc_rows + nnew) * TEP, (size_t)h.lat_tc_rows * TEP);
      if (nlat > 0)
        hipLaunchKernelGGL((k_lat_tmat<P, float>), dim3(nlat), dim3(64), 0, h.stream, h.lat_tc_keys.p,
                           h.lat_Tf.p + (size_t)h.lat_tc_rows * TEP);
    } else {
      constexpr size_t TEP = TPad<P, double>::TEP;
      grow_keep_rows(h, h.lat_T, (size_t)(h.lat_tc_rows + nnew) * TEP, (size_t)h.lat_tc_rows * TEP);
      if (nlat > 0)
        hipLaunchKernelGGL((k_lat_tmat<P, double>), dim3(nlat), dim3(64), 0, h.stream, h.lat_tc_keys.p,
                           h.lat_T.p + (size_t)h.lat_tc_rows * TEP);
    }
    h.lat_tc_rows += nnew;
  }
  EXA_HIP(hipGetLastError());
}

// The set-up, queued before P2P so that it runs while the P2P list is
// grouped, before P2P fills the GPU.
template <int P>
static void lattice_begin(Handle &h) {
  const bool f32 = h.cfg.precision == 1;
  // Source multipoles scaled per cell and the tiles (independent of the
  // lists; already queued behind the radii when the upward pass was split).
  if (!h.lat_ms_ready) mscale_impl<P>(h, h.stream);
  h.lat_ms_ready = false;
  if (h.lat_tiles_ready)
    EXA_HIP(hipStreamWaitEvent(h.stream, h.ev_tiles, 0));
  else
    run_lattice_tiles(h, h.stream);
  h.lat_tiles_ready = false;
  if (h.lat_tc_P != P || h.lat_tc_f32 != f32 || h.lat_tc_keyn != lat_keys(h) ||
      (int64_t)h.lat_ntiles * h.lat_noff > INT_MAX)
    tc_reset(h, P, f32);
  lattice_steps<P>(h);
  if (h.lat_noff == 0) {  // no offset known yet: register them before P2P fills the GPU
    EXA_HIP(hipEventSynchronize(h.ev_cnt));
    if (reinterpret_cast<const LatState *>(h.hpin + kPinLat)->unknown) {
      lattice_register<P>(h);
      lattice_steps<P>(h);
    }
  }
  h.lat_begun = true;
}

template <int P>
static void lattice_run(Handle &h, M2LList &irr) {
  using S = MfmaShape<P>;
  const int64_t np = h.nm2l;
  const int TPB = 256;
  const int gp = div_up(np, TPB);
  if (!h.lat_begun) lattice_begin<P>(h);
  h.lat_begun = false;
  const LatState *ls = reinterpret_cast<const LatState *>(h.hpin + kPinLat);
  const int ntiles = h.lat_ntiles;
  h.lat_stats_tiles = 0;
  join_multipoles(h);  // the set-up above did not need them
  // Irregular pairs are expected: they are grouped and translated on the third
  // stream beside the contraction, and the reduction adds to their result
  // (lattice_finish).  Behind the reduction on the main stream instead, a box
  // of 64^3 bodies (237000 of 11.5 M pairs irregular) took 5.09 ms, not 4.81,
  // and 4.2 M clustered bodies 22.7 ms, not 22.2.
  const bool irregular = (h.cfg.images > 0 || h.cfg.builder == 1) && !h.serial_heavy;
  // The contraction (timed by ev[12..13]) and the reduction: queued on the
  // set-up as it is; both do nothing if it met an unknown offset, and are
  // queued again after that offset has its row.
  for (int again = 0;; again++) {
    h.lat_run_ntiles = 0;
    if (h.lat_noff > 0 && ntiles > 0) {
      h.lat_part.resize((size_t)ntiles * kLatSeg * S::RB * 16 * 64);
      // One workgroup per item, or lat_wg_cu workgroups per CU looping over
      // the items (room left on every CU for the P2P waves of the other stream).
      const int nitems = ntiles * kLatSeg;
      int ngrid = nitems;
      if (h.lat_wg_cu > 0) ngrid = std::min(ngrid, std::max(kLatSeg, (h.lat_wg_cu * h.ncu) / kLatSeg * kLatSeg));
      h.lat_run_ntiles = ntiles;
      h.lat_run_ngrid = ngrid;
      if (h.serial_heavy) EXA_HIP(hipStreamWaitEvent(h.stream, h.ev[10], 0));  // P2P's end (second stream)
      EXA_HIP(hipEventRecord(h.ev[12], h.stream));
      h.lat_timed = true;
      lattice_contract<P>(h);
      EXA_HIP(hipEventRecord(h.ev[13], h.stream));
      if (!irregular) lattice_reduce<P>(h);
    }
    EXA_HIP(hipEventSynchronize(h.ev_cnt));
    if (!ls->unknown) break;
    if (again) throw Error(EXAFMM_HIP_EDEVICE, "lattice M2L: offsets unknown after their registration");
    lattice_register<P>(h);
    lattice_steps<P>(h);
  }
  const int nirr = ls->nirr;
  h.lat_stats_steps = h.lat_run_ntiles ? ls->nsteps : 0;
  h.lat_stats_tiles = h.lat_run_ntiles ? ls->ntiles : 0;
  h.lat_stats_noff = h.lat_run_ntiles ? ls->noffs : 0;
  h.lat_reduce_pending = irregular && h.lat_run_ntiles > 0;
  int nitl = 0;
  if (nirr) {
    if (h.lat_reduce_pending) EXA_HIP(hipStreamWaitEvent(h.stream3, h.ev_cnt, 0));
    group_irregular(h, h.lat_reduce_pending ? h.stream3 : h.stream, nirr, nitl);
  }
  irr = M2LList{h.irr_tgt.p, nitl, h.irr_off.p, h.irr_src.p, h.irr_img.p, nirr};
  h.lat_stats_pairs = np - nirr;
  EXA_HIP(hipGetLastError());
}

// The reduction left by run_m2l_lattice, behind the per-pair kernel on the
// third stream.
void lattice_finish(Handle &h) {
  if (!h.lat_reduce_pending) return;
  h.lat_reduce_pending = false;
  EXA_HIP(hipEventRecord(h.ev_image, h.stream3));
  EXA_HIP(hipStreamWaitEvent(h.stream, h.ev_image, 0));
  switch (h.cfg.P) {
    case 4: lattice_reduce<4>(h); break;
    case 6: lattice_reduce<6>(h); break;
    case 8: lattice_reduce<8>(h); break;
    case 10: lattice_reduce<10>(h); break;
    case 12: lattice_reduce<12>(h); break;
  }
}

bool lattice_applies(const Handle &h) {
  return h.cfg.basis == 0 && !h.cfg.mass && h.lattice_m2l && h.cfg.P >= 4 && h.cfg.P <= 12 && (h.cfg.P % 2) == 0;
}

// Scaled source multipoles for the lattice contraction, queued on stream st
// right behind the multipoles (the split upward pass).
void run_lattice_mscale(Handle &h, hipStream_t st) {
  if (!lattice_applies(h)) return;
  switch (h.cfg.P) {
    case 4: mscale_impl<4>(h, st); break;
    case 6: mscale_impl<6>(h, st); break;
    case 8: mscale_impl<8>(h, st); break;
    case 10: mscale_impl<10>(h, st); break;
    case 12: mscale_impl<12>(h, st); break;
  }
  EXA_HIP(hipGetLastError());
  h.lat_ms_ready = true;
}

void m2l_begin(Handle &h) {
  h.lat_begun = false;
  if (!lattice_applies(h) || h.nm2l == 0) {
    h.lat_ms_ready = h.lat_tiles_ready = false;  // queued scaled multipoles and tiles (if any) go unused
    return;
  }
  switch (h.cfg.P) {
    case 4: lattice_begin<4>(h); break;
    case 6: lattice_begin<6>(h); break;
    case 8: lattice_begin<8>(h); break;
    case 10: lattice_begin<10>(h); break;
    case 12: lattice_begin<12>(h); break;
  }
  EXA_HIP(hipGetLastError());
}

// The lattice contraction and reduction again on the current multipoles,
// with the set-up of the last run_m2l_lattice (same tree and lists).
void lattice_replay(Handle &h) {
  if (!lattice_applies(h) || h.nm2l == 0 || h.lat_run_ntiles == 0) return;
  switch (h.cfg.P) {
    case 4: lattice_contract<4>(h); lattice_reduce<4>(h); break;
    case 6: lattice_contract<6>(h); lattice_reduce<6>(h); break;
    case 8: lattice_contract<8>(h); lattice_reduce<8>(h); break;
    case 10: lattice_contract<10>(h); lattice_reduce<10>(h); break;
    case 12: lattice_contract<12>(h); lattice_reduce<12>(h); break;
  }
}

void lattice_reset(Handle &h) {
  h.lat_timed = h.lat_reduce_pending = false;
  h.lat_run_ntiles = 0;
  h.lat_stats_pairs = 0;
  h.lat_stats_tiles = h.lat_stats_noff = 0;
  h.lat_stats_steps = 0;
}

bool run_m2l_lattice(Handle &h, M2LList &irr) {
  if (!lattice_applies(h) || h.nm2l == 0) {
    h.lat_ms_ready = h.lat_tiles_ready = false;
    return false;
  }
  switch (h.cfg.P) {
    case 4: lattice_run<4>(h, irr); return true;
    case 6: lattice_run<6>(h, irr); return true;
    case 8: lattice_run<8>(h, irr); return true;
    case 10: lattice_run<10>(h, irr); return true;
    case 12: lattice_run<12>(h, irr); return true;
    default: return false;
  }
}

}  // namespace exafmm
