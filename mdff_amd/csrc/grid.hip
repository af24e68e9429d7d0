// grid.hip -- reciprocal-space Ewald sums through a uniform grid (grid.h).
//
// The structure factors of all k = 2 pi B n, |n_a| <= kmax_a, are a
// non-uniform Fourier transform of the moments, and the field at the atoms
// its adjoint.  With a kernel phi of support W grid cells whose transform is
// phi^:
//
//   G(l)  = sum_j (q_j + mu_j . d/dr_j) prod_a phi(y_aj - l_a)      spread
//   S(n)  = sum_l G(l) e^{2 pi i n.l/M} / phi^(n)                   transform
//   b(l)  = sum_n A_n S(n) e^{-2 pi i n.l/M} / phi^(n)              back
//   psi(r)= sum_l b(l) prod_a phi(y_a - l_a)                        interpolate
//
// and the field and its gradient are the first and second derivatives of
// phi in the last sum.  This evaluates the very sum over the k mesh that the
// direct kernels evaluate (no Ewald term is approximated); the error is that
// of the kernel, set below the rounding of the arithmetic type: the kernel
// sqrt(1-z^2) I1(beta sqrt(1-z^2)), z = 2x/W, beta = pi W (1 - 1/(2 sigma)),
// on a grid of M >= 1.95 (2 kmax + 1) points per axis (sigma = M /
// (2 kmax + 1)) leaves 3e-15, 4e-15 and 9e-15 relative in psi and its first
// and second derivatives at W = 17 (7e-14 in the second at W = 16), and
// 8e-10, 9e-9 and 9e-8 at W = 10.  The derivatives have polynomials of their
// own (fitted in long double), so that no digit is lost by differentiating a
// fit.  Errors of a whole evaluation against a plain FP64 sum over every k,
// 24,576 atoms, kmax 24 (direct kernels in brackets): FP64 forces 1.5e-14
// (1.2e-14), EFGs 1.2e-14 (1.1e-14); mixed forces 5.4e-7 (5.4e-7), dipoles
// 3.5e-7 (5.4e-7).
//
// Work: 2 W^3 terms per atom and O(M^3 kmax) for the transforms, against
// O(kmax^3) per atom for the direct sum: at 24,576 atoms and kmax 24
// (58,824 k) 1e4 against 6e5 terms per atom.  Evaluations of 12 Ewald calls
// with the direct sums and with the grid in one build, ms: 24,576 atoms at
// kmax 20 7.79 / 2.26 FP64, 1.90 / 1.17 mixed; 3000 at kmax 24 2.53 / 0.96,
// 1.80 / 0.80; 3072 at kmax 10 1.25 / 0.84, 1.23 / 0.65.
//
// Every step is a gather (a workgroup owns its tile of the grid, a wave its
// atom) with a fixed order of summation: results are bitwise reproducible.
//
// The transforms keep only the 2 kmax + 1 modes of each axis and are dense
// products with the cosine and sine tables on the matrix cores
// (v_mfma_f64_16x16x4), each axis folded to its even and odd halves (a
// quarter of the products of the complex form).  The grid points sit at
// half-integer positions l + 1/2, so that an even axis folds onto M/2 pairs
// without fixed points.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "grid.h"
#include "kernels.h"

namespace mdff {
namespace grid {

constexpr int TX = 16, TY = 8, TZ = 8;  // tile of the grid owned by a workgroup
constexpr int MMAX = 448;               // grid points per axis (LDS of the transforms)
constexpr int W64 = 17, W32 = 10;       // kernel support, FP64 / FP32
constexpr int DEG64 = 22, DEG32 = 13;   // degree of its polynomial pieces
constexpr int HS = 40;                  // LDS row of the (y, n3) planes: 32 + bank offset

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename R>
struct Mat;
template <>
struct Mat<double> {
  typedef v4d acc;
  // ZV: z per lane of the interpolation; PADZ: padding of the potential's
  // rows, at least W - 1
  static constexpr int W = W64, DEG = DEG64, ZV = 1, PADZ = 20;
  static __device__ __forceinline__ v4d mma(double a, double b, v4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // row of accumulator element i in lane l (column l & 15)
  static __device__ __forceinline__ int row(int l, int i) { return 4 * i + (l >> 4); }
};
template <>
struct Mat<float> {
  typedef v4f acc;
  static constexpr int W = W32, DEG = DEG32, ZV = 2, PADZ = 12;
  static __device__ __forceinline__ v4f mma(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int l, int i) { return 4 * (l >> 4) + i; }
};

// Extents of a plan, passed to every kernel by value.
struct Ext {
  int M[3];    // grid points per axis: M1 a multiple of 16, M2 and M3 of 8
  int k[3];    // kmax
  int nt[3];   // tiles per axis (also the bins)
  int ntile;   // tiles of one configuration
  int N2f;     // 2 k2 + 1
  int N3c;     // k3 + 1
  int NCC;     // N2f N3c columns of the (n2, n3) plane
  int np[3];   // modes 0..k of an axis, padded to 16 (column stride of F)
  int xp[3];   // folded points M/2, padded to 16 (column stride of T)
  int nseg;
  size_t ng;   // M1 M2 M3
  size_t nm;   // (2 k1 + 1) NCC
};

// Twiddles of an axis, half-point phases t = 2 pi n (l + 1/2) / M:
//   Fc, Fs [l < xp][np]    cos t, sin t (zero past M/2 and kmax)
//   Tc, Ts [n < np][xp]    the same transposed (zero past kmax and M/2)
struct Tw {
  const double *Fc[3], *Fs[3], *Tc[3], *Ts[3];
};

struct Plan {
  Ext e;
  bool fp64 = true;
  std::vector<Seg> segs;
  int natom = 0;            // atoms of all configurations
  std::vector<void*> allocs;
  Seg* d_seg = nullptr;
  Tw tw;
  double* d_phat = nullptr;  // 1 / phi^ of modes 0..k, axis after axis
  int phoff[3] = {0, 0, 0};
  void* d_poly = nullptr;    // [axis][phi, phi', phi''][DEG + 1][W]
  void* d_G = nullptr;       // grids, [seg][x][y][z]
  double2* d_T = nullptr;    // [seg][x][n2][n3]
  double* d_D = nullptr;     // Ewald factors / phi^^2, [seg][n1][n2][n3]
  void* d_tab = nullptr;     // [atom][axis][phi, phi'][W]
  void* d_tab2 = nullptr;    // [atom][axis][W], phi''
  int4* d_l0 = nullptr;      // first points of the supports
  void* d_P = nullptr;       // potentials, [seg][x][y][M3 + PADZ]
  // bins: two classes (active atoms, the others) of nseg x ntile bins
  int *d_key = nullptr, *d_start = nullptr, *d_cur = nullptr, *d_perm0 = nullptr,
      *d_perm = nullptr;
  int margin[3] = {0, 0, 0};
  // tile lists one after the other, each with room for its candidates at the
  // binning: the first slots (one more than tiles), their number and the
  // slots allocated; per tile (first slot, active atoms, all atoms)
  int* d_off = nullptr;
  unsigned long long* d_total = nullptr;
  long long slots = 0;
  int2* d_ov = nullptr;
  int4* d_cnt = nullptr;
  int nact = 0;           // active atoms
  int split = 1;          // partial grids of the spread
  bool is_binned = false;
  const int* cfg = nullptr;  // configuration of each atom (the caller's), or null: one
};

// ---------------------------------------------------------------------------
// host side: the kernel, its polynomials and its transform

typedef long double LD;

// phi, phi', phi'' at x (in cells, |x| <= W/2): the power series of
// s I1(beta s) in s^2 = 1 - z^2 has positive terms only, so that value and
// derivatives keep full relative precision.
struct Kernel {
  LD h;
  std::vector<LD> c;
  Kernel(int W, LD beta) : h(W / (LD)2) {
    LD t = beta / 2, mx = 0, sum = 0;
    for (int m = 0;; ++m) {
      c.push_back(t);
      sum += t;
      mx = std::max(mx, t);
      if (m > beta && t < 1e-25L * mx) break;
      t = t * (beta / 2) * (beta / 2) / ((LD)(m + 1) * (m + 2));
    }
    for (LD& v : c) v /= sum;
  }
  void eval(LD x, LD out[3]) const {
    const LD z = x / h, q = 1 - z * z;
    LD g = 0, g1 = 0, g2 = 0;
    for (size_t k = c.size(); k-- > 0;) {
      g2 = g2 * q + 2 * g1;
      g1 = g1 * q + g;
      g = g * q + c[k];
    }
    const LD F1 = g + q * g1, F2 = 2 * g1 + q * g2;
    out[0] = q * g;
    out[1] = -2 * z * F1 / h;
    out[2] = (-2 * F1 + 4 * z * z * F2) / (h * h);
  }
};

// Monomial coefficients (in u in [-1, 1]) of the Chebyshev interpolants of
// phi, phi', phi'' on each cell x = (u + 1)/2 + p - W/2, layout [f][deg+1][W].
static void fit(const Kernel& K, int W, int deg, std::vector<LD>& out) {
  const int n = deg + 1;
  const LD pi = acosl(-1.0L);
  out.assign((size_t)3 * n * W, 0);
  std::vector<LD> cs((size_t)n * n), v(3 * n);  // cos(k theta_j)
  for (int k = 0; k < n; ++k)
    for (int j = 0; j < n; ++j) cs[(size_t)k * n + j] = cosl(k * (pi * (j + 0.5L) / n));
  for (int p = 0; p < W; ++p) {
    for (int j = 0; j < n; ++j) {
      LD f[3];
      K.eval((cs[n + j] + 1) / 2 + p - K.h, f);
      for (int d = 0; d < 3; ++d) v[d * n + j] = f[d];
    }
    for (int d = 0; d < 3; ++d) {
      std::vector<LD> a(n, 0), t0(n, 0), t1(n, 0), t2(n);
      t0[0] = 1;
      if (n > 1) t1[1] = 1;
      for (int k = 0; k < n; ++k) {
        LD s = 0;
        for (int j = 0; j < n; ++j) s += v[d * n + j] * cs[(size_t)k * n + j];
        s *= (k ? 2.0L : 1.0L) / n;
        const std::vector<LD>& T = k == 0 ? t0 : t1;
        for (int m = 0; m < n; ++m) a[m] += s * T[m];
        if (k >= 1) {
          for (int m = 0; m < n; ++m) t2[m] = (m ? 2 * t1[m - 1] : 0) - t0[m];
          t0 = t1;
          t1 = t2;
        }
      }
      for (int m = 0; m < n; ++m) out[((size_t)d * n + m) * W + p] = a[m];
    }
  }
}

// phi^(n) = int phi(x) cos(2 pi n x / M) dx, Gauss-Legendre on each cell.
static void transform(const Kernel& K, int W, int M, int kmax, std::vector<double>& out) {
  constexpr int NG = 40;
  const LD pi = acosl(-1.0L);
  LD x[NG], w[NG];
  for (int i = 0; i < NG; ++i) {
    LD t = cosl(pi * (i + 0.75L) / (NG + 0.5L)), d = 1;
    for (int it = 0; it < 100; ++it) {
      LD p0 = 1, p1 = t;
      for (int k = 2; k <= NG; ++k) {
        const LD p2 = ((2 * k - 1) * t * p1 - (k - 1) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      d = NG * (t * p1 - p0) / (t * t - 1);
      const LD dt = p1 / d;
      t -= dt;
      if (fabsl(dt) < 1e-19L) break;
    }
    x[i] = t;
    w[i] = 2 / ((1 - t * t) * d * d);
  }
  std::vector<LD> s(kmax + 1, 0);
  for (int p = 0; p < W; ++p)
    for (int i = 0; i < NG; ++i) {
      const LD xx = (x[i] + 1) / 2 + p - K.h;
      LD f[3];
      K.eval(xx, f);
      // cos(n t) by its recurrence
      const LD c = cosl(2 * pi * xx / M);
      LD c0 = 1, c1 = c;
      for (int n = 0; n <= kmax; ++n) {
        s[n] += w[i] / 2 * f[0] * c0;
        const LD c2 = 2 * c * c1 - c0;
        c0 = c1;
        c1 = c2;
      }
    }
  out.resize(kmax + 1);
  for (int n = 0; n <= kmax; ++n) out[n] = (double)(1 / s[n]);
}

// ---------------------------------------------------------------------------
// device helpers

// Grid coordinate, first point of the support and the piece coordinate u of
// a fractional coordinate: points l0 .. l0 + W - 1 (l0 reduced mod M), point
// a at piece W - 1 - a, all at the same u in [-1, 1].
template <int W>
__device__ __forceinline__ int support(double s, int M, double& u) {
  const double y = (s - floor(s)) * M - 0.5;
  const double c = ceil(y - 0.5 * W);
  u = 2.0 * (y - c - 0.5 * W) + 1.0;
  int l = (int)c;
  l = l < 0 ? l + M : l;
  return min(max(l, 0), M - 1);  // also for coordinates that are not finite
}

__device__ __forceinline__ int wrap(int x, int M) { return x < 0 ? x + M : (x >= M ? x - M : x); }

// ---------------------------------------------------------------------------
// binning (at a list build)

template <int W>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_bin(int n, Ext e, const double4* __restrict__ s4,
                                                         const int* __restrict__ typ,
                                                         const int* __restrict__ cfg,
                                                         unsigned active, int* __restrict__ key,
                                                         int* __restrict__ cnt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double4 s = s4[i];
  double u;
  const int bx = support<W>(s.x, e.M[0], u) / TX, by = support<W>(s.y, e.M[1], u) / TY,
            bz = support<W>(s.z, e.M[2], u) / TZ;
  const int cls = ((active >> typ[i]) & 1u) ? 0 : 1;
  const int seg = cfg ? cfg[i] : 0;
  const int k = (cls * e.nseg + seg) * e.ntile + (bx * e.nt[1] + by) * e.nt[2] + bz;
  key[i] = k;
  atomicAdd(&cnt[k + 1], 1);  // k_cell_scan turns these into bin starts
}

// Bins a tile's candidates may sit in, along one axis: atoms whose support
// starts within W - 1 points before the tile or in it, give or take margin.
struct BinRange {
  int lo, n;
};
template <int W>
__device__ __forceinline__ BinRange bin_range(int t, int T, int nt, int margin) {
  const int before = (W - 1 + margin + T - 1) / T;        // whole bins before the tile
  const int after = (T - 1 + margin) / T;                 // and after it
  const int n = min(before + after + 1, nt);
  int lo = t - before;
  lo %= nt;
  return {lo < 0 ? lo + nt : lo, n};
}

// Row r of a tile's candidate rows: bins (bx, by) fixed, the bz range as one
// or two runs of consecutive bins (part 0 / 1); returns its atoms as
// [first, first + len) of the bin order.
template <int W>
struct Cands {
  BinRange x, y, z;
  int rows;
  __device__ __forceinline__ Cands(const Ext& e, const int* m, int tile) {
    const int tz = tile % e.nt[2], ty = (tile / e.nt[2]) % e.nt[1],
              tx = tile / (e.nt[2] * e.nt[1]);
    x = bin_range<W>(tx, TX, e.nt[0], m[0]);
    y = bin_range<W>(ty, TY, e.nt[1], m[1]);
    z = bin_range<W>(tz, TZ, e.nt[2], m[2]);
    rows = 2 * x.n * y.n;
  }
  __device__ __forceinline__ int2 run(const Ext& e, const int* start, int base, int r) const {
    const int part = r & 1, q = r >> 1;
    int bx = x.lo + q / y.n, by = y.lo + q % y.n;
    bx -= bx >= e.nt[0] ? e.nt[0] : 0;
    by -= by >= e.nt[1] ? e.nt[1] : 0;
    const int b = base + (bx * e.nt[1] + by) * e.nt[2];
    const int end = z.lo + z.n;
    const int b0 = part ? 0 : z.lo, b1 = part ? max(0, end - e.nt[2]) : min(end, e.nt[2]);
    const int s = start[b + b0];
    return make_int2(s, start[b + b1] - s);
  }
};

struct Margin {
  int m[3];
};

// Candidates of every tile (room[tile + 1], for k_cell_scan) and of all.
template <int W>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_cap(Ext e, Margin mg,
                                                         const int* __restrict__ start,
                                                         int* __restrict__ room,
                                                         unsigned long long* __restrict__ total) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= e.ntile * e.nseg) return;
  const Cands<W> c(e, mg.m, t % e.ntile);
  int tot = 0;
  for (int cls = 0; cls < 2; ++cls)
    for (int r = 0; r < c.rows; ++r)
      tot += c.run(e, start, (cls * e.nseg + t / e.ntile) * e.ntile, r).y;
  if (t == 0) room[0] = 0;
  room[t + 1] = tot;
  atomicAdd(total, (unsigned long long)tot);
}

// ---------------------------------------------------------------------------
// per evaluation: tile lists and kernel values

// The atoms whose support overlaps a tile, active atoms first, each class in
// bin order, as (atom, offsets of the support's start from the tile + 64 in
// three bytes); cnt = (first slot, active, all).  One workgroup per tile tests the
// candidates of the neighbouring bins and compacts the hits with ballots, so
// that the order is fixed.
template <int W>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_lists(
    Ext e, Margin mg, const double4* __restrict__ s4, const int* __restrict__ start,
    const int* __restrict__ perm, const int* __restrict__ off, int2* __restrict__ ov,
    int4* __restrict__ cnt) {
  __shared__ int first[MDFF_BLOCK], pre[MDFF_BLOCK + 1], wsum[4];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int tile = blockIdx.x, seg = blockIdx.y;
  const size_t at = (size_t)seg * e.ntile + tile;
  const int first_slot = off[at], cap = off[at + 1] - first_slot;
  const int z0 = (tile % e.nt[2]) * TZ, y0 = ((tile / e.nt[2]) % e.nt[1]) * TY,
            x0 = tile / (e.nt[2] * e.nt[1]) * TX;
  const Cands<W> c(e, mg.m, tile);
  int nov = 0, act = 0;
  for (int cls = 0; cls < 2; ++cls) {
    for (int r0 = 0; r0 < c.rows; r0 += MDFF_BLOCK) {
      int2 run = make_int2(0, 0);
      if (r0 + t < c.rows) run = c.run(e, start, (cls * e.nseg + seg) * e.ntile, r0 + t);
      // inclusive prefix of the run lengths
      int inc = run.y;
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
      }
      if (lane == 63) wsum[wv] = inc;
      __syncthreads();
      for (int k = 0; k < wv; ++k) inc += wsum[k];
      first[t] = run.x;
      pre[t + 1] = inc;
      if (t == 0) pre[0] = 0;
      __syncthreads();
      const int total = pre[MDFF_BLOCK];
      for (int v0 = 0; v0 < total; v0 += MDFF_BLOCK) {
        const int v = v0 + t;
        bool o = false;
        int2 ent = make_int2(0, 0);
        if (v < total) {
          int r = 0;
          for (int step = MDFF_BLOCK / 2; step > 0; step >>= 1)
            if (pre[r + step] <= v) r += step;
          const int a = perm[first[r] + v - pre[r]];
          const double4 s = s4[a];
          double u;
          int dx = wrap(support<W>(s.x, e.M[0], u) - x0, e.M[0]);
          int dy = wrap(support<W>(s.y, e.M[1], u) - y0, e.M[1]);
          int dz = wrap(support<W>(s.z, e.M[2], u) - z0, e.M[2]);
          o = true;
          if (dx >= TX) {
            o = o && dx > e.M[0] - W;
            dx -= e.M[0];
          }
          if (dy >= TY) {
            o = o && dy > e.M[1] - W;
            dy -= e.M[1];
          }
          if (dz >= TZ) {
            o = o && dz > e.M[2] - W;
            dz -= e.M[2];
          }
          ent = make_int2(a, (dx + 64) | (dy + 64) << 8 | (dz + 64) << 16);
        }
        const unsigned long long bo = __ballot(o);
        if (lane == 0) wsum[wv] = __popcll(bo);
        __syncthreads();
        int po = nov + __popcll(bo & ((1ull << lane) - 1ull));
        for (int k = 0; k < 4; ++k) {
          if (k < wv) po += wsum[k];
          nov += wsum[k];
        }
        if (o && po < cap) ov[(size_t)first_slot + po] = ent;
        __syncthreads();
      }
      __syncthreads();
    }
    if (cls == 0) act = nov;
  }
  if (t == 0) cnt[at] = make_int4(first_slot, min(act, cap), min(nov, cap), 0);
}

// Kernel values of every atom: tab[atom][axis][phi, phi'][W] and
// tab2[atom][axis][phi''][W], and the first points l0[atom] of its support.
// One thread per (atom, axis, point); the coefficients in LDS with the piece
// fastest, so that the lanes of an atom read consecutive words.
template <typename R>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_tab(int n, Ext e, const double4* __restrict__ s4,
                                                         const R* __restrict__ poly,
                                                         R* __restrict__ tab,
                                                         R* __restrict__ tab2,
                                                         int* __restrict__ l0) {
  constexpr int W = Mat<R>::W, D = Mat<R>::DEG + 1;
  __shared__ R pc[9 * D * W];
  for (int k = threadIdx.x; k < 9 * D * W; k += MDFF_BLOCK) pc[k] = poly[k];
  __syncthreads();
  const long long total = (long long)n * 3 * W;
  for (long long g = (long long)blockIdx.x * MDFF_BLOCK + threadIdx.x; g < total;
       g += (long long)gridDim.x * MDFF_BLOCK) {
    const int a = (int)(g % W);
    const int ax = (int)(g / W % 3);
    const int i = (int)(g / (3 * W));
    const double* sp = reinterpret_cast<const double*>(s4 + i);
    double ud;
    const int l = support<W>(sp[ax], e.M[ax], ud);
    if (a == 0) l0[4 * (size_t)i + ax] = l;
    const R u = (R)ud;
    const R* c = pc + (size_t)ax * 3 * D * W + (W - 1 - a);
    R f0 = 0, f1 = 0, f2 = 0;
#pragma unroll
    for (int m = D - 1; m >= 0; --m) {
      f0 = f0 * u + c[m * W];
      f1 = f1 * u + c[(D + m) * W];
      f2 = f2 * u + c[(2 * D + m) * W];
    }
    R* o = tab + ((size_t)i * 3 + ax) * 2 * W + a;
    o[0] = f0;
    o[W] = f1;
    tab2[((size_t)i * 3 + ax) * W + a] = f2;
  }
}

// Tiles in an order that keeps the tiles of one XCD (blocks b, b + 8, ..)
// next to each other: their grid regions and atoms then share its L2.
__device__ __forceinline__ int xcd_tile(int b, int n) {
  const int per = (n + 7) / 8;
  return (b & 7) * per + (b >> 3);
}
static int xcd_blocks(int n) { return (n + 7) / 8 * 8; }

// ---------------------------------------------------------------------------
// spread

// A workgroup owns a 16 x 8 x 8 tile of the grid and sums its overlapping
// atoms as a matrix product on the matrix cores: rows are the 16 x points,
// columns the 64 (y, z) points (wave w: y = 2 w, 2 w + 1), and K runs over
// the atoms, two terms each for dipoles:
//   G = sum_j (mx phi'_x) (phi_y phi_z) + phi_x ((q phi_y + my phi'_y) phi_z + phi_y mz phi'_z).
// The factors of 32 atoms at a time are expanded to the tile's points in LDS
// (zero outside an atom's support), the next 32 loaded while the current
// ones multiply; no zeroed grid and no atomics.  The tile shape makes
// (W + 15)(W + 7)^2 / W^3 products per term of the support: 3.7 at W = 17,
// 7.2 at W = 10.  Where the grid
// has few tiles, gridDim.z (one or two) blocks share a tile's atoms and write partial
// grids, which the forward transform adds.
constexpr int SCH = 32;  // atoms per LDS chunk

template <typename R, bool CHG, bool DIP>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_spread(
    Ext e, const Seg* __restrict__ segs, const double* __restrict__ q,
    const double* __restrict__ mu, int n, const R* __restrict__ tab,
    const int2* __restrict__ list, const int4* __restrict__ cnt, int act,
    R* __restrict__ G) {
  constexpr int W = Mat<R>::W;
  typedef typename Mat<R>::acc acc_t;
  struct R2 {
    R x, y;
  };
  __shared__ R lx[SCH][2][TX];
  __shared__ R2 ly[SCH][TY], lz[SCH][TZ];
  const int tile = xcd_tile(blockIdx.x, e.ntile), seg = blockIdx.y;
  if (tile >= e.ntile) return;
  const size_t at = (size_t)seg * e.ntile + tile;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int4 cc = cnt[at];
  // this block's share of the list (gridDim.z partial grids)
  const int tot = act ? cc.y : cc.z;
  const int lo = (int)((long long)tot * blockIdx.z / gridDim.z);
  const int m = (int)((long long)tot * (blockIdx.z + 1) / gridDim.z) - lo;
  const int2* lst = list + (size_t)cc.x + lo;
  const int z0 = (tile % e.nt[2]) * TZ, y0 = ((tile / e.nt[2]) % e.nt[1]) * TY,
            x0 = tile / (e.nt[2] * e.nt[1]) * TX;
  const Cell& cell = segs[seg].cell;
  const int al = t >> 3, pp = t & 7;  // 8 threads expand an atom
  // this thread's share of a chunk as loaded, every load unconditional (a
  // masked one is waited for at the end of its branch), masked and multiplied
  // when it goes to LDS; the list entry a chunk further ahead, so that the
  // loads that depend on it issue at once
  R tx[2][2], ty[2], tz[2];
  double m0 = 0.0, m1 = 0.0, m2 = 0.0, qi = 0.0;
  int2 cur, nxt = lst[min(al, max(m - 1, 0))];
  auto dist = [](int d, int M) { return d < 0 ? d + M : d; };
  auto load = [&](int c0) {
    cur = nxt;
    nxt = lst[min(c0 + SCH + al, max(m - 1, 0))];
    const int i = cur.x;
    const R* T = tab + (size_t)i * 6 * W;
    const int ox = (cur.y & 255) - 64, oy = (cur.y >> 8 & 255) - 64, oz = (cur.y >> 16 & 255) - 64;
    if (DIP) {
      m0 = mu[i];
      m1 = mu[i + n];
      m2 = mu[i + 2 * (size_t)n];
    }
    if (CHG) qi = q[i];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int d = min(dist(pp + 8 * k - ox, e.M[0]), W - 1);
      tx[k][1] = T[d];
      if (DIP) tx[k][0] = T[W + d];
    }
    const int dy = min(dist(pp - oy, e.M[1]), W - 1), dz = min(dist(pp - oz, e.M[2]), W - 1);
    ty[0] = T[2 * W + dy];
    tz[0] = T[4 * W + dz];
    if (DIP) {
      ty[1] = T[3 * W + dy];
      tz[1] = T[5 * W + dz];
    }
  };
  acc_t acc = {0, 0, 0, 0};
  const int row = lane & 15, kk = lane >> 4;
  const int yy = 2 * wv + (row >> 3), zz = row & 7;
  if (m > 0) load(0);
  for (int c0 = 0; c0 < m; c0 += SCH) {
    {
      const int ox = (cur.y & 255) - 64, oy = (cur.y >> 8 & 255) - 64,
                oz = (cur.y >> 16 & 255) - 64;
      const bool in = c0 + al < m;
      R mg[3] = {R(0), R(0), R(0)};
      if (DIP)
        for (int a = 0; a < 3; ++a)
          mg[a] = (R)(e.M[a] *
                      (cell.B[3 * a] * m0 + cell.B[3 * a + 1] * m1 + cell.B[3 * a + 2] * m2));
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const R on = in && dist(pp + 8 * k - ox, e.M[0]) < W ? R(1) : R(0);
        if (DIP) lx[al][0][pp + 8 * k] = on * mg[0] * tx[k][0];
        lx[al][1][pp + 8 * k] = on * tx[k][1];
      }
      const R ony = dist(pp - oy, e.M[1]) < W ? R(1) : R(0);
      const R onz = dist(pp - oz, e.M[2]) < W ? R(1) : R(0);
      R y1 = CHG ? (R)qi * ty[0] : R(0);
      if (DIP) y1 += mg[1] * ty[1];
      ly[al][pp] = {ony * ty[0], ony * y1};
      lz[al][pp] = {onz * tz[0], DIP ? onz * mg[2] * tz[1] : R(0)};
    }
    __syncthreads();
    if (c0 + SCH < m) load(c0 + SCH);
    const int left = min(SCH, m - c0);
    if (DIP) {
      // lane's K slot: atom 2 s + (kk >> 1), term kk & 1
      const int sl = kk & 1;
      for (int s0 = 0; 2 * s0 < left; s0 += 4) {
        R x[4], b[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int a = 2 * (s0 + s) + (kk >> 1);
          const R2 fy = ly[a][yy], fz = lz[a][zz];
          b[s] = sl ? fy.y * fz.x + fy.x * fz.y : fy.x * fz.x;
          x[s] = lx[a][sl][row];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = Mat<R>::mma(x[s], b[s], acc);
      }
    } else {
      for (int s0 = 0; 4 * s0 < left; s0 += 4) {
        R x[4], b[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int a = 4 * (s0 + s) + kk;
          b[s] = ly[a][yy].y * lz[a][zz].x;
          x[s] = lx[a][1][row];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = Mat<R>::mma(x[s], b[s], acc);
      }
    }
    __syncthreads();
  }
  R* g = G + ((size_t)blockIdx.z * e.nseg + seg) * e.ng + (size_t)(y0 + yy) * e.M[2] + z0 + zz;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    g[(size_t)(x0 + Mat<R>::row(lane, i)) * e.M[1] * e.M[2]] = acc[i];
}

// The sources of the displaced moments, d/de of q_j, mu_j at r_j + e g_j: dipoles
// q g and quadrupoles g mu,
//   G = sum_j (g . d/dr_j)(q_j + mu_j . d/dr_j) prod phi,
// as k_grid_spread with three terms per atom (phi_x, phi'_x, phi''_x) of the
// four of a matrix step.  Once per gradient evaluation: not pipelined.
template <typename R>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_spread_adj(
    Ext e, const Seg* __restrict__ segs, const double* __restrict__ q,
    const double* __restrict__ mu, const double* __restrict__ gv, int n,
    const R* __restrict__ tab, const R* __restrict__ tab2, const int2* __restrict__ list,
    const int4* __restrict__ cnt, R* __restrict__ G) {
  constexpr int W = Mat<R>::W;
  typedef typename Mat<R>::acc acc_t;
  __shared__ R lx[SCH][3][TX], ly[SCH][3][TY], lz[SCH][3][TZ];
  // per x term the coefficients of f f, f' f, f f', f'' f, f f'', f' f' in (y, z)
  __shared__ R co[SCH][4][6];
  const int tile = xcd_tile(blockIdx.x, e.ntile), seg = blockIdx.y;
  if (tile >= e.ntile) return;
  const size_t at = (size_t)seg * e.ntile + tile;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int4 cc = cnt[at];
  const int m = cc.z;
  const int2* lst = list + (size_t)cc.x;
  const int z0 = (tile % e.nt[2]) * TZ, y0 = ((tile / e.nt[2]) % e.nt[1]) * TY,
            x0 = tile / (e.nt[2] * e.nt[1]) * TX;
  const Cell& cell = segs[seg].cell;
  const int al = t >> 3, pp = t & 7;
  const int row = lane & 15, kk = lane >> 4;
  const int yy = 2 * wv + (row >> 3), zz = row & 7;
  acc_t acc = {0, 0, 0, 0};
  for (int c0 = 0; c0 < m; c0 += SCH) {
    const bool in = c0 + al < m;
    const int2 en = lst[min(c0 + al, m - 1)];
    const int i = en.x;
    const R* T = tab + (size_t)i * 6 * W;
    const R* T2 = tab2 + (size_t)i * 3 * W;
    const int o[3] = {(en.y & 255) - 64, (en.y >> 8 & 255) - 64, (en.y >> 16 & 255) - 64};
    auto point = [&](int ax, int p, R* f, int stride) {
      int d = p - o[ax];
      d += d < 0 ? e.M[ax] : 0;
      const R on = in && d < W ? R(1) : R(0);
      d = min(d, W - 1);
      f[0] = on * T[2 * ax * W + d];
      f[stride] = on * T[(2 * ax + 1) * W + d];
      f[2 * stride] = on * T2[ax * W + d];
    };
    point(0, pp, &lx[al][0][pp], TX);
    point(0, pp + 8, &lx[al][0][pp + 8], TX);
    point(1, pp, &ly[al][0][pp], TY);
    point(2, pp, &lz[al][0][pp], TZ);
    if (pp == 0) {
      double gg[3], mm[3];
      for (int a = 0; a < 3; ++a) {
        const double* b = cell.B + 3 * a;
        gg[a] = e.M[a] * (b[0] * gv[i] + b[1] * gv[i + n] + b[2] * gv[i + 2 * (size_t)n]);
        mm[a] = e.M[a] * (b[0] * mu[i] + b[1] * mu[i + n] + b[2] * mu[i + 2 * (size_t)n]);
      }
      const double qi = q[i];
      R(*c)[6] = co[al];
      for (int k = 0; k < 4; ++k)
        for (int j = 0; j < 6; ++j) c[k][j] = R(0);
      c[0][1] = (R)(qi * gg[1]);
      c[0][2] = (R)(qi * gg[2]);
      c[0][3] = (R)(gg[1] * mm[1]);
      c[0][4] = (R)(gg[2] * mm[2]);
      c[0][5] = (R)(gg[1] * mm[2] + gg[2] * mm[1]);
      c[1][0] = (R)(qi * gg[0]);
      c[1][1] = (R)(gg[0] * mm[1] + gg[1] * mm[0]);
      c[1][2] = (R)(gg[0] * mm[2] + gg[2] * mm[0]);
      c[2][0] = (R)(gg[0] * mm[0]);
    }
    __syncthreads();
    const int left = min(SCH, m - c0);
    for (int a = 0; a < left; ++a) {
      const R* c = co[a][kk];
      const R f = ly[a][0][yy], f1 = ly[a][1][yy], f2 = ly[a][2][yy];
      const R h = lz[a][0][zz], h1 = lz[a][1][zz], h2 = lz[a][2][zz];
      const R b = c[0] * f * h + c[1] * f1 * h + c[2] * f * h1 + c[3] * f2 * h + c[4] * f * h2 +
                  c[5] * f1 * h1;
      acc = Mat<R>::mma(lx[a][min(kk, 2)][row], b, acc);
    }
    __syncthreads();
  }
  R* g = G + (size_t)seg * e.ng + (size_t)(y0 + yy) * e.M[2] + z0 + zz;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    g[(size_t)(x0 + Mat<R>::row(lane, i)) * e.M[1] * e.M[2]] = acc[i];
}

// ---------------------------------------------------------------------------
// transforms (FP64 matrix cores)

__device__ __forceinline__ v4d mma(double a, double b, v4d c) { return Mat<double>::mma(a, b, c); }

// Forward z and y transforms of one x plane, 16 n3 at a time:
//   H(y, n3) = sum_z G(y, z) e^{i t3},  T(x, n2, n3) = sum_y H e^{i t2}.
// Waves take 16-row tiles of y, then (16 n2, 8 n3) tiles.
// The K loops of the three transform kernels take 16 points (4 matrix steps)
// at a time, loaded together before they multiply: the tables are padded with
// zeros to whole groups, the data indexes clamped.
template <typename R>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_fwd(Ext e, Tw tw, int split,
                                                         const R* __restrict__ G,
                                                         double2* __restrict__ T) {
  extern __shared__ double H[];  // [M2][HS], column 2 n3 + (re, im)
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 15, kk = lane >> 4;
  const int x = blockIdx.x, ch = blockIdx.y, seg = blockIdx.z;
  const int M2 = e.M[1], M3 = e.M[2];
  const R* g = G + (size_t)seg * e.ng + (size_t)x * M2 * M3;
  for (int rt = wv; rt * 16 < M2; rt += 4) {
    const R* gr = g + (size_t)min(rt * 16 + col, M2 - 1) * M3;
    v4d C = {0, 0, 0, 0}, S = {0, 0, 0, 0};
    const double* fc = tw.Fc[2] + ch * 16 + col;
    const double* fs = tw.Fs[2] + ch * 16 + col;
    for (int z0 = 0; z0 < e.xp[2]; z0 += 16) {
      double a[4], b[4], c[4], s[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int z = z0 + 4 * u + kk, zc = min(z, M3 / 2 - 1);
        a[u] = (double)gr[zc];
        b[u] = (double)gr[M3 - 1 - zc];
        c[u] = fc[z * e.np[2]];
        s[u] = fs[z * e.np[2]];
      }
      for (int sp = 1; sp < split; ++sp) {
        const R* gs = gr + (size_t)sp * e.nseg * e.ng;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int zc = min(z0 + 4 * u + kk, M3 / 2 - 1);
          a[u] += (double)gs[zc];
          b[u] += (double)gs[M3 - 1 - zc];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        C = mma(a[u] + b[u], c[u], C);
        S = mma(a[u] - b[u], s[u], S);
      }
    }
    for (int i = 0; i < 4; ++i) {
      const int y = rt * 16 + Mat<double>::row(lane, i);
      if (y < M2) {
        H[y * HS + 2 * col] = C[i];
        H[y * HS + 2 * col + 1] = S[i];
      }
    }
  }
  __syncthreads();
  const int nr = e.np[1] / 16;
  for (int j = wv; j < 2 * nr; j += 4) {
    const int r = j >> 1, h = j & 1;
    v4d C = {0, 0, 0, 0}, S = {0, 0, 0, 0};
    const double* fc = tw.Fc[1] + r * 16 + col;
    const double* fs = tw.Fs[1] + r * 16 + col;
    const double* hc = H + 16 * h + col;
    for (int y0 = 0; y0 < e.xp[1]; y0 += 16) {
      double a[4], b[4], c[4], s[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int y = y0 + 4 * u + kk, yc = min(y, M2 / 2 - 1);
        c[u] = fc[y * e.np[1]];
        s[u] = fs[y * e.np[1]];
        a[u] = hc[yc * HS];
        b[u] = hc[(M2 - 1 - yc) * HS];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        C = mma(c[u], a[u] + b[u], C);
        S = mma(s[u], a[u] - b[u], S);
      }
    }
    const int n3 = ch * 16 + 8 * h + (col >> 1);
    const int p = col & 1;
    double* o = reinterpret_cast<double*>(T + ((size_t)seg * e.M[0] + x) * e.NCC) + 2 * n3 + p;
    for (int i = 0; i < 4; ++i) {
      const double so = __shfl_xor(S[i], 1, 64);
      const int n2 = r * 16 + Mat<double>::row(lane, i);
      if (n2 <= e.k[1] && n3 <= e.k[2]) {
        // C +- i S
        const double d = p ? so : -so;
        o[(size_t)(e.k[1] + n2) * e.N3c * 2] = C[i] + d;
        if (n2 > 0) o[(size_t)(e.k[1] - n2) * e.N3c * 2] = C[i] - d;
      }
    }
  }
}

// The x transform of 8 (n2, n3) columns, the product with the Ewald factors
// and the x transform back, in place.  With EN the energy and stress sums of
// the half space: |S|^2 A_k and (delta_ab - kcoe k_a k_b) |S|^2 A_k.
struct EnArgs {
  Cell cell;
  double alpha;
  double* pout;
};

template <bool EN>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_mid(Ext e, Tw tw, const double* __restrict__ D,
                                                         double2* __restrict__ T, EnArgs en) {
  extern __shared__ double sh[];
  const int K1 = e.np[0];
  double* Cb = sh;            // [K1][16]
  double* Sb = sh + K1 * 16;  // [K1][16]
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 15, kk = lane >> 4;
  const int c0 = blockIdx.x * 8, seg = blockIdx.y;
  const int M1 = e.M[0];
  const bool ok = c0 + (col >> 1) < e.NCC;
  const size_t rs = (size_t)e.NCC * 2;
  double* t = reinterpret_cast<double*>(T + (size_t)seg * M1 * e.NCC) +
              2 * (ok ? c0 + (col >> 1) : e.NCC - 1) + (col & 1);
  for (int j = wv; j < 2 * (K1 / 16); j += 4) {
    const int r = j >> 1, sc = j & 1;
    const double* f = (sc ? tw.Fs[0] : tw.Fc[0]) + r * 16 + col;
    const double sg = sc ? -1.0 : 1.0;
    v4d A = {0, 0, 0, 0};
    for (int x0 = 0; x0 < e.xp[0]; x0 += 16) {
      double a[4], b[4], c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int x = x0 + 4 * u + kk, xc = min(x, M1 / 2 - 1);
        a[u] = t[xc * rs];
        b[u] = t[(M1 - 1 - xc) * rs];
        c[u] = f[x * K1];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) A = mma(c[u], a[u] + sg * b[u], A);
    }
    double* o = sc ? Sb : Cb;
    for (int i = 0; i < 4; ++i) o[(r * 16 + Mat<double>::row(lane, i)) * 16 + col] = A[i];
  }
  __syncthreads();
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  const double* Ds = D + (size_t)seg * e.nm;
  for (int k = threadIdx.x; k < K1 * 8; k += MDFF_BLOCK) {
    const int n1 = k >> 3, c = k & 7, cc = c0 + c;
    double Er = 0, Ei = 0, Or = 0, Oi = 0;
    double* cb = Cb + n1 * 16 + 2 * c;
    double* sb = Sb + n1 * 16 + 2 * c;
    if (n1 <= e.k[0] && cc < e.NCC) {
      const double pr = cb[0] - sb[1], pi = cb[1] + sb[0];
      const double mr = cb[0] + sb[1], mi = cb[1] - sb[0];
      const double dp = Ds[(size_t)(e.k[0] + n1) * e.NCC + cc];
      const double dm = n1 > 0 ? Ds[(size_t)(e.k[0] - n1) * e.NCC + cc] : 0.0;
      Er = dp * pr + dm * mr;
      Ei = dp * pi + dm * mi;
      Or = n1 > 0 ? dp * pr - dm * mr : 0.0;
      Oi = n1 > 0 ? dp * pi - dm * mi : 0.0;
      if (EN) {
        const int n3 = cc % e.N3c, n2 = cc / e.N3c - e.k[1];
        const double wgt = n3 > 0 ? 1.0 : 0.5;  // the plane n3 = 0 holds k and -k
        const double* B = en.cell.B;
        for (int sgn = 0; sgn < 2; ++sgn) {
          const double str =
              wgt * (sgn ? dm * (mr * mr + mi * mi) : dp * (pr * pr + pi * pi));
          if (str == 0.0) continue;
          double kv[3], k2 = 0.0;
          for (int a = 0; a < 3; ++a) {
            kv[a] = 2.0 * MDFF_PI *
                    ((sgn ? -n1 : n1) * B[a] + n2 * B[a + 3] + n3 * B[a + 6]);
            k2 += kv[a] * kv[a];
          }
          const double kc = 2.0 * (1.0 / k2 + 0.25 / (en.alpha * en.alpha));
          acc[0] += str;
          acc[1] += (1.0 - kc * kv[0] * kv[0]) * str;
          acc[2] += (1.0 - kc * kv[1] * kv[1]) * str;
          acc[3] += (1.0 - kc * kv[2] * kv[2]) * str;
          acc[4] -= kc * kv[0] * kv[1] * str;
          acc[5] -= kc * kv[0] * kv[2] * str;
          acc[6] -= kc * kv[1] * kv[2] * str;
        }
      }
    }
    cb[0] = Er;
    cb[1] = Ei;
    sb[0] = Or;
    sb[1] = Oi;
  }
  __syncthreads();
  const int p = col & 1;
  for (int r = wv; r * 16 < M1 / 2; r += 4) {
    v4d C = {0, 0, 0, 0}, S = {0, 0, 0, 0};
    const double* tc = tw.Tc[0] + r * 16 + col;
    const double* ts = tw.Ts[0] + r * 16 + col;
    for (int n0 = 0; n0 <= e.k[0]; n0 += 16) {
      double c[4], s[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + 4 * u + kk;
        c[u] = tc[n * e.xp[0]];
        s[u] = ts[n * e.xp[0]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + 4 * u + kk;
        C = mma(c[u], Cb[n * 16 + col], C);
        S = mma(s[u], Sb[n * 16 + col], S);
      }
    }
    for (int i = 0; i < 4; ++i) {
      const double so = __shfl_xor(S[i], 1, 64);
      const int x = r * 16 + Mat<double>::row(lane, i);
      const double d = p ? -so : so;  // C -+ i S
      if (ok && x < M1 / 2) {
        t[x * rs] = C[i] + d;
        t[(M1 - 1 - x) * rs] = C[i] - d;
      }
    }
  }
  if (EN) {
    __syncthreads();
    block_sum<7>(acc, sh);
    if (threadIdx.x == 0)
      for (int k = 0; k < 7; ++k) en.pout[(size_t)k * gridDim.x + blockIdx.x] = acc[k];
  }
}

// Back transforms over n2 and n3 for 16 folded y rows (and their mirrors) of
// one x plane: W(y, n3) = sum_n2 V e^{-i t2}, b(y, z) = Re sum_n3 c W e^{-i t3}
// with c = 1 for n3 = 0, else 2 (the other half space).
template <typename R>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_inv(Ext e, Tw tw, const double2* __restrict__ T,
                                                         R* __restrict__ P) {
  extern __shared__ double sh[];
  const int KZ = e.np[2], KS = KZ + 1;
  double* Wr = sh;                // [2][16][KS]
  double* Wi = sh + 2 * 16 * KS;  // [2][16][KS]
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 15, kk = lane >> 4;
  const int x = blockIdx.x, yt = blockIdx.y, seg = blockIdx.z;
  const int M2 = e.M[1], M3 = e.M[2];
  const double* t = reinterpret_cast<const double*>(T + ((size_t)seg * e.M[0] + x) * e.NCC);
  const int p = col & 1;
  for (int ct = wv; ct * 16 < 2 * KZ; ct += 4) {
    const int n3 = ct * 8 + (col >> 1);
    const bool ok = n3 < e.N3c;
    const double* tp = t + 2 * (ok ? n3 : 0) + p;
    v4d C = {0, 0, 0, 0}, S = {0, 0, 0, 0};
    const double* tc = tw.Tc[1] + yt * 16 + col;
    const double* ts = tw.Ts[1] + yt * 16 + col;
    for (int n0 = 0; n0 <= e.k[1]; n0 += 16) {
      double a[4], b[4], c[4], s[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + 4 * u + kk, nn = min(n, e.k[1]);
        a[u] = tp[(size_t)(e.k[1] + nn) * e.N3c * 2];
        b[u] = tp[(size_t)(e.k[1] - nn) * e.N3c * 2];
        c[u] = tc[n * e.xp[1]];
        s[u] = ts[n * e.xp[1]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double bb = n0 + 4 * u + kk > 0 ? b[u] : 0.0;  // n2 = 0 once
        C = mma(c[u], a[u] + bb, C);
        S = mma(s[u], a[u] - bb, S);
      }
    }
    const double c = !ok ? 0.0 : (n3 > 0 ? 2.0 : 1.0);
    double* o = (p ? Wi : Wr) + n3;
    for (int i = 0; i < 4; ++i) {
      const double so = __shfl_xor(S[i], 1, 64);
      const double d = p ? -so : so;
      const int row = Mat<double>::row(lane, i);
      if (n3 < KZ) {
        o[row * KS] = c * (C[i] + d);
        o[(16 + row) * KS] = c * (C[i] - d);
      }
    }
  }
  __syncthreads();
  const int P3 = M3 + Mat<R>::PADZ;
  R* g = P + ((size_t)seg * e.M[0] + x) * M2 * P3;
  const int nz = (M3 / 2 + 15) / 16;
  for (int j = wv; j < 2 * nz; j += 4) {
    const int m = j & 1, zt = j >> 1;
    v4d C = {0, 0, 0, 0}, S = {0, 0, 0, 0};
    const double* tc = tw.Tc[2] + zt * 16 + col;
    const double* ts = tw.Ts[2] + zt * 16 + col;
    const double* wr = Wr + (m * 16 + col) * KS;
    const double* wi = Wi + (m * 16 + col) * KS;
    for (int n0 = 0; n0 < KZ; n0 += 16) {
      double c[4], s[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + 4 * u + kk;
        c[u] = tc[n * e.xp[2]];
        s[u] = ts[n * e.xp[2]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int n = n0 + 4 * u + kk;
        C = mma(wr[n], c[u], C);
        S = mma(wi[n], s[u], S);
      }
    }
    const int z = zt * 16 + col;
    for (int i = 0; i < 4; ++i) {
      int y = yt * 16 + Mat<double>::row(lane, i);
      if (y >= M2 / 2 || z >= M3 / 2) continue;
      if (m) y = M2 - 1 - y;
      R* o = g + (size_t)y * P3;
      const R lo = (R)(C[i] + S[i]), hi = (R)(C[i] - S[i]);
      o[z] = lo;
      o[M3 - 1 - z] = hi;
      if (z < Mat<R>::PADZ) o[M3 + z] = lo;
      if (M3 - 1 - z < Mat<R>::PADZ) o[2 * M3 - 1 - z] = hi;
    }
  }
}

// Ewald factors over the squared kernel transform (set_cells).
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_factors(Ext e, const Seg* __restrict__ segs,
                                                             const double* __restrict__ ph, int o2,
                                                             int o3, double* __restrict__ D) {
  const size_t i = (size_t)blockIdx.x * MDFF_BLOCK + threadIdx.x;
  if (i >= e.nm) return;
  const int seg = blockIdx.y;
  const int cc = (int)(i % e.NCC), n1 = (int)(i / e.NCC) - e.k[0];
  const int n3 = cc % e.N3c, n2 = cc / e.N3c - e.k[1];
  const double* B = segs[seg].cell.B;
  const double al = segs[seg].alpha;
  double k2 = 0.0;
  for (int a = 0; a < 3; ++a) {
    const double k = 2.0 * MDFF_PI * (n1 * B[a] + n2 * B[a + 3] + n3 * B[a + 6]);
    k2 += k * k;
  }
  const double p = ph[abs(n1)] * ph[o2 + abs(n2)] * ph[o3 + n3];
  const bool zero = n1 == 0 && n2 == 0 && n3 == 0;
  D[(size_t)seg * e.nm + i] = zero ? 0.0 : exp(-k2 * 0.25 / (al * al)) / k2 * p * p;
}

// ---------------------------------------------------------------------------
// interpolation

// Sum over the wave, uniform: DPP adds within rows, then across them.
template <int CTRL>
__device__ __forceinline__ float dpp0(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp0(double x) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true),
      __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane63(float x) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
__device__ __forceinline__ double lane63(double x) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 63),
                          __builtin_amdgcn_readlane(__double2loint(x), 63));
}
template <typename R>
__device__ __forceinline__ R wave_total(R x) {
  x += dpp0<0x111>(x);  // row_shr 1, 2, 4, 8
  x += dpp0<0x112>(x);
  x += dpp0<0x114>(x);
  x += dpp0<0x118>(x);
  x += dpp0<0x142>(x);  // row_bcast 15, 31
  x += dpp0<0x143>(x);
  return lane63(x);
}

// A wave takes an atom, its lanes the support's W x ceil(W / ZV) groups of ZV
// neighbouring z at one y, each summing its columns over x against phi_x,
// phi'_x (phi''_x), then over its z.  The potentials are read where they lie
// (their rows padded with their own beginning, so that a group never wraps):
// consecutive waves take atoms in bin order, which share most of their
// support in the caches.  16,384 atoms on 96^3 points: 13 us at W = 10, 59 us
// at W = 17, the latter bound by the lines it takes through L2 (9.5 M requests,
// 2.0 per row of 136 bytes, 97 % hits; the same with one to five passes'
// loads in flight).  With the region of a tile staged in LDS 15 and 52 us
// (the FP64 SCF instance 61 against 62), but 12 us instead of 5 for 2,000
// atoms on 48^3 (few workgroups, each first waiting for its region).
//
// IND (an SCF field of one configuration, no surface term): the field of
// k_combine64<ES_IND> is formed here too, with the block partials of its
// residual (or p.Ap) rows in ca.rpart: 15 and 62 us, against 5.6 us more in a
// launch of its own.
// VAL: also the potential psi itself, in row 3.
template <typename R, bool SECOND, bool IND, int BA, bool VAL = false>
__global__ __launch_bounds__(MDFF_BLOCK) void k_grid_gather(
    Ext e, const R* __restrict__ P, const int4* __restrict__ l0, const R* __restrict__ tab,
    const R* __restrict__ tab2, const int* __restrict__ perm, const int* __restrict__ cfg,
    int count, int apw, int n, double* __restrict__ out, CombineArgs ca) {
  constexpr int W = Mat<R>::W, ZV = Mat<R>::ZV, NG = (W + ZV - 1) / ZV;
  constexpr int IT = (W * NG + 63) / 64;
  constexpr int NV = SECOND ? 9 : VAL ? 4 : 3;
  __shared__ double red[2][4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int per = 4 * apw;
  const int nb = (count + per - 1) / per;
  const int blk = xcd_tile(blockIdx.x, nb);
  if (blk >= nb) return;
  const int P3 = e.M[2] + Mat<R>::PADZ;
  const size_t px = (size_t)e.M[1] * P3;
  // BA atoms of a wave at a time, their loads issued together: a dependent
  // load here costs a microsecond (the data was written by other XCDs)
  double acc0 = 0.0, acc1 = 0.0;
  const double c1 = 1.0 / (4.0 * MDFF_PI), c2 = -1.0 / (8.0 * MDFF_PI * MDFF_PI);
  const double Mx = e.M[0], My = e.M[1], Mz = e.M[2];
  const size_t N = n;
  for (int k0 = 0; k0 < apw; k0 += BA) {
    const int h0 = (blk * 4 + wv) * apw + k0;
    const int left = min(min(count - h0, apw - k0), BA);
    if (left <= 0) break;
    // lanes 3 j + r: component r of atom j in the combine
    const int ej = min(lane / 3, left - 1), er3 = lane % 3;
    const int ei = perm[h0 + ej];
    int id[BA], lx[BA], ly[BA], lz[BA];
    {
      const int4 l = l0[ei];
#pragma unroll
      for (int j = 0; j < BA; ++j) {
        id[j] = __builtin_amdgcn_readlane(ei, 3 * j);
        lx[j] = __builtin_amdgcn_readlane(l.x, 3 * j);
        ly[j] = __builtin_amdgcn_readlane(l.y, 3 * j);
        lz[j] = __builtin_amdgcn_readlane(l.z, 3 * j);
      }
    }
    double m0 = 0, m1 = 0, m2 = 0, efd = 0, est = 0;
    int ety = 0;
    if (IND) {
      m0 = ca.mu[ei];
      m1 = ca.mu[ei + N];
      m2 = ca.mu[ei + 2 * N];
      efd = ca.ef_dir[ei + er3 * N];
      ety = ca.typ[ei];
      if (!ca.cg_Ap) est = ca.E_stat[ei + er3 * N];
    }
    R v[BA][NV];
#pragma unroll
    for (int j = 0; j < BA; ++j)
#pragma unroll
      for (int c = 0; c < NV; ++c) v[j][c] = R(0);
    // not unrolled at W = 17: five passes' loads would leave two waves per SIMD
#pragma unroll IT > 2 ? 1 : IT
    for (int it = 0; it < IT; ++it) {
      const int c = lane + 64 * it;
      const bool in = c < W * NG;
      const int b = in ? c / NG : 0, zg = in ? c % NG * ZV : 0;
      R x[BA][W][ZV], fy[BA], gy[BA], hy[BA], fz[BA][ZV], gz[BA][ZV], hz[BA][ZV];
#pragma unroll
      for (int j = 0; j < BA; ++j) {
        const R* T = tab + (size_t)id[j] * 6 * W;
        const R* T2 = tab2 + (size_t)id[j] * 3 * W;
        const R* s = P + (cfg ? (size_t)cfg[id[j]] * e.M[0] * px : 0) +
                     (size_t)wrap(ly[j] + b, e.M[1]) * P3 + lz[j] + zg;
#pragma unroll
        for (int a = 0; a < W; ++a)
          __builtin_memcpy(x[j][a], s + wrap(lx[j] + a, e.M[0]) * px, sizeof(x[j][a]));
        fy[j] = T[2 * W + b];
        gy[j] = T[3 * W + b];
        if (SECOND) hy[j] = T2[W + b];
#pragma unroll
        for (int z = 0; z < ZV; ++z) {
          const int d = min(zg + z, W - 1);
          fz[j][z] = T[4 * W + d];
          gz[j][z] = T[5 * W + d];
          if (SECOND) hz[j][z] = T2[2 * W + d];
        }
      }
#pragma unroll
      for (int j = 0; j < BA; ++j) {
        const R* T = tab + (size_t)id[j] * 6 * W;
        const R* T2 = tab2 + (size_t)id[j] * 3 * W;
#pragma unroll
        for (int z = 0; z < ZV; ++z) {
          R s0 = 0, s1 = 0, s2 = 0;
#pragma unroll
          for (int a = 0; a < W; ++a) {
            s0 += T[a] * x[j][a][z];
            s1 += T[W + a] * x[j][a][z];
            if (SECOND) s2 += T2[a] * x[j][a][z];
          }
          const R on = in && zg + z < W ? R(1) : R(0);
          s0 *= on;
          s1 *= on;
          s2 *= on;
          v[j][0] += s1 * (fy[j] * fz[j][z]);
          v[j][1] += s0 * (gy[j] * fz[j][z]);
          v[j][2] += s0 * (fy[j] * gz[j][z]);
          if (VAL) v[j][3] += s0 * (fy[j] * fz[j][z]);
          if (SECOND) {
            v[j][3] += s2 * (fy[j] * fz[j][z]);
            v[j][4] += s0 * (hy[j] * fz[j][z]);
            v[j][5] += s0 * (fy[j] * hz[j][z]);
            v[j][6] += s1 * (gy[j] * fz[j][z]);
            v[j][7] += s1 * (fy[j] * gz[j][z]);
            v[j][8] += s0 * (gy[j] * gz[j][z]);
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < BA; ++j)
#pragma unroll
      for (int c = 0; c < NV; ++c) v[j][c] = wave_total(v[j][c]);
    // the sums of this lane's atom
    R w[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      w[c] = v[0][c];
#pragma unroll
      for (int j = 1; j < BA; ++j) w[c] = ej == j ? v[j][c] : w[c];
    }
    const double u0 = c1 * Mx * (double)w[0], u1 = c1 * My * (double)w[1],
                 u2 = c1 * Mz * (double)w[2];
    if (lane >= 3 * left) continue;
    if (IND) {
      const int r = er3;
      const double* B = ca.cell.B;
      const double b0 = r == 0 ? B[0] : r == 1 ? B[1] : B[2],
                   b1 = r == 0 ? B[3] : r == 1 ? B[4] : B[5],
                   b2 = r == 0 ? B[6] : r == 1 ? B[7] : B[8];
      const double fe = -2.0 * ca.fpi_V * (2.0 * MDFF_PI);
      const double er = fe * (b0 * u0 + b1 * u1 + b2 * u2);
      const double mr = r == 0 ? m0 : r == 1 ? m1 : m2;
      const double ef = (efd + er) + 2.0 * ca.selfa2 * mr;
      if (ca.cg_Ap) {
        // Ap = alpha^-1 p - T p and p.Ap
        const double* ip = ca.T->invpol[ety];
        const double ap = ip[r] * m0 + ip[r + 3] * m1 + ip[r + 6] * m2 - ef;
        ca.cg_Ap[ei + r * N] = ap;
        acc0 += mr * ap;
      } else {
        // E and the stopping criterion's rows (resid_terms)
        const double E = est + ef;
        ca.E[ei + r * N] = E;
        const double pa = ca.T->pol[ety][r + 3 * r];
        const double d = pa == 0.0 ? 0.0 : mr / pa - E;
        acc0 += d * d;
        if (r == 0) acc1 += 1.0;
      }
    } else if (er3 == 0) {
      double* r = out + ei;
      r[0] = u0;
      r[N] = u1;
      r[2 * N] = u2;
      if (VAL) r[3 * N] = (double)w[3];
      if (SECOND) {
        r[3 * N] = c2 * Mx * Mx * (double)w[3];
        r[4 * N] = c2 * My * My * (double)w[4];
        r[5 * N] = c2 * Mz * Mz * (double)w[5];
        r[6 * N] = c2 * Mx * My * (double)w[6];
        r[7 * N] = c2 * Mx * Mz * (double)w[7];
        r[8 * N] = c2 * My * Mz * (double)w[8];
      }
    }
  }
  if (IND) {
    acc0 = wave_total(acc0);
    acc1 = wave_total(acc1);
    if (lane == 0) {
      red[0][wv] = acc0;
      red[1][wv] = acc1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      ca.rpart[blk] = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
      ca.rpart[nb + blk] = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
    }
  }
}

// ---------------------------------------------------------------------------
// host

static int extent(int kmax, int mult, int W) {
  const int need = std::max((int)std::ceil(1.95 * (2 * kmax + 1)), W);
  return (need + mult - 1) / mult * mult;
}

bool supported(const int kmax[3]) {
  for (int a = 0; a < 3; ++a)
    if (kmax[a] < 1 || extent(kmax[a], 16, W64) > MMAX) return false;
  return true;
}

static int extent(int axis, const int kmax[3], bool fp64) {
  return extent(kmax[axis], axis == 0 ? TX : TY, fp64 ? W64 : W32);
}

Size size(const int kmax[3], bool fp64) {
  double M[3], k[3];
  for (int a = 0; a < 3; ++a) {
    M[a] = extent(a, kmax, fp64);
    k[a] = kmax[a] + 1;
  }
  Size z;
  z.points = (size_t)(M[0] * M[1] * M[2]);
  z.tiles = (int)(M[0] / TX * (M[1] / TY) * (M[2] / TZ));
  // the six folded cosine / sine products of the three axes, forward and back
  z.flops = 4.0 * (M[0] * M[1] * M[2] * k[2] + 2.0 * M[0] * M[1] * k[1] * k[2] +
                   2.0 * M[0] * k[0] * (2.0 * k[1] - 1.0) * k[2]);
  return z;
}

template <typename T>
static bool take(Plan* p, T** d, size_t count) {
  void* v = nullptr;
  if (hipMalloc(&v, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess) return false;
  p->allocs.push_back(v);
  *d = static_cast<T*>(v);
  return true;
}
static void release(Plan* p, void* d) {
  if (!d) return;
  (void)hipFree(d);
  p->allocs.erase(std::find(p->allocs.begin(), p->allocs.end(), d));
}

template <typename R>
static bool setup(Plan* p) {
  constexpr int W = Mat<R>::W, DEG = Mat<R>::DEG;
  Ext& e = p->e;
  std::vector<R> poly;
  std::vector<double> ph, tw;
  size_t off[3][4];
  const LD pi = acosl(-1.0L);
  for (int a = 0; a < 3; ++a) {
    p->phoff[a] = (int)ph.size();
    int same = 0;
    while (e.M[same] != e.M[a] || e.k[same] != e.k[a]) ++same;
    if (same < a) {
      // an axis of the same extents: the same kernel
      const size_t np = (size_t)3 * (DEG + 1) * W;
      for (size_t k = 0; k < np; ++k) poly.push_back(poly[same * np + k]);
      for (int n = 0; n <= e.k[a]; ++n) ph.push_back(ph[p->phoff[same] + n]);
    } else {
      const LD sigma = (LD)e.M[a] / (2 * e.k[a] + 1);
      const Kernel K(W, pi * W * (1 - 1 / (2 * sigma)));
      std::vector<LD> f;
      fit(K, W, DEG, f);
      for (LD v : f) poly.push_back((R)v);
      std::vector<double> t;
      transform(K, W, e.M[a], e.k[a], t);
      ph.insert(ph.end(), t.begin(), t.end());
    }
    const int M2 = e.M[a] / 2, np = e.np[a], xp = e.xp[a];
    for (int k = 0; k < 4; ++k) {
      off[a][k] = tw.size();
      tw.resize(tw.size() + (size_t)np * xp, 0.0);
    }
    for (int l = 0; l < M2; ++l) {
      const LD th = 2 * pi * (l + 0.5L) / e.M[a], c1 = cosl(th), s1 = sinl(th);
      LD cn = 1, sn = 0;
      for (int n = 0; n <= e.k[a]; ++n) {
        const double c = (double)cn, s = (double)sn;
        const LD t = cn * c1 - sn * s1;
        sn = sn * c1 + cn * s1;
        cn = t;
        tw[off[a][0] + (size_t)l * np + n] = c;
        tw[off[a][1] + (size_t)l * np + n] = s;
        tw[off[a][2] + (size_t)n * xp + l] = c;
        tw[off[a][3] + (size_t)n * xp + l] = s;
      }
    }
  }
  double* d_tw = nullptr;
  R *d_poly = nullptr, *d_G = nullptr, *d_P = nullptr, *d_tab = nullptr, *d_tab2 = nullptr;
  if (!take(p, &d_tw, tw.size()) || !take(p, &p->d_phat, ph.size()) ||
      !take(p, &d_poly, poly.size()) || !take(p, &d_G, e.ng * e.nseg * p->split) || !take(p, &p->d_l0, p->natom) ||
      !take(p, &d_P, (size_t)e.nseg * e.M[0] * e.M[1] * (e.M[2] + Mat<R>::PADZ)) ||
      !take(p, &d_tab, (size_t)p->natom * 6 * W) || !take(p, &d_tab2, (size_t)p->natom * 3 * W))
    return false;
  p->d_poly = d_poly;
  p->d_G = d_G;
  p->d_P = d_P;
  p->d_tab = d_tab;
  p->d_tab2 = d_tab2;
  for (int a = 0; a < 3; ++a) {
    p->tw.Fc[a] = d_tw + off[a][0];
    p->tw.Fs[a] = d_tw + off[a][1];
    p->tw.Tc[a] = d_tw + off[a][2];
    p->tw.Ts[a] = d_tw + off[a][3];
  }
  return hipMemcpy(d_tw, tw.data(), tw.size() * sizeof(double), hipMemcpyHostToDevice) ==
             hipSuccess &&
         hipMemcpy(p->d_phat, ph.data(), ph.size() * sizeof(double), hipMemcpyHostToDevice) ==
             hipSuccess &&
         hipMemcpy(d_poly, poly.data(), poly.size() * sizeof(R), hipMemcpyHostToDevice) ==
             hipSuccess;
}

// blocks of k_grid_mid: 8 columns of the (n2, n3) plane each
static int mid_blocks(const Ext& e) { return (e.NCC + 7) / 8; }

// dynamic LDS of the kernels
static size_t lds_fwd(const Ext& e) { return (size_t)e.M[1] * HS * sizeof(double); }
static size_t lds_mid(const Ext& e) {
  return std::max<size_t>((size_t)e.np[0] * 32, 4 * 7) * sizeof(double);
}
static size_t lds_inv(const Ext& e) {
  return (size_t)4 * 16 * (e.np[2] + 1) * sizeof(double);
}

Plan* create(hipStream_t st, const std::vector<Seg>& segs, const int kmax[3], bool fp64) {
  if (!supported(kmax) || segs.empty()) return nullptr;
  Plan* p = new Plan();
  p->fp64 = fp64;
  Ext& e = p->e;
  e.nseg = (int)segs.size();
  e.ng = 1;
  for (int a = 0; a < 3; ++a) {
    e.k[a] = kmax[a];
    e.M[a] = extent(a, kmax, fp64);
    e.nt[a] = e.M[a] / (a == 0 ? TX : TY);
    e.np[a] = (kmax[a] + 1 + 15) / 16 * 16;
    e.xp[a] = (e.M[a] / 2 + 15) / 16 * 16;
    e.ng *= e.M[a];
  }
  e.ntile = e.nt[0] * e.nt[1] * e.nt[2];
  // two workgroups per CU of the spread, but at most two partial grids: at
  // 48^3 points (108 tiles) spread and forward transform, which reads them
  // all from a few dozen CUs, take 11.7 + 6.1 us with one, 7.7 + 7.7 with two
  // and 6.8 + 10.7 with four
  p->split = std::max(1, std::min(2, 512 / (e.ntile * e.nseg)));
  e.N2f = 2 * kmax[1] + 1;
  e.N3c = kmax[2] + 1;
  e.NCC = e.N2f * e.N3c;
  e.nm = (size_t)(2 * kmax[0] + 1) * e.NCC;
  for (const Seg& s : segs) p->natom = std::max(p->natom, s.off + s.n);
  const size_t nb = (size_t)2 * e.nseg * e.ntile;
  bool ok = fp64 ? setup<double>(p) : setup<float>(p);
  ok = ok && take(p, &p->d_seg, segs.size()) && take(p, &p->d_T, (size_t)e.nseg * e.M[0] * e.NCC) &&
       take(p, &p->d_D, e.nseg * e.nm) && take(p, &p->d_key, p->natom) &&
       take(p, &p->d_start, nb + 1) && take(p, &p->d_cur, nb + 1) &&
       take(p, &p->d_perm0, p->natom) && take(p, &p->d_perm, p->natom) &&
       take(p, &p->d_total, 1) && take(p, &p->d_off, (size_t)e.nseg * e.ntile + 1) &&
       take(p, &p->d_cnt, (size_t)e.nseg * e.ntile);
  // more LDS than the default limit of a launch
  const std::pair<const void*, size_t> big[] = {
      {fp64 ? (void*)k_grid_fwd<double> : (void*)k_grid_fwd<float>, lds_fwd(e)},
      {(void*)k_grid_mid<false>, lds_mid(e)},
      {(void*)k_grid_mid<true>, lds_mid(e)},
      {fp64 ? (void*)k_grid_inv<double> : (void*)k_grid_inv<float>, lds_inv(e)}};
  for (const auto& b : big)
    if (b.second > 65536)
      ok = ok && hipFuncSetAttribute(b.first, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)b.second) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    destroy(p);
    return nullptr;
  }
  set_cells(p, st, segs);
  return p;
}

void destroy(Plan* p) {
  if (!p) return;
  for (void* v : p->allocs) (void)hipFree(v);
  delete p;
}

void set_cells(Plan* p, hipStream_t st, const std::vector<Seg>& segs) {
  p->segs = segs;
  p->is_binned = false;
  (void)hipMemcpyAsync(p->d_seg, p->segs.data(), segs.size() * sizeof(Seg), hipMemcpyHostToDevice,
                       st);
  const dim3 g((unsigned)((p->e.nm + MDFF_BLOCK - 1) / MDFF_BLOCK), p->e.nseg);
  k_grid_factors<<<g, MDFF_BLOCK, 0, st>>>(p->e, p->d_seg, p->d_phat, p->phoff[1], p->phoff[2],
                                           p->d_D);
}


size_t partials(const Plan* p) {
  // seven energy and stress rows of k_grid_mid, two rows of the SCF
  // interpolation (at most a block per four atoms)
  return std::max<size_t>((size_t)7 * mid_blocks(p->e), (size_t)2 * ((p->natom + 3) / 4));
}
bool binned(const Plan* p) { return p->is_binned; }
void unbin(Plan* p) { p->is_binned = false; }

bool bin(Plan* p, hipStream_t st, const double4* s4, const int* typ, const int* cfg,
         unsigned active, double drift) {
  p->is_binned = false;  // until everything below has succeeded
  const Ext& e = p->e;
  const int n = p->natom;
  const int gn = (n + MDFF_BLOCK - 1) / MDFF_BLOCK;
  const int nb = 2 * e.nseg * e.ntile;
  // grid cells an atom may cross: a displacement d changes s_a by at most
  // |B_a| d
  Margin mg;
  for (int a = 0; a < 3; ++a) {
    double w = 0.0;
    for (const Seg& s : p->segs) {
      const double* b = s.cell.B + 3 * a;
      w = std::max(w, std::sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]));
    }
    mg.m[a] = drift > 0.0 ? (int)std::min<double>(e.M[a], std::ceil(drift * w * e.M[a]) + 1) : 0;
    p->margin[a] = mg.m[a];
  }
  k_cell_zero<<<(nb + 1 + MDFF_BLOCK - 1) / MDFF_BLOCK, MDFF_BLOCK, 0, st>>>(nb + 1, p->d_start);
  k_cell_zero<<<1, MDFF_BLOCK, 0, st>>>(2, reinterpret_cast<int*>(p->d_total));
  if (p->fp64)
    k_grid_bin<W64><<<gn, MDFF_BLOCK, 0, st>>>(n, e, s4, typ, cfg, active, p->d_key, p->d_start);
  else
    k_grid_bin<W32><<<gn, MDFF_BLOCK, 0, st>>>(n, e, s4, typ, cfg, active, p->d_key, p->d_start);
  k_cell_scan<<<1, 1024, 0, st>>>(nb, p->d_start, p->d_cur);
  k_cell_fill<<<gn, MDFF_BLOCK, 0, st>>>(n, p->d_key, p->d_cur, p->d_perm0);
  k_cell_order<<<gn, MDFF_BLOCK, 0, st>>>(n, p->d_key, p->d_start, p->d_perm0, p->d_perm, nullptr);
  const int ntile = e.nseg * e.ntile;
  const int gt = (ntile + MDFF_BLOCK - 1) / MDFF_BLOCK;
  if (p->fp64)
    k_grid_cap<W64><<<gt, MDFF_BLOCK, 0, st>>>(e, mg, p->d_start, p->d_off, p->d_total);
  else
    k_grid_cap<W32><<<gt, MDFF_BLOCK, 0, st>>>(e, mg, p->d_start, p->d_off, p->d_total);
  k_cell_scan<<<1, 1024, 0, st>>>(ntile, p->d_off, p->d_cur);
  unsigned long long total = 0;
  if (hipMemcpyAsync(&total, p->d_total, sizeof(total), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(&p->nact, p->d_start + nb / 2, sizeof(int), hipMemcpyDeviceToHost, st) !=
          hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return false;
  if (total > (unsigned long long)INT_MAX) return false;  // slots are ints
  if ((long long)total + 1 > p->slots) {
    release(p, p->d_ov);
    p->d_ov = nullptr;
    p->slots = 0;
    // one slot past the last list: a tile without atoms reads it, unused
    const size_t c = total + total / 8 + 8;
    if (!take(p, &p->d_ov, c)) {
      (void)hipGetLastError();
      return false;
    }
    p->slots = (long long)c;
  }
  p->cfg = cfg;
  p->is_binned = true;
  return true;
}

void prepare(Plan* p, mdffgpu_ctx* ctx, hipStream_t st, const double4* s4) {
  ProfScope _ps(ctx, K_GRID_PREP);
  const Ext& e = p->e;
  Margin mg;
  for (int a = 0; a < 3; ++a) mg.m[a] = p->margin[a];
  const dim3 g(e.ntile, e.nseg);
  const long long work = (long long)p->natom * 3 * (p->fp64 ? W64 : W32);
  const int gt = (int)std::min<long long>((work + MDFF_BLOCK - 1) / MDFF_BLOCK, 2048);
  if (p->fp64) {
    k_grid_lists<W64><<<g, MDFF_BLOCK, 0, st>>>(e, mg, s4, p->d_start, p->d_perm, p->d_off, p->d_ov,
                                                p->d_cnt);
    k_grid_tab<double><<<gt, MDFF_BLOCK, 0, st>>>(p->natom, e, s4, (const double*)p->d_poly,
                                                  (double*)p->d_tab, (double*)p->d_tab2, (int*)p->d_l0);
  } else {
    k_grid_lists<W32><<<g, MDFF_BLOCK, 0, st>>>(e, mg, s4, p->d_start, p->d_perm, p->d_off, p->d_ov,
                                                p->d_cnt);
    k_grid_tab<float><<<gt, MDFF_BLOCK, 0, st>>>(p->natom, e, s4, (const float*)p->d_poly,
                                                 (float*)p->d_tab, (float*)p->d_tab2, (int*)p->d_l0);
  }
}

// Spread grids to potentials: the three transform kernels.
template <typename R>
static void convolve(Plan* p, mdffgpu_ctx* ctx, hipStream_t st, int split, double* pout) {
  ProfScope _ps(ctx, K_GRID_FT);
  const Ext& e = p->e;
  const R* G = static_cast<const R*>(p->d_G);
  R* P = static_cast<R*>(p->d_P);
  const dim3 gf(e.M[0], (e.N3c + 15) / 16, e.nseg);
  k_grid_fwd<R><<<gf, MDFF_BLOCK, lds_fwd(e), st>>>(e, p->tw, split, G, p->d_T);
  const dim3 gm(mid_blocks(e), e.nseg);
  EnArgs en;
  std::memset(&en, 0, sizeof(en));
  if (pout) {
    en.cell = p->segs[0].cell;
    en.alpha = p->segs[0].alpha;
    en.pout = pout;
    k_grid_mid<true><<<gm, MDFF_BLOCK, lds_mid(e), st>>>(e, p->tw, p->d_D, p->d_T, en);
  } else {
    k_grid_mid<false><<<gm, MDFF_BLOCK, lds_mid(e), st>>>(e, p->tw, p->d_D, p->d_T, en);
  }
  const dim3 gi(e.M[0], (e.M[1] / 2 + 15) / 16, e.nseg);
  k_grid_inv<R><<<gi, MDFF_BLOCK, lds_inv(e), st>>>(e, p->tw, p->d_T, P);
}

template <typename R>
static int sums_t(Plan* p, mdffgpu_ctx* ctx, hipStream_t st, const double* q,
                  const double* mu, bool chg, bool dip, bool second, bool src_active, bool dst_active,
                  double* out, double* pout, const CombineArgs* ind) {
  const Ext& e = p->e;
  const int n = p->natom;
  R* G = static_cast<R*>(p->d_G);
  const R* P = static_cast<const R*>(p->d_P);
  const R* tab = static_cast<const R*>(p->d_tab);
  const R* tab2 = static_cast<const R*>(p->d_tab2);
  const dim3 gt(xcd_blocks(e.ntile), e.nseg, p->split);
  const int sa = src_active ? 1 : 0;
  {
    ProfScope _ps(ctx, K_GRID_SPREAD);
    if (chg && dip)
      k_grid_spread<R, true, true><<<gt, MDFF_BLOCK, 0, st>>>(e, p->d_seg, q, mu, n, tab, p->d_ov,
                                                              p->d_cnt, sa, G);
    else if (dip)
      k_grid_spread<R, false, true><<<gt, MDFF_BLOCK, 0, st>>>(e, p->d_seg, q, mu, n, tab,
                                                               p->d_ov, p->d_cnt, sa, G);
    else
      k_grid_spread<R, true, false><<<gt, MDFF_BLOCK, 0, st>>>(e, p->d_seg, q, mu, n, tab,
                                                               p->d_ov, p->d_cnt, sa, G);
  }
  convolve<R>(p, ctx, st, p->split, pout);
  ProfScope _ps(ctx, K_GRID_GATHER);
  const int count = dst_active ? p->nact : n;
  // about 4096 waves of a large system take the atoms in turn
  const int apw = std::max(1, count / (sizeof(R) == 8 ? 8192 : 4096));
  const int nb = (count + 4 * apw - 1) / (4 * apw);
  if (count == 0) return ind ? 0 : mid_blocks(e);
  const int gg = xcd_blocks(nb);
  CombineArgs ca;
  std::memset(&ca, 0, sizeof(ca));
  if (ind) ca = *ind;
  auto go = [&](auto kernel) {
    kernel<<<gg, MDFF_BLOCK, 0, st>>>(e, P, p->d_l0, tab, tab2, p->d_perm, p->cfg, count, apw, n,
                                      out, ca);
  };
  // FP32 waves that take several atoms load four at once (registers)
  constexpr int BA = sizeof(R) == 4 ? 4 : 1;
  if (ind && apw > 1)
    go(k_grid_gather<R, false, true, BA>);
  else if (ind)
    go(k_grid_gather<R, false, true, 1>);
  else if (second)
    go(k_grid_gather<R, true, false, 1>);
  else if (apw > 1)
    go(k_grid_gather<R, false, false, BA>);
  else
    go(k_grid_gather<R, false, false, 1>);
  return ind ? nb : mid_blocks(e);
}

int sums(Plan* p, mdffgpu_ctx* ctx, hipStream_t st, const double* q,
         const double* mu, bool chg, bool dip,
         bool second, bool src_active, bool dst_active, double* out, double* pout,
         const CombineArgs* ind) {
  return p->fp64 ? sums_t<double>(p, ctx, st, q, mu, chg, dip, second, src_active, dst_active, out, pout, ind)
                 : sums_t<float>(p, ctx, st, q, mu, chg, dip, second, src_active, dst_active, out, pout, ind);
}

template <typename R>
static void adjoint_t(Plan* p, hipStream_t st, const double* q, const double* mu, const double* g,
                      double* out) {
  const Ext& e = p->e;
  const int n = p->natom;
  const R* tab = static_cast<const R*>(p->d_tab);
  const R* tab2 = static_cast<const R*>(p->d_tab2);
  k_grid_spread_adj<R><<<dim3(xcd_blocks(e.ntile), e.nseg), MDFF_BLOCK, 0, st>>>(
      e, p->d_seg, q, mu, g, n, tab, tab2, p->d_ov, p->d_cnt, static_cast<R*>(p->d_G));
  convolve<R>(p, nullptr, st, 1, nullptr);
  CombineArgs ca;
  std::memset(&ca, 0, sizeof(ca));
  k_grid_gather<R, false, false, 1, true><<<xcd_blocks((n + 3) / 4), MDFF_BLOCK, 0, st>>>(
      e, static_cast<const R*>(p->d_P), p->d_l0, tab, tab2, p->d_perm, p->cfg, n, 1, n, out, ca);
}

void adjoint_sums(Plan* p, hipStream_t st, const double* q, const double* mu, const double* g,
                  double* out) {
  if (p->fp64)
    adjoint_t<double>(p, st, q, mu, g, out);
  else
    adjoint_t<float>(p, st, q, mu, g, out);
}

}  // namespace grid
}  // namespace mdff
