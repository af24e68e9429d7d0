// grid.h -- reciprocal-space Ewald sums through a uniform grid: the sums over
// every k vector of the half-space mesh, evaluated as a non-uniform Fourier
// transform (spread the moments onto a grid, transform, multiply by the
// Ewald factors, transform back, interpolate) instead of one term per
// (atom, k).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "common.h"

struct mdffgpu_ctx;

namespace mdff {
struct CombineArgs;
namespace grid {

// One configuration: its cell and Ewald alpha and its atoms in the caller's
// arrays.
struct Seg {
  Cell cell;
  double alpha;
  int off, n;
};

struct Plan;

// Whether a plan exists for these kmax (grid extents within the kernels'
// limits).
bool supported(const int kmax[3]);

// Plan for configurations that share kmax; fp64: grid and kernel tables in
// double (support 17), else in float (support 10; transforms in double).
// Null when device memory runs out (the caller has the direct sums).
Plan* create(hipStream_t st, const std::vector<Seg>& segs, const int kmax[3], bool fp64);
void destroy(Plan* p);

// New cells (and alpha) of the configurations; the binning has to be redone.
void set_cells(Plan* p, hipStream_t st, const std::vector<Seg>& segs);

// Bins of the current positions (fractional coordinates s4, one per atom).
// Atoms of a species with its bit in `active` come first in their own bins:
// the calls over the active atoms alone read those.  Until the next call no
// atom may move by more than drift (a length).  Waits for the stream; false
// when device memory runs out: the plan is of no use then.
bool bin(Plan* p, hipStream_t st, const double4* s4, const int* typ, const int* cfg,
         unsigned active, double drift);
bool binned(const Plan* p);
void unbin(Plan* p);

// Kernel values and tile lists at the current positions: once per
// evaluation.  ctx (here and below) brackets the launches for its
// instrumentation, or null.
void prepare(Plan* p, mdffgpu_ctx* ctx, hipStream_t st, const double4* s4);

// The reciprocal sums of one Ewald call with charges q (chg) and dipoles mu
// (dip; SoA of stride n): U_a = sum_k A_k n_a Im(S conj e^{ikr}) and, with
// second, V_ab = sum_k A_k n_a n_b Re(..) over the half-space mesh into
// out[row * n + atom], rows U1 U2 U3 V11 V22 V33 V12 V13 V23.  src_active:
// only the active atoms carry moments; dst_active: rows of the active atoms
// only.  With pout (one configuration), block partials of the energy and
// stress sums go to pout[row * nblocks + block] (7 rows); returns nblocks.
// With ind (an SCF call of one configuration, no surface term) the combine of
// k_combine64<ES_IND> is done here instead of writing out; returns the number
// of block partials per row of ind->rpart.
int sums(Plan* p, mdffgpu_ctx* ctx, hipStream_t st, const double* q, const double* mu, bool chg,
         bool dip, bool second, bool src_active, bool dst_active, double* out, double* pout,
         const CombineArgs* ind = nullptr);

// Potentials of the displaced sources, d/de at r_j + e g_j of all atoms (g SoA
// of stride n): out rows U1 U2 U3 as above and, row 3, psi = sum over every k
// of A_k S e^{-ikr}.
void adjoint_sums(Plan* p, hipStream_t st, const double* q, const double* mu, const double* g,
                  double* out);

// What one configuration's grid takes with these kmax, for the choice between
// it and the direct sums: points, tiles of the spread, flops of the
// transforms of one call (without padding).
struct Size {
  size_t points;
  int tiles;
  double flops;
};
Size size(const int kmax[3], bool fp64);

// Doubles that pout and ind->rpart need at most.
size_t partials(const Plan* p);

}  // namespace grid
}  // namespace mdff
