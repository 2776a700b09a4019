// ed_batch.hpp -- batched solves of many sectors (parameter points of a VCA /
// CDMFT sweep).  An item that fits in LDS runs as one workgroup, a whole
// Lanczos ground state or LanczosGreen continued fraction; larger items
// ("wide") advance together, one Lanczos step of every item per launch.
#pragma once

#include <vector>

#include "ed_common.hpp"

namespace ed {

struct Instance;

// device view of one factorized sector: per-spin merged one-body tables (CSR
// with values, both triangles) and the full diagonal, label order
// I = i_up + dim_up * i_dn
struct BatchSector {
  uint32_t du = 0, dd = 0;
  const uint32_t *up_ptr = nullptr, *up_col = nullptr, *dn_ptr = nullptr, *dn_col = nullptr;
  const double *up_val = nullptr, *dn_val = nullptr, *diag = nullptr;
};

// Lanczos ground state of one sector (LanczosEigenvalue + LanczosEigenvector,
// src_ed/Hamiltonian/Lanczos.hpp:41-143): start vector normal_draw(seed, .)
// normalized, Ritz stop |z_last beta| <= accur, eigenvector by replaying the
// recurrence
struct BatchGSItem {
  BatchSector S;
  uint64_t seed = 0;
  double *gs = nullptr;   // dim: normalized ground state (output)
  double *tri = nullptr;  // kTriArrays (max_iter + 2), for items whose arrays are not in LDS
  double *out = nullptr;  // E0, iterations, status (0 ok, 1 not converged)
};

// LanczosGreen (src_ed/Hamiltonian/Lanczos.hpp:156-183) from
// psi = c_o1 |gs> (+ c_o2 |gs>), built in the kernel from half-basis maps
struct BatchCFItem {
  BatchSector S;              // target sector
  const double *gs = nullptr; // source state
  uint32_t du_s = 0;          // source up dimension
  int spin = 0, norb = 1;
  const int32_t *map[2] = {nullptr, nullptr};
  const int8_t *sgn[2] = {nullptr, nullptr};
  const int8_t *upar = nullptr;  // spin-down orbitals: (-1)^(up occupation)
  double *a = nullptr;        // max_cf
  double *b = nullptr;        // max_cf + 1 (b[0] = 1)
  double *out = nullptr;      // n (-1: psi vanishes), ||psi||^2
};

// tridiagonal work arrays of a ground-state item, each max_iter + 2 long
constexpr int kTriArrays = 6;
// largest LDS footprint of an item run from LDS
constexpr size_t kBatchLdsCap = 64 * 1024;

// LDS bytes of one item held entirely in LDS: nvec Lanczos vectors and ntri
// tridiagonal doubles, then the sector's diagonal and one-body tables (nu, nd
// entries); the kernels carve their LDS in this order
__host__ __device__ inline size_t batch_lds_bytes(int nvec, size_t ntri, uint32_t du, uint32_t dd, uint32_t nu,
                                                  uint32_t nd) {
  const size_t dim = (size_t)du * dd;
  return 8 * ((size_t)nvec * dim + ntri + dim + nu + nd) + 4 * ((size_t)du + 1 + nu + dd + 1 + nd);
}
constexpr int kGsVectors = 3;  // two Lanczos vectors, ground state
constexpr int kCfVectors = 2;  // two Lanczos vectors

// One wide item.  Its vectors are stored with the larger half basis as the
// fast index ("lanes", nl states; the other half is "rows", nr states):
// J = lane + nl * row, which is the label order unless swap.  dg is the
// diagonal in that order.
struct WideItem {
  const uint32_t *lp = nullptr, *lc = nullptr, *rp = nullptr, *rc = nullptr;  // lane / row one-body tables (CSR)
  const double *lv = nullptr, *rv = nullptr, *dg = nullptr;
  double *u = nullptr;     // 2 dim: the two Lanczos vectors (a ground state: 3 dim, the eigenvector last)
  double *part = nullptr;  // 2 nwg: dot and norm partials
  double *a = nullptr;     // alpha_k at a[k]
  double *b = nullptr;     // beta_{k-1} at b[k], k >= 1
  double *sc = nullptr;    // kWideScalars, see ed_batch.hip
};
constexpr int kWideScalars = 8;

// items of one shape (nl x nr), advanced together
struct WideShape {
  uint32_t nl = 0, nr = 0;
  int swap = 0;
  int rows = 1;     // rows per workgroup
  int rpt = 1;      // rows per thread
  int nwg = 1;      // workgroups per item
  uint32_t emax = 0;  // longest row of the row tables
  bool stage = true;  // rows fit in LDS (else read from memory)
  size_t lds = 0;
};
WideShape wide_shape(uint32_t du, uint32_t dd, uint32_t emax);

// continued fractions of n items of one shape; src[k] is item k's start state
void wide_cf(const WideShape &W, const WideItem *items, const BatchCFItem *src, int n, int max_cf, double acc,
             hipStream_t s);
// ground states of n items of one shape: src[k].gs and src[k].out as for
// batch_gs; item k's a is its kTriArrays tridiagonal arrays (max_iter + 2 long
// each: alpha, beta, ...) and b points one before the second of them
void wide_gs(const WideShape &W, const WideItem *items, const BatchGSItem *src, int n, int max_iter, double accur,
             hipStream_t s);

// items run from LDS, lds dynamic bytes each; block: 64 or 256 threads per item
// (tri_lds: the tridiagonal arrays among them, else in each item's tri)
void batch_gs(const BatchGSItem *d_items, int n, int block, size_t lds, bool tri_lds, int max_iter, double accur,
              hipStream_t s);
void batch_cf(const BatchCFItem *d_items, int n, int block, size_t lds, int max_cf, double acc, hipStream_t s);

// fractions of sectors of at most 16 rt down and 16 ct up half states (rt, ct
// in 1, 2): vectors in registers, one wave an item
void tile_cf(const BatchCFItem *d_items, int n, int rt, int ct, int max_cf, double acc, hipStream_t s);

// writes item k's continued fraction (out[2k] = n steps, out[2k + 1] =
// ||psi||^2), transformed with the state's energy e0[k], weight w[k] and
// electron / hole pm[k], into a continued-fraction store at off[fid[k]]
void batch_cf_store(int nitems, int max_cf, const double *out, const double *a, const double *b, const int *fid,
                    const int *off, const double *e0, const double *w, const int8_t *pm, double *A, double *B,
                    hipStream_t s);

// solves the ground state (and with want_gf the Green function) of every
// instance; factorizable instances using Lanczos + continued fractions run
// batched, the others through their own solve
void solve_batch(const std::vector<Instance *> &insts, bool want_gf);

// One LanczosGreen run: alpha_n and beta_{n-1} (b[0] = 1, one entry more than
// a) and the start vector's squared norm; empty where that vanishes.
struct Fraction {
  std::vector<double> a, b;
  double norm2 = 0.0;
};
struct State;
struct TermList;
// whether an instance's fractions of npairs orbital pairs from state st, at most
// max_cf levels each, run as a batch (the same recurrence and stop rule as
// lanczos_green, all pairs together)
bool fractions_together(const Instance &I, const TermList &T, const State &st, int spin, size_t npairs, long max_cf);
// the fractions of c^{pm}_o1 (+ c^{pm}_o2) |st> for the given pairs, at most
// max_cf levels: entry 2 k + (pm < 0) for pair k; the hole and the electron
// part run together.  Empty where the target sector is invalid or empty.
std::vector<Fraction> state_fractions(const Instance &I, const TermList &T, const State &st, int spin,
                                      const std::vector<std::pair<int, int>> &pairs, int max_cf);

}  // namespace ed
