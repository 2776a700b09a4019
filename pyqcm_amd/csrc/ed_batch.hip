// ed_batch.hip -- batched Lanczos ground states and LanczosGreen continued
// fractions.  An item whose sector fits (tables, diagonal, Lanczos vectors and
// tridiagonal arrays within kBatchLdsCap) is one workgroup that runs the whole
// recurrence from LDS, so that a sweep over hundreds of parameter points x
// sectors is a single launch.  Larger ("wide") items keep their vectors in
// memory and advance in lockstep, two launches per Lanczos step for all items
// of a shape (ground states three).  The projected tridiagonal problem is solved on the device by
// one wave per item; every reduction has a fixed order.
#include "ed_batch.hpp"

#include <cfloat>

#include "ed_rng.hpp"

namespace ed {
namespace {

constexpr int kW = 64;

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kW);
  return v;
}
__device__ __forceinline__ double wmin(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, kW));
  return v;
}
__device__ __forceinline__ double wmax(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, kW));
  return v;
}

// workgroup sum, the result in every thread
template <int BS>
__device__ __forceinline__ double bsum(double v, double *sh) {
  v = wsum(v);
  if (BS == kW) return v;
  const int lane = threadIdx.x & (kW - 1), w = threadIdx.x / kW;
  __syncthreads();
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < BS / kW; ++i) r += sh[i];
  return r;
}

// 1/x: the hardware estimate refined by one Newton step (relative error a
// few ulp); used only where a sign depends on it (Sturm counts)
__device__ __forceinline__ double frcp(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  return fma(r, fma(-x, r, 1.0), r);
}

// i_dn of label I = i_up + du * i_dn, from a double-precision reciprocal of
// du corrected to the exact quotient
__device__ __forceinline__ uint32_t label_dn(uint32_t I, uint32_t du, double rdu) {
  uint32_t q = (uint32_t)((double)I * rdu);
  const uint64_t qd = (uint64_t)q * du;
  if (qd > I) --q;
  else if (I - qd >= du) ++q;
  return q;
}

// walks the labels I = t, t + BS, ... of one thread with their (i_dn, i_up)
struct LabelWalk {
  uint32_t I, id, iu, sd, su, du;
  __device__ __forceinline__ LabelWalk(uint32_t t, uint32_t step, uint32_t du_, double rdu) : I(t), du(du_) {
    id = label_dn(t, du, rdu);
    iu = t - id * du;
    sd = label_dn(step, du, rdu);
    su = step - sd * du;
  }
  __device__ __forceinline__ void next(uint32_t step) {
    I += step;
    iu += su;
    id += sd;
    if (iu >= du) {
      iu -= du;
      ++id;
    }
  }
};

// (H x)[I] for one label I = iu + du * id
__device__ __forceinline__ double hx(const BatchSector &S, const double *x, uint32_t I, uint32_t id, uint32_t iu) {
  double acc = S.diag[I] * x[I];
  const double *xr = x + (size_t)S.du * id;
  for (uint32_t e = S.up_ptr[iu]; e < S.up_ptr[iu + 1]; ++e) acc += S.up_val[e] * xr[S.up_col[e]];
  const double *xc = x + iu;
  for (uint32_t e = S.dn_ptr[id]; e < S.dn_ptr[id + 1]; ++e) acc += S.dn_val[e] * xc[(size_t)S.du * S.dn_col[e]];
  return acc;
}

// copies a sector's diagonal and one-body tables to LDS (doubles at d, words
// at u, in the order batch_lds_bytes counts them) and returns the LDS view;
// the caller synchronizes before use
template <int BS>
__device__ BatchSector stage_sector(const BatchSector &G, double *d, uint32_t *u) {
  const uint32_t dim = G.du * G.dd, nu = G.up_ptr[G.du], nd = G.dn_ptr[G.dd];
  double *diag = d, *uval = d + dim, *dval = uval + nu;
  uint32_t *uptr = u, *ucol = uptr + G.du + 1, *dptr = ucol + nu, *dcol = dptr + G.dd + 1;
  for (uint32_t i = threadIdx.x; i < dim; i += BS) diag[i] = G.diag[i];
  for (uint32_t i = threadIdx.x; i < nu; i += BS) {
    uval[i] = G.up_val[i];
    ucol[i] = G.up_col[i];
  }
  for (uint32_t i = threadIdx.x; i < nd; i += BS) {
    dval[i] = G.dn_val[i];
    dcol[i] = G.dn_col[i];
  }
  for (uint32_t i = threadIdx.x; i <= G.du; i += BS) uptr[i] = G.up_ptr[i];
  for (uint32_t i = threadIdx.x; i <= G.dd; i += BS) dptr[i] = G.dn_ptr[i];
  BatchSector L;
  L.du = G.du;
  L.dd = G.dd;
  L.diag = diag;
  L.up_val = uval;
  L.dn_val = dval;
  L.up_ptr = uptr;
  L.up_col = ucol;
  L.dn_ptr = dptr;
  L.dn_col = dcol;
  return L;
}

// One Lanczos step on (v, vp), in place: vp <- w = H v - bprev vp - alpha v,
// alpha = <Hv - bprev vp, v>, beta = ||w|| (H v reads only v, and vp[I] only
// at I, so w can overwrite vp).  Returns alpha and beta in every thread; the
// caller scales vp by 1 / beta and swaps the two names.
template <int BS>
__device__ __forceinline__ void lanczos_step(const BatchSector &S, double rdu, uint32_t dim, const double *v,
                                             double *vp, double bprev, double *sh, double &alpha, double &beta) {
  double dot = 0.0;
  for (LabelWalk L(threadIdx.x, BS, S.du, rdu); L.I < dim; L.next(BS)) {
    const double t = hx(S, v, L.I, L.id, L.iu) - bprev * vp[L.I];
    vp[L.I] = t;
    dot += t * v[L.I];
  }
  alpha = bsum<BS>(dot, sh);
  double n2 = 0.0;
  for (uint32_t I = threadIdx.x; I < dim; I += BS) {
    const double t = vp[I] - alpha * v[I];
    vp[I] = t;
    n2 += t * t;
  }
  beta = sqrt(bsum<BS>(n2, sh));
}

// number of eigenvalues of the tridiagonal (a, b^2 = bb) below x
__device__ __forceinline__ int sturm_below(int n, const double *a, const double *bb, double x) {
  int cnt = 0;
  double q = a[0] - x;
  if (q < 0.0) ++cnt;
  for (int i = 1; i < n; ++i) {
    if (q == 0.0) q = -1e-300;
    q = fma(-bb[i - 1], frcp(q), a[i] - x);
    if (q < 0.0) ++cnt;
  }
  return cnt;
}

// Lowest eigenpair of the tridiagonal (a[0..n), b[0..n-1), bb = b^2), run by
// the 64 lanes of wave 0.
//  * Bracket [lo, hi] of the lowest eigenvalue by Sturm counts: Gershgorin
//    below; above, `*hi_io` when it is a number (an upper bound from the
//    previous, one row shorter tridiagonal: the lowest Ritz value never
//    increases as the tridiagonal grows), probed first on a geometric grid
//    so that a nearly converged value is bracketed in one round; then
//    multisection (64 counts per round, the interval shrinks 65x) until its
//    width is below 1e-8 of the norm.
//  * Lane 0: two sweeps of inverse iteration from (1, ..., 1) with the shift
//    sigma = lo, below the spectrum, so that the unpivoted LDL^T of T - sigma
//    is positive definite; the recurrences carry their last value in a
//    register.  The eigenvector's contamination shrinks as
//    ((lambda - sigma) / gap)^2, and the Rayleigh quotient z^T T z gives the
//    eigenvalue to rounding.
// z[0..n) receives the normalized eigenvector; lane 0 writes *lam (the
// Rayleigh quotient), *zlast and *hi_io (an upper bound of the eigenvalue
// for the next call).  D and l are n-long scratch arrays.
__device__ __forceinline__ void tri_lowest_wave(int n, const double *a, const double *b, const double *bb,
                                                double *hi_io, double *z, double *D, double *l, double *lam,
                                                double *zlast) {
  const int lane = threadIdx.x;
  if (n == 1) {
    // a one-step space: the eigenpair is a_0 and the unit vector (a zero
    // a_0 would otherwise leave no scale for the shifted factorization)
    if (lane == 0) {
      z[0] = 1.0;
      *lam = a[0];
      *zlast = 1.0;
      *hi_io = a[0] + 4.0 * DBL_EPSILON * fabs(a[0]) + 1e-300;
    }
    return;
  }
  double lo = 1e300, hi = -1e300, nrm = 0.0;
  for (int i = lane; i < n; i += kW) {
    const double r = (i > 0 ? fabs(b[i - 1]) : 0.0) + (i < n - 1 ? fabs(b[i]) : 0.0);
    lo = fmin(lo, a[i] - r);
    hi = fmax(hi, a[i] + r);
    nrm = fmax(nrm, fabs(a[i]) + r);
  }
  lo = wmin(lo);
  hi = wmax(hi);
  nrm = wmax(nrm);
  const double eps = DBL_EPSILON;
  hi += 1e-300 + 4.0 * eps * nrm;
  lo -= 1e-300 + 4.0 * eps * nrm;
  const double prev = *hi_io;
  if (prev == prev && prev < hi && prev > lo) {
    hi = prev;
    // x_l = hi - (hi - lo) 2^(-0.9 l): distances from the full width down to ~1e-17 of it
    const double x = hi - (hi - lo) * exp2(-0.9 * (double)lane);
    const unsigned long long mask = __ballot(sturm_below(n, a, bb, x) >= 1);
    if (mask == 0ull) {
      lo = __shfl(x, kW - 1, kW);
    } else {
      const int f = __ffsll((long long)mask) - 1;
      hi = __shfl(x, f, kW);
      if (f > 0) lo = __shfl(x, f - 1, kW);
    }
  }
  for (int round = 0; round < 64; ++round) {
    if (hi - lo <= 1e-8 * nrm) break;
    const double x = lo + (hi - lo) * (double)(lane + 1) / (double)(kW + 1);
    const bool below = sturm_below(n, a, bb, x) >= 1;
    const unsigned long long mask = __ballot(below);
    const double x63 = __shfl(x, kW - 1, kW);
    if (mask == 0ull) {
      lo = x63;
    } else {
      const int f = __ffsll((long long)mask) - 1;
      const double xf = __shfl(x, f, kW);
      const double xl = __shfl(x, f > 0 ? f - 1 : 0, kW);
      hi = xf;
      if (f > 0) lo = xl;
    }
  }
  if (lane == 0) {
    // D holds the reciprocal pivots of T - sigma
    double sigma = lo - 4.0 * eps * nrm - 1e-300, delta = 4.0 * (double)(n > 16 ? n : 16) * eps * fmax(nrm, 1e-300);
    for (int attempt = 0; attempt < 40; ++attempt) {
      bool ok = true;
      double p = a[0] - sigma;
      for (int i = 0; i < n - 1; ++i) {
        if (!(p > 0.0)) {
          ok = false;
          break;
        }
        const double ip = 1.0 / p;
        D[i] = ip;
        l[i] = b[i] * ip;
        p = a[i + 1] - sigma - l[i] * b[i];
      }
      if (ok && p > 0.0) {
        D[n - 1] = 1.0 / p;
        break;
      }
      sigma -= delta;
      delta *= 8.0;
    }
    double scale = 1.0;
    for (int sweep = 0; sweep < 2; ++sweep) {
      // forward: y_i = x_i - l_{i-1} y_{i-1}, stored as y_i / d_i
      double y = 0.0;
      for (int i = 0; i < n; ++i) {
        const double xi = sweep == 0 ? 1.0 : scale * z[i];
        y = i > 0 ? fma(-l[i - 1], y, xi) : xi;
        z[i] = y * D[i];
      }
      // backward: x_i = y_i / d_i - l_i x_{i+1}
      double x = z[n - 1], ss = x * x;
      for (int i = n - 2; i >= 0; --i) {
        x = fma(-l[i], x, z[i]);
        z[i] = x;
        ss = fma(x, x, ss);
      }
      scale = 1.0 / sqrt(ss);
    }
    // normalize; Rayleigh quotient z^T T z
    double rq = 0.0, zp = 0.0;
    for (int i = 0; i < n; ++i) {
      const double zi = z[i] * scale;
      z[i] = zi;
      rq = fma(a[i] * zi, zi, rq);
      if (i > 0) rq = fma(2.0 * b[i - 1] * zp, zi, rq);
      zp = zi;
    }
    *lam = rq;
    *zlast = zp;
    *hi_io = fmin(hi, rq + 4.0 * eps * nrm);
  }
}

constexpr int kRitzEvery = 4;
constexpr uint32_t kRitzEach = 48;
// TRI: the tridiagonal arrays in LDS too; else (more steps allowed than fit
// beside the sector) the item's own in memory
template <int BS, bool TRI>
__global__ __launch_bounds__(BS) void k_batch_gs(const BatchGSItem *items, int max_iter, double accur) {
  extern __shared__ double smem[];
  __shared__ double sh[BS / kW];
  __shared__ double s_lam, s_zl, s_hi;
  const BatchGSItem &it = items[blockIdx.x];
  const BatchSector G = it.S;
  const uint32_t dim = G.du * G.dd;
  const double rdu = 1.0 / (double)G.du;
  const int M = max_iter + 2;
  double *v = smem, *vp = v + dim, *gs = vp + dim, *tri = TRI ? gs + dim : it.tri;
  const uint32_t nu = G.up_ptr[G.du], nd = G.dn_ptr[G.dd];
  double *sd = gs + dim + (TRI ? (size_t)kTriArrays * M : 0);
  const BatchSector S = stage_sector<BS>(G, sd, reinterpret_cast<uint32_t *>(sd + dim + nu + nd));
  double *al = tri, *be = al + M, *bb = be + M, *z = bb + M, *D = z + M, *l = D + M;
  // start vector (the same draws as the single-sector path)
  double nn = 0.0;
  for (uint32_t I = threadIdx.x; I < dim; I += BS) {
    const double r = normal_draw(it.seed, I);
    v[I] = r;
    vp[I] = 0.0;
    nn += r * r;
  }
  const double inv0 = 1.0 / sqrt(bsum<BS>(nn, sh));
  for (uint32_t I = threadIdx.x; I < dim; I += BS) v[I] *= inv0;
  if (threadIdx.x == 0) s_hi = __builtin_nan("");
  __syncthreads();
  int k = 0, status = 0;
  double bprev = 0.0;
  for (;;) {
    double alpha, beta;
    lanczos_step<BS>(S, rdu, dim, v, vp, bprev, sh, alpha, beta);
    if (threadIdx.x == 0) {
      al[k] = alpha;
      be[k] = beta;
      bb[k] = beta * beta;
    }
    __syncthreads();
    ++k;
    // The Ritz pair is a serial chain of one wave, longer than the step itself:
    // found every kRitzEvery steps, and at each one where the Krylov space may be
    // exhausted (as many steps as states, a small beta) or the run ends.  512 points
    // of 2x3 (300 to 400 states): every step 13.5 ms, every 4th 5.7; 12 of 2x2 with a
    // bath orbital (50 and 100 states), whole solve: 2.24 and 1.54 ms.  The smallest
    // sectors converge as their Krylov space ends, and past that point a pair may
    // look unconverged again (128 points of 2x2, 24 and 36 states: at each step 26
    // steps at most, 0.28 ms, at every 4th 42, 0.31): there at each step.
    if (dim < kRitzEach || k <= kRitzEvery || k % kRitzEvery == 0 || (uint32_t)k >= dim || !(beta > 1e-6 * be[0]) ||
        k > max_iter) {
      if (threadIdx.x < kW) tri_lowest_wave(k, al, be, bb, &s_hi, z, D, l, &s_lam, &s_zl);
      __syncthreads();
      // a zero beta: the Krylov space is exhausted (one-state sectors end here)
      if (!(beta > 0.0) || fabs(s_zl * beta) <= accur) break;
      if (k > max_iter) {
        status = 1;
        break;
      }
    }
    const double ib = 1.0 / beta;
    for (uint32_t I = threadIdx.x; I < dim; I += BS) vp[I] *= ib;
    double *t = v;
    v = vp;
    vp = t;
    bprev = beta;
    __syncthreads();
  }
  const double lam = s_lam;
  // eigenvector: replay the recurrence, gs = sum_j z_j v_j
  for (uint32_t I = threadIdx.x; I < dim; I += BS) {
    const double x0 = normal_draw(it.seed, I) * inv0;
    v[I] = x0;
    vp[I] = 0.0;
    gs[I] = z[0] * x0;
  }
  __syncthreads();
  for (int j = 1; j < k; ++j) {
    const double bp = j >= 2 ? be[j - 2] : 0.0, aj = al[j - 1], ib = 1.0 / be[j - 1], zj = z[j];
    for (LabelWalk L(threadIdx.x, BS, S.du, rdu); L.I < dim; L.next(BS)) {
      const double w = (hx(S, v, L.I, L.id, L.iu) - bp * vp[L.I] - aj * v[L.I]) * ib;
      vp[L.I] = w;
      gs[L.I] += zj * w;
    }
    double *t = v;
    v = vp;
    vp = t;
    __syncthreads();
  }
  double g2 = 0.0;
  for (uint32_t I = threadIdx.x; I < dim; I += BS) g2 += gs[I] * gs[I];
  const double ig = 1.0 / sqrt(bsum<BS>(g2, sh));
  for (uint32_t I = threadIdx.x; I < dim; I += BS) it.gs[I] = gs[I] * ig;
  if (threadIdx.x == 0) {
    it.out[0] = lam;
    it.out[1] = (double)k;
    it.out[2] = (double)status;
  }
}

template <int BS>
__global__ __launch_bounds__(BS) void k_batch_cf(const BatchCFItem *items, int max_cf, double acc) {
  extern __shared__ double smem[];
  __shared__ double sh[BS / kW];
  // item fields in registers (the two-orbital arrays are read by name, not
  // by a run-time index, so nothing is spilled to scratch)
  const BatchCFItem &itg = items[blockIdx.x];
  const BatchSector G = itg.S;
  const double *gs = itg.gs;
  const uint32_t du_s = itg.du_s;
  const int spin = itg.spin, norb = itg.norb;
  const int32_t *map0 = itg.map[0], *map1 = itg.map[1];
  const int8_t *sgn0 = itg.sgn[0], *sgn1 = itg.sgn[1], *upar = itg.upar;
  double *av = itg.a, *bv = itg.b, *out = itg.out;
  const uint32_t dim = G.du * G.dd;
  const double rdu = 1.0 / (double)G.du;
  double *v = smem, *vp = v + dim;
  const uint32_t nu = G.up_ptr[G.du], nd = G.dn_ptr[G.dd];
  double *sd = vp + dim;
  const BatchSector S = stage_sector<BS>(G, sd, reinterpret_cast<uint32_t *>(sd + dim + nu + nd));
  // psi = c_o1 |gs> (+ c_o2 |gs>), gathered over the target sector
  double nn = 0.0;
  for (LabelWalk L(threadIdx.x, BS, G.du, rdu); L.I < dim; L.next(BS)) {
    const uint32_t id = L.id, iu = L.iu;
    double val = 0.0;
    if (spin == 0) {
      const int32_t s0 = map0[iu];
      if (s0 >= 0) val += (double)sgn0[iu] * gs[(size_t)s0 + (size_t)du_s * id];
      if (norb == 2) {
        const int32_t s1 = map1[iu];
        if (s1 >= 0) val += (double)sgn1[iu] * gs[(size_t)s1 + (size_t)du_s * id];
      }
    } else {
      const double pu = (double)upar[iu];
      const int32_t s0 = map0[id];
      if (s0 >= 0) val += (double)sgn0[id] * pu * gs[iu + (size_t)du_s * s0];
      if (norb == 2) {
        const int32_t s1 = map1[id];
        if (s1 >= 0) val += (double)sgn1[id] * pu * gs[iu + (size_t)du_s * s1];
      }
    }
    v[L.I] = val;
    vp[L.I] = 0.0;
    nn += val * val;
  }
  nn = bsum<BS>(nn, sh);
  if (!(nn > 1e-14)) {
    if (threadIdx.x == 0) {
      out[0] = -1.0;
      out[1] = nn;
    }
    return;
  }
  const double inv = 1.0 / sqrt(nn);
  for (uint32_t I = threadIdx.x; I < dim; I += BS) v[I] *= inv;
  if (threadIdx.x == 0) bv[0] = 1.0;
  __syncthreads();
  int n = 0;
  double bprev = 0.0, prod = 1.0, blast = 1.0;
  while (prod > acc && fabs(blast) > acc && n < max_cf) {
    double alpha, beta;
    lanczos_step<BS>(S, rdu, dim, v, vp, bprev, sh, alpha, beta);
    if (threadIdx.x == 0) {
      av[n] = alpha;
      bv[n + 1] = beta;
    }
    prod *= fabs(beta);
    blast = beta;
    ++n;
    if (!(prod > acc && fabs(blast) > acc && n < max_cf)) break;
    const double ib = 1.0 / beta;
    for (uint32_t I = threadIdx.x; I < dim; I += BS) vp[I] *= ib;
    double *t = v;
    v = vp;
    vp = t;
    bprev = beta;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = (double)n;
    out[1] = nn;
  }
}

// ---------------------------------------------------------------------------
// Tile kernel: continued fractions of sectors of at most 32 x 32 half states.
// One wave holds the vector X[i_dn][i_up] in registers as RT x CT tiles of
// 16 x 16 and applies the one-body operators as small dense products on the
// FP64 matrix cores: Y = K_dn X + X K_up^T on top of diag o X - beta X_prev as
// the accumulator's start.  v_mfma_f64_16x16x4: lane l supplies A(l % 16,
// l / 16) and B(l / 16, l % 16), and register r of D holds (4 r + l / 16,
// l % 16), so register s % 4 of X's tile row s / 4 already is the B operand
// of K_dn X's k-step s; only X K_up^T needs X in A order, one pass through
// LDS.  No barriers, no table reads in a step: the sparse form read 12 bytes
// of tables from LDS per hop beside 8 of the vector.
// ---------------------------------------------------------------------------
typedef double f64x4 __attribute__((ext_vector_type(4)));

// x moved across lanes by a DPP control; lanes without a source give 0
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp0(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return __longlong_as_double((long long)hi << 32 | (unsigned)lo);
}
// wave sum, the same in every lane: shifts within rows of 16, then the row
// sums handed on (no LDS permutes: their latency is most of a tile step)
__device__ __forceinline__ double wsum_dpp(double v) {
  v += dpp0<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v += dpp0<0x112, 0xf>(v);
  v += dpp0<0x114, 0xf>(v);
  v += dpp0<0x118, 0xf>(v);
  v += dpp0<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
  v += dpp0<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double((long long)hi << 32 | (unsigned)lo);
}

// operand k[t][s] = K(16 t + lane % 16, 4 s + lane / 16) of the CSR matrix K
// (n rows), spread densely over xt (16 T x 16 T, stride 16 T + 1) on the way
template <int T>
__device__ __forceinline__ void tile_operand(uint32_t n, const uint32_t *ptr, const uint32_t *col, const double *val,
                                             double *xt, double (*k)[4 * T]) {
  constexpr int S = 16 * T + 1;
  const int lane = threadIdx.x;
  __syncthreads();
  for (int i = lane; i < 16 * T * S; i += kW) xt[i] = 0.0;
  __syncthreads();
  if ((uint32_t)lane < n)
    for (uint32_t e = ptr[lane]; e < ptr[lane + 1]; ++e) xt[lane * S + col[e]] = val[e];
  __syncthreads();
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int s = 0; s < 4 * T; ++s) k[t][s] = xt[(16 * t + lane % 16) * S + 4 * s + lane / 16];
}

template <int RT, int CT>
__global__ __launch_bounds__(kW) void k_tile_cf(const BatchCFItem *items, int max_cf, double acc) {
  constexpr int MT = RT > CT ? RT : CT, S = 16 * CT + 1;
  __shared__ double xt[16 * MT * (16 * MT + 1)];
  const BatchCFItem &itg = items[blockIdx.x];
  const BatchSector G = itg.S;
  const int lane = threadIdx.x, lr = lane / 16, lc = lane % 16;
  double kd[RT][4 * RT], ku[CT][4 * CT];
  tile_operand<RT>(G.dd, G.dn_ptr, G.dn_col, G.dn_val, xt, kd);
  tile_operand<CT>(G.du, G.up_ptr, G.up_col, G.up_val, xt, ku);
  const int nkr = (int)(G.dd + 3) / 4, nkc = (int)(G.du + 3) / 4;
  // psi = c_o1 |gs> (+ c_o2 |gs>); padding stays zero throughout
  f64x4 v[RT][CT], vp[RT][CT], dg[RT][CT];
  double nn = 0.0;
  {
    const double *gs = itg.gs;
    const uint32_t du_s = itg.du_s;
    const int spin = itg.spin, norb = itg.norb;
    const int32_t *map0 = itg.map[0], *map1 = itg.map[1];
    const int8_t *sgn0 = itg.sgn[0], *sgn1 = itg.sgn[1], *upar = itg.upar;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t id = 16 * t + 4 * r + lr, iu = 16 * c + lc;
          double x = 0.0, d = 0.0;
          if (id < G.dd && iu < G.du) {
            d = G.diag[id * G.du + iu];
            const uint32_t im = spin == 0 ? iu : id;
            const int32_t s0 = map0[im];
            if (s0 >= 0)
              x += (double)sgn0[im] * gs[spin == 0 ? (size_t)s0 + (size_t)du_s * id : iu + (size_t)du_s * s0];
            if (norb == 2) {
              const int32_t s1 = map1[im];
              if (s1 >= 0)
                x += (double)sgn1[im] * gs[spin == 0 ? (size_t)s1 + (size_t)du_s * id : iu + (size_t)du_s * s1];
            }
            if (spin == 1) x *= (double)upar[iu];
          }
          v[t][c][r] = x;
          vp[t][c][r] = 0.0;
          dg[t][c][r] = d;
          nn += x * x;
        }
  }
  nn = wsum_dpp(nn);
  if (!(nn > 1e-14)) {
    if (lane == 0) {
      itg.out[0] = -1.0;
      itg.out[1] = nn;
    }
    return;
  }
  const double inv = 1.0 / sqrt(nn);
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) v[t][c] *= inv;
  double *av = itg.a, *bv = itg.b;
  if (lane == 0) bv[0] = 1.0;
  int n = 0;
  double bprev = 0.0, prod = 1.0, blast = 1.0;
  while (prod > acc && fabs(blast) > acc && n < max_cf) {
    f64x4 y[RT][CT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        y[t][c] = dg[t][c] * v[t][c] - bprev * vp[t][c];
#pragma unroll
        for (int r = 0; r < 4; ++r) xt[(16 * t + 4 * r + lr) * S + 16 * c + lc] = v[t][c][r];
      }
#pragma unroll
    for (int s = 0; s < 4 * RT; ++s)
      if (s < nkr)
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
          for (int c = 0; c < CT; ++c)
            y[t][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(kd[t][s], v[s / 4][c][s % 4], y[t][c], 0, 0, 0);
    __syncthreads();  // one wave: orders the LDS writes before the reads
#pragma unroll
    for (int s = 0; s < 4 * CT; ++s)
      if (s < nkc)
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          const double a = xt[(16 * t + lc) * S + 4 * s + lr];
#pragma unroll
          for (int c = 0; c < CT; ++c) y[t][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, ku[c][s], y[t][c], 0, 0, 0);
        }
    __syncthreads();
    double dot = 0.0;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) dot += y[t][c][r] * v[t][c][r];
    const double alpha = wsum_dpp(dot);
    double n2 = 0.0;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        y[t][c] -= alpha * v[t][c];
#pragma unroll
        for (int r = 0; r < 4; ++r) n2 += y[t][c][r] * y[t][c][r];
      }
    const double beta = sqrt(wsum_dpp(n2));
    if (lane == 0) {
      av[n] = alpha;
      bv[n + 1] = beta;
    }
    prod *= fabs(beta);
    blast = beta;
    bprev = beta;
    ++n;
    const double ib = 1.0 / beta;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        vp[t][c] = v[t][c];
        v[t][c] = y[t][c] * ib;
      }
  }
  if (lane == 0) {
    itg.out[0] = (double)n;
    itg.out[1] = nn;
  }
}

// ---------------------------------------------------------------------------
// wide items.  The vectors stay unnormalized as in the device-driven
// single-sector recurrence: U_k = beta_{k-1} v_k (U_0 the start vector, its
// norm in place of beta_{-1}), buffer k & 1 holding U_k.  Step k is
//   hv:  t = H U_k / n_k - (n_k / n_{k-1}) U_{k-1} over U_{k-1}, n_k = |U_k|
//        folded from the previous launch's partials; partials of <t, U_k>
//   upd: alpha_k = <t, U_k> / n_k, U_{k+1} = t - (alpha_k / n_k) U_k over t;
//        partials of |U_{k+1}|^2
// Every workgroup of an item folds the same partials in the same order, so
// all take the same branch when the stop rule ends the item; workgroup 0
// stores the scalars, which other workgroups read from the next launch on.
// Memory bound: 6 vector accesses a step plus the neighbour rows, which hit
// the XCD's L2 because an item's workgroups are numbered onto one XCD or a run
// of them (wide_place).  Rows of U_k are staged in LDS for the lane
// part; a lane's table entries are loaded once for RPT rows, since they are
// 12 bytes a hop against 8 of the vector.
// ---------------------------------------------------------------------------
enum { SC_N = 0, SC_NN = 1, SC_PROD = 2 /* two, by parity */, SC_HI = 4, SC_LAM = 5, SC_STATUS = 6 };
constexpr double kRunning = -2.0;
constexpr int kWideBlock = 256;
constexpr int kXcd = 8;
constexpr size_t kWideSpread = size_t(1) << 17;
constexpr size_t kWideLdsMax = 144 * 1024;  // longest row staged in LDS
constexpr size_t kTriLdsMax = 144 * 1024;   // largest tridiagonal in LDS (3 072 steps)

// Item and workgroup of a block.  Block b runs on XCD b % 8.  Items are dealt out
// to the XCDs whole (grid: kXcd * ceil(n / kXcd) * nwg blocks), so that what one
// launch writes the next finds in its own L2, or (kWideSpread states or more, nwg
// negated) XCD x takes the x-th run of all items' workgroups (kXcd * ceil(n nwg /
// kXcd) blocks), so that fewer than 8 items, or 9, fill the chip too.  ms of a
// Green function, whole / in runs / one fraction after the other:
//   3 920 states    1 fraction a part  4.8 /  5.4 /  17    10 fractions   5.0 /  5.5 / 180
//   15 876          1                 17.6 / 20.5 /  39     6            19.9 / 22.7 / 250
//   52 920          1                  6.5 /  6.2 /  21    10            10.1 / 10.7 / 228
//   213 444         1                 47   / 35   /  46     6            52.9 / 47.4 / 295
//   731 808         1                 44.9 / 26.1 /  24.9  10           150   / 108  / 252
__device__ __forceinline__ bool wide_place(int n, int &nwg, int &item, int &w) {
  const int b = blockIdx.x, j = b / kXcd;
  if (nwg < 0) {
    nwg = -nwg;
    const int t = (int)(b % kXcd * (gridDim.x / kXcd)) + j;
    item = t / nwg;
    w = t - item * nwg;
  } else {
    item = (j / nwg) * kXcd + b % kXcd;
    w = j % nwg;
  }
  return item < n;
}

// sum of nwg partials, the same in every lane of every workgroup
__device__ __forceinline__ double wide_fold(const double *p, int nwg) {
  double s = 0.0;
  for (int i = threadIdx.x & (kW - 1); i < nwg; i += kW) s += p[i];
  return wsum(s);
}

// MODE 0: step k of a continued fraction; 1: of a ground state; 2: step k
// (>= 1) of the ground state's eigenvector replay on normalized vectors (max_k
// is then the length of a tridiagonal array)
template <int MODE, int RPT, bool RG1, bool STAGE>
__global__ __launch_bounds__(kWideBlock) void k_wide_hv(const WideItem *items, int n, int nwg, uint32_t nl,
                                                        uint32_t nr, int rg_n, uint32_t emax, int k, int max_k,
                                                        double acc) {
  extern __shared__ double smem[];
  __shared__ double sh[kWideBlock / kW];
  int item, w;
  if (!wide_place(n, nwg, item, w)) return;
  const WideItem it = items[item];
  const size_t dim = (size_t)nl * nr;
  const double *C = it.u + (MODE == 2 ? (size_t)((k - 1) & 1) : (size_t)(k & 1)) * dim;
  double *P = it.u + (MODE == 2 ? (size_t)(k & 1) : (size_t)((k + 1) & 1)) * dim;
  double c_h, c_p, c_x = 0.0, z = 0.0;  // t = c_h H x - c_p P - c_x x
  if (MODE == 2) {
    if (k >= (int)it.sc[SC_N]) return;
    const double ib = 1.0 / it.b[k];
    c_h = ib;
    c_p = k >= 2 ? it.b[k - 1] * ib : 0.0;
    c_x = it.a[k - 1] * ib;
    z = it.a[3 * (size_t)max_k + k];  // the tridiagonal arrays start at a: alpha, beta, beta^2, z, ...
  } else {
    if (it.sc[SC_N] != kRunning) return;
    const double s2 = wide_fold(it.part + nwg, nwg), nk = sqrt(s2);
    bool stop;
    if (k == 0) {
      stop = MODE == 0 ? !(s2 > 1e-14) : !(s2 > 0.0);
      if (w == 0 && threadIdx.x == 0) {
        it.sc[SC_NN] = s2;
        if (stop) it.sc[SC_N] = -1.0;
      }
    } else {
      const double prod = it.sc[SC_PROD + ((k - 1) & 1)] * nk;
      stop = MODE == 0 ? !(prod > acc && nk > acc && k < max_k) : !(nk > 0.0);
      if (w == 0 && threadIdx.x == 0) {
        it.b[k] = nk;
        it.sc[SC_PROD + (k & 1)] = prod;
        if (stop) it.sc[SC_N] = (double)k;
      }
    }
    if (stop) return;
    c_h = 1.0 / nk;
    c_p = k == 0 ? 0.0 : nk / (k >= 2 ? it.b[k - 1] : sqrt(it.sc[SC_NN]));
  }
  const bool first = MODE == 2 ? k == 1 : k == 0;  // no previous vector: its buffer is not read
  const uint32_t RG = RG1 ? 1u : (uint32_t)rg_n, R = RG * RPT;
  const uint32_t d0 = (uint32_t)w * R;
  const uint32_t nrow = d0 < nr ? min(R, nr - d0) : 0u;
  const size_t base = (size_t)d0 * nl;
  // staged: the neighbour lists of the R rows, padded to emax entries (own
  // row, value 0), and the rows themselves
  double *nval = smem, *xs = smem + (size_t)R * emax + (R * emax + 1) / 2;
  uint32_t *ncol = reinterpret_cast<uint32_t *>(smem + (size_t)R * emax);
  for (uint32_t f = threadIdx.x; f < R * emax; f += kWideBlock) {
    const uint32_t r = f / emax, q = f - r * emax, d = min(d0 + r, nr - 1);
    const uint32_t e = it.rp[d] + q;
    const bool in = r < nrow && e < it.rp[d + 1];
    ncol[f] = in ? it.rc[e] : d;
    nval[f] = in ? it.rv[e] : 0.0;
  }
  if (STAGE)
    for (uint32_t f = threadIdx.x; f < nrow * nl; f += kWideBlock) xs[f] = C[base + f];
  __syncthreads();
  const double *X = STAGE ? xs : C + base;
  double dot = 0.0;
  const uint32_t rg = RG1 ? 0u : threadIdx.x / nl;
  for (uint32_t il = RG1 ? threadIdx.x : threadIdx.x - rg * nl; il < nl && rg < RG; il += RG1 ? kWideBlock : nl) {
    // (rows past the last one repeat it, so that every load is in range; their
    // results are not used)
    uint32_t ro[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j) ro[j] = min(rg + RG * j, nrow - 1);
    double h[RPT], pv[RPT];
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const size_t I = base + (size_t)ro[j] * nl + il;
      h[j] = it.dg[I];
      pv[j] = first ? 0.0 : P[I];
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) h[j] *= X[(size_t)ro[j] * nl + il];
    const uint32_t e1 = it.lp[il + 1];
    uint32_t e = it.lp[il];
    for (; e + 4 <= e1; e += 4) {
      uint32_t c[4];
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        c[q] = it.lc[e + q];
        v[q] = it.lv[e + q];
      }
#pragma unroll
      for (int j = 0; j < RPT; ++j) {
        const double *xr = X + (size_t)ro[j] * nl;
#pragma unroll
        for (int q = 0; q < 4; ++q) h[j] += v[q] * xr[c[q]];
      }
    }
    for (; e < e1; ++e) {
      const uint32_t c = it.lc[e];
      const double v = it.lv[e];
#pragma unroll
      for (int j = 0; j < RPT; ++j) h[j] += v * X[(size_t)ro[j] * nl + c];
    }
    // the row part: one neighbour of each of the RPT rows at a time, their
    // loads in flight together
#pragma unroll 2
    for (uint32_t q = 0; q < emax; ++q) {
      double x[RPT];
#pragma unroll
      for (int j = 0; j < RPT; ++j) x[j] = C[(size_t)ncol[ro[j] * emax + q] * nl + il];
#pragma unroll
      for (int j = 0; j < RPT; ++j) h[j] += nval[ro[j] * emax + q] * x[j];
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const uint32_t r = rg + RG * j;
      if (r >= nrow) continue;
      const size_t I = base + (size_t)r * nl + il;
      const double x = X[(size_t)r * nl + il];
      double t = c_h * h[j] - c_p * pv[j];
      if (MODE == 2) t -= c_x * x;
      P[I] = t;
      if (MODE == 2) it.u[2 * dim + I] += z * t;
      else dot += t * x;
    }
    if (!RG1) break;
  }
  if (MODE != 2) {
    dot = bsum<kWideBlock>(dot, sh);
    if (threadIdx.x == 0) it.part[w] = dot;
  }
}

__global__ __launch_bounds__(kWideBlock) void k_wide_upd(const WideItem *items, int n, int nwg, size_t dim, int k) {
  __shared__ double sh[kWideBlock / kW];
  int item, w;
  if (!wide_place(n, nwg, item, w)) return;
  const WideItem it = items[item];
  if (it.sc[SC_N] != kRunning) return;
  const double inv = 1.0 / (k >= 1 ? it.b[k] : sqrt(it.sc[SC_NN]));
  const double alpha = wide_fold(it.part, nwg) * inv;
  if (w == 0 && threadIdx.x == 0) it.a[k] = alpha;
  const double c = alpha * inv;
  const double *C = it.u + (size_t)(k & 1) * dim;
  double *T = it.u + (size_t)((k + 1) & 1) * dim;
  const size_t chunk = (dim + nwg - 1) / nwg, i0 = (size_t)w * chunk, i1 = min(dim, i0 + chunk);
  double s = 0.0;
  for (size_t i = i0 + threadIdx.x; i < i1; i += kWideBlock) {
    const double t = T[i] - c * C[i];
    T[i] = t;
    s += t * t;
  }
  s = bsum<kWideBlock>(s, sh);
  if (threadIdx.x == 0) it.part[nwg + w] = s;
}

// U_0 of a continued fraction: psi = c_o1 |gs> (+ c_o2 |gs>)
__global__ __launch_bounds__(kWideBlock) void k_wide_cf_init(const WideItem *items, const BatchCFItem *src, int n,
                                                             int nwg, uint32_t nl, uint32_t nr, int swap) {
  __shared__ double sh[kWideBlock / kW];
  int item, w;
  if (!wide_place(n, nwg, item, w)) return;
  const WideItem it = items[item];
  const BatchCFItem &q = src[item];
  const double *gs = q.gs;
  const uint32_t du_s = q.du_s;
  const int spin = q.spin, norb = q.norb;
  const int32_t *map0 = q.map[0], *map1 = q.map[1];
  const int8_t *sgn0 = q.sgn[0], *sgn1 = q.sgn[1], *upar = q.upar;
  const size_t dim = (size_t)nl * nr, chunk = (dim + nwg - 1) / nwg, i0 = (size_t)w * chunk;
  const size_t i1 = min(dim, i0 + chunk);
  double s = 0.0;
  for (size_t J = i0 + threadIdx.x; J < i1; J += kWideBlock) {
    const uint32_t r = (uint32_t)(J / nl), l = (uint32_t)(J - (size_t)r * nl);
    const uint32_t iu = swap ? r : l, id = swap ? l : r;
    const uint32_t im = spin == 0 ? iu : id;
    double val = 0.0;
    const int32_t s0 = map0[im];
    if (s0 >= 0) val += (double)sgn0[im] * gs[spin == 0 ? (size_t)s0 + (size_t)du_s * id : iu + (size_t)du_s * s0];
    if (norb == 2) {
      const int32_t s1 = map1[im];
      if (s1 >= 0) val += (double)sgn1[im] * gs[spin == 0 ? (size_t)s1 + (size_t)du_s * id : iu + (size_t)du_s * s1];
    }
    if (spin == 1) val *= (double)upar[iu];
    it.u[J] = val;
    s += val * val;
  }
  s = bsum<kWideBlock>(s, sh);
  if (threadIdx.x == 0) {
    it.part[nwg + w] = s;
    if (w == 0) {
      it.sc[SC_N] = kRunning;
      it.sc[SC_PROD] = 1.0;
    }
  }
}

// U_0 of a ground state: normal draws in label order.  replay: the draws
// normalized, and the eigenvector's first term z_0 v_0
__global__ __launch_bounds__(kWideBlock) void k_wide_gs_init(const WideItem *items, const BatchGSItem *src, int n,
                                                             int nwg, uint32_t nl, uint32_t nr, int swap, int M,
                                                             int replay) {
  __shared__ double sh[kWideBlock / kW];
  int item, w;
  if (!wide_place(n, nwg, item, w)) return;
  const WideItem it = items[item];
  const uint64_t seed = src[item].seed;
  const size_t dim = (size_t)nl * nr, chunk = (dim + nwg - 1) / nwg, i0 = (size_t)w * chunk;
  const size_t i1 = min(dim, i0 + chunk);
  const double inv = replay ? 1.0 / sqrt(it.sc[SC_NN]) : 1.0, z0 = replay ? it.a[3 * (size_t)M] : 0.0;
  double s = 0.0;
  for (size_t J = i0 + threadIdx.x; J < i1; J += kWideBlock) {
    const uint32_t r = (uint32_t)(J / nl), l = (uint32_t)(J - (size_t)r * nl);
    const size_t I = swap ? (size_t)r + (size_t)nr * l : J;
    const double x = normal_draw(seed, I) * inv;
    it.u[J] = x;
    if (replay) it.u[2 * dim + J] = z0 * x;
    s += x * x;
  }
  if (replay) return;
  s = bsum<kWideBlock>(s, sh);
  if (threadIdx.x == 0) {
    it.part[nwg + w] = s;
    if (w == 0) {
      it.sc[SC_N] = kRunning;
      it.sc[SC_PROD] = 1.0;
      it.sc[SC_HI] = __builtin_nan("");
      it.sc[SC_STATUS] = 0.0;
    }
  }
}

// after step k: the Ritz pair of the (k + 1) x (k + 1) tridiagonal and the
// stop rule of the ground state, one wave per item.  LDS: the tridiagonal in
// LDS, since the Sturm counts and the inverse iteration walk it serially; else
// (more steps than fit) on the item's own arrays.
template <bool LDS>
__global__ __launch_bounds__(kW) void k_wide_ritz(const WideItem *items, int nwg, int M, int k, int max_iter,
                                                  double accur) {
  extern __shared__ double smem[];
  __shared__ double s_lam, s_zl, s_hi;
  const WideItem it = items[blockIdx.x];
  if (it.sc[SC_N] != kRunning) return;
  const size_t len = LDS ? (size_t)k + 1 : (size_t)M;
  double *al = LDS ? smem : it.a;
  double *be = al + len, *bb = be + len, *z = bb + len, *D = z + len, *l = D + len;
  double *be_g = it.a + M, *z_g = it.a + 3 * (size_t)M;
  const double beta = sqrt(wide_fold(it.part + nwg, nwg));
  if (LDS)
    for (int i = threadIdx.x; i <= k; i += kW) {
      const double bi = i < k ? be_g[i] : beta;
      al[i] = it.a[i];
      be[i] = bi;
      bb[i] = bi * bi;
    }
  else
    for (int i = threadIdx.x; i < k; i += kW) bb[i] = be[i] * be[i];  // (the LDS form leaves none)
  if (threadIdx.x == 0) {
    be_g[k] = beta;
    if (!LDS) bb[k] = beta * beta;
    s_hi = it.sc[SC_HI];
  }
  __syncthreads();
  tri_lowest_wave(k + 1, al, be, bb, &s_hi, z, D, l, &s_lam, &s_zl);
  __syncthreads();
  if (LDS)
    for (int i = threadIdx.x; i <= k; i += kW) z_g[i] = z[i];
  if (threadIdx.x == 0) {
    it.sc[SC_HI] = s_hi;
    it.sc[SC_LAM] = s_lam;
    if (!(beta > 0.0) || fabs(s_zl * beta) <= accur) it.sc[SC_N] = (double)(k + 1);
    else if (k + 1 > max_iter) {
      it.sc[SC_STATUS] = 1.0;
      it.sc[SC_N] = (double)(k + 1);
    }
  }
}

// norm partials of the eigenvector, then (scale) the normalized eigenvector in
// label order and the item's results
__global__ __launch_bounds__(kWideBlock) void k_wide_gs_out(const WideItem *items, const BatchGSItem *src, int n,
                                                            int nwg, uint32_t nl, uint32_t nr, int swap, int scale) {
  __shared__ double sh[kWideBlock / kW];
  int item, w;
  if (!wide_place(n, nwg, item, w)) return;
  const WideItem it = items[item];
  const size_t dim = (size_t)nl * nr, chunk = (dim + nwg - 1) / nwg, i0 = (size_t)w * chunk;
  const size_t i1 = min(dim, i0 + chunk);
  const double *g = it.u + 2 * dim;
  if (!scale) {
    double s = 0.0;
    for (size_t J = i0 + threadIdx.x; J < i1; J += kWideBlock) s += g[J] * g[J];
    s = bsum<kWideBlock>(s, sh);
    if (threadIdx.x == 0) it.part[w] = s;
    return;
  }
  const double ig = 1.0 / sqrt(wide_fold(it.part, nwg));
  double *gs = src[item].gs;
  for (size_t J = i0 + threadIdx.x; J < i1; J += kWideBlock) {
    const uint32_t r = (uint32_t)(J / nl), l = (uint32_t)(J - (size_t)r * nl);
    gs[swap ? (size_t)r + (size_t)nr * l : J] = g[J] * ig;
  }
  if (w == 0 && threadIdx.x == 0) {
    src[item].out[0] = it.sc[SC_LAM];
    src[item].out[1] = it.sc[SC_N];
    src[item].out[2] = it.sc[SC_STATUS];
  }
}

__global__ void k_wide_cf_out(const WideItem *items, const BatchCFItem *src, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  src[k].out[0] = items[k].sc[SC_N];
  src[k].out[1] = items[k].sc[SC_NN];
}

// number of items still running
__global__ __launch_bounds__(kW) void k_wide_running(const WideItem *items, int n, int *count) {
  int c = 0;
  for (int k = threadIdx.x; k < n; k += kW) c += items[k].sc[SC_N] == kRunning;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, kW);
  if (threadIdx.x == 0) *count = c;
}

// writes item k's fraction, transformed as the continued_fraction ctor
// (src_ed/continued_fraction.cpp:33-42) does, at off[fid[k]] of the store:
// a_i - E0 (electrons, pm > 0) or E0 - a_i (holes) in A; b_0 = ||psi||^2 w
// and b_i^2 (0 < i < n) in B
__global__ void k_cf_store(int nitems, int max_cf, const double *out, const double *a, const double *b,
                           const int *fid, const int *off, const double *e0, const double *w, const int8_t *pm,
                           double *A, double *B) {
  const int k = blockIdx.x;
  if (k >= nitems) return;
  const int n = (int)out[2 * (size_t)k];
  if (n <= 0) return;
  const double *ak = a + (size_t)max_cf * k, *bk = b + (size_t)(max_cf + 1) * k;
  const size_t o = (size_t)off[fid[k]];
  const double E = e0[k], b0 = out[2 * (size_t)k + 1] * w[k];
  const bool el = pm[k] > 0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    A[o + i] = el ? ak[i] - E : E - ak[i];
    B[o + i] = i == 0 ? b0 : bk[i] * bk[i];
  }
}

}  // namespace

void batch_gs(const BatchGSItem *d_items, int n, int block, size_t lds, bool tri_lds, int max_iter, double accur,
              hipStream_t s) {
  if (n <= 0) return;
  if (lds > kBatchLdsCap) fail(ED_ERR_INVALID, "batch_gs: LDS request above the cap");
#define ED_GS(BS, TRI) \
  hipLaunchKernelGGL((k_batch_gs<BS, TRI>), dim3(n), dim3(BS), lds, s, d_items, max_iter, accur)
  if (block == 256) {
    if (tri_lds) ED_GS(256, true);
    else ED_GS(256, false);
  } else {
    if (tri_lds) ED_GS(64, true);
    else ED_GS(64, false);
  }
#undef ED_GS
  ED_HIP(hipGetLastError());
}

void batch_cf(const BatchCFItem *d_items, int n, int block, size_t lds, int max_cf, double acc, hipStream_t s) {
  if (n <= 0) return;
  if (lds > kBatchLdsCap) fail(ED_ERR_INVALID, "batch_cf: LDS request above the cap");
  if (block == 256)
    hipLaunchKernelGGL((k_batch_cf<256>), dim3(n), dim3(256), lds, s, d_items, max_cf, acc);
  else
    hipLaunchKernelGGL((k_batch_cf<64>), dim3(n), dim3(64), lds, s, d_items, max_cf, acc);
  ED_HIP(hipGetLastError());
}

WideShape wide_shape(uint32_t du, uint32_t dd, uint32_t emax) {
  WideShape W;
  W.emax = emax;
  W.swap = dd > du;
  W.nl = W.swap ? dd : du;
  W.nr = W.swap ? du : dd;
  const size_t row = W.nl * sizeof(double);
  W.stage = row <= kWideLdsMax;
  // rows longer than half a workgroup: one row at a time per thread column,
  // four rows sharing a table load; shorter ones several side by side.  The
  // split depends on the sector alone, so an item's sums, and its fraction to
  // the last bit, do not depend on what runs beside it.
  const int rg = W.nl > (uint32_t)kWideBlock / 2 ? 1 : kWideBlock / (int)W.nl;
  W.rpt = rg > 1 ? 2 : 4;
  while (W.rpt > 1 && (!W.stage || W.rpt * row > 64 * 1024)) W.rpt /= 2;
  W.rows = rg * W.rpt;
  W.nwg = (int)((W.nr + W.rows - 1) / W.rows);
  W.lds = ((size_t)W.rows * emax + ((size_t)W.rows * emax + 1) / 2) * sizeof(double) + (W.stage ? W.rows * row : 0);
  return W;
}

namespace {
bool wide_spread(const WideShape &W) { return (size_t)W.nl * W.nr >= kWideSpread; }
// the kernels' nwg (negated: workgroups in runs, see wide_place) and their grid
int wide_nwg(const WideShape &W) { return wide_spread(W) ? -W.nwg : W.nwg; }
unsigned wide_grid(const WideShape &W, int n) {
  if (wide_spread(W)) return (unsigned)(((size_t)n * W.nwg + kXcd - 1) / kXcd * kXcd);
  return (unsigned)(kXcd * ((n + kXcd - 1) / kXcd) * W.nwg);
}

template <int MODE>
void wide_hv(const WideShape &W, const WideItem *items, int n, int k, int max_k, double acc, hipStream_t s) {
  const int rg = W.rows / W.rpt;
#define ED_WIDE(RPT, RG1, STG)                                                                                    \
  do {                                                                                                            \
    if (W.lds > 64 * 1024)                                                                                        \
      ED_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_wide_hv<MODE, RPT, RG1, STG>),                  \
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)W.lds));                        \
    hipLaunchKernelGGL((k_wide_hv<MODE, RPT, RG1, STG>), dim3(wide_grid(W, n)), dim3(kWideBlock), W.lds, s,       \
                       items, n, wide_nwg(W), W.nl, W.nr, rg, W.emax, k, max_k, acc);                            \
  } while (0)
  if (!W.stage) ED_WIDE(1, true, false);
  else if (rg > 1) ED_WIDE(2, false, true);
  else if (W.rpt == 4) ED_WIDE(4, true, true);
  else if (W.rpt == 2) ED_WIDE(2, true, true);
  else ED_WIDE(1, true, true);
#undef ED_WIDE
}

void wide_upd(const WideShape &W, const WideItem *items, int n, int k, hipStream_t s) {
  hipLaunchKernelGGL(k_wide_upd, dim3(wide_grid(W, n)), dim3(kWideBlock), 0, s, items, n, wide_nwg(W),
                     (size_t)W.nl * W.nr, k);
}

// items still running, asked of the device every kWideCheck steps
constexpr int kWideCheck = 16;
bool wide_running(const WideItem *items, int n, DevBuf<int> &count, hipStream_t s) {
  check_cancel();
  hipLaunchKernelGGL(k_wide_running, dim3(1), dim3(kW), 0, s, items, n, count.p);
  ED_HIP(hipGetLastError());
  return count.to_host()[0] > 0;
}
}  // namespace

void wide_cf(const WideShape &W, const WideItem *items, const BatchCFItem *src, int n, int max_cf, double acc,
             hipStream_t s) {
  if (n <= 0) return;
  DevBuf<int> count(1);
  hipLaunchKernelGGL(k_wide_cf_init, dim3(wide_grid(W, n)), dim3(kWideBlock), 0, s, items, src, n, wide_nwg(W), W.nl, W.nr,
                     W.swap);
  for (int k = 0; k <= max_cf; ++k) {
    wide_hv<0>(W, items, n, k, max_cf, acc, s);  // k == max_cf only ends the items
    if (k == max_cf) break;
    wide_upd(W, items, n, k, s);
    if ((k + 1) % kWideCheck == 0 && !wide_running(items, n, count, s)) break;
  }
  hipLaunchKernelGGL(k_wide_cf_out, dim3((n + 255) / 256), dim3(256), 0, s, items, src, n);
  ED_HIP(hipGetLastError());
}

void wide_gs(const WideShape &W, const WideItem *items, const BatchGSItem *src, int n, int max_iter, double accur,
             hipStream_t s) {
  if (n <= 0) return;
  DevBuf<int> count(1);
  const int M = max_iter + 2;
  const unsigned g = wide_grid(W, n);
  hipLaunchKernelGGL(k_wide_gs_init, dim3(g), dim3(kWideBlock), 0, s, items, src, n, wide_nwg(W), W.nl, W.nr, W.swap, M, 0);
  int k = 0;
  for (;; ++k) {
    wide_hv<1>(W, items, n, k, 0, 0.0, s);
    wide_upd(W, items, n, k, s);
    const size_t tri = (size_t)kTriArrays * (k + 1) * sizeof(double);
    if (tri <= kTriLdsMax) {
      if (tri > 64 * 1024)
        ED_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_wide_ritz<true>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)tri));
      hipLaunchKernelGGL((k_wide_ritz<true>), dim3(n), dim3(kW), tri, s, items, W.nwg, M, k, max_iter, accur);
    } else {
      hipLaunchKernelGGL((k_wide_ritz<false>), dim3(n), dim3(kW), 0, s, items, W.nwg, M, k, max_iter, accur);
    }
    // (k_wide_ritz ends every item by step max_iter)
    if ((k >= max_iter || (k + 1) % kWideCheck == 0) && !wide_running(items, n, count, s)) break;
  }
  hipLaunchKernelGGL(k_wide_gs_init, dim3(g), dim3(kWideBlock), 0, s, items, src, n, wide_nwg(W), W.nl, W.nr, W.swap, M, 1);
  for (int j = 1; j <= k; ++j) wide_hv<2>(W, items, n, j, M, 0.0, s);
  for (int scale = 0; scale < 2; ++scale)
    hipLaunchKernelGGL(k_wide_gs_out, dim3(g), dim3(kWideBlock), 0, s, items, src, n, wide_nwg(W), W.nl, W.nr, W.swap,
                       scale);
  ED_HIP(hipGetLastError());
}

void tile_cf(const BatchCFItem *d_items, int n, int rt, int ct, int max_cf, double acc, hipStream_t s) {
  if (n <= 0) return;
  if (rt < 1 || rt > 2 || ct < 1 || ct > 2) fail(ED_ERR_INTERNAL, "tile_cf: sector beyond 32 x 32 half states");
#define ED_TILE(R, C) hipLaunchKernelGGL((k_tile_cf<R, C>), dim3(n), dim3(kW), 0, s, d_items, max_cf, acc)
  if (rt == 1 && ct == 1) ED_TILE(1, 1);
  else if (rt == 1) ED_TILE(1, 2);
  else if (ct == 1) ED_TILE(2, 1);
  else ED_TILE(2, 2);
#undef ED_TILE
  ED_HIP(hipGetLastError());
}

void batch_cf_store(int nitems, int max_cf, const double *out, const double *a, const double *b, const int *fid,
                    const int *off, const double *e0, const double *w, const int8_t *pm, double *A, double *B,
                    hipStream_t s) {
  if (nitems <= 0) return;
  hipLaunchKernelGGL(k_cf_store, dim3(nitems), dim3(64), 0, s, nitems, max_cf, out, a, b, fid, off, e0, w, pm, A, B);
  ED_HIP(hipGetLastError());
}

}  // namespace ed
