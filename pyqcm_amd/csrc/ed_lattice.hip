// ed_lattice.hip -- (frequency, wavevector) grid sums for CPT and the
// self-energy functional: per (frequency, k) the d x d matrix V(k) G is formed
// and factored with partial pivoting, LU for log|det(V G - 1)|, Gauss-Jordan
// for (1 - V G)^{-1}; sums over k run in a fixed order, so results do not
// depend on scheduling.  Two kernels: k_lattice_reg (d <= 6) keeps one matrix
// per lane in registers, k_lattice (d = 7, 8, where a matrix no longer fits
// beside its temporaries) one matrix per wave in LDS.
#include "ed_lattice.hpp"

#include <cmath>
#include <cstring>

namespace ed {

long KGrid::count() const {
  long n = 1;
  for (int a = 0; a < dim; ++a) n *= nk[a];
  return n;
}

// The elements go to the device grouped as the kernel for this d reads them, all
// parts in one block of doubles: V0, the values, R, then the integer lists.  Up
// to kRegDim by neighbor vector (one phase serves a group); above by position,
// since there a lane owns one.
SuperlatticeDev::SuperlatticeDev(const Superlattice &S) : d(S.d), nnbr((int)S.R.size() / 3) {
  const int dd = d * d;
  const bool reg = d <= kRegDim;
  const size_t ne = S.nbr.size(), ng = reg ? (size_t)nnbr : (size_t)dd;
  const auto group = [&](size_t r) { return reg ? S.nbr[r] : S.row[r] + d * S.col[r]; };
  std::vector<int> eptr(ng + 1, 0), epos(std::max<size_t>(ne, 1), 0);
  std::vector<double> ev(2 * std::max<size_t>(ne, 1), 0.0);
  std::vector<char> used(dd, 0);
  for (int e = 0; e < dd; ++e) used[e] = S.V0[2 * e] != 0.0 || S.V0[2 * e + 1] != 0.0;
  for (size_t r = 0; r < ne; ++r) {
    ++eptr[group(r) + 1];
    used[S.row[r] + d * S.col[r]] = 1;
  }
  for (size_t n = 0; n < ng; ++n) eptr[n + 1] += eptr[n];
  std::vector<int> fill(eptr.begin(), eptr.end() - 1), plist, slot(dd, 0);
  for (int e = 0; e < dd; ++e)
    if (used[e]) {
      slot[e] = (int)plist.size();
      plist.push_back(e);
      if (dd <= 64) mask |= 1ull << e;  // larger d: refused when a sum is asked for
    }
  npos = (int)plist.size();
  for (size_t r = 0; r < ne; ++r) {
    const int at = fill[group(r)]++;
    epos[at] = reg ? slot[S.row[r] + d * S.col[r]] : S.nbr[r];
    ev[2 * at] = S.val[2 * r];
    ev[2 * at + 1] = S.val[2 * r + 1];
  }
  std::vector<double> blob(S.V0.begin(), S.V0.begin() + 2 * dd);
  auto put_d = [&](const std::vector<double> &v) {
    const size_t at = blob.size();
    blob.insert(blob.end(), v.begin(), v.end());
    return at;
  };
  auto put_i = [&](const std::vector<int> &v) {
    const size_t at = blob.size();
    blob.resize(at + (v.size() + 1) / 2 + 1);
    std::memcpy(blob.data() + at, v.data(), v.size() * sizeof(int));
    return at;
  };
  const size_t ov = put_d(ev), oR = put_d(S.R), op = put_i(eptr), oe = put_i(epos), ol = put_i(plist);
  mem.upload(blob);
  V0 = mem.p;
  val = mem.p + ov;
  R = mem.p + oR;
  eptr_d = reinterpret_cast<const int *>(mem.p + op);
  epos_d = reinterpret_cast<const int *>(mem.p + oe);
  plist_d = reinterpret_cast<const int *>(mem.p + ol);
}

namespace {

constexpr long kLatticeWaves = 4096;  // waves a launch is cut into (1024 SIMDs x 4)

struct Arg {
  int d, nnbr, dim, nk0, nk1, nk2, npos;
  unsigned long long mask;
  double off;
  long nk, kchunk;
  const double *V0, *val, *R;
  const int *eptr, *epos, *plist;
};

__device__ __forceinline__ void cmul(double ar, double ai, double br, double bi, double &r, double &i) {
  r = ar * br - ai * bi;
  i = ar * bi + ai * br;
}

// exp(2 pi i k . R_n) of grid point kk
__device__ __forceinline__ void phase(const Arg &A, long kk, int n, double &cs, double &sn) {
  const long a0 = kk % A.nk0, a1 = (kk / A.nk0) % A.nk1, a2 = kk / ((long)A.nk0 * A.nk1);
  const double kx = A.dim >= 1 ? ((double)a0 + A.off) / A.nk0 : 0.0;
  const double ky = A.dim >= 2 ? ((double)a1 + A.off) / A.nk1 : 0.0;
  const double kz = A.dim >= 3 ? ((double)a2 + A.off) / A.nk2 : 0.0;
  const double ang = 2.0 * M_PI * (kx * A.R[3 * n] + ky * A.R[3 * n + 1] + kz * A.R[3 * n + 2]);
  sincos(ang, &sn, &cs);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <int D>
__device__ __forceinline__ void cond_swap(bool sw, double &a, double &b) {
  const double t = sw ? b : a;
  b = sw ? a : b;
  a = t;
}

// Register kernel, d = D <= 6: one wave per (zc frequencies, chunk of k
// points), one k point per lane.  V(k) is formed once per k point at the
// npos positions it can be nonzero and kept in LDS (a lane reads only its own
// column: no conflicts, no barriers); G is uniform over the wave and comes
// from scalar loads; V G and the factorization are unrolled over static
// registers.  FP64 VALU bound: 4 x 4 log-determinants take ~500 and 6 x 6
// inverses ~2300 vector instructions per 64 points, against one matrix per
// group of 16-64 lanes in LDS, where a d = 4 factorization was a chain of
// ~40 barrier-separated steps with 6-16 of 64 lanes doing arithmetic.
// Whole calls on the MI355X: 2 x 96 frequencies x 128^2 points of 4 x 4
// log-determinants 2.57 -> 0.43 ms, 256 x 64^2 inverses of 6 x 6 3.21 -> 0.47.
// MODE 0: part[iz][chunk] = sum over the chunk of log|det(V G - 1)|
// MODE 1: part[iz][chunk][e] = sum over the chunk of ((1 - V G)^{-1})_e
template <int MODE, int D>
__global__ __launch_bounds__(64) void k_lattice_reg(Arg A, int nz, int zc, const double *__restrict__ Gz,
                                                    double *__restrict__ part) {
  constexpr int DD = D * D, W = MODE == 0 ? 1 : 2 * DD;
  extern __shared__ double lds[];
  __shared__ double sred[MODE == 0 ? 1 : 16 * 65];
  double2 *sV = reinterpret_cast<double2 *>(lds);  // [npos][64]
  double *sAcc = lds + (size_t)A.npos * 128;       // [zc][W]
  const int lane = threadIdx.x, iz0 = blockIdx.y * zc, nzc = min(zc, nz - iz0);
  for (int t = lane; t < nzc * W; t += 64) sAcc[t] = 0.0;
  const long k0 = (long)blockIdx.x * A.kchunk, k1 = k0 + A.kchunk < A.nk ? k0 + A.kchunk : A.nk;
  for (long kb = k0; kb < k1; kb += 64) {
    const bool valid = kb + lane < k1;
    const long kk = valid ? kb + lane : k1 - 1;
    for (int p = 0; p < A.npos; ++p) {
      const int e = A.plist[p];
      sV[p * 64 + lane] = make_double2(A.V0[2 * e], A.V0[2 * e + 1]);
    }
    for (int n = 0; n < A.nnbr; ++n) {
      double cs, sn;
      phase(A, kk, n, cs, sn);
      for (int r = A.eptr[n]; r < A.eptr[n + 1]; ++r) {
        double2 &v = sV[A.epos[r] * 64 + lane];
        double tr, ti;
        cmul(A.val[2 * r], A.val[2 * r + 1], cs, sn, tr, ti);
        v.x += tr;
        v.y += ti;
      }
    }
    for (int z = 0; z < nzc; ++z) {
      const double *G = Gz + 2 * (size_t)(iz0 + z) * DD;
      double mr[DD], mi[DD];  // column-major, as G
#pragma unroll
      for (int e = 0; e < DD; ++e) mr[e] = mi[e] = 0.0;
      int p = 0;
#pragma unroll
      for (int l = 0; l < D; ++l) {
        if (!((A.mask >> (l * D)) & ((1ull << D) - 1ull))) continue;
        double gr[D], gi[D];
#pragma unroll
        for (int j = 0; j < D; ++j) {
          gr[j] = G[2 * (l + j * D)];
          gi[j] = G[2 * (l + j * D) + 1];
        }
#pragma unroll
        for (int i = 0; i < D; ++i) {
          if (!((A.mask >> (i + l * D)) & 1ull)) continue;
          const double2 v = sV[p * 64 + lane];
          ++p;
#pragma unroll
          for (int j = 0; j < D; ++j) {
            mr[i + j * D] += v.x * gr[j] - v.y * gi[j];
            mi[i + j * D] += v.x * gi[j] + v.y * gr[j];
          }
        }
      }
#pragma unroll
      for (int e = 0; e < DD; ++e) {
        if (MODE == 1) {
          mr[e] = -mr[e];
          mi[e] = -mi[e];
        }
        if (e % D == e / D) mr[e] += MODE == 0 ? -1.0 : 1.0;
      }
      double prod = 1.0, logdet = 0.0;
      int piv[D];
#pragma unroll
      for (int c = 0; c < D; ++c) {
        // pivot row: the first largest |M(r, c)|, r >= c; the rows are
        // exchanged by selects, skipped where no lane of the wave needs them
        double q2 = mr[c + c * D] * mr[c + c * D] + mi[c + c * D] * mi[c + c * D];
        int pr = c;
#pragma unroll
        for (int r = c + 1; r < D; ++r) {
          const double m2 = mr[r + c * D] * mr[r + c * D] + mi[r + c * D] * mi[r + c * D];
          if (m2 > q2) {
            q2 = m2;
            pr = r;
          }
        }
        piv[c] = pr;
#pragma unroll
        for (int r = c + 1; r < D; ++r) {
          if (!__any(pr == r)) continue;
#pragma unroll
          for (int j = MODE == 0 ? c : 0; j < D; ++j) {
            cond_swap<D>(pr == r, mr[c + j * D], mr[r + j * D]);
            cond_swap<D>(pr == r, mi[c + j * D], mi[r + j * D]);
          }
        }
        if (MODE == 0) {
          // the product of the squared pivots is kept within range
          const double p2 = prod * q2;
          if (p2 < 1e100 && p2 > 1e-100) {
            prod = p2;
          } else {
            logdet += log(prod) + log(q2);
            prod = 1.0;
          }
          if (c == D - 1) break;
        }
        const double iq = 1.0 / q2, ir = mr[c + c * D] * iq, ii = -mi[c + c * D] * iq;
        if (MODE == 0) {
#pragma unroll
          for (int r = c + 1; r < D; ++r) {
            double fr, fi;
            cmul(mr[r + c * D], mi[r + c * D], ir, ii, fr, fi);
#pragma unroll
            for (int j = c + 1; j < D; ++j) {
              mr[r + j * D] -= fr * mr[c + j * D] - fi * mi[c + j * D];
              mi[r + j * D] -= fr * mi[c + j * D] + fi * mr[c + j * D];
            }
          }
        } else {
          // Gauss-Jordan in place: column c becomes that of the inverse
          mr[c + c * D] = 1.0;
          mi[c + c * D] = 0.0;
#pragma unroll
          for (int j = 0; j < D; ++j) {
            double tr, ti;
            cmul(mr[c + j * D], mi[c + j * D], ir, ii, tr, ti);
            mr[c + j * D] = tr;
            mi[c + j * D] = ti;
          }
#pragma unroll
          for (int r = 0; r < D; ++r) {
            if (r == c) continue;
            const double fr = mr[r + c * D], fi = mi[r + c * D];
            mr[r + c * D] = 0.0;
            mi[r + c * D] = 0.0;
#pragma unroll
            for (int j = 0; j < D; ++j) {
              mr[r + j * D] -= fr * mr[c + j * D] - fi * mi[c + j * D];
              mi[r + j * D] -= fr * mi[c + j * D] + fi * mr[c + j * D];
            }
          }
        }
      }
      if (MODE == 0) {
        logdet = 0.5 * (logdet + log(prod));
        const double s = wave_sum(valid ? logdet : 0.0);
        if (lane == 0) sAcc[z] += s;
      } else {
        // the row exchanges, undone as column exchanges in reverse order
#pragma unroll
        for (int c = D - 1; c >= 0; --c)
#pragma unroll
          for (int r = c + 1; r < D; ++r) {
            if (!__any(piv[c] == r)) continue;
#pragma unroll
            for (int i = 0; i < D; ++i) {
              cond_swap<D>(piv[c] == r, mr[i + c * D], mr[i + r * D]);
              cond_swap<D>(piv[c] == r, mi[i + c * D], mi[i + r * D]);
            }
          }
        // sum over the lanes, 16 values at a time through LDS: four lanes add
        // sixteen points each of one value
#pragma unroll
        for (int g = 0; g < (W + 15) / 16; ++g) {
          __syncthreads();
#pragma unroll
          for (int t = 0; t < 16; ++t) {
            const int w = g * 16 + t;
            if (w < W) sred[t * 65 + lane] = valid ? (w & 1 ? mi[w / 2] : mr[w / 2]) : 0.0;
          }
          __syncthreads();
          const int t = lane >> 2, qd = lane & 3, w = g * 16 + t;
          double s = 0.0;
          if (w < W)
#pragma unroll
            for (int j = 0; j < 16; ++j) s += sred[t * 65 + qd * 16 + j];
          s += __shfl_xor(s, 1, 64);
          s += __shfl_xor(s, 2, 64);
          if (qd == 0 && w < W) sAcc[z * W + w] += s;
        }
      }
    }
  }
  __syncthreads();
  for (int t = lane; t < nzc * W; t += 64)
    part[((size_t)(iz0 + t / W) * gridDim.x + blockIdx.x) * W + t % W] = sAcc[t];
}

// index of the largest value over the wave (ties: the smaller index)
__device__ __forceinline__ int wave_argmax(double v, int who) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double v2 = __shfl_xor(v, o, 64);
    const int w2 = __shfl_xor(who, o, 64);
    if (v2 > v || (v2 == v && w2 < who)) {
      v = v2;
      who = w2;
    }
  }
  return who;
}

// LDS kernel for d = 7, 8 (a matrix of 49-64 complex entries and its
// temporaries do not fit one lane's registers): one wave per (frequency,
// chunk of k points), one column-major matrix at a time, lane e < d^2 holding
// element (e mod d, e / d).  Same sums as k_lattice_reg.
template <int MODE>
__global__ __launch_bounds__(64) void k_lattice(Arg A, const double *Gz, double *part) {
  __shared__ double sG[2 * kLatticeMaxDim * kLatticeMaxDim];
  __shared__ double sV[2 * 64], sM[2 * 64], sB[2 * 64];
  __shared__ double sph[2 * kLatticeMaxNbr];
  const int iz = blockIdx.y, chunk = blockIdx.x, e = threadIdx.x, d = A.d, dd = d * d;
  const bool act = e < dd;
  const int i = act ? e % d : 0, j = act ? e / d : 0;
  const long nchunk = gridDim.x;
  if (act) {
    sG[2 * e] = Gz[2 * ((size_t)iz * dd + e)];
    sG[2 * e + 1] = Gz[2 * ((size_t)iz * dd + e) + 1];
  }
  double acc = 0.0, accr = 0.0, acci = 0.0;
  const long k0 = (long)chunk * A.kchunk, k1 = k0 + A.kchunk < A.nk ? k0 + A.kchunk : A.nk;
  for (long kk = k0; kk < k1; ++kk) {
    if (e < A.nnbr) phase(A, kk, e, sph[2 * e], sph[2 * e + 1]);
    __syncthreads();
    if (act) {
      double vr = A.V0[2 * e], vi = A.V0[2 * e + 1];
      for (int r = A.eptr[e]; r < A.eptr[e + 1]; ++r) {
        const int n = A.epos[r];
        double tr, ti;
        cmul(A.val[2 * r], A.val[2 * r + 1], sph[2 * n], sph[2 * n + 1], tr, ti);
        vr += tr;
        vi += ti;
      }
      sV[2 * e] = vr;
      sV[2 * e + 1] = vi;
    }
    __syncthreads();
    if (act) {
      double pr = 0.0, pi = 0.0;
      for (int l = 0; l < d; ++l) {
        double tr, ti;
        cmul(sV[2 * (i + l * d)], sV[2 * (i + l * d) + 1], sG[2 * (l + j * d)], sG[2 * (l + j * d) + 1], tr, ti);
        pr += tr;
        pi += ti;
      }
      const double one = i == j ? 1.0 : 0.0;
      sM[2 * e] = MODE == 0 ? pr - one : one - pr;
      sM[2 * e + 1] = MODE == 0 ? pi : -pi;
      if (MODE == 1) {
        sB[2 * e] = one;
        sB[2 * e + 1] = 0.0;
      }
    }
    __syncthreads();
    double logdet = 0.0;
    for (int c = 0; c < d; ++c) {
      // pivot row: the largest |M(r, c)|, r >= c
      double mag = -1.0;
      if (act && j == c && i >= c) mag = sM[2 * e] * sM[2 * e] + sM[2 * e + 1] * sM[2 * e + 1];
      const int p = wave_argmax(mag, act ? i : d);
      // swap rows c and p (nothing to do where p == c)
      double mr = 0.0, mi = 0.0, br = 0.0, bi = 0.0;
      const bool sw = act && p != c && (i == c || i == p);
      if (sw) {
        const int o = (i == c ? p : c) + j * d;
        mr = sM[2 * o];
        mi = sM[2 * o + 1];
        if (MODE == 1) {
          br = sB[2 * o];
          bi = sB[2 * o + 1];
        }
      }
      __syncthreads();
      if (sw) {
        sM[2 * e] = mr;
        sM[2 * e + 1] = mi;
        if (MODE == 1) {
          sB[2 * e] = br;
          sB[2 * e + 1] = bi;
        }
      }
      __syncthreads();
      const int pc = c + c * d;
      const double qr = sM[2 * pc], qi = sM[2 * pc + 1], q2 = qr * qr + qi * qi;
      logdet += 0.5 * log(q2);
      // 1 / pivot
      const double ir = qr / q2, ii = -qi / q2;
      if (MODE == 0) {
        // LU: rows below the pivot, columns right of it
        double nr = 0.0, ni = 0.0;
        const bool up = act && i > c && j > c;
        if (up) {
          double fr, fi, tr, ti;
          cmul(sM[2 * (i + c * d)], sM[2 * (i + c * d) + 1], ir, ii, fr, fi);
          cmul(fr, fi, sM[2 * (c + j * d)], sM[2 * (c + j * d) + 1], tr, ti);
          nr = sM[2 * e] - tr;
          ni = sM[2 * e + 1] - ti;
        }
        __syncthreads();
        if (up) {
          sM[2 * e] = nr;
          sM[2 * e + 1] = ni;
        }
        __syncthreads();
      } else {
        // Gauss-Jordan on [M | B]: row c scaled by 1 / pivot, eliminated from every other row
        double nmr = 0.0, nmi = 0.0, nbr = 0.0, nbi = 0.0;
        if (act) {
          double cr, ci, dr, di;
          cmul(sM[2 * (c + j * d)], sM[2 * (c + j * d) + 1], ir, ii, cr, ci);
          cmul(sB[2 * (c + j * d)], sB[2 * (c + j * d) + 1], ir, ii, dr, di);
          if (i == c) {
            nmr = cr;
            nmi = ci;
            nbr = dr;
            nbi = di;
          } else {
            const double fr = sM[2 * (i + c * d)], fi = sM[2 * (i + c * d) + 1];
            double tr, ti;
            cmul(fr, fi, cr, ci, tr, ti);
            nmr = sM[2 * e] - tr;
            nmi = sM[2 * e + 1] - ti;
            cmul(fr, fi, dr, di, tr, ti);
            nbr = sB[2 * e] - tr;
            nbi = sB[2 * e + 1] - ti;
          }
        }
        __syncthreads();
        if (act) {
          sM[2 * e] = nmr;
          sM[2 * e + 1] = nmi;
          sB[2 * e] = nbr;
          sB[2 * e + 1] = nbi;
        }
        __syncthreads();
      }
    }
    if (MODE == 0) {
      acc += logdet;
    } else if (act) {
      accr += sB[2 * e];
      acci += sB[2 * e + 1];
    }
    __syncthreads();
  }
  if (MODE == 0) {
    if (e == 0) part[(size_t)iz * nchunk + chunk] = acc;
  } else if (act) {
    const size_t o = ((size_t)iz * nchunk + chunk) * dd + e;
    part[2 * o] = accr;
    part[2 * o + 1] = acci;
  }
}

// the chunks' sums, one workgroup per frequency: four groups of lanes take
// every fourth chunk, then the groups in order.  MODE 1 multiplies the summed
// inverse by G from the left: sum_k G M_k^{-1} = G sum_k M_k^{-1}.
template <int MODE>
__global__ __launch_bounds__(256) void k_lattice_fold(int d, int nchunk, double scale, const double *Gz,
                                                      const double *part, double *out) {
  __shared__ double red[4][2 * 64];
  const int iz = blockIdx.x, dd = d * d, width = MODE == 0 ? 1 : 2 * dd;
  const int t = threadIdx.x & 63, g = threadIdx.x >> 6;
  if (MODE == 0) {
    double s = 0.0;
    for (int c = g * 64 + t; c < nchunk; c += 256) s += part[(size_t)iz * nchunk + c];
    s = wave_sum(s);
    if (t == 0) red[g][0] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[iz] = ((red[0][0] + red[1][0]) + (red[2][0] + red[3][0])) * scale;
    return;
  }
  double sr = 0.0, si = 0.0;
  if (t < dd)
    for (int c = g; c < nchunk; c += 4) {
      const double *p = part + ((size_t)iz * nchunk + c) * width;
      sr += p[2 * t];
      si += p[2 * t + 1];
    }
  red[g][2 * t] = sr;
  red[g][2 * t + 1] = si;
  __syncthreads();
  if (g == 0) {
    sr = (red[0][2 * t] + red[1][2 * t]) + (red[2][2 * t] + red[3][2 * t]);
    si = (red[0][2 * t + 1] + red[1][2 * t + 1]) + (red[2][2 * t + 1] + red[3][2 * t + 1]);
    red[0][2 * t] = sr * scale;
    red[0][2 * t + 1] = si * scale;
  }
  __syncthreads();
  if (g == 0 && t < dd) {
    const int i = t % d, j = t / d;
    const double *G = Gz + 2 * (size_t)iz * dd;
    double xr = 0.0, xi = 0.0;
    for (int l = 0; l < d; ++l) {
      double tr, ti;
      cmul(G[2 * (i + l * d)], G[2 * (i + l * d) + 1], red[0][2 * (l + j * d)], red[0][2 * (l + j * d) + 1], tr, ti);
      xr += tr;
      xi += ti;
    }
    out[2 * ((size_t)iz * dd + t)] = xr;
    out[2 * ((size_t)iz * dd + t) + 1] = xi;
  }
}

template <int MODE, int D>
void launch_reg(const Arg &A, int nz, int zc, long nchunk, size_t lds, const double *dG, double *part) {
  if (lds > 64 * 1024)
    ED_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_lattice_reg<MODE, D>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL((k_lattice_reg<MODE, D>), dim3((unsigned)nchunk, (unsigned)((nz + zc - 1) / zc)), dim3(64), lds,
                     stream(), A, nz, zc, dG, part);
}

template <int MODE>
void run(const SuperlatticeDev &S, const KGrid &K, int nz, const double *dG, double *out) {
  if (S.d < 1 || S.d > kLatticeMaxDim)
    fail(ED_ERR_UNSUPPORTED, "lattice sums: Green-function dimension " + std::to_string(S.d) + " outside 1.." +
                                 std::to_string(kLatticeMaxDim));
  if (S.nnbr > kLatticeMaxNbr) fail(ED_ERR_UNSUPPORTED, "lattice sums: more than 64 superlattice neighbors");
  if (K.dim < 0 || K.dim > 3) fail(ED_ERR_INVALID, "lattice sums: wavevector grid dimension outside 0..3");
  for (int a = 0; a < K.dim; ++a)
    if (K.nk[a] < 1) fail(ED_ERR_INVALID, "lattice sums: empty wavevector grid");
  if (nz <= 0) return;
  Arg A;
  A.d = S.d;
  A.nnbr = S.nnbr;
  A.dim = K.dim;
  A.nk0 = K.dim >= 1 ? K.nk[0] : 1;
  A.nk1 = K.dim >= 2 ? K.nk[1] : 1;
  A.nk2 = K.dim >= 3 ? K.nk[2] : 1;
  A.npos = S.npos;
  A.mask = S.mask;
  A.off = K.offset;
  A.nk = K.count();
  if (nz > 65535) fail(ED_ERR_INVALID, "lattice sums: more than 65535 frequencies per call");
  A.V0 = S.V0;
  A.val = S.val;
  A.R = S.R;
  A.eptr = S.eptr_d;
  A.epos = S.epos_d;
  A.plist = S.plist_d;
  const int width = MODE == 0 ? 1 : 2 * S.d * S.d;
  const bool reg = S.d <= kRegDim;
  // about kLatticeWaves waves; in the register kernel a wave takes up to 8
  // frequencies of the same 64 points first (V(k) is formed once for them),
  // then more points
  long nchunk;
  int zc = 1;
  if (reg) {
    const long nb = (A.nk + 63) / 64, per = std::max<long>(1, (nb * nz + kLatticeWaves - 1) / kLatticeWaves);
    zc = (int)std::min<long>(std::min<long>(per, 8), nz);
    A.kchunk = 64 * std::min(nb, std::max<long>(1, per / zc));
  } else {
    nchunk = std::max<long>(1, std::min<long>(A.nk, (kLatticeWaves + nz - 1) / nz));
    A.kchunk = (A.nk + nchunk - 1) / nchunk;
  }
  nchunk = (A.nk + A.kchunk - 1) / A.kchunk;
  DevBuf<double> part((size_t)nz * nchunk * width), dout((size_t)nz * width);
  if (reg) {
    const size_t lds = ((size_t)A.npos * 128 + (size_t)zc * width) * sizeof(double);
    switch (S.d) {
      case 1: launch_reg<MODE, 1>(A, nz, zc, nchunk, lds, dG, part.p); break;
      case 2: launch_reg<MODE, 2>(A, nz, zc, nchunk, lds, dG, part.p); break;
      case 3: launch_reg<MODE, 3>(A, nz, zc, nchunk, lds, dG, part.p); break;
      case 4: launch_reg<MODE, 4>(A, nz, zc, nchunk, lds, dG, part.p); break;
      case 5: launch_reg<MODE, 5>(A, nz, zc, nchunk, lds, dG, part.p); break;
      default: launch_reg<MODE, 6>(A, nz, zc, nchunk, lds, dG, part.p); break;
    }
  } else {
    hipLaunchKernelGGL((k_lattice<MODE>), dim3((unsigned)nchunk, (unsigned)nz), dim3(64), 0, stream(), A, dG, part.p);
  }
  ED_HIP(hipGetLastError());
  hipLaunchKernelGGL((k_lattice_fold<MODE>), dim3(nz), dim3(256), 0, stream(), S.d, (int)nchunk, 1.0 / (double)A.nk,
                     dG, part.p, dout.p);
  ED_HIP(hipGetLastError());
  dout.download(out, (size_t)nz * width);
}

}  // namespace

void lattice_logdet(const SuperlatticeDev &S, const KGrid &K, int nz, const double *dG, double *out) {
  run<0>(S, K, nz, dG, out);
}

void lattice_cpt_average(const SuperlatticeDev &S, const KGrid &K, int nz, const double *dG, double *out) {
  run<1>(S, K, nz, dG, out);
}

}  // namespace ed
