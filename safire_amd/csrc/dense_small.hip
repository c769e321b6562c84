// Batched small dense kernels: one wavefront per matrix.
//
//  * lu_inverse_logdet: Gauss-Jordan inversion with partial pivoting (pivot = first maximum of
//    |re| + |im|, the getrf choice), producing the inverse and log det of each n x n complex
//    matrix.  The pivots are exactly getrf's U diagonal, so the log det follows
//    log_determinant_from_getrf (determinants_impl.hpp:33-75): sum_i log(+-U_ii + DBL_MIN) with
//    the sign flipped on swapped rows, added to the running value, imaginary part wrapped into
//    [-pi, pi].  A singular matrix yields a zero inverse (getri_or_zero,
//    nda_functions.hpp:422-437).
//  * chol_upper_inverse: Cholesky S = R^H R (R upper, positive real diagonal) of a Hermitian
//    positive-definite Gram matrix and R^{-1}; the building block of the Cholesky-QR2
//    orthogonalization.
//
// n <= 64.  All LDS traffic of one workgroup is program-ordered, and explicit barriers separate
// the phases that read another lane's data.
#include "afq_internal.hpp"

namespace afq {

namespace {

constexpr double kPi = 3.14159265358979323846;

// log of a complex number (principal branch)
__device__ inline void clog(double re, double im, double& lr, double& li) {
  lr = log(hypot(re, im));
  li = atan2(im, re);
}

// lu_inverse_logdet: one wavefront per matrix, lane r holds row r in registers (n <= 64).
// Rows are never moved: each lane tracks the position its row would occupy in getrf's swapped
// order, the pivot of step j is the unused row of largest |re|+|im| in column j with ties going
// to the lowest position (getrf's first maximum), and the row at position j trades positions
// with it. Gauss-Jordan then eliminates column j from every other row with the pivot row read
// from the pivot lane's registers (readlane).  The columns move down by one register as they are
// updated, so column j is always the first, its result enters at the end and one loop body serves
// every step: code unrolled over the steps ran at the rate at which a cold instruction cache is
// filled.  Without the inverse, columns <= j are dead after step j and are not updated. The
// log det
// takes log(+-U_jj + DBL_MIN) with the sign flipped exactly on getrf's swapped steps; the
// in-place result Y gives A^{-1}[k][c] = Y[p_k][s_c] (p_k = pivot row of step k, s_c = step at
// which row c pivoted), applied while storing.
//
// Bound by the chain of its steps: most calls have no more matrices than the machine has SIMDs, so one
// wavefront's latency is the time.  A step's own chain (the largest of a column, the pivot's
// reciprocal) is started before the columns of the step before are updated: column j + 1 is
// updated first and its pivot picked while the other columns' independent products fill the
// gaps.  Inverse of 512 matrices of n = 24: 28 -> 19 us, 128 of n = 40: 48 -> 41 us, 256 of n = 10:
// 16.6 -> 11.7 us; the triangular inverse of 1024 of n = 40: 95 -> 61 us.  What is left is the issue
// of eight instructions a column and step.  The largest entry is found with DPP moves inside the rows of 16 lanes, which cost a few
// cycles each where a shuffle through LDS costs over a hundred.
__device__ inline double rdl(double v, int src) {
  int lo = __double2loint(v), hi = __double2hiint(v);
  lo = __builtin_amdgcn_readlane(lo, src);
  hi = __builtin_amdgcn_readlane(hi, src);
  return __hiloint2double(hi, lo);
}

// ovlp[b] = scale * wrap(ovlp[b] + (lr, li)) + add, the imaginary part wrapped into [-pi, pi]
__device__ inline void ov_update(z64* ovlp, long b, double lr, double li, double ov_scale,
                                 double ov_add_re, double ov_add_im) {
  z64 o = ovlp[b];
  double re = o.re + lr, im = o.im + li;
  if (im > kPi) {
    while (im > kPi) im -= 2 * kPi;
  } else if (im < -kPi) {
    while (im < -kPi) im += 2 * kPi;
  }
  ovlp[b] = {ov_scale * re + ov_add_re, ov_scale * im + ov_add_im};
}

// v of the lane that DPP control CTRL names (rows outside ROWS keep their own)
template <int CTRL, int ROWS = 0xF>
__device__ inline int dpp(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS = 0xF>
__device__ inline double dpp_max(double v) {
  const double o = __hiloint2double(dpp<CTRL, ROWS>(__double2hiint(v)),
                                    dpp<CTRL, ROWS>(__double2loint(v)));
  return fmax(v, o);
}
// The maximum (minimum) over lanes 0 .. L - 1 rounded up to whole rows of 16, in every lane.  DPP:
// lanes exchanged in pairs, quads, halves and whole rows, then lane 15 of row 0 (2) broadcast to
// row 1 (3) and lane 31 to rows 2 and 3.
template <int L>
__device__ inline double lanes_max(double v) {
  v = dpp_max<0xB1>(v);
  v = dpp_max<0x4E>(v);
  v = dpp_max<0x141>(v);
  if (L > 8) v = dpp_max<0x140>(v);
  if (L > 16) v = dpp_max<0x142, 0xA>(v);
  if (L > 32) v = dpp_max<0x143, 0xC>(v);
  return rdl(v, L > 32 ? 63 : L > 16 ? 31 : 0);
}
template <int L>
__device__ inline int lanes_min(int v) {
  v = min(v, dpp<0xB1>(v));
  v = min(v, dpp<0x4E>(v));
  v = min(v, dpp<0x141>(v));
  if (L > 8) v = min(v, dpp<0x140>(v));
  if (L > 16) v = min(v, dpp<0x142, 0xA>(v));
  if (L > 32) v = min(v, dpp<0x143, 0xC>(v));
  return __builtin_amdgcn_readlane(v, L > 32 ? 63 : L > 16 ? 31 : 0);
}

// keep_ldet != nullptr: the raw log det sum (before the update of ovlp) of matrix b is stored
// there.  reuse (INV only): keepT holds the matrix whose inverse (at Ainv) and raw log det (at
// keep_ldet) were kept; when matrix b matches it bit for bit (no NaN), the kept values are
// exact for it: ovlp is updated from keep_ldet and nothing else is written.  Otherwise keepT
// takes matrix b and the factors are recomputed into Ainv and keep_ldet.
// NOPIV: no pivoting, for upper triangular matrices only (the Cholesky factor's inverse): row j
// is zero left of column j at step j, so each column of the inverse is stored when its step ends.
// WV = 2 (INV only): two wavefronts hold the even and the odd columns; both pick every pivot, the
// column it is picked from passes through LDS.  WAVES: wavefronts that have to fit on a SIMD.
template <int NMAX, bool INV, bool NOPIV = false, int WV = 1, int WAVES = 1>
__global__ void __launch_bounds__(64 * WV, WAVES)
    k_lu_rows(const z64* __restrict__ A, long a_bs, int n, z64* __restrict__ Ainv, long i_bs,
              z64* __restrict__ ovlp, double ov_scale, double ov_add_re, double ov_add_im,
              z64* __restrict__ keepT, z64* __restrict__ keep_ldet, int reuse) {
  constexpr bool FULL = INV && !NOPIV;  // every column stays live
  constexpr int NC = NMAX / WV;         // columns of a wavefront
  static_assert(WV == 1 || FULL, "two wavefronts: the pivoted inverse only");
  __shared__ int pivrow[64];
  __shared__ double2 colj[WV == 2 ? 2 : 1][64];
  const int lane = threadIdx.x & 63;
  const int wv = WV == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long b = blockIdx.x;
  const z64* Ab = A + b * a_bs;
  double xr[NC], xi[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int m = c * WV + wv;
    z64 v = (lane < n && m < n) ? Ab[(long)lane * n + m] : z64{0.0, 0.0};
    xr[c] = v.re;
    xi[c] = v.im;
  }
  // (rows of 64 columns fill the register file: no kept factors there)
  if constexpr (INV && !NOPIV && NMAX <= 48) {
    if (reuse) {
      z64* Kb = keepT + b * a_bs;
      bool same = true;
      if (lane < n) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int m = c * WV + wv;
          const z64 k = m < n ? Kb[(long)lane * n + m] : z64{xr[c], xi[c]};
          same = same & (xr[c] == xr[c]) & (xi[c] == xi[c]) &
                 (__double_as_longlong(k.re) == __double_as_longlong(xr[c])) &
                 (__double_as_longlong(k.im) == __double_as_longlong(xi[c]));
        }
      }
      if (WV == 1 ? __ballot(!same) == 0 : __syncthreads_and(same) != 0) {  // uniform
        if (ovlp != nullptr && threadIdx.x == 0) {
          const z64 l = keep_ldet[b];
          ov_update(ovlp, b, l.re, l.im, ov_scale, ov_add_re, ov_add_im);
        }
        return;
      }
      if (lane < n) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int m = c * WV + wv;
          if (m < n) Kb[(long)lane * n + m] = z64{xr[c], xi[c]};
        }
      }
    }
  }
  bool used = lane >= n;
  int pos = lane;         // position of my row in getrf's order
  int mystep = n;         // step at which my row pivoted
  int step_row = -1;      // the row that pivoted in step `lane`
  double ur = 1.0, ui = 0.0;  // my pivot value with getrf's sign (+-U_jj)
  bool singular = false;
  // the pivot of the current step: its lane, its value, and what every row is updated with
  int p = 0;
  double dr = 0.0, di = 0.0, hr = 0.0, hi = 0.0, njr = 0.0, nji = 0.0;
  // picks the pivot of step j, given the rows' entries in column j (j = n: changes no row)
  auto pick = [&](int j, double fr, double fi) {
    int bpos = j;
    if constexpr (NOPIV) {
      p = j & 63;
    } else {
      // max |re|+|im| over unused rows, ties to the lowest position (a NaN entry ranks below every
      // number but above used rows, so the reduction stays well defined and uniform)
      const double mag = fabs(fr) + fabs(fi);
      const double best = used ? -1.0 : (mag == mag ? mag : -0.5);
      const double top = lanes_max<NMAX>(best);
      bpos = lanes_min<NMAX>(!used && best == top ? pos : 64);
      // the pivot row is the lane at position bpos; the row at position j moves to bpos's slot
      const unsigned long long owner = __ballot(!used && pos == bpos);
      p = __builtin_amdgcn_readfirstlane(owner ? __ffsll(owner) - 1 : 0);
    }
    const bool mine = lane == p && !used, swapped = bpos != j;
    pos = mine ? j : !used && pos == j ? bpos : pos;
    dr = rdl(fr, p);
    di = rdl(fi, p);
    ur = mine ? (swapped ? -dr : dr) : ur;
    ui = mine ? (swapped ? -di : di) : ui;
    mystep = mine ? j : mystep;
    used = used || mine;
    step_row = lane == j ? p : step_row;
    const double den = dr * dr + di * di;
    const double ir = dr / den, ii = -di / den;
    // h = g / d with g = d - 1 on the pivot row (which becomes the pivot row / d), f elsewhere
    const double gr = (lane == p) ? dr - 1.0 : fr, gi = (lane == p) ? di : fi;
    hr = gr * ir - gi * ii;
    hi = gr * ii + gi * ir;
    // column j of the result: 1/d on the pivot row, -f/d elsewhere
    njr = (lane == p) ? ir : -(fr * ir - fi * ii);
    nji = (lane == p) ? ii : -(fr * ii + fi * ir);
  };
  // x - h y as four fused multiply-adds, y the entry of lane q (scalar reads of the pivot lane's
  // registers: no LDS round trip)
  auto reduce = [&](double& vr, double& vi, int q, double gr, double gi) {
    const double yr = rdl(vr, q), yi = rdl(vi, q);
    const double nr = fma(gi, yi, fma(-gr, yr, vr));
    vi = fma(-gi, yr, fma(-gr, yi, vi));
    vr = nr;
  };
  z64* Ib = Ainv + b * i_bs;
  // column j, which its wavefront holds first
  auto column = [&](int j, double& fr, double& fi) {
    if constexpr (WV == 1) {
      fr = xr[0];
      fi = xi[0];
    } else {
      if (wv == (j & 1)) colj[j & 1][lane] = double2{xr[0], xi[0]};
      __syncthreads();
      const double2 f = colj[j & 1][lane];
      fr = f.x;
      fi = f.y;
    }
  };
  double fr, fi;
  column(0, fr, fi);
  pick(0, fr, fi);
  int j = 0;
#pragma unroll 1
  for (; j < n && (dr != 0.0 || di != 0.0); ++j) {
    const int q = p;
    const double gr = hr, gi = hi, cr = njr, ci = nji;
    // (the column is final: later pivot rows are zero there)
    if (NOPIV && lane < n) Ib[(long)lane * n + j] = {cr, ci};
    if constexpr (WV == 1) {
      // the next column and its pivot
      reduce(xr[1], xi[1], q, gr, gi);
      xr[0] = xr[1];
      xi[0] = xi[1];
      pick(j + 1, xr[0], xi[0]);
#pragma unroll
      for (int k = 0; k < NMAX; k += 8) {
        if (!FULL && k >= NMAX - 1 - j) break;  // uniform: nothing live from column k + 1 on
#pragma unroll
        for (int c = max(k, 1); c < k + 8; ++c) {
          if (c + 1 == NMAX) {
            xr[c] = cr;
            xi[c] = ci;
          } else {
            xr[c] = xr[c + 1];
            xi[c] = xi[c + 1];
            reduce(xr[c], xi[c], q, gr, gi);
          }
        }
      }
    } else {
      // the other wavefront sends the next column, meanwhile this one updates EARLY columns
      constexpr int EARLY = NC / 4;
      const bool own = wv == (j & 1);
      auto move_down = [&](int c0, int c1) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
          if (c >= c0 && c < c1) {
            xr[c] = c + 1 < NC ? xr[c + 1] : cr;
            xi[c] = c + 1 < NC ? xi[c + 1] : ci;
            if (c + 1 < NC) reduce(xr[c], xi[c], q, gr, gi);
          }
      };
      if (own) move_down(0, EARLY);
      else reduce(xr[0], xi[0], q, gr, gi);
      column(j + 1, fr, fi);
      if (own) {
        pick(j + 1, fr, fi);
        move_down(EARLY, NC);
      } else {
        pick(j + 1, fr, fi);
#pragma unroll
        for (int c = 1; c < NC; ++c) reduce(xr[c], xi[c], q, gr, gi);
      }
    }
  }
  // A zero pivot: its step is skipped and the inverse will be zero.  The log det still takes the
  // later pivots.
  singular = j < n;
#pragma unroll 1
  for (; j < n; ++j) {
    if (dr != 0.0 || di != 0.0) {
#pragma unroll
      for (int c = 0; c < NC; ++c) reduce(xr[c], xi[c], p, hr, hi);
    }
    if (wv == j % WV) {
#pragma unroll
      for (int c = 1; c < NC; ++c) {
        xr[c - 1] = xr[c];
        xi[c - 1] = xi[c];
      }
    }
    column(j + 1, fr, fi);
    pick(j + 1, fr, fi);
  }
  if (ovlp != nullptr || keep_ldet != nullptr) {
    double lr = 0.0, li = 0.0;
    if (lane < n) clog(ur + 2.2250738585072014e-308, ui, lr, li);
    lr = wave_sum(lr);
    li = wave_sum(li);
    if (threadIdx.x == 0) {
      if (keep_ldet != nullptr) keep_ldet[b] = {lr, li};
      if (ovlp != nullptr) ov_update(ovlp, b, lr, li, ov_scale, ov_add_re, ov_add_im);
    }
  }
  if constexpr (NOPIV) {
    if (singular && lane < n) {
#pragma unroll 1
      for (int c = 0; c < n; ++c) Ib[(long)lane * n + c] = {0.0, 0.0};
    }
  } else if constexpr (INV) {
    pivrow[lane] = step_row;
    __syncthreads();
    if (lane < n && mystep < n) {
      // (its steps have brought a wavefront's column k to NC - steps + k)
      const int first = NC - (n - wv + WV - 1) / WV;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int m = (c - first) * WV + wv;
        const int col = c >= first && m < n ? pivrow[m] : -1;
        if (col >= 0 && col < n)
          Ib[(long)mystep * n + col] = singular ? z64{0.0, 0.0} : z64{xr[c], xi[c]};
      }
    }
  }
}

constexpr int kLuThreads = 256;
// Workgroup Cholesky: S = R^H R with R upper triangular (positive real diagonal), written to R
// with zeros below the diagonal.
__global__ void __launch_bounds__(kLuThreads)
    k_chol_blk(const z64* __restrict__ S, int n, z64* __restrict__ R) {
  extern __shared__ double2 sm2[];
  const int ld = n + 1;
  double2* a = sm2;
  const int tid = threadIdx.x;
  const long b = blockIdx.x;
  const z64* Sb = S + b * (long)n * n;
  for (int e = tid; e < n * n; e += kLuThreads) {
    z64 v = Sb[e];
    a[(e / n) * ld + e % n] = make_double2(v.re, v.im);
  }
  __syncthreads();
  for (int j = 0; j < n; ++j) {
    const double d = sqrt(a[j * ld + j].x);
    __syncthreads();
    for (int c = tid; c < n; c += kLuThreads) {
      if (c == j) {
        a[j * ld + c] = make_double2(d, 0.0);
      } else if (c > j) {
        double2 x = a[j * ld + c];
        a[j * ld + c] = make_double2(x.x / d, x.y / d);
      }
    }
    __syncthreads();
    // A[i][c] -= conj(R[j][i]) R[j][c] for j < i <= c
    const int m = n - j - 1;
    for (int e = tid; e < m * m; e += kLuThreads) {
      const int i = j + 1 + e / m, c = j + 1 + e % m;
      if (c < i) continue;
      const double2 ri = a[j * ld + i], rc = a[j * ld + c];
      double2 x = a[i * ld + c];
      x.x -= ri.x * rc.x + ri.y * rc.y;
      x.y -= ri.x * rc.y - ri.y * rc.x;
      a[i * ld + c] = x;
    }
    __syncthreads();
  }
  z64* Rb = R + b * (long)n * n;
  for (int e = tid; e < n * n; e += kLuThreads) {
    const int r = e / n, c = e % n;
    double2 v = a[r * ld + c];
    Rb[e] = (c >= r) ? z64{v.x, v.y} : z64{0.0, 0.0};
  }
}

// Cholesky of a Hermitian positive-definite S (upper R, S = R^H R) and the inverse of R.
// Rinv is written as a full n x n matrix (zeros below the diagonal). ldet += sum_i log R_ii.
__global__ void __launch_bounds__(64)
    k_chol_upper_inverse(const z64* __restrict__ S, int n, z64* __restrict__ Rinv,
                         z64* __restrict__ ldet) {
  extern __shared__ double smem[];
  const int ld = n + 1;
  double* a = smem;  // [n][ld] complex
  const int lane = threadIdx.x;
  const long b = blockIdx.x;
  const z64* Sb = S + b * (long)n * n;
  for (int e = lane; e < n * n; e += 64) {
    int r = e / n, c = e % n;
    z64 v = Sb[e];
    a[2 * (r * ld + c)] = v.re;
    a[2 * (r * ld + c) + 1] = v.im;
  }
  __syncthreads();
  double lsum = 0.0;
  // right-looking upper Cholesky: row j of R
  for (int j = 0; j < n; ++j) {
    double d = sqrt(a[2 * (j * ld + j)]);
    lsum += log(d);
    __syncthreads();
    for (int c = lane; c < n; c += 64) {
      if (c == j) {
        a[2 * (j * ld + c)] = d;
        a[2 * (j * ld + c) + 1] = 0.0;
      } else if (c > j) {
        a[2 * (j * ld + c)] /= d;
        a[2 * (j * ld + c) + 1] /= d;
      }
    }
    __syncthreads();
    // trailing update: A[i][c] -= conj(R[j][i]) R[j][c] for j < i <= c
    for (int c = lane; c < n; c += 64) {
      if (c <= j) continue;
      double rcr = a[2 * (j * ld + c)], rci = a[2 * (j * ld + c) + 1];
      for (int i = j + 1; i <= c; ++i) {
        double rir = a[2 * (j * ld + i)], rii = -a[2 * (j * ld + i) + 1];  // conj(R[j][i])
        a[2 * (i * ld + c)] -= rir * rcr - rii * rci;
        a[2 * (i * ld + c) + 1] -= rir * rci + rii * rcr;
      }
    }
    __syncthreads();
  }
  // inverse of the upper triangle, lane = column c: X[c][c] = 1/R[c][c];
  // X[i][c] = -(sum_{k=i+1..c} R[i][k] X[k][c]) / R[i][i]
  // (each lane writes and re-reads only its own column of Rinv in global memory)
  z64* Rb = Rinv + b * (long)n * n;
  for (int c = lane; c < n; c += 64) {
    for (int i = c + 1; i < n; ++i) Rb[(long)i * n + c] = {0.0, 0.0};
    Rb[(long)c * n + c] = {1.0 / a[2 * (c * ld + c)], 0.0};
    for (int i = c - 1; i >= 0; --i) {
      double sr = 0.0, si = 0.0;
      for (int k = i + 1; k <= c; ++k) {
        double rr = a[2 * (i * ld + k)], ri = a[2 * (i * ld + k) + 1];
        z64 x = Rb[(long)k * n + c];
        sr += rr * x.re - ri * x.im;
        si += rr * x.im + ri * x.re;
      }
      double rd = a[2 * (i * ld + i)];
      Rb[(long)i * n + c] = {-sr / rd, -si / rd};
    }
  }
  if (lane == 0 && ldet != nullptr) {
    z64 o = ldet[b];
    ldet[b] = {o.re + lsum, o.im};
  }
}

}  // namespace

void lu_inverse_logdet(hipStream_t s, const z64* A, long a_bs, int nb, int n, z64* Ainv,
                       long i_bs, z64* ovlp, double ov_scale, z64 ov_add, bool want_inverse,
                       const LuKeep* keep, bool reuse) {
  AFQ_CHECK(n >= 1 && n <= 64, kErrShape, "n must be in [1, 64]");
  AFQ_CHECK(!keep || (want_inverse && n <= 48 && Ainv == keep->Tinv && a_bs == (long)n * n &&
                      i_bs == (long)n * n && (reuse || A == keep->T)),
            kErrArg, "kept factors: n <= 48, the inverse in the kept buffer, [nb][n][n] layouts");
  if (nb <= 0) return;
  z64* kT = keep && reuse ? keep->T : nullptr;
  z64* kl = keep ? keep->ldet : nullptr;
  const int ru = keep && reuse ? 1 : 0;
#define AFQ_LU(NM, INV, WV, WAVES)                                                               \
  hipLaunchKernelGGL((k_lu_rows<NM, INV, false, WV, WAVES>), dim3(nb), dim3(64 * WV), 0, s, A,   \
                     a_bs, n, Ainv, i_bs, ovlp, ov_scale, ov_add.re, ov_add.im, kT, kl, ru)
#define AFQ_LU_ROWS(NM)                \
  do {                                 \
    if (want_inverse) AFQ_LU(NM, true, 1, 1); \
    else AFQ_LU(NM, false, 1, 1);      \
  } while (0)
  if (n <= 8)
    AFQ_LU_ROWS(8);
  else if (n <= 16)
    AFQ_LU_ROWS(16);
  else if (n <= 24)
    AFQ_LU_ROWS(24);
  else if (n <= 32)
    AFQ_LU_ROWS(32);
  else if (n <= 40)
    AFQ_LU_ROWS(40);
  else if (n <= 48)
    AFQ_LU_ROWS(48);
  else if (!want_inverse)
    AFQ_LU(64, false, 1, 1);
  // One wavefront cannot hold rows of 64 and the next step's pivot beside them (the density matrix
  // of 300 walkers, n = 50 and 64: 216 and 269 us, two wavefronts 137 and 172).  Where the matrices
  // outnumber what 256 registers a lane let run at once, two workgroups on a SIMD pay for the
  // spills (3000 walkers, n = 64: 1104 against 1076 us).  Up to 48 columns two wavefronts are
  // slower, the pivot's chain being the same (n = 32: 68 against 78 us).
  else if (nb <= 768)
    AFQ_LU(64, true, 2, 1);
  else
    AFQ_LU(64, true, 2, 2);
#undef AFQ_LU_ROWS
#undef AFQ_LU
  AFQ_LAUNCH_CHECK();
}

void chol_upper_inverse(hipStream_t s, const z64* S, int nb, int n, z64* Rinv, z64* ldet) {
  AFQ_CHECK(n >= 1 && n <= 64, kErrShape, "n must be in [1, 64]");
  if (nb <= 0) return;
  size_t lds = sizeof(double2) * ((size_t)n * (n + 1) + n);
  AFQ_CHECK(lds <= 160 * 1024, kErrShape, "matrix too large for one workgroup's LDS");
  if (lds > 65536)  // n = 64
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k_chol_blk),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  // R is written into Rinv, then inverted in place (upper triangular: no pivoting needed);
  // the inversion's log det is sum_i log R_ii (R_ii real and positive).
  hipLaunchKernelGGL(k_chol_blk, dim3(nb), dim3(kLuThreads), lds, s, S, n, Rinv);
  AFQ_LAUNCH_CHECK();
  const long nn = (long)n * n;
  if (n <= 8)
    hipLaunchKernelGGL((k_lu_rows<8, true, true>), dim3(nb), dim3(64), 0, s, Rinv, nn, n, Rinv, nn,
                       ldet, 1.0, 0.0, 0.0, nullptr, nullptr, 0);
  else if (n <= 16)
    hipLaunchKernelGGL((k_lu_rows<16, true, true>), dim3(nb), dim3(64), 0, s, Rinv, nn, n, Rinv, nn,
                       ldet, 1.0, 0.0, 0.0, nullptr, nullptr, 0);
  else if (n <= 24)
    hipLaunchKernelGGL((k_lu_rows<24, true, true>), dim3(nb), dim3(64), 0, s, Rinv, nn, n, Rinv, nn,
                       ldet, 1.0, 0.0, 0.0, nullptr, nullptr, 0);
  else if (n <= 32)
    hipLaunchKernelGGL((k_lu_rows<32, true, true>), dim3(nb), dim3(64), 0, s, Rinv, nn, n, Rinv, nn,
                       ldet, 1.0, 0.0, 0.0, nullptr, nullptr, 0);
  else if (n <= 40)
    hipLaunchKernelGGL((k_lu_rows<40, true, true>), dim3(nb), dim3(64), 0, s, Rinv, nn, n, Rinv, nn,
                       ldet, 1.0, 0.0, 0.0, nullptr, nullptr, 0);
  else if (n <= 48)
    hipLaunchKernelGGL((k_lu_rows<48, true, true>), dim3(nb), dim3(64), 0, s, Rinv, nn, n, Rinv, nn,
                       ldet, 1.0, 0.0, 0.0, nullptr, nullptr, 0);
  else
    hipLaunchKernelGGL((k_lu_rows<64, true, true>), dim3(nb), dim3(64), 0, s, Rinv, nn, n, Rinv, nn,
                       ldet, 1.0, 0.0, 0.0, nullptr, nullptr, 0);
  AFQ_LAUNCH_CHECK();
}

}  // namespace afq
