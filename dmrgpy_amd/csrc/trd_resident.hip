// Householder tridiagonalisation with the matrix held in registers: one
// launch reduces a symmetric (or Hermitian) matrix of order m to tridiagonal
// form, unblocked (LAPACK dsytd2 / zhetd2, lower), with one exchange between
// the workgroups per column.
//
// The launch-per-column reduction (sytrd.hip) is bound by latency -- two
// dependent launches and their memory round trips per column, 9 ... 13 us --
// and, from order ~2000 on, by streaming the trailing matrix.  Here each of G
// workgroups keeps RW consecutive rows of the matrix in registers (the
// chip's register files hold 128 MB; order 2588 takes 54), so a column costs
// no memory traffic but the exchange of two vectors, and the rank-2 update
// (free of memory traffic too) needs no panel.  Per column J, every
// workgroup redundantly holds the column a = A[:, J] spread over its threads:
//
//   x = a[J+2:];  A x and |x|^2 for its own rows;  publish A x;
//   tau, beta, scale from |x|, v = e_{J+1} + scale x, and the previous column's
//   A -= v w^T + w v^T on its own rows, while the exchange is under way;
//   read all of A x and row J+1 of A (published by its owner): q = A v;
//   w = tau q - (tau^2 (q.v) / 2) v;   next column  A[:, J+1] - v w_1 - w.
//
// A x is taken with the matrix before the previous column's update and
// corrected by v (w.x) + w (v.x), as in the blocked reduction's panels, so
// that neither the update nor the reflector's divisions sit between one
// exchange and the next.
//
// Exchange: every published word goes to its own address in a buffer that a
// preceding kernel filled with one NaN pattern; readers poll each word
// (relaxed device-scope atomics) until it differs.  A word carries its own
// validity, so no fence, flag or cache write-back is needed.  Measured with
// 16 / 32 / 64 / 128 / 256 workgroups exchanging 760 words: 1.6 / 2.1 / 2.5 /
// 3.0 / 3.2 us.  All waits are bounded: a workgroup that waits longer than
// the context's limit (other work holding the CUs its peers need) gives up, as
// then do the others (at once where they had not started), the input is
// untouched and the caller runs the launch-per-column reduction instead.  Where
// the other work stays, every attempt would cost a wait, so after a failure the
// context passes over the next reductions (1, 2, 4 ... 64, until one succeeds):
// a wasted wait of 50 ms is as long as 5000 columns by panels.
//
// Measured per column, launch-per-column / resident (us): real order 128
// 8.7 / 2.45, 380 9.8 / 2.6, 2588 (930 columns reduced) 16.2 / 5.9; complex
// order 1200 14.5 / 5.6 (with the update and the reflector before the
// publication: 2.8, 2.9, 6.3, 5.7).  What bounds a column is the exchange,
// then the chain of two workgroup-wide reductions.
#include "dmrg_internal.h"
#include "wave_reduce.h"

#include <algorithm>
#include <cstring>

namespace dmrg {

constexpr unsigned long long RES_EMPTY = ~0ull;                  // a NaN no arithmetic produces; see publish()
constexpr unsigned long long RES_NAN = 0x7FF8000000000000ull;
constexpr int RES_CHECK = 32, RES_CHECK_MIN = 64;                 // early-stop checks: every 32 columns from 64 on

struct ResArgs {
  const double* A;             // m x m, row pitch lda, imaginary plane at +pA
  long long lda, pA;
  int m, mp;                   // order, order padded to a multiple of 16
  int col0, n;                 // absolute column of the first one, order of the whole matrix
  unsigned long long* X;       // exchange: per column [2 (row, q)][planes][mp]
  unsigned long long* chk;     // per early-stop check [2][gridDim.x]
  double* R;                   // reflectors: row J, columns J+2 ... (m x m, planes m*m apart)
  double *d, *e, *tau;         // at col0 (tau interleaved when complex)
  int early;
  double tol2, total2;         // stop once |trailing|_F^2 <= tol2 * total2 (total2 < 0: of this matrix)
  long long limit;             // longest wait, wall-clock ticks; 0: none, the first unmet word gives up
  int* status;                 // [0] 1 = gave up, [1] columns reduced
  double* trace;               // trace of the block left when stopped early
};

__device__ __forceinline__ void publish(unsigned long long* p, double x) {
  unsigned long long u = (unsigned long long)__double_as_longlong(x);
  if (u == RES_EMPTY) u = RES_NAN;
  __hip_atomic_store(p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long peek(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One wait for words published by other workgroups: over() after each look
// that missed some, true once the limit has passed (ANY: the argument's, else
// the default one; see either_launch)
constexpr long long RES_DEFAULT = 5000000;   // wall-clock ticks (100 MHz): 50 ms, as Ctx::trd_wait
template <bool ANY>
struct Patience {
  int spin = 0;
  long long t0 = 0;
  __device__ __forceinline__ bool over(const ResArgs& g) {
    if (ANY && g.limit == 0) return true;
    if ((++spin & 63) != 0) return false;
    const long long t = wall_clock64();
    if (t0 == 0) t0 = t;
    return t - t0 > (ANY ? g.limit : RES_DEFAULT);
  }
};
__device__ __forceinline__ void give_up(const ResArgs& g) {
  __hip_atomic_store(g.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// T threads, thread t holds columns t, t + T, ... (CC of them) of RW rows.
template <bool CX, int T, int CC, int RW, bool ANY>
__global__ __launch_bounds__(T) void trd_resident_k(ResArgs g) {
  constexpr int NP = CX ? 2 : 1, NW = T / 64, NS = NP * RW;
  // 16 sums per column: A x of the own rows, |x|^2 at NS and, real, w.x and v.x
  // of the previous column after it (complex: four more, reduced apart)
  static_assert(CX ? NS <= 15 : NS <= 13, "reduction holds 16 values");
  __shared__ double red[NW * 16], red2[NW * 4], red4[NW * 4];
  __shared__ double sa[2][NP][16], sq[NP][16];
  __shared__ double2 svw[NW][NP][16];   // (v, w) of the own rows, one copy per wave
  __shared__ double s_a0[NP], s_d;
  __shared__ int s_bad;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wg = blockIdx.x, G = gridDim.x, m = g.m, mp = g.mp;
  const int row0 = wg * RW, last = min(row0 + RW, m) - 1;
  const bool writer = wg == G - 1;
  // an attempt already given up before this workgroup found a place: leave at
  // once, or workgroups that run one after the other would each wait a limit
  if (tid == 0) s_bad = __hip_atomic_load(g.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (s_bad) return;

  // own rows (conj(buffer) when complex: the reduction works on the column-major view)
  double M[NP][RW][CC], a[NP][CC], v[NP][CC], w[NP][CC];
#pragma unroll
  for (int k = 0; k < CC; ++k) {
    const int c = tid + T * k;
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const bool ok = c < m && row0 + i < m;
      const long long o = (long long)(row0 + i) * g.lda + c;
      M[0][i][k] = ok ? g.A[o] : 0.0;
      if (CX) M[NP - 1][i][k] = ok ? -g.A[o + g.pA] : 0.0;
    }
    a[0][k] = c < m ? g.A[c] : 0.0;
    if (CX) a[NP - 1][k] = c < m ? g.A[c + g.pA] : 0.0;
#pragma unroll
    for (int p = 0; p < NP; ++p) v[p][k] = w[p][k] = 0.0;
  }
  double total2 = g.total2;
  bool passed = false;   // the last early-stop check
  double tr = 0.0, ti = 0.0, Kr = 0.0, Ki = 0.0, scr = 0.0, sci = 0.0;   // tau, w = tau q + K v, v = scale a

  // On entry to column J: a = column J; v, w = column J-1's, not yet applied to M.
  for (int J = 0;; ++J) {
    const int par = J & 1;
    unsigned long long* Xc = g.X + (long long)J * (2 * NP * mp);
    unsigned long long* Xq = Xc + NP * mp;
    // ---- v and w of the own rows (column J-1; rows from J on), lane i for row i
    double ovr = 0.0, ovi = 0.0, owr = 0.0, owi = 0.0;
    if (J > 0 && lane < RW) {
      const int r = row0 + lane;
      if (r >= J && r < m) {
        const double ar = sa[par ^ 1][0][lane], ai = CX ? sa[par ^ 1][NP - 1][lane] : 0.0;
        ovr = r == J ? 1.0 : scr * ar - sci * ai;
        ovi = r == J ? 0.0 : scr * ai + sci * ar;
        const double qr = sq[0][lane], qi = CX ? sq[NP - 1][lane] : 0.0;
        owr = tr * qr - ti * qi + Kr * ovr - Ki * ovi;
        owi = tr * qi + ti * qr + Kr * ovi + Ki * ovr;
      }
    }
    if (lane < RW) {
      svw[wave][0][lane] = double2{ovr, owr};
      if (CX) svw[wave][NP - 1][lane] = double2{ovi, owi};
    }
    // ---- row J+1 for everybody (with column J-1 applied)
    const int i1 = J + 1 - row0;
    if (i1 >= 0 && i1 < RW && J + 1 < m) {
      const double pvr = lane_value(ovr, i1), pwr = lane_value(owr, i1);
      const double pvi = CX ? lane_value(ovi, i1) : 0.0, pwi = CX ? lane_value(owi, i1) : 0.0;
#pragma unroll
      for (int i = 0; i < RW; ++i)
        if (i == i1) {
#pragma unroll
          for (int k = 0; k < CC; ++k) {
            const int c = tid + T * k;
            if (c > J && c < m) {
              if (!CX) {
                publish(Xc + c, M[0][i][k] - (pvr * w[0][k] + pwr * v[0][k]));
              } else {
                const double wr = w[0][k], wi = w[NP - 1][k], vr = v[0][k], vi = v[NP - 1][k];
                publish(Xc + c, M[0][i][k] - (pvr * wr + pvi * wi + pwr * vr + pwi * vi));
                publish(Xc + mp + c, M[NP - 1][i][k] - (pvi * wr - pvr * wi + pwi * vr - pwr * vi));
              }
            }
          }
        }
    }
    // ---- A x of the own rows, x = a[J+2:], with the A before column J-1:
    // column J-1's update is taken off the sums below and applied to M later,
    // while the exchange is under way
    double acc[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) acc[t] = 0.0;
    double wxr = 0.0, wxi = 0.0, vxr = 0.0, vxi = 0.0;   // w^H x, v^H x
#pragma unroll
    for (int k = 0; k < CC; ++k) {
      const int c = tid + T * k;
      if (c == J) s_d = a[0][k];
      if (c == J + 1) {
#pragma unroll
        for (int p = 0; p < NP; ++p) s_a0[p] = a[p][k];
      }
      if (c >= row0 && c < row0 + RW) {
#pragma unroll
        for (int p = 0; p < NP; ++p) sa[par][p][c - row0] = a[p][k];
      }
#pragma unroll
      for (int p = 0; p < NP; ++p) {   // from here on only a[J+2:] is wanted
        a[p][k] = c >= J + 2 ? a[p][k] : 0.0;
        acc[NS] += a[p][k] * a[p][k];
        wxr += w[p][k] * a[p][k];
        vxr += v[p][k] * a[p][k];
      }
      if (CX) {
        wxi += w[0][k] * a[NP - 1][k] - w[NP - 1][k] * a[0][k];
        vxi += v[0][k] * a[NP - 1][k] - v[NP - 1][k] * a[0][k];
      }
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        if (!CX) {
          acc[i] += M[0][i][k] * a[0][k];
        } else {
          acc[i] += M[0][i][k] * a[0][k] - M[NP - 1][i][k] * a[NP - 1][k];
          acc[RW + i] += M[0][i][k] * a[NP - 1][k] + M[NP - 1][i][k] * a[0][k];
        }
      }
    }
    if (!CX) {
      acc[14] = wxr;
      acc[15] = vxr;
    } else {
      wave_sums4(wxr, wxi, vxr, vxi);
      if (lane < 4) red4[wave * 4 + lane] = lane == 0 ? wxr : (lane == 1 ? wxi : (lane == 2 ? vxr : vxi));
    }
    {
      const double s = wave_sums16(acc, lane);
      if ((lane & 3) == 0) red[wave * 16 + sum_index(lane)] = s;
    }
    __syncthreads();
    double tot = 0.0;
    if (lane < 16) {
#pragma unroll
      for (int u = 0; u < NW; ++u) tot += red[u * 16 + lane];
    }
    if (wave == 0) {   // publish A x; q = A v = (row J+1) + scale (A x) is formed by the readers
      double yr = tot, yi = CX ? __shfl(tot, (RW + lane) & 63) : 0.0;
      if (!CX) {
        yr -= ovr * lane_value(tot, 14) + owr * lane_value(tot, 15);
      } else {
        double t4 = 0.0;
        if (lane < 4) {
#pragma unroll
          for (int u = 0; u < NW; ++u) t4 += red4[u * 4 + lane];
        }
        const double xr = lane_value(t4, 0), xi = lane_value(t4, 1), zr = lane_value(t4, 2), zi = lane_value(t4, 3);
        yr -= ovr * xr - ovi * xi + owr * zr - owi * zi;
        yi -= ovr * xi + ovi * xr + owr * zi + owi * zr;
      }
      const int r = row0 + lane;
      if (lane < RW && r > J && r < m) {
        publish(Xq + r, yr);
        if (CX) publish(Xq + mp + r, yi);
      }
    }
    // ---- column J-1's rank-2 update
    if (J > 0) {
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const double2 pr = svw[wave][0][i];
        const double2 pi = CX ? svw[wave][NP - 1][i] : double2{0.0, 0.0};
#pragma unroll
        for (int k = 0; k < CC; ++k) {
          if (!CX) {
            M[0][i][k] -= pr.x * w[0][k] + pr.y * v[0][k];
          } else {   // B -= v conj(w) + w conj(v)
            const double wr = w[0][k], wi = w[NP - 1][k], vr = v[0][k], vi = v[NP - 1][k];
            M[0][i][k] -= pr.x * wr + pi.x * wi + pr.y * vr + pi.y * vi;
            M[NP - 1][i][k] -= pi.x * wr - pr.x * wi + pi.y * vr - pr.y * vi;
          }
        }
      }
    }
    // ---- early stop: |A[J:, J:]|_F^2 against the whole matrix's
    const int s_abs = g.col0 + J;
    const bool first = J == 0 && g.early && total2 < 0.0;
    if (first || (g.early && J > 0 && s_abs >= RES_CHECK_MIN && s_abs % RES_CHECK == 0 && s_abs < g.n - 1)) {
      double q2 = 0.0, dg = 0.0;
#pragma unroll
      for (int i = 0; i < RW; ++i)
#pragma unroll
        for (int k = 0; k < CC; ++k) {
          const int c = tid + T * k, r = row0 + i;
          if (r >= J && c >= J) {   // zero past the order
#pragma unroll
            for (int p = 0; p < NP; ++p) q2 += M[p][i][k] * M[p][i][k];
            if (r == c) dg += M[0][i][k];
          }
        }
      const double s = wave_sums2(q2, dg);
      if (lane == 0) red2[wave * 2] = s;
      if (lane == 32) red2[wave * 2 + 1] = s;
      __syncthreads();
      unsigned long long* ck = g.chk + (long long)(s_abs / RES_CHECK) * 2 * G;
      if (tid < 2) {
        double t = 0.0;
#pragma unroll
        for (int u = 0; u < NW; ++u) t += red2[u * 2 + tid];
        publish(ck + tid * G + wg, t);
      }
      __syncthreads();
      double f2 = 0.0, tc = 0.0;
      for (int o = J / RW + tid; o < G; o += T) {   // the workgroups that hold rows from J on
        unsigned long long y0, y1;
        Patience<ANY> wait;
        for (;;) {
          y0 = peek(ck + o);
          y1 = peek(ck + G + o);
          if (y0 != RES_EMPTY && y1 != RES_EMPTY) break;
          if (wait.over(g)) {
            s_bad = 1;
            break;
          }
        }
        f2 += as_d(y0);
        tc += as_d(y1);
      }
      const double ss = wave_sums2(f2, tc);
      if (lane == 0) red2[wave * 2] = ss;
      if (lane == 32) red2[wave * 2 + 1] = ss;
      __syncthreads();
      f2 = tc = 0.0;
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        f2 += red2[u * 2];
        tc += red2[u * 2 + 1];
      }
      const bool bad = s_bad != 0;
      __syncthreads();
      if (bad) {
        if (tid == 0) give_up(g);
        return;
      }
      if (first) {
        total2 = f2;
      } else if (passed) {   // one check after the first to pass, as the panel path stops
        if (writer && tid == 0) {
          g.status[1] = J;
          g.trace[0] = tc;
        }
        return;
      } else {
        passed = f2 <= g.tol2 * total2;
      }
    }
    // ---- reflector of column J (every workgroup, the same sums in the same order;
    // |x|^2 is the plain sum of squares, as in the panels)
    const double xn2 = lane_value(tot, NS);
    const double a0r = s_a0[0], a0i = CX ? s_a0[NP - 1] : 0.0;
    double beta;
    if (!CX) {
      tr = 0.0;
      beta = a0r;
      scr = 0.0;
      if (xn2 != 0.0) {
        const double h2 = a0r * a0r + xn2;
        beta = -copysign(h2 > 1e-280 && h2 < 1e280 ? sqrt(h2) : hypot(a0r, sqrt(xn2)), a0r);
        tr = (beta - a0r) / beta;
        scr = 1.0 / (a0r - beta);
      }
    } else {
      // an exactly zero sub-column with a real a0 takes the reflection
      // tau = 2, v = e_{J+1}, as in the launch-per-column reduction
      tr = 2.0;
      ti = 0.0;
      beta = -a0r;
      scr = sci = 0.0;
      if (xn2 != 0.0 || a0i != 0.0) {
        const double h2 = a0r * a0r + a0i * a0i + xn2;
        beta = -copysign(h2 > 1e-280 && h2 < 1e280 ? sqrt(h2) : hypot(hypot(a0r, a0i), sqrt(xn2)), a0r);
        tr = (beta - a0r) / beta;
        ti = -a0i / beta;
        const double dr = a0r - beta, di = a0i, den = dr * dr + di * di;
        scr = dr / den;
        sci = -di / den;
      }
    }
    double* Rj = g.R + (long long)J * m;
#pragma unroll
    for (int k = 0; k < CC; ++k) {
      const int c = tid + T * k;
      const double ar = a[0][k], ai = CX ? a[NP - 1][k] : 0.0;   // zero up to J+1 and past the order
      v[0][k] = c == J + 1 ? 1.0 : scr * ar - sci * ai;
      if (CX) v[NP - 1][k] = scr * ai + sci * ar;
      if (writer && c >= J + 2 && c < m) {
#pragma unroll
        for (int p = 0; p < NP; ++p) Rj[(long long)p * m * m + c] = v[p][k];
      }
    }
    if (writer && tid == 0) {
      g.d[J] = s_d;
      g.e[J] = beta;
      if (CX) {
        g.tau[2 * J] = tr;
        g.tau[2 * J + 1] = ti;
      } else {
        g.tau[J] = tr;
      }
    }
    // ---- everybody's A x, and row J+1, loaded together (the row was published
    // well before and is looked at last: one round trip for both)
    double cv[NP][CC], qv[NP][CC], q1[NP], c1[NP];
    {
      int idx[CC];
#pragma unroll
      for (int k = 0; k < CC; ++k) {
        const int c = tid + T * k;
        idx[k] = c > J && c < m ? c : J + 1;
      }
      unsigned long long uc[NP][CC], uq[NP][CC], u1[NP], e1[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        e1[p] = peek(Xc + p * mp + J + 1);
#pragma unroll
        for (int k = 0; k < CC; ++k) uc[p][k] = peek(Xc + p * mp + idx[k]);
      }
      Patience<ANY> wait;
      bool ok = true, miss;
      do {
        miss = false;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          u1[p] = peek(Xq + p * mp + J + 1);
#pragma unroll
          for (int k = 0; k < CC; ++k) uq[p][k] = peek(Xq + p * mp + idx[k]);
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          miss |= u1[p] == RES_EMPTY;
#pragma unroll
          for (int k = 0; k < CC; ++k) miss |= uq[p][k] == RES_EMPTY;
        }
        if (miss && wait.over(g)) ok = false;
      } while (miss && ok);
      do {
        miss = false;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          if (e1[p] == RES_EMPTY) {
            miss = true;
            e1[p] = peek(Xc + p * mp + J + 1);
          }
#pragma unroll
          for (int k = 0; k < CC; ++k)
            if (uc[p][k] == RES_EMPTY) {
              miss = true;
              uc[p][k] = peek(Xc + p * mp + idx[k]);
            }
        }
        if (miss && wait.over(g)) ok = false;
      } while (miss && ok);
      if (!ok) s_bad = 1;
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const double sg = p ? -1.0 : 1.0;   // column J+1 is the conjugate of row J+1
        q1[p] = as_d(u1[p]);
        c1[p] = sg * as_d(e1[p]);
#pragma unroll
        for (int k = 0; k < CC; ++k) {
          qv[p][k] = as_d(uq[p][k]);
          cv[p][k] = sg * as_d(uc[p][k]);
        }
      }
    }
    // q = A v = A e_{J+1} + scale A x;  q^H v (v is zero up to J and past the order)
    double sr = 0.0, si = 0.0;
#pragma unroll
    for (int k = 0; k < CC; ++k) {
      const double yr = qv[0][k], yi = CX ? qv[NP - 1][k] : 0.0;
      qv[0][k] = cv[0][k] + scr * yr - sci * yi;
      sr += qv[0][k] * v[0][k];
      if (CX) {
        qv[NP - 1][k] = cv[NP - 1][k] + scr * yi + sci * yr;
        sr += qv[NP - 1][k] * v[NP - 1][k];
        si += qv[0][k] * v[NP - 1][k] - qv[NP - 1][k] * v[0][k];
      }
      const int c = tid + T * k;
      if (c >= row0 && c < row0 + RW) {
#pragma unroll
        for (int p = 0; p < NP; ++p) sq[p][c - row0] = qv[p][k];
      }
    }
    {
      const double s = wave_sums2(sr, si);
      if (lane == 0) red2[wave * 2] = s;
      if (lane == 32) red2[wave * 2 + 1] = s;
    }
    __syncthreads();
    if (s_bad) {
      if (tid == 0) give_up(g);
      return;
    }
    sr = si = 0.0;
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      sr += red2[u * 2];
      if (CX) si += red2[u * 2 + 1];
    }
    // K = -(tau / 2) (w0^H v) with w0 = tau q:  w0^H v = conj(tau) q^H v
    const double zr = tr * sr + ti * si, zi = tr * si - ti * sr;
    Kr = -0.5 * (tr * zr - ti * zi);
    Ki = -0.5 * (tr * zi + ti * zr);
    const double y1r = q1[0], y1i = CX ? q1[NP - 1] : 0.0;
    const double q1r = c1[0] + scr * y1r - sci * y1i, q1i = CX ? c1[NP - 1] + scr * y1i + sci * y1r : 0.0;
    const double w1r = tr * q1r - ti * q1i + Kr, w1i = tr * q1i + ti * q1r + Ki;
#pragma unroll
    for (int k = 0; k < CC; ++k) {
      const int c = tid + T * k;
      const bool in = c > J && c < m;
      const double vr = v[0][k], vi = CX ? v[NP - 1][k] : 0.0;
      const double qr = qv[0][k], qi = CX ? qv[NP - 1][k] : 0.0;
      w[0][k] = in ? tr * qr - ti * qi + Kr * vr - Ki * vi : 0.0;
      if (CX) w[NP - 1][k] = in ? tr * qi + ti * qr + Kr * vi + Ki * vr : 0.0;
      // column J+1 - v conj(w_1) - w
      a[0][k] = in ? cv[0][k] - (vr * w1r + vi * w1i) - w[0][k] : 0.0;
      if (CX) a[NP - 1][k] = in ? cv[NP - 1][k] - (vi * w1r - vr * w1i) - w[NP - 1][k] : 0.0;
      if (J == m - 2 && writer && c == m - 1) g.d[m - 1] = a[0][k];
    }
    if (J == m - 2 || last < J + 1) return;
  }
}

// every word of the exchange and of the checks empty, status cleared
__global__ void trd_resident_fill_k(unsigned long long* __restrict__ X, long long nx, unsigned long long* __restrict__ chk,
                                    long long nc, int* __restrict__ status, int m) {
  const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x, st = (long long)gridDim.x * blockDim.x;
  for (long long i = i0; i < nx; i += st) X[i] = RES_EMPTY;
  for (long long i = i0; i < nc; i += st) chk[i] = RES_EMPTY;
  if (i0 == 0) {
    status[0] = 0;
    status[1] = m - 1;
  }
}

// the reflectors into the rows of the matrix (row j, columns j+2 ...)
__global__ __launch_bounds__(256) void trd_resident_store_k(const double* __restrict__ R, int m, int done,
                                                            double* __restrict__ A, long long lda, long long pA,
                                                            int planes) {
  const int j = blockIdx.x;
  if (j >= done) return;
  for (int p = 0; p < planes; ++p)
    for (int c = j + 2 + threadIdx.x; c < m; c += 256)
      A[(long long)p * pA + (long long)j * lda + c] = R[((long long)p * m + j) * m + c];
}

template <bool CX, int T, int CC, int RW, bool ANY = true>
static bool resident_launch(Ctx* c, const ResArgs& g, int G) {
  // every workgroup must be resident at once: they wait for each other
  int per_cu = 0, cus = 0;
  DMRG_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, trd_resident_k<CX, T, CC, RW, ANY>, T, 0));
  DMRG_CHECK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
  if ((long long)per_cu * cus < G) return false;
  trd_resident_k<CX, T, CC, RW, ANY><<<G, T, 0, c->stream>>>(g);
  DMRG_CHECK_HIP(hipGetLastError());
  return true;
}

// The default limit as a constant of the code (ANY = false) where the variant
// fills the registers: as one more argument it takes order 2588 from 5.57 to 5.9
// us per column, complex 1700 from 6.58 to 6.7 and 1200 from 5.61 to 5.67.
template <bool CX, int T, int CC, int RW>
static bool either_launch(Ctx* c, const ResArgs& g, int G) {
  return g.limit == RES_DEFAULT ? resident_launch<CX, T, CC, RW, false>(c, g, G) : resident_launch<CX, T, CC, RW>(c, g, G);
}

int trd_resident_max(int field) { return field == CPLX ? 256 * 7 : 256 * 12; }

// Reduces A[s0:, s0:] of the n x n matrix A (in place: reflectors into its
// rows) as sytrd_lower / hetrd_lower do; false (nothing changed) when the
// order is out of range, the workgroups do not all fit, or a wait ran out (now
// or shortly before).
// *done: absolute number of columns reduced; *dropped: trace of the rest.
bool trd_resident(Ctx* c, int field, double* A, int n, int s0, double* d, double* e, double* tau, double stop_tol,
                  double total2, int* done, double* dropped) {
  const bool cx = field == CPLX;
  const int m = n - s0, np = cx ? 2 : 1;
  if (m < 3 || m > trd_resident_max(field) || !c->trd_backoff.allowed()) return false;
  // workgroup size and rows per workgroup: 13 rows (7 complex) fill the
  // 16-value reduction; larger orders take 12 so that the rows fit the
  // registers (512 threads, 256 registers each)
  const int T = m <= 256 ? 256 : 512, CC = (m + T - 1) / T;
  const int RW = cx ? 7 : (CC <= 2 ? 13 : 12);
  const int G = (m + RW - 1) / RW;
  ResArgs g;
  g.A = A + (long long)s0 * n + s0;
  g.lda = n;
  g.pA = (long long)n * n;
  g.m = m;
  g.mp = (m + 15) / 16 * 16;
  g.col0 = s0;
  g.n = n;
  const long long nx = (long long)(m - 1) * 2 * np * g.mp;
  const long long nc = (long long)(n / RES_CHECK + 1) * 2 * G;
  unsigned char* buf = (unsigned char*)ws_get(c, WS_TRD_X, 8 * (size_t)(nx + nc) + 64);
  g.X = (unsigned long long*)buf;
  g.chk = g.X + nx;
  g.status = (int*)(g.chk + nc);
  g.trace = (double*)(g.status + 2);
  g.R = (double*)ws_get(c, WS_TRD_R, sizeof(double) * np * (size_t)m * m);
  g.d = d + s0;
  g.e = e + s0;
  g.tau = tau + (size_t)np * s0;
  g.early = stop_tol > 0.0 ? 1 : 0;
  g.tol2 = stop_tol * stop_tol;
  g.total2 = total2;
  g.limit = c->trd_wait;
  trd_resident_fill_k<<<2048, 256, 0, c->stream>>>(g.X, nx, g.chk, nc, g.status, m);
  DMRG_CHECK_HIP(hipGetLastError());
  bool ok = false;
  if (!cx) {
    if (T == 256) ok = resident_launch<false, 256, 1, 13>(c, g, G);
    else switch (CC) {
      case 1: ok = resident_launch<false, 512, 1, 13>(c, g, G); break;
      case 2: ok = resident_launch<false, 512, 2, 13>(c, g, G); break;
      case 3: ok = resident_launch<false, 512, 3, 12>(c, g, G); break;
      case 4: ok = resident_launch<false, 512, 4, 12>(c, g, G); break;
      case 5: ok = resident_launch<false, 512, 5, 12>(c, g, G); break;
      case 6: ok = either_launch<false, 512, 6, 12>(c, g, G); break;
    }
  } else {
    if (T == 256) ok = resident_launch<true, 256, 1, 7>(c, g, G);
    else switch (CC) {
      case 1: ok = resident_launch<true, 512, 1, 7>(c, g, G); break;
      case 2: ok = resident_launch<true, 512, 2, 7>(c, g, G); break;
      case 3: ok = either_launch<true, 512, 3, 7>(c, g, G); break;
      case 4: ok = either_launch<true, 512, 4, 7>(c, g, G); break;
    }
  }
  if (!ok) return false;
  DMRG_CHECK_HIP(hipMemcpyAsync(c->host_scalars + 36, g.status, 16, hipMemcpyDeviceToHost, c->stream));
  DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
  int st[2];
  std::memcpy(st, c->host_scalars + 36, sizeof(st));
  if (st[0] != 0) {
    ++c->trd_counts[2];
    c->trd_backoff.failed();
    return false;
  }
  ++c->trd_counts[1];
  c->trd_backoff.succeeded();
  trd_resident_store_k<<<st[1], 256, 0, c->stream>>>(g.R, m, st[1], A + (long long)s0 * n + s0, n, g.pA, np);
  DMRG_CHECK_HIP(hipGetLastError());
  *done = s0 + st[1];
  if (st[1] < m - 1 && dropped) *dropped = std::max(0.0, c->host_scalars[37]);
  return true;
}

}  // namespace dmrg
