// Householder tridiagonalisation of real orders up to 128 (LAPACK dsytd2,
// lower) in one workgroup, the matrix in its registers.
//
// At these orders the register-resident reduction across workgroups
// (trd_resident.hip) is bound by its exchange, one device-wide round trip per
// column.  128 x 128 doubles fill a quarter of one compute unit's registers,
// so one workgroup does it with one barrier per column and no polling, no
// failure path and no workspace.
//
// The matrix sits at the end of a 128 x 128 frame: rows and columns
// J0 = 128 - m ... 127.  Four waves hold 32 rows each, a lane the columns
// lane and lane + 64 of them.  Every wave holds the column vectors x, v, w
// whole, two elements per lane, and once more the elements of its own rows,
// one per lane of 16, from where a row broadcast brings them to the update:
//
//   M -= v w^T + w v^T (previous column) and y = M x in one pass over the
//   registers, with beta, tau, scale of this column beside it;  the wave's
//   part of y, and row J+1, to LDS;  barrier;
//   y from its parts;  q = M v = M e_{J+1} + scale y;  q.v by one wave sum;
//   w = tau q + K v;  next column M e_{J+1} - v w_1 - w;  its x, |x|^2.
//
// The second part is done by every wave for itself (same values, same order),
// which saves the second barrier.  Waves whose rows are all reduced only keep
// the barriers.  What bounds a column is the chain: the pass (1300 cycles of
// 288 instructions), the two wave sums, the reflector's divisions and the LDS
// round trip.
//
// Order 128, across workgroups / here: 314 / 205 us.  The complex form (eight
// waves, 1.1 us of pass per column) measured 312 us against 298 across
// workgroups and is not kept.
#include "dmrg_internal.h"
#include "wave_reduce.h"

#include <algorithm>
#include <utility>

namespace dmrg {

constexpr int SGL_N = 128, SGL_RW = 32, SGL_RG = SGL_N / SGL_RW;
static_assert(SGL_RG == 4, "y is added up from four parts");
constexpr int SGL_CHECK = 32, SGL_CHECK_MIN = 64;   // early-stop checks as in trd_resident.hip

struct SingleArgs {
  double* A;             // m x m, row pitch lda
  long long lda;
  int m;
  double *d, *e, *tau;
  int early;
  double tol2;           // stop once |trailing|_F^2 <= tol2 |A|_F^2
  int* status;           // pinned host memory: columns reduced; read when early
  double* trace;         // likewise: trace of the block left
};

// the value of lane I of each row of 16
template <int I>
__device__ __forceinline__ double row_lane(double x) {
  return __builtin_amdgcn_update_dpp(0.0, x, 0x150 + I, 0xf, 0xf, true);
}

struct SingleState {
  double M[SGL_RW][2];
  // elements: lane, lane + 64, rows of the group 16 apart
  double v[4], w[4], x[4];
  double y[2];
};

template <int I>
__device__ __forceinline__ void single_row(SingleState& s) {
  constexpr int E = 2 + I / 16, L = I % 16;
  const double vr = row_lane<L>(s.v[E]), wr = row_lane<L>(s.w[E]), xr = row_lane<L>(s.x[E]);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const double b = s.M[I][k] - vr * s.w[k] - wr * s.v[k];
    s.M[I][k] = b;
    s.y[k] += b * xr;
  }
}

template <int FROM, int... I>
__device__ __forceinline__ void single_rows(SingleState& s, std::integer_sequence<int, I...>) {
  (single_row<FROM + I>(s), ...);
}

// row i of the group, i uniform: a tree of scalar branches
template <int LO, int N>
__device__ __forceinline__ void pick_row(const SingleState& s, int i, double (&out)[2]) {
  if constexpr (N == 1) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      out[k] = s.M[LO][k];
      // each leaf its own: merged, the row would be an address and M in memory
      asm volatile("; row %1" : "+v"(out[k]) : "n"(LO));
    }
  } else if (i < LO + N / 2) {
    pick_row<LO, N / 2>(s, i, out);
  } else {
    pick_row<LO + N / 2, N / 2>(s, i, out);
  }
}

// num / den where some, else 0, without a branch around the division
__device__ __forceinline__ double quotient(bool some, double num, double den) {
  double q = num / (some ? den : 1.0);
  asm volatile("" : "+v"(q));
  return some ? q : 0.0;
}

__global__ __launch_bounds__(256) void trd_single_k(SingleArgs g) {
  __shared__ double part[2][SGL_RG][SGL_N];
  __shared__ double col[2][SGL_N];
  __shared__ double out[3][SGL_N];   // d, e, tau
  __shared__ double chk[SGL_RG][2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int J0 = SGL_N - g.m, r0 = wave * SGL_RW, rmax = r0 + SGL_RW - 1;
  const bool writer = wave == SGL_RG - 1;
  const int idx[4] = {lane, lane + 64, r0 + (lane & 15), r0 + 16 + (lane & 15)};
  SingleState s;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int c = idx[k];
#pragma unroll
    for (int i = 0; i < SGL_RW; ++i)
      s.M[i][k] = c >= J0 && r0 + i >= J0 ? g.A[(long long)(r0 + i - J0) * g.lda + c - J0] : 0.0;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    s.x[t] = idx[t] >= J0 ? g.A[idx[t] - J0] : 0.0;
    s.v[t] = s.w[t] = 0.0;
  }
  // no part from waves before the matrix
#pragma unroll
  for (int u = 0; u < 2; ++u) part[u][wave][lane] = part[u][wave][lane + 64] = 0.0;
  double total2 = -1.0, dJ = 0.0, a0 = 0.0;   // column J: its diagonal, the entry below it
  bool passed = false;

  double* refl = g.A + (lane - J0);   // the lane's place in row J
  auto finish = [&](int done) {   // by the wave that wrote them
    for (int i = lane; i < done; i += 64) {
      g.d[i] = out[0][i];
      g.e[i] = out[1][i];
      g.tau[i] = out[2][i];
    }
  };
  // early stop: |A[J:, J:]|_F^2 against the whole matrix's; true: stop here
  auto check = [&](int J, bool active) -> bool {
    const int sa = J - J0;
    if (!g.early || !(sa == 0 || (sa >= SGL_CHECK_MIN && sa % SGL_CHECK == 0))) return false;
    double q2 = 0.0, dg = 0.0;
    int ln = lane, rr = r0;   // opaque, or their comparisons would be kept in registers across the columns
    asm volatile("" : "+v"(ln), "+s"(rr));
    if (active) {   // rows and columns from J + 1 on
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int c = ln + 64 * k;
#pragma unroll
        for (int i = 0; i < SGL_RW; ++i)
          if (rr + i > J && c > J) {
            q2 += s.M[i][k] * s.M[i][k];
            if (rr + i == c) dg += s.M[i][k];
          }
      }
      if (writer) {   // column and row J
        q2 += 2.0 * (s.x[0] * s.x[0] + s.x[1] * s.x[1]);
        if (lane == 0) {
          q2 += dJ * dJ + 2.0 * a0 * a0;
          dg += dJ;
        }
      }
    }
    const double both = wave_sums2(q2, dg);
    if (lane == 0) chk[wave][0] = both;
    if (lane == 32) chk[wave][1] = both;
    __syncthreads();
    double f2 = 0.0, tc = 0.0;
#pragma unroll
    for (int u = 0; u < SGL_RG; ++u) {
      f2 += chk[u][0];
      tc += chk[u][1];
    }
    __syncthreads();
    if (sa == 0) {
      total2 = f2;
    } else if (passed) {   // one check after the first to pass, as the panel path stops
      if (writer) {
        finish(sa);
        if (lane == 0) {
          g.status[0] = sa;
          g.trace[0] = tc;
        }
      }
      return true;
    } else {
      passed = f2 <= g.tol2 * total2;
    }
    return false;
  };

  int J = J0;
  for (; J < SGL_N - 1 && rmax > J; ++J) {
    const int par = J & 1, sa = J - J0, l1 = (J + 1) & 63;
    const bool hi = J + 1 >= 64;
    // s.x holds column J from its diagonal on; x = the part from J + 2 on
    dJ = lane_value(J >= 64 ? s.x[1] : s.x[0], J & 63);
    a0 = lane_value(hi ? s.x[1] : s.x[0], l1);
#pragma unroll
    for (int t = 0; t < 4; ++t) s.x[t] = idx[t] >= J + 2 ? s.x[t] : 0.0;
    s.y[0] = s.y[1] = 0.0;
    // the pass over the registers in three parts, a third of the reflector's
    // chain of dependent operations beside each
    double xx = s.x[0] * s.x[0] + s.x[1] * s.x[1];
    xx = lane_value(wave_sums2(xx, xx), 0);
    single_rows<0>(s, std::make_integer_sequence<int, 8>{});
    __builtin_amdgcn_sched_barrier(0);
    const bool some = xx != 0.0;
    double beta;
    {
      const double h2 = a0 * a0 + xx;
      // powers of two keep a0^2 and the root in range; xx is the plain sum of
      // squares, as in the panels: entries of x below 1e-154 lose digits in
      // it, and below 1e-162 they count as zero
      const double up = h2 > 1e-280 ? (h2 < 1e280 ? 1.0 : 0x1p-600) : 0x1p600;
      const double dn = h2 > 1e-280 ? (h2 < 1e280 ? 1.0 : 0x1p600) : 0x1p-600;
      const double b = a0 * up;
      beta = some ? -copysign(sqrt(b * b + xx * up * up) * dn, a0) : a0;
    }
    single_rows<8>(s, std::make_integer_sequence<int, 10>{});
    __builtin_amdgcn_sched_barrier(0);
    const double tau = quotient(some, beta - a0, beta), scale = quotient(some, 1.0, a0 - beta);
    single_rows<18>(s, std::make_integer_sequence<int, 14>{});
    part[par][wave][lane] = s.y[0];
    part[par][wave][lane + 64] = s.y[1];
    if (wave == (J + 1) / SGL_RW) {   // row J+1 = column J+1
      double r1[2];
      pick_row<0, SGL_RW>(s, (J + 1) % SGL_RW, r1);
      col[par][lane] = r1[0];
      col[par][lane + 64] = r1[1];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) s.v[t] = idx[t] == J + 1 ? 1.0 : scale * s.x[t];
    __syncthreads();
    if (check(J, true)) return;
    // q = M v = M e_{J+1} + scale y; q.v
    double cv[4], q[4], yp[4][SGL_RG];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      cv[t] = col[par][idx[t]];
#pragma unroll
      for (int u = 0; u < SGL_RG; ++u) yp[t][u] = part[par][u][idx[t]];
    }
    __builtin_amdgcn_sched_barrier(0);   // all loads under way before the first is waited for
#pragma unroll
    for (int t = 0; t < 4; ++t)
      q[t] = idx[t] > J ? cv[t] + scale * ((yp[t][0] + yp[t][1]) + (yp[t][2] + yp[t][3])) : 0.0;
    double qv = q[0] * s.v[0] + q[1] * s.v[1];
    qv = lane_value(wave_sums2(qv, qv), 0);
    // w = w0 + K v, K = -(tau / 2) (w0.v) with w0 = tau q
    const double K = -0.5 * tau * tau * qv;
#pragma unroll
    for (int t = 0; t < 4; ++t) s.w[t] = tau * q[t] + K * s.v[t];
    const double w1 = lane_value(hi ? s.w[1] : s.w[0], l1);
#pragma unroll
    for (int t = 0; t < 4; ++t) s.x[t] = cv[t] - s.v[t] * w1 - s.w[t];   // column J+1
    if (writer) {
      if (lane == 0) {
        out[0][sa] = dJ;
        out[1][sa] = beta;
        out[2][sa] = tau;
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)   // the reflector, into row J of the matrix
        if (idx[t] >= J + 2) refl[64 * t] = s.v[t];
      refl += g.lda;
    }
  }
  for (; J < SGL_N - 1; ++J) {   // reduced: keep the barriers
    if (J == rmax) part[J & 1][wave][lane] = part[J & 1][wave][lane + 64] = 0.0;   // nothing more from this wave
    __syncthreads();
    if (check(J, false)) return;
  }
  if (writer) {
    if (lane == 63) g.d[g.m - 1] = s.x[1];
    finish(g.m - 1);
    if (g.early && lane == 0) g.status[0] = g.m - 1;
  }
}

int trd_single_max() { return SGL_N; }

// Reduces the real n x n matrix A as sytrd_lower does; *done: columns reduced,
// *dropped: trace of the rest when stopped early.
void trd_single(Ctx* c, double* A, int n, double* d, double* e, double* tau, double stop_tol, int* done,
                double* dropped) {
  DMRG_REQUIRE(n >= 2 && n <= SGL_N, "trd_single: order out of range");
  SingleArgs g;
  g.A = A;
  g.lda = n;
  g.m = n;
  g.d = d;
  g.e = e;
  g.tau = tau;
  g.early = stop_tol > 0.0 ? 1 : 0;
  g.tol2 = stop_tol * stop_tol;
  g.status = (int*)(c->host_scalars + 36);
  g.trace = c->host_scalars + 37;
  trd_single_k<<<1, 256, 0, c->stream>>>(g);
  DMRG_CHECK_HIP(hipGetLastError());
  *done = n - 1;
  if (g.early) {
    DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
    *done = *(volatile int*)g.status;
    if (*done < n - 1 && dropped) *dropped = std::max(0.0, c->host_scalars[37]);
  }
}

}  // namespace dmrg
