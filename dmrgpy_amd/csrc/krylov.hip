// Krylov solvers on the device: Lanczos ground state and Lanczos matrix
// exponential, both with full re-orthogonalisation.  Vectors stay in HBM
// (FP64, planar complex); only the projected tridiagonal matrix and a handful
// of scalars per iteration come to the host, once per iteration.
//
// Vector work per iteration k (n elements per plane, sizeof = 8): three
// kernels after the apply (kry_alpha_k, kry_project_k, kry_clean_k), about
// (2k + 8) * n * 8 bytes of HBM traffic -- bandwidth bound for long vectors,
// launch bound for short ones.
#include "dmrg_internal.h"
#include "host_eig.h"
#include "wave_reduce.h"

#include <cfloat>
#include <cmath>
#include <complex>
#include <random>

namespace dmrg {

// ---------------------------------------------------------------------------
// device kernels
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

// part[j*nblk + blk] (re) and part[(k+j)*nblk + blk] (im): block-partial
// sums of conj(Q_j) . w over a contiguous chunk of the vector.
template <bool CX>
__global__ __launch_bounds__(256) void dot_block_k(const double* __restrict__ Q, long long ldq, int k,
                                                   const double* __restrict__ w, long long n,
                                                   double* __restrict__ part, int nblk) {
  __shared__ double red[2][4];
  const long long chunk = (n + nblk - 1) / nblk;
  const long long beg = (long long)blockIdx.x * chunk;
  const long long end = beg + chunk < n ? beg + chunk : n;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int j = 0; j < k; ++j) {
    const double* q = Q + (long long)j * ldq;
    double sr = 0, si = 0;
    for (long long i = beg + threadIdx.x; i < end; i += 256) {
      const double qr = q[i], wr = w[i];
      if (CX) {
        const double qi = q[i + n], wi = w[i + n];
        sr += qr * wr + qi * wi;
        si += qr * wi - qi * wr;
      } else {
        sr += qr * wr;
      }
    }
    sr = wave_sum(sr);
    if (CX) si = wave_sum(si);
    if (lane == 0) {
      red[0][wv] = sr;
      red[1][wv] = si;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      part[(long long)j * nblk + blockIdx.x] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
      if (CX) part[(long long)(k + j) * nblk + blockIdx.x] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    }
    __syncthreads();
  }
}

// out[row] = sum_b part[row*nblk + b]  (fixed order: deterministic)
__global__ __launch_bounds__(256) void reduce_rows_k(const double* __restrict__ part, int nblk,
                                                     double* __restrict__ out) {
  __shared__ double red[4];
  const int row = blockIdx.x;
  double s = 0;
  for (int b = threadIdx.x; b < nblk; b += 256) s += part[(long long)row * nblk + b];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[row] = red[0] + red[1] + red[2] + red[3];
}

// w -= sum_j coef_j Q_j (coef complex when CX: re[0..k), im[k..2k))
template <bool CX>
__global__ __launch_bounds__(256) void sub_block_k(const double* __restrict__ Q, long long ldq, int k,
                                                   const double* __restrict__ coef, double* __restrict__ w,
                                                   long long n) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long stride = (long long)gridDim.x * 256;
  for (; i < n; i += stride) {
    double ar = w[i], ai = CX ? w[i + n] : 0.0;
    for (int j = 0; j < k; ++j) {
      const double* q = Q + (long long)j * ldq;
      const double cr = coef[j];
      const double qr = q[i];
      if (CX) {
        const double ci = coef[k + j], qi = q[i + n];
        ar -= cr * qr - ci * qi;
        ai -= cr * qi + ci * qr;
      } else {
        ar -= cr * qr;
      }
    }
    w[i] = ar;
    if (CX) w[i + n] = ai;
  }
}

// x = scale * sum_j coef_j Q_j, coef real (COEF_CX false) or complex
template <bool CX, bool COEF_CX>
__global__ __launch_bounds__(256) void combine_k(const double* __restrict__ Q, long long ldq, int k,
                                                 const double* __restrict__ coef, double scale,
                                                 double* __restrict__ x, long long n) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long stride = (long long)gridDim.x * 256;
  for (; i < n; i += stride) {
    double ar = 0, ai = 0;
    for (int j = 0; j < k; ++j) {
      const double* q = Q + (long long)j * ldq;
      const double cr = coef[j], ci = COEF_CX ? coef[k + j] : 0.0;
      const double qr = q[i], qi = CX ? q[i + n] : 0.0;
      ar += cr * qr - ci * qi;
      ai += cr * qi + ci * qr;
    }
    x[i] = scale * ar;
    if (CX) x[i + n] = scale * ai;
  }
}

__global__ void scale_copy_k(const double* __restrict__ src, double* __restrict__ dst, double s, long long n) {
  long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long stride = (long long)gridDim.x * 256;
  for (; i < n; i += stride) dst[i] = s * src[i];
}

static unsigned vgrid(long long n) {
  long long b = (n + 255) / 256;
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return (unsigned)b;
}

static int dot_blocks(long long n) {
  long long b = (n + 2047) / 2048;
  if (b > 1024) b = 1024;
  if (b < 1) b = 1;
  return (int)b;
}

void vec_dot_block(Ctx* c, int field, const double* Q, long long ldq, int k, const double* w, long long n,
                   double* out) {
  if (k <= 0) return;
  // bytes: the k basis vectors and w read once
  ProfScope ps(c, 3, 0.0, 8.0 * (field == CPLX ? 2 : 1) * (double)(k + 1) * (double)n);
  const int nb = dot_blocks(n);
  const int rows = (field == CPLX ? 2 : 1) * k;
  double* part = (double*)ws_get(c, WS_KRYLOV_RED, sizeof(double) * (size_t)rows * nb);
  if (field == CPLX) dot_block_k<true><<<nb, 256, 0, c->stream>>>(Q, ldq, k, w, n, part, nb);
  else dot_block_k<false><<<nb, 256, 0, c->stream>>>(Q, ldq, k, w, n, part, nb);
  DMRG_CHECK_HIP(hipGetLastError());
  reduce_rows_k<<<rows, 256, 0, c->stream>>>(part, nb, out);
  DMRG_CHECK_HIP(hipGetLastError());
}

void vec_sub_block(Ctx* c, int field, const double* Q, long long ldq, int k, const double* coef, double* w,
                   long long n) {
  if (k <= 0) return;
  // bytes: the k basis vectors read once, w read and written
  ProfScope ps(c, 3, 0.0, 8.0 * (field == CPLX ? 2 : 1) * (double)(k + 2) * (double)n);
  if (field == CPLX) sub_block_k<true><<<vgrid(n), 256, 0, c->stream>>>(Q, ldq, k, coef, w, n);
  else sub_block_k<false><<<vgrid(n), 256, 0, c->stream>>>(Q, ldq, k, coef, w, n);
  DMRG_CHECK_HIP(hipGetLastError());
}

void vec_combine(Ctx* c, int field, const double* Q, long long ldq, int k, const double* coef, int coef_cplx,
                 double scale, double* x, long long n) {
  DMRG_REQUIRE(!(coef_cplx && field == REAL), "combine: complex coefficients need a complex vector");
  if (field == CPLX) {
    if (coef_cplx) combine_k<true, true><<<vgrid(n), 256, 0, c->stream>>>(Q, ldq, k, coef, scale, x, n);
    else combine_k<true, false><<<vgrid(n), 256, 0, c->stream>>>(Q, ldq, k, coef, scale, x, n);
  } else {
    combine_k<false, false><<<vgrid(n), 256, 0, c->stream>>>(Q, ldq, k, coef, scale, x, n);
  }
  DMRG_CHECK_HIP(hipGetLastError());
}

static void scale_copy(Ctx* c, const double* src, double* dst, double s, long long ntot) {
  scale_copy_k<<<vgrid(ntot), 256, 0, c->stream>>>(src, dst, s, ntot);
  DMRG_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// One Krylov step's vector work.  With w = H q_k on entry:
//   alpha = Re <q_k|w>;  w -= alpha q_k + beta q_{k-1};
//   c_j = <q_j|w> for the basis vectors to re-orthogonalise against;
//   w -= sum_j c_j q_j;  |w|^2.
// A sum over workgroups ends one kernel and the next one's workgroups each
// add up the partial sums (in the same fixed order: deterministic); the last
// one's and alpha go straight to pinned host memory, where the host adds them
// up after its one synchronisation per step.  The separate dot / reduce /
// subtract kernels and scalar copies this replaces were 15 launches; the
// block dot product walked the basis one vector at a time, with a
// workgroup-wide sum after each (complex n = 16384, 20 vectors: 19 us, now 5).
// ---------------------------------------------------------------------------
constexpr int KRY_T = 256;
constexpr int KRY_MAXBLK = 1024;

// Workgroups: enough for short vectors to fill the chip (256 elements each),
// few enough that re-reading the partial sums of every basis vector in every
// workgroup stays small next to the vectors themselves (the larger counts are
// for vectors of at least 2M / 8M elements).
static int kry_blocks(long long n) {
  const long long cap = n >= (8LL << 20) ? 1024 : (n >= (2LL << 20) ? 512 : 256);
  return (int)std::max<long long>(1, std::min<long long>(cap, (n + KRY_T - 1) / KRY_T));
}

// this workgroup's elements [beg, end)
__device__ __forceinline__ void kry_range(long long n, long long& beg, long long& end) {
  long long chunk = (n + gridDim.x - 1) / gridDim.x;
  chunk = (chunk + KRY_T - 1) / KRY_T * KRY_T;
  beg = (long long)blockIdx.x * chunk;
  end = beg + chunk < n ? beg + chunk : n;
}

// sum of one value per thread over the workgroup; valid in thread 0
__device__ __forceinline__ double kry_block_sum(double x, double* sh) {
  x = wave_sums2(x, 0.0);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
  __syncthreads();
  return threadIdx.x == 0 ? sh[0] + sh[1] + sh[2] + sh[3] : 0.0;
}

// part[0..nb) added up by every wave (the same order everywhere)
__device__ __forceinline__ double kry_sum_parts(const double* __restrict__ part, int nb) {
  double x = 0.0;
  for (int b = threadIdx.x & 63; b < nb; b += 64) x += part[b];
  return lane_value(wave_sums2(x, 0.0), 0);
}

// part[block] = sum of Re(conj(a) b) over the workgroup's elements
template <bool CX>
__global__ __launch_bounds__(KRY_T) void kry_alpha_k(const double* __restrict__ a, const double* __restrict__ b,
                                                     long long n, double* __restrict__ part) {
  __shared__ double sh[4];
  long long beg, end;
  kry_range(n, beg, end);
  double s = 0.0;
#pragma unroll 4
  for (long long i = beg + threadIdx.x; i < end; i += KRY_T) {
    s += a[i] * b[i];
    if (CX) s += a[i + n] * b[i + n];
  }
  s = kry_block_sum(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// Partial dot products of the NB basis vectors from j0 on (those past the
// last: repeated, not stored) with this workgroup's elements of w
template <bool CX, int NB>
__device__ __forceinline__ void kry_dots(const double* __restrict__ Q, long long ldq, int j0, int k,
                                         const double* __restrict__ w, long long n, long long beg, long long end,
                                         double* red, double* __restrict__ part2) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double acc[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) acc[t] = 0.0;
  for (long long i = beg + tid; i < end; i += KRY_T) {
    const double wr = w[i], wi = CX ? w[i + n] : 0.0;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const double* v = Q + (long long)min(j0 + t, k - 1) * ldq;
      const double vr = v[i];
      if (CX) {
        const double vi = v[i + n];
        acc[t] += vr * wr + vi * wi;
        acc[(NB + t) & 15] += vr * wi - vi * wr;
      } else {
        acc[t] += vr * wr;
      }
    }
  }
  const double s = wave_sums16(acc, lane);
  __syncthreads();   // the previous batch's sums are read
  if ((lane & 3) == 0) red[wave * 16 + sum_index(lane)] = s;
  __syncthreads();
  if (tid < (CX ? 2 * NB : NB)) {
    const int j = j0 + tid % NB;
    if (j < k)
      part2[(long long)(tid < NB ? j : k + j) * gridDim.x + blockIdx.x] =
          red[tid] + red[16 + tid] + red[32 + tid] + red[48 + tid];
  }
}

// alpha from part1 (to host_alpha); w -= alpha q + beta qp (qp null: no second
// term); then the partial dot products c_j of Q_0 .. Q_{k-1} with w, k x nblk
// (imaginary parts after the k real rows), or with k = 0 the partial |w|^2
template <bool CX>
__global__ __launch_bounds__(KRY_T) void kry_project_k(const double* __restrict__ q, const double* __restrict__ qp,
                                                       double beta, const double* __restrict__ part1, int nb1,
                                                       const double* __restrict__ Q, long long ldq, int k, double* w,
                                                       long long n, double* __restrict__ part2,
                                                       double* __restrict__ host_alpha) {
  __shared__ double red[4 * 16];
  const int tid = threadIdx.x;
  const double alpha = kry_sum_parts(part1, nb1);
  if (blockIdx.x == 0 && tid == 0) *host_alpha = alpha;
  long long beg, end;
  kry_range(n, beg, end);
  double nrm = 0.0;
#pragma unroll 2
  for (long long i = beg + tid; i < end; i += KRY_T) {   // each thread reads back only its own elements below
    double wr = w[i] - alpha * q[i], wi = CX ? w[i + n] - alpha * q[i + n] : 0.0;
    if (qp) {
      wr -= beta * qp[i];
      if (CX) wi -= beta * qp[i + n];
    }
    w[i] = wr;
    nrm += wr * wr;
    if (CX) {
      w[i + n] = wi;
      nrm += wi * wi;
    }
  }
  if (k == 0) {
    nrm = kry_block_sum(nrm, red);
    if (tid == 0) part2[blockIdx.x] = nrm;
    return;
  }
  // batches of up to 16 sums, the last one rounded up to a power of two
  constexpr int MAXB = CX ? 8 : 16;
  int j0 = 0;
  for (; k - j0 > MAXB / 2; j0 += MAXB) kry_dots<CX, MAXB>(Q, ldq, j0, k, w, n, beg, end, red, part2);
  const int rest = k - j0;
  if (rest <= 0) return;
  if (!CX && rest > 4) kry_dots<CX, CX ? 4 : 8>(Q, ldq, j0, k, w, n, beg, end, red, part2);
  else if (rest > 2) kry_dots<CX, 4>(Q, ldq, j0, k, w, n, beg, end, red, part2);
  else if (rest > 1) kry_dots<CX, 2>(Q, ldq, j0, k, w, n, beg, end, red, part2);
  else kry_dots<CX, 1>(Q, ldq, j0, k, w, n, beg, end, red, part2);
}

// c_j from part2 (k x nb); w -= sum_j c_j Q_j; partial |w|^2 to host_norm
constexpr int KRY_COEF = 512;   // coefficients held at a time
template <bool CX>
__global__ __launch_bounds__(KRY_T) void kry_clean_k(const double* __restrict__ Q, long long ldq, int k,
                                                     const double* __restrict__ part2, int nb, double* w, long long n,
                                                     double* __restrict__ host_norm) {
  __shared__ double cr[KRY_COEF], ci[CX ? KRY_COEF : 1];
  __shared__ double sh[4];
  const int tid = threadIdx.x, wave = tid >> 6;
  long long beg, end;
  kry_range(n, beg, end);
  double nrm = 0.0;
  for (int j0 = 0; j0 < k; j0 += KRY_COEF) {
    const int kb = min(KRY_COEF, k - j0);
    __syncthreads();   // the previous coefficients are used
    for (int r = wave; r < (CX ? 2 * kb : kb); r += 4) {
      const int row = r < kb ? j0 + r : k + j0 + (r - kb);
      const double x = kry_sum_parts(part2 + (long long)row * nb, nb);
      if ((tid & 63) == 0) {
        if (r < kb) cr[r] = x;
        else ci[CX ? r - kb : 0] = x;
      }
    }
    __syncthreads();
    const bool last = j0 + KRY_COEF >= k;
    for (long long i = beg + tid; i < end; i += KRY_T) {
      double wr = w[i], wi = CX ? w[i + n] : 0.0;
#pragma unroll 8
      for (int j = 0; j < kb; ++j) {
        const double* v = Q + (long long)(j0 + j) * ldq;
        const double vr = v[i];
        if (CX) {
          const double vi = v[i + n];
          wr -= cr[j] * vr - ci[j] * vi;
          wi -= cr[j] * vi + ci[j] * vr;
        } else {
          wr -= cr[j] * vr;
        }
      }
      w[i] = wr;
      if (CX) w[i + n] = wi;
      if (last) {
        nrm += wr * wr;
        if (CX) nrm += wi * wi;
      }
    }
  }
  nrm = kry_block_sum(nrm, sh);
  if (tid == 0) host_norm[blockIdx.x] = nrm;
}

static double sum_host(const double* p, int nb) {
  double s = 0.0;
  for (int b = 0; b < nb; ++b) s += p[b];
  return s;
}

// |x| (one kernel, the partial sums added up on the host)
static double krylov_norm(Ctx* c, int field, const double* x, long long n) {
  const int nb = kry_blocks(n);
  double* hp = c->host_parts;
  {
    ProfScope ps(c, 3, 0.0, 8.0 * (field == CPLX ? 2 : 1) * (double)n);
    if (field == CPLX) kry_alpha_k<true><<<nb, KRY_T, 0, c->stream>>>(x, x, n, hp);
    else kry_alpha_k<false><<<nb, KRY_T, 0, c->stream>>>(x, x, n, hp);
    DMRG_CHECK_HIP(hipGetLastError());
  }
  DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
  return std::sqrt(std::max(sum_host(hp, nb), 0.0));
}

// The step above for basis vector `it`, re-orthogonalising against the first
// k of Q; returns alpha, and |w| in *beta_new
static double krylov_step(Ctx* c, int field, const double* Q, long long ldq, int it, int k, double beta, double* w,
                          long long n, double* beta_new) {
  const int nb = kry_blocks(n), np = field == CPLX ? 2 : 1;
  double* part = (double*)ws_get(c, WS_KRYLOV_RED, sizeof(double) * ((size_t)np * std::max(k, 1) + 1) * nb);
  double* part2 = part + nb;
  double* hp = c->host_parts;   // [nb] |w|^2, then alpha
  double* dst = k == 0 ? hp : part2;
  const double* q = Q + (long long)it * ldq;
  const double* qp = it > 0 ? q - ldq : nullptr;
  {
    // bytes: alpha reads q and w; the projection q, q_{k-1}, w, the basis, and
    // writes w; the clean-up reads the basis and w and writes w
    ProfScope ps(c, 3, 0.0, 8.0 * np * (double)n * (2 + (it > 0 ? 4 : 3) + (k > 0 ? 2 * k + 2 : 0)));
    if (field == CPLX) {
      kry_alpha_k<true><<<nb, KRY_T, 0, c->stream>>>(q, w, n, part);
      kry_project_k<true><<<nb, KRY_T, 0, c->stream>>>(q, qp, beta, part, nb, Q, ldq, k, w, n, dst, hp + KRY_MAXBLK);
      if (k > 0) kry_clean_k<true><<<nb, KRY_T, 0, c->stream>>>(Q, ldq, k, part2, nb, w, n, hp);
    } else {
      kry_alpha_k<false><<<nb, KRY_T, 0, c->stream>>>(q, w, n, part);
      kry_project_k<false><<<nb, KRY_T, 0, c->stream>>>(q, qp, beta, part, nb, Q, ldq, k, w, n, dst, hp + KRY_MAXBLK);
      if (k > 0) kry_clean_k<false><<<nb, KRY_T, 0, c->stream>>>(Q, ldq, k, part2, nb, w, n, hp);
    }
    DMRG_CHECK_HIP(hipGetLastError());
  }
  DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
  *beta_new = std::sqrt(std::max(sum_host(hp, nb), 0.0));
  return hp[KRY_MAXBLK];
}

// Re <a|b> with a host round trip (used outside the hot loop)
double vec_dot_real(Ctx* c, int field, const double* a, const double* b, long long n) {
  double* out = (double*)ws_get(c, WS_KRYLOV_COEF, sizeof(double) * 4);
  vec_dot_block(c, field, a, 0, 1, b, n, out);
  DMRG_CHECK_HIP(hipMemcpyAsync(c->host_scalars, out, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
  return c->host_scalars[0];
}

// The host-side small eigenproblems (tridiag_eig, jacobi_eig,
// tridiag_expm_col0) are in host_eig.h.

// ---------------------------------------------------------------------------
// Lanczos ground state
// ---------------------------------------------------------------------------
static double lowest_tridiag(const std::vector<double>& al, const std::vector<double>& be) {
  std::vector<double> d(al);
  tridiag_eig(d, be, nullptr);
  return d[0];
}

static void dense_ground(Ctx* c, const HeffOp& h, double* x, double* energy) {
  const int field = h.d.field;
  const long long n = h.n;
  const int np = field == CPLX ? 2 : 1;
  const int dim = (int)n;
  double* e = (double*)ws_get(c, WS_KRYLOV_W, sizeof(double) * n * np * 2);
  std::vector<double> hcol((size_t)n * np), hm((size_t)dim * np * dim * np, 0.0), host_e(n * np);
  const int N = dim * np;  // real embedding size
  for (int col = 0; col < N; ++col) {
    std::fill(host_e.begin(), host_e.end(), 0.0);
    host_e[col] = 1.0;  // unit vector (real or imaginary part)
    DMRG_CHECK_HIP(hipMemcpyAsync(e, host_e.data(), sizeof(double) * n * np, hipMemcpyHostToDevice, c->stream));
    heff_apply(c, h, e, e + n * np);
    DMRG_CHECK_HIP(hipMemcpyAsync(hcol.data(), e + n * np, sizeof(double) * n * np, hipMemcpyDeviceToHost,
                                  c->stream));
    DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
    for (int row = 0; row < N; ++row) hm[(size_t)row * N + col] = hcol[row];
  }
  // symmetrise ((H + H^dag)/2 of the reference is the symmetric part of the
  // real embedding)
  for (int i = 0; i < N; ++i)
    for (int j = i + 1; j < N; ++j) {
      const double s = 0.5 * (hm[(size_t)i * N + j] + hm[(size_t)j * N + i]);
      hm[(size_t)i * N + j] = hm[(size_t)j * N + i] = s;
    }
  std::vector<double> w, v;
  jacobi_eig(hm, N, w, v);
  int k = 0;
  for (int i = 1; i < N; ++i)
    if (w[i] < w[k]) k = i;
  std::vector<double> xv(N);
  for (int i = 0; i < N; ++i) xv[i] = v[(size_t)i * N + k];
  DMRG_CHECK_HIP(hipMemcpyAsync(x, xv.data(), sizeof(double) * N, hipMemcpyHostToDevice, c->stream));
  DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
  *energy = w[k];
}

void lanczos_ground(Ctx* c, const HeffOp& h, double* x, int maxiter, double tol, double res_tol, double* energy,
                    int* iters) {
  const int field = h.d.field;
  const int np = field == CPLX ? 2 : 1;
  const long long n = h.n, ntot = n * np;
  if (n <= 3) {
    dense_ground(c, h, x, energy);
    if (iters) *iters = 0;
    return;
  }
  const int m = (int)std::min<long long>(maxiter, n);
  DMRG_REQUIRE(m >= 1, "lanczos: maxiter must be >= 1");
  const long long ldq = ntot;
  double* Q = (double*)ws_get(c, WS_KRYLOV_Q, sizeof(double) * (size_t)ldq * m);
  double* w = (double*)ws_get(c, WS_KRYLOV_W, sizeof(double) * ntot);
  double* coef = (double*)ws_get(c, WS_KRYLOV_COEF, sizeof(double) * 2 * (size_t)m);

  double beta0 = krylov_norm(c, field, x, n);
  if (beta0 == 0.0) {
    // zero start vector: seeded Gaussian restart (dmrg.py:102-105)
    std::mt19937_64 gen(0);
    std::normal_distribution<double> nd;
    std::vector<double> r(ntot, 0.0);
    for (long long i = 0; i < n; ++i) r[i] = nd(gen);
    DMRG_CHECK_HIP(hipMemcpyAsync(x, r.data(), sizeof(double) * ntot, hipMemcpyHostToDevice, c->stream));
    DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
    double s2 = 0;
    for (long long i = 0; i < n; ++i) s2 += r[i] * r[i];
    beta0 = std::sqrt(s2);
  }
  scale_copy(c, x, Q, 1.0 / beta0, ntot);

  std::vector<double> al, be;
  // first step
  double beta = 0.0;
  heff_apply(c, h, Q, w);
  al.push_back(krylov_step(c, field, Q, ldq, 0, 0, 0.0, w, n, &beta));
  double prev = al[0];
  int k = 1;
  for (int it = 1; it < m; ++it) {
    if (beta < tol) break;
    be.push_back(beta);
    double* q = Q + (long long)it * ldq;
    scale_copy(c, w, q, 1.0 / beta, ntot);
    heff_apply(c, h, q, w);
    // full re-orthogonalisation against q_0..q_{it-1} (dmrg.py:128-129)
    al.push_back(krylov_step(c, field, Q, ldq, it, it, beta, w, n, &beta));
    k = it + 1;
    const double cur = lowest_tridiag(al, be);
    if (std::fabs(cur - prev) < tol * std::max(1.0, std::fabs(cur))) break;
    if (res_tol > 0.0) {
      // Ritz residual |H y - theta y| = beta_k |last component of the
      // lowest tridiagonal eigenvector|: the stop for reduced-precision
      // operators, whose Ritz values stall at the rounding floor
      std::vector<double> dd(al), zz;
      tridiag_eig(dd, be, &zz);
      const double res = beta * std::fabs(zz[(size_t)(k - 1) * k + 0]);
      if (res <= res_tol * std::max(1.0, std::fabs(cur))) break;
    }
    prev = cur;
  }
  // Ritz vector x = Q v
  std::vector<double> d(al), z;
  std::vector<double> ee(be.begin(), be.begin() + (k - 1));
  d.resize(k);
  tridiag_eig(d, ee, &z);
  std::vector<double> v(k);
  for (int i = 0; i < k; ++i) v[i] = z[(size_t)i * k + 0];
  DMRG_CHECK_HIP(hipMemcpyAsync(coef, v.data(), sizeof(double) * k, hipMemcpyHostToDevice, c->stream));
  vec_combine(c, field, Q, ldq, k, coef, 0, 1.0, x, n);
  DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
  *energy = d[0];
  if (iters) *iters = k;
}

double rayleigh(Ctx* c, const HeffOp& h, const double* x) {
  const int np = h.d.field == CPLX ? 2 : 1;
  double* y = (double*)ws_get(c, WS_REFINE, sizeof(double) * h.n * np);
  heff_apply(c, h, x, y);
  const double xy = vec_dot_real(c, h.d.field, x, y, h.n);
  const double xx = vec_dot_real(c, h.d.field, x, x, h.n);
  return xy / xx;
}

// ---------------------------------------------------------------------------
// Krylov exponential
// ---------------------------------------------------------------------------
void krylov_expm(Ctx* c, const HeffOp& h, double* x, std::complex<double> coeff, int maxiter, double tol,
                 double errgoal, int* iters) {
  const int field = h.d.field;
  const int np = field == CPLX ? 2 : 1;
  const long long n = h.n, ntot = n * np;
  DMRG_REQUIRE(field == CPLX || coeff.imag() == 0.0, "expm: complex coefficient needs a complex vector");
  const int m = (int)std::min<long long>(maxiter, n);
  DMRG_REQUIRE(m >= 1, "expm: maxiter must be >= 1");
  const long long ldq = ntot;
  double* Q = (double*)ws_get(c, WS_KRYLOV_Q, sizeof(double) * (size_t)ldq * m);
  double* w = (double*)ws_get(c, WS_KRYLOV_W, sizeof(double) * ntot);
  double* coef = (double*)ws_get(c, WS_KRYLOV_COEF, sizeof(double) * 2 * (size_t)m);

  const double beta0 = krylov_norm(c, field, x, n);
  if (beta0 == 0.0) {
    if (iters) *iters = 0;
    return;
  }
  scale_copy(c, x, Q, 1.0 / beta0, ntot);
  std::vector<double> al, be;
  double beta = 0.0;
  for (int it = 0; it < m; ++it) {
    heff_apply(c, h, Q + (long long)it * ldq, w);
    // w -= Q_k (Q_k^dag w) over every basis vector so far (tdvp.py:138-139)
    al.push_back(krylov_step(c, field, Q, ldq, it, it + 1, beta, w, n, &beta));
    // first column of exp(coeff T_k)
    const int k = it + 1;
    const std::vector<std::complex<double>> col = tridiag_expm_col0(al, be, coeff);
    if (beta < tol || it == m - 1 || beta0 * beta * std::abs(col[k - 1]) < errgoal) {
      std::vector<double> cc(2 * (size_t)k);
      for (int r = 0; r < k; ++r) {
        cc[r] = col[r].real();
        cc[k + r] = col[r].imag();
      }
      DMRG_CHECK_HIP(hipMemcpyAsync(coef, cc.data(), sizeof(double) * 2 * k, hipMemcpyHostToDevice, c->stream));
      vec_combine(c, field, Q, ldq, k, coef, field == CPLX ? 1 : 0, beta0, x, n);
      DMRG_CHECK_HIP(hipStreamSynchronize(c->stream));
      if (iters) *iters = k;
      return;
    }
    be.push_back(beta);
    scale_copy(c, w, Q + (long long)(it + 1) * ldq, 1.0 / beta, ntot);
  }
  throw Error("expm: unreachable");
}

}  // namespace dmrg
