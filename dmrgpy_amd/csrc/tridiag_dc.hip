// Eigenpairs of a real symmetric tridiagonal matrix by divide and conquer
// (Cuppen's rank-one tearing; deflation and secular roots as in LAPACK's
// dlaed2 / dlaed4; eigenvectors from the recomputed updating vector of Gu and
// Eisenstat, SIAM J. Matrix Anal. Appl. 16, 172 (1995)): the middle step of
// the Gram eigensolver, between the tridiagonalisation and the
// back-transformation.
//
// The matrix is cut into 2^L blocks of B <= 12 rows (padded at its end with
// decoupled rows whose eigenvalues sort below all others), one wave solves
// each by implicit QL, and L levels merge pairs of blocks, all merges of a
// level in the same launches:
//   dc_deflate_k   one workgroup per merge: z, the merged order, deflation
//   dc_secular_k   one wave per root of the secular equation
//   dc_lowner_k    one wave per entry of the recomputed z; ranks
//   dc_vectors_k   one wave per eigenvector of the rank-one problem
//   one batched MFMA product: (each block's vectors) x its half of those
// The last level's vectors and products run for the kept eigenvectors only
// (tridiag_dc_vectors), once the host has seen the eigenvalues.  Rotations
// from deflating close poles are folded into the vectors of the rank-one
// problem, so the products keep their block structure.
//
// Bound by the latency of its chain of small launches (five per level, 4 to 18
// us each).  rocSOLVER's dstedc, which it replaces, spent its time in serial
// loops: 0.65 / 1.0 / 3.1 / 4.0 ms at orders 128 / 224 / 930 / 1200 (up to
// 480 us per level in its secular equations), against 0.15 / 0.2 / 0.4 / 0.4
// ms here.  Blocks of at most 12: QL runs about 0.4 us per rotation, 418 us
// for blocks of 32, 38 for 8, and a level of merges costs 30.
//
// A NaN or infinity in the matrix, or an iteration that runs out of steps, is
// reported through a status word and leaves every eigenvalue NaN.
#include "dmrg_internal.h"
#include "secular_root.h"
#include "wave_reduce.h"

#include <algorithm>

namespace dmrg {

constexpr int DC_LEAF = 12, DC_MAX = 4096;
constexpr double DC_EPS = 1.1102230246251565e-16;   // 2^-53
// Couplings of the scaled matrix below this are taken as zero (a part that far
// below the rest is diagonal then), and poles or weights of a merge below
// DC_FLOOR of its size are deflated.  A root then lies at least 1e-120 of the
// merge's size from its pole, so that the squares of z / (d - x), at most
// 1e300, stay in range.
constexpr double DC_TINY = 1e-70, DC_FLOOR = 1e-40;
constexpr double DC_FAIL = 1e-10;                    // relative residual of a root that was not found
constexpr double DC_PAD = -3.5;                      // below every eigenvalue of the scaled matrix (|lambda| <= 3)

// One level's merges; every array holds `merges` rows of N entries (N = 2 S)
struct DcLevel {
  int S, N, n;                 // half size, merged size, order of the matrix
  const double* e;             // off-diagonal of the matrix (unscaled)
  const double* scale;         // [0] the matrix was divided by this
  const double* D;             // eigenvalues of the halves, each ascending
  const double* Q;             // [2 merges][S][S], row = coordinate
  double* lam;                 // merged eigenvalues, ascending
  double *dl, *zl, *zh, *tau;  // survivors: pole, z, recomputed z, root - dl[org]
  int* org;
  int* sidx;                   // survivor -> index
  int *rep;                    // index -> survivor it follows (-1: none)
  double* g;                   // and its weight there
  double* dd;                  // deflated: eigenvalue,
  int *didx, *drot;            // index, rotation that deflated it (-1: none)
  double *rc, *rs;             // rotations
  int *rbase, *rlen;           // rotation -> first of its chain; at a chain's first, its length
  int *ichain, *ipos;          // index -> first rotation of its chain (-1: none), position in it
  int* col;                    // ascending position -> survivor j or N + deflated k
  int* K;                      // survivors per merge
  int* stat;                   // [blocks] nonzero: failed
};

__device__ __forceinline__ double dc_coupling(double e) { return fabs(e) < DC_TINY ? 0.0 : e; }

// ---------------------------------------------------------------------------
// Blocks: implicit QL with shifts, one wave per block.  Every lane runs the
// scalar recurrence; lane i applies the rotations to row i of the vectors.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void dc_leaf_k(const double* __restrict__ d, const double* __restrict__ e, int n,
                                                int B, double* __restrict__ D, double* __restrict__ Q,
                                                double* __restrict__ scale, int* __restrict__ stat) {
  __shared__ double sd[DC_LEAF], se[DC_LEAF + 1], Z[DC_LEAF][DC_LEAF + 1];
  const int lane = threadIdx.x, b0 = blockIdx.x * B;
  double mx = 0.0;
  bool finite = true;
  for (int i = lane; i < n; i += 64) {
    mx = fmax(mx, fabs(d[i]));
    finite &= isfinite(d[i]);
    if (i < n - 1) {
      mx = fmax(mx, fabs(e[i]));
      finite &= isfinite(e[i]);
    }
  }
  if (__any(!finite)) {   // in every block alike
    if (lane < B) D[b0 + lane] = __builtin_nan("");
    if (lane == 0) {
      stat[blockIdx.x] = 1;
      if (blockIdx.x == 0) scale[0] = 1.0;
    }
    return;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
  const double sc = mx > 0.0 ? fmax(mx, 1e-300) : 1.0, inv = 1.0 / sc;
  if (blockIdx.x == 0 && lane == 0) scale[0] = sc;
  auto off = [&](int i) { return i >= 0 && i < n - 1 ? dc_coupling(e[i] * inv) : 0.0; };   // of i and i + 1
  // a block graded downwards is turned upside down: QL keeps the small
  // eigenvalues' accuracy when the small entries come first
  auto diag = [&](int i) {
    double x = i < n ? d[i] * inv : DC_PAD;
    if (i == b0) x -= fabs(off(b0 - 1));               // tearing at the block's two ends
    if (i == b0 + B - 1) x -= fabs(off(b0 + B - 1));
    return x;
  };
  const bool flip = fabs(diag(b0)) > fabs(diag(b0 + B - 1));
  if (lane < B) {
    const int i = flip ? b0 + B - 1 - lane : b0 + lane;
    sd[lane] = diag(i);
    se[lane] = lane < B - 1 ? off(flip ? i - 1 : i) : 0.0;
    for (int k = 0; k < B; ++k) Z[lane][k] = k == lane ? 1.0 : 0.0;
  }
  __syncthreads();
  bool failed = false;
  for (int l = 0; l < B; ++l) {
    bool found = false;
    for (int iter = 0; iter < 60; ++iter) {
      int m = l;
      for (; m < B - 1; ++m) {
        const double t = fabs(sd[m]) + fabs(sd[m + 1]);
        if (fabs(se[m]) <= DC_EPS * t) break;
      }
      found = m == l;
      if (found) break;
      double p = (sd[l + 1] - sd[l]) / (2.0 * se[l]);
      double r = sqrt(p * p + 1.0);
      if (!(fabs(p) < 1e150)) r = fabs(p);
      double gg = sd[m] - sd[l] + se[l] / (p + copysign(r, p));
      double s = 1.0, c = 1.0, q = 0.0;
      bool split = false;
      for (int i = m - 1; i >= l; --i) {
        const double f = s * se[i], bb = c * se[i];
        const double di1 = sd[i + 1], di = sd[i];
        double fu = f, gu = gg, dn = 1.0, r2 = f * f + gg * gg;
        if (r2 < 1e-280) {   // squares out of range: by a power of two
          fu *= 0x1p500;
          gu *= 0x1p500;
          dn = 0x1p-500;
          r2 = fu * fu + gu * gu;
        }
        const double rin = r2 > 0.0 ? rsqrt(r2) : 0.0;
        r = r2 * rin * dn;
        __syncthreads();   // every lane has read what lane 0 now replaces
        if (lane == 0) se[i + 1] = r;
        if (r == 0.0) {
          if (lane == 0) {
            sd[i + 1] = di1 - q;
            se[m] = 0.0;
          }
          split = true;
          __syncthreads();
          break;
        }
        s = fu * rin;
        c = gu * rin;
        const double h = di1 - q;
        const double t = (di - h) * s + 2.0 * c * bb;
        q = s * t;
        if (lane == 0) sd[i + 1] = h + q;
        gg = c * t - bb;
        if (lane < B) {
          const double z1 = Z[lane][i + 1], z0 = Z[lane][i];
          Z[lane][i + 1] = s * z0 + c * z1;
          Z[lane][i] = c * z0 - s * z1;
        }
      }
      __syncthreads();
      if (!split && lane == 0) {
        sd[l] -= q;
        se[l] = gg;
        se[m] = 0.0;
      }
      __syncthreads();
    }
    failed |= !found;
  }
  if (lane == 0) stat[blockIdx.x] = failed;
  // ascending order by rank
  if (lane < B) {
    const double x = sd[lane];
    int rank = 0;
    for (int k = 0; k < B; ++k) rank += sd[k] < x || (sd[k] == x && k < lane);
    D[b0 + rank] = x;
    double* Qb = Q + (size_t)blockIdx.x * B * B;
    for (int r = 0; r < B; ++r) Qb[r * B + rank] = Z[flip ? B - 1 - r : r][lane];
  }
}

// exclusive prefix count of `flag` over the workgroup (256 threads) plus base;
// every thread gets the total added to base
__device__ __forceinline__ int block_rank(bool flag, int& base, int* sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long b = __ballot(flag);
  const int before = __popcll(b & ((1ull << lane) - 1));
  __syncthreads();
  if (lane == 0) sh[wave] = __popcll(b);
  __syncthreads();
  int off = base;
  for (int w = 0; w < wave; ++w) off += sh[w];
  base += sh[0] + sh[1] + sh[2] + sh[3];
  return off + before;
}

// Two poles p < n too close to tell apart: rotating z_p away leaves an
// off-diagonal entry below the rounding of the two poles themselves, or the floor
__device__ __forceinline__ bool dc_close(double dp, double zp, double dn, double zn, double floor) {
  return fabs((dn - dp) * zp * zn) <= (DC_EPS * (fabs(dp) + fabs(dn)) + floor) * (zp * zp + zn * zn);
}

__global__ __launch_bounds__(256) void dc_deflate_k(DcLevel L) {
  extern __shared__ double lds[];
  const int N = L.N, S = L.S, m = blockIdx.x, tid = threadIdx.x;
  double* sd = lds;            // sorted poles
  double* sz = sd + N;         // and their z
  int* sp = (int*)(sz + N);    // sorted -> index
  int* sc = sp + N;            // candidates (past the first deflation) -> sorted
  unsigned long long* fl = (unsigned long long*)(sc + N);   // candidate pairs to look at, one bit each
  __shared__ int sh[4];
  __shared__ double mxs[4];
  const size_t o = (size_t)m * N;
  const double* D = L.D + o;
  const double* Q1 = L.Q + (size_t)(2 * m) * S * S;
  const double* Q2 = Q1 + (size_t)S * S;
  const int cut = m * N + S;   // first row of the lower block
  const double beta = cut < L.n ? dc_coupling(L.e[cut - 1] / L.scale[0]) : 0.0;
  const double rho = 2.0 * fabs(beta), sg = beta < 0.0 ? -0.70710678118654752440 : 0.70710678118654752440;
  for (int i = tid; i < N; i += 256) {   // every slot valid whatever the values (NaN) do to the order
    sd[i] = sz[i] = 0.0;
    sp[i] = i;
  }
  __syncthreads();
  // merged ascending order of the halves (each ascending)
  double md = 0.0;
  for (int i = tid; i < N; i += 256) {
    const bool lower = i >= S;
    const double x = D[i];
    const double* other = lower ? D : D + S;
    int lo = 0, hi = S;   // entries of the other half before x (ties: the upper block first)
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (lower ? other[mid] <= x : other[mid] < x) lo = mid + 1;
      else hi = mid;
    }
    const int r = (lower ? i - S : i) + lo;
    const double z = lower ? sg * Q2[i - S] : 0.70710678118654752440 * Q1[(size_t)(S - 1) * S + i];
    sd[r] = x;
    sz[r] = z;
    sp[r] = i;
    if (x > DC_PAD + 0.25) md = fmax(md, fabs(x));
    L.ichain[o + i] = -1;
    L.rep[o + i] = -1;
    L.g[o + i] = 0.0;
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) {
    md = fmax(md, __shfl_xor(md, w, 64));
  }
  if ((tid & 63) == 0) mxs[tid >> 6] = md;
  __syncthreads();
  md = fmax(fmax(mxs[0], mxs[1]), fmax(mxs[2], mxs[3]));
  // Deflation is relative to the pole it concerns, not to the matrix norm as
  // in LAPACK: Gram matrices are graded, and their small eigenvalues (the
  // ones a truncation decides on) keep their own accuracy.  It costs little
  // here, where the products take the full order anyway.
  const double floor = DC_FLOOR * fmax(md, rho);
  // ---- poles the update hardly touches
  int nc = 0, nd = 0;
  for (int b = 0; b < N; b += 256) {
    const int i = b + tid;
    const bool in = i < N, cand = in && rho * fabs(sz[in ? i : 0]) > fmax(DC_EPS * fabs(sd[in ? i : 0]), floor);
    const int c0 = block_rank(cand, nc, sh);
    const int d0 = block_rank(in && !cand, nd, sh);
    if (cand) sc[c0] = i;
    else if (in) {
      L.dd[o + d0] = sd[i];
      L.didx[o + d0] = sp[i];
      L.drot[o + d0] = -1;
    }
  }
  __syncthreads();
  // ---- pairs of neighbours too close to tell apart: flagged in parallel, then
  // rotated one after the other (a rotation changes the pair that follows it)
  for (int b = 0; b < nc; b += 256) {
    const int j = b + tid;
    const bool f = j > 0 && j < nc && dc_close(sd[sc[j - 1]], sz[sc[j - 1]], sd[sc[j]], sz[sc[j]], floor);
    const unsigned long long w = __ballot(f);
    if ((tid & 63) == 0) fl[j >> 6] = w;
  }
  __syncthreads();
  if (tid == 0) {
    int nr = 0;
    const int words = (nc + 63) >> 6;
    int last = 0;   // pairs up to here are done
    for (int w = 0; w < words; ++w) {
      unsigned long long bits = fl[w];
      while (bits) {
        int j = (w << 6) + __ffsll((long long)bits) - 1;
        bits &= bits - 1;
        if (j <= last) continue;
        const int base = nr;
        while (j < nc) {
          const int a = sc[j - 1], b = sc[j];
          if (!dc_close(sd[a], sz[a], sd[b], sz[b], floor)) break;
          const double t = sqrt(sz[a] * sz[a] + sz[b] * sz[b]);
          const double c = sz[b] / t, s = -sz[a] / t;
          const double da = sd[a], db = sd[b];
          sz[b] = t;
          sz[a] = 0.0;
          sd[a] = da * c * c + db * s * s;
          sd[b] = da * s * s + db * c * c;
          L.rc[o + nr] = c;
          L.rs[o + nr] = s;
          L.rbase[o + nr] = base;
          if (nr == base) {
            L.ichain[o + sp[a]] = base;
            L.ipos[o + sp[a]] = 0;
          }
          L.ichain[o + sp[b]] = base;
          L.ipos[o + sp[b]] = nr - base + 1;
          L.dd[o + nd + nr] = sd[a];
          L.didx[o + nd + nr] = sp[a];
          L.drot[o + nd + nr] = nr;
          sc[j - 1] = -1 - a;   // deflated
          ++nr;
          ++j;
        }
        last = j;
        if (nr > base) L.rlen[o + base] = nr - base;
      }
    }
  }
  __syncthreads();
  // ---- survivors
  int k = 0;
  for (int b = 0; b < nc; b += 256) {
    const int j = b + tid;
    const bool alive = j < nc && sc[j] >= 0;
    const int r = block_rank(alive, k, sh);
    if (alive) {
      const int i = sc[j];
      L.dl[o + r] = sd[i];
      L.zl[o + r] = sz[i];
      L.sidx[o + r] = sp[i];
      L.rep[o + sp[i]] = r;
      L.g[o + sp[i]] = 1.0;
    }
  }
  if (tid == 0) L.K[m] = k;
  __threadfence_block();
  __syncthreads();
  // ---- weights of the members of a chain of rotations in its survivor
  for (int r = tid; r < k; r += 256) {
    const int last = L.sidx[o + r], base = L.ichain[o + last];
    if (base < 0) continue;
    const int R = L.rlen[o + base];
    double v = 1.0;
    for (int q = R - 1; q >= 0; --q) {   // rotation q joins positions q and q + 1
      const int who = q == R - 1 ? last : L.didx[o + nd + base + q + 1];
      L.rep[o + who] = r;
      L.g[o + who] = L.rc[o + base + q] * v;
      v *= -L.rs[o + base + q];
    }
    const int who = L.didx[o + nd + base];
    L.rep[o + who] = r;
    L.g[o + who] = v;
  }
}

// Every root of the secular equation (secular_root.h), one wave per root
__global__ __launch_bounds__(256) void dc_secular_k(DcLevel L) {
  const int m = blockIdx.y, lane = threadIdx.x & 63;
  const int j = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t o = (size_t)m * L.N;
  const int K = L.K[m];
  if (j >= K) return;
  const double* dl = L.dl + o;
  const double* zl = L.zl + o;
  const double rinv = 0.5 / fabs(L.e[m * L.N + L.S - 1] / L.scale[0]);
  const bool end = j == K - 1;
  double z2 = 0.0;
  if (end) {
    double u1 = 0.0, u2 = 0.0, u3 = 0.0;
    for (int i = lane; i < K; i += 64) z2 += zl[i] * zl[i];
    wave_sums4(z2, u1, u2, u3);
  }
  const int jn = end ? j : j + 1;
  const SecularRoot r = secular_root(end, dl[j], dl[jn], zl[j], zl[jn], z2, rinv, [&](double origin, double tau) {
    SecularSums s = {0.0, 0.0, 0.0, 0.0};
    for (int i = lane; i < K; i += 64) {
      const double z = zl[i], t = z / ((dl[i] - origin) - tau);
      if (i <= j) {
        s.psi += z * t;
        s.dpsi += t * t;
      } else {
        s.phi += z * t;
        s.dphi += t * t;
      }
    }
    wave_sums4(s.psi, s.dpsi, s.phi, s.dphi);
    return s;
  });
  if (lane == 0) {
    if (!(r.residual < DC_FAIL)) L.stat[0] = 1;   // not found: the iteration's own ends leave a rounding's worth
    L.tau[o + j] = r.tau;
    L.org[o + j] = j + r.next;
  }
}

// The z for which the computed roots are exact, and the ascending position of
// every eigenvalue; one wave per entry
__global__ __launch_bounds__(256) void dc_lowner_k(DcLevel L) {
  const int m = blockIdx.y, lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = L.N;
  if (i >= N) return;
  const size_t o = (size_t)m * N;
  const int K = L.K[m], nd = N - K;
  const double* dl = L.dl + o;
  if (i < K) {
    const double di = dl[i];
    double p = 1.0;
    for (int j = lane; j < K; j += 64) {
      const double x = (di - dl[L.org[o + j]]) - L.tau[o + j];
      p *= j == i ? x : x / (di - dl[j]);
    }
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) p *= __shfl_xor(p, w, 64);
    const double lam = dl[L.org[o + i]] + L.tau[o + i];
    int less = 0;
    for (int k = lane; k < nd; k += 64) less += L.dd[o + k] < lam;
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) less += __shfl_xor(less, w, 64);
    if (lane == 0) {
      L.zh[o + i] = copysign(sqrt(fabs(p)), L.zl[o + i]);
      L.lam[o + i + less] = lam;
      L.col[o + i + less] = i;
    }
  } else {
    const int k0 = i - K;
    const double x = L.dd[o + k0];
    int less = 0;
    for (int j = lane; j < K; j += 64) less += dl[L.org[o + j]] + L.tau[o + j] <= x;
    for (int k = lane; k < nd; k += 64) less += L.dd[o + k] < x || (L.dd[o + k] == x && k < k0);
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) less += __shfl_xor(less, w, 64);
    if (lane == 0) {
      L.lam[o + less] = x;
      L.col[o + less] = N + k0;
    }
  }
}

// The eigenvectors at the ascending positions first .. first + rows - 1 of the
// rank-one problem, in the basis of the two blocks' eigenvectors:
// Ut[merge][half][r][S]; one wave per vector
__global__ __launch_bounds__(256) void dc_vectors_k(DcLevel L, int first, int rows, double* __restrict__ Ut) {
  const int m = blockIdx.y, lane = threadIdx.x & 63, N = L.N, S = L.S;
  const int r = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (r >= rows) return;
  const size_t o = (size_t)m * N;
  double* top = Ut + ((size_t)(2 * m) * rows + r) * S;
  double* bot = Ut + ((size_t)(2 * m + 1) * rows + r) * S - S;   // index x >= S at bot[x]
  const int code = min(max(L.col[o + first + r], 0), 2 * N - 1);
  if (code < N) {
    const int K = L.K[m], j = min(code, max(K - 1, 0));
    const double* dl = L.dl + o;
    const double origin = dl[K > 0 ? L.org[o + j] : 0], tau = L.tau[o + j];
    double s = 0.0, u1 = 0.0, u2 = 0.0, u3 = 0.0;
    for (int i = lane; i < K; i += 64) {
      const double u = L.zh[o + i] / ((dl[i] - origin) - tau);
      s += u * u;
    }
    wave_sums4(s, u1, u2, u3);
    const double inv = 1.0 / sqrt(s);
    for (int x = lane; x < N; x += 64) {
      const int i = L.rep[o + x];
      (x < S ? top : bot)[x] = i >= 0 ? L.g[o + x] * (L.zh[o + i] / ((dl[i] - origin) - tau)) * inv : 0.0;
    }
  } else {
    const int k = code - N, who = L.didx[o + k], rot = k < N - L.K[m] ? L.drot[o + k] : -1;
    for (int x = lane; x < N; x += 64) {
      double u = x == who ? 1.0 : 0.0;
      if (rot >= 0) {   // deflated by a rotation: a vector of its chain
        const int base = L.rbase[o + rot];
        u = 0.0;
        if (L.ichain[o + x] == base) {
          const int t = L.ipos[o + x], q1 = rot - base;   // rotation q joins positions q and q + 1
          if (t == q1 + 1) {
            u = L.rs[o + rot];
          } else if (t <= q1) {
            u = L.rc[o + rot];
            for (int q = t; q < q1; ++q) u *= -L.rs[o + base + q];
            if (t > 0) u *= L.rc[o + base + t - 1];
          }
        }
      }
      (x < S ? top : bot)[x] = u;
    }
  }
}

// eigenvalues past the padding, scaled back (all NaN after a failure), and the
// status of the whole solve
__global__ __launch_bounds__(256) void dc_values_k(const double* __restrict__ lam, int np, int n,
                                                   const double* __restrict__ scale, double* __restrict__ w,
                                                   const int* __restrict__ stat, int blocks, int* __restrict__ info) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  int bad = 0;
  for (int b = threadIdx.x; b < blocks; b += 256) bad |= stat[b];
  bad = __syncthreads_or(bad);
  if (i < n) w[i] = bad ? __builtin_nan("") : lam[np - n + i] * scale[0];
  if (i == 0) *info = bad;
}

// Zt[r][i] = Q[i][first + r]: the vectors of a matrix that is one block
__global__ void dc_rows_k(const double* __restrict__ Q, int B, int n, int first, int rows, double* __restrict__ Zt,
                          int ldz) {
  for (int x = blockIdx.x * 256 + threadIdx.x; x < rows * n; x += gridDim.x * 256) {
    const int r = x / n, i = x % n;
    Zt[(size_t)r * ldz + i] = Q[i * B + first + r];
  }
}

// sorted poles, z, two index lists, one bit per pair (whole rounds of 256)
static size_t dc_deflate_lds(int N) {
  return (size_t)N * (2 * sizeof(double) + 2 * sizeof(int)) + 32 * (size_t)((N + 255) / 256);
}

// orders up to 4096 would pad to the arrays' limit; 4032 is the largest one tested
bool tridiag_dc_ok(int n) { return n >= 1 && n <= DC_MAX - 64; }

// [Q ping][Q pong][Ut][D ping][D pong][arrays of a level][scale][status of up to 512 blocks]
static size_t dc_ws_bytes(int np) { return sizeof(double) * (3 * (size_t)np * np + 18 * (size_t)np + 64 + 256); }

static DcLevel dc_level(int n, const double* e, int S, double* ws, int np) {
  DcLevel L;
  L.S = S;
  L.N = 2 * S;
  L.n = n;
  L.e = e;
  double* p = ws;
  auto dbl = [&]() { double* q = p; p += np; return q; };
  L.dl = dbl(); L.zl = dbl(); L.zh = dbl(); L.tau = dbl(); L.g = dbl(); L.dd = dbl(); L.rc = dbl(); L.rs = dbl();
  int* q = (int*)p;
  auto itg = [&]() { int* r = q; q += np; return r; };
  L.org = itg(); L.sidx = itg(); L.rep = itg(); L.didx = itg(); L.drot = itg(); L.rbase = itg(); L.rlen = itg();
  L.ichain = itg(); L.ipos = itg(); L.col = itg(); L.K = itg();
  return L;
}

// Eigenvalues (ascending, into w[n], device) of the tridiagonal matrix d, e
// (device, read only); keeps what tridiag_dc_vectors needs in the context's
// workspace.  *info (device): 0, or 1 when the matrix holds NaN or infinity or
// an iteration did not converge.
void tridiag_dc_values(Ctx* c, int n, const double* d, const double* e, double* w, int* info) {
  DMRG_REQUIRE(tridiag_dc_ok(n), "tridiag_dc: order out of range");
  int levels = 0;
  while ((DC_LEAF << levels) < n) ++levels;
  const int blocks = 1 << levels, B = (n + blocks - 1) / blocks, np = B * blocks;
  const size_t nq = (size_t)np * np;
  double* ws = (double*)ws_get(c, WS_TRD_DC, dc_ws_bytes(np));
  double* Q[2] = {ws, ws + nq};
  double* Ut = Q[1] + nq;
  double* D[2] = {Ut + nq, Ut + nq + np};
  double* arr = D[1] + np;
  double* scale = arr + 16 * (size_t)np;
  int* stat = (int*)(scale + 64);
  DMRG_REQUIRE(blocks <= 512, "tridiag_dc: too many blocks");
  dc_leaf_k<<<blocks, 64, 0, c->stream>>>(d, e, n, B, D[0], Q[0], scale, stat);
  DMRG_CHECK_HIP(hipGetLastError());
  int cur = 0;
  for (int l = 0; l < levels; ++l) {
    const int S = B << l, N = 2 * S, merges = blocks >> (l + 1);
    DcLevel L = dc_level(n, e, S, arr, np);
    L.scale = scale;
    L.stat = stat;
    L.D = D[cur];
    L.Q = Q[cur];
    L.lam = D[cur ^ 1];
    const size_t lds = dc_deflate_lds(N);
    if (lds > 48 * 1024)
      DMRG_CHECK_HIP(hipFuncSetAttribute((const void*)dc_deflate_k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)dc_deflate_lds(DC_MAX)));
    dc_deflate_k<<<merges, 256, lds, c->stream>>>(L);
    DMRG_CHECK_HIP(hipGetLastError());
    const dim3 per((N + 3) / 4, merges);
    dc_secular_k<<<per, 256, 0, c->stream>>>(L);
    DMRG_CHECK_HIP(hipGetLastError());
    dc_lowner_k<<<per, 256, 0, c->stream>>>(L);
    DMRG_CHECK_HIP(hipGetLastError());
    if (l < levels - 1) {
      dc_vectors_k<<<per, 256, 0, c->stream>>>(L, 0, N, Ut);
      DMRG_CHECK_HIP(hipGetLastError());
      // coordinates of every block: (block's vectors) x (its half of the new ones)
      GemmDesc g = gdesc(S, N, S, S, S, N, REAL, 4);
      g.transB = true;
      g.batch = 2 * merges;
      g.sA = (long long)S * S;
      g.sB = g.sC = (long long)S * N;
      gemm_f64(c, g, Q[cur], Ut, Q[cur ^ 1]);
    }
    cur ^= 1;
  }
  dc_values_k<<<(n + 255) / 256, 256, 0, c->stream>>>(D[cur], np, n, scale, w, stat, blocks, info);
  DMRG_CHECK_HIP(hipGetLastError());
  c->dc_n = n;
}

// Rows of Zt (keep x n, row pitch ldz): the eigenvectors of the `keep` largest
// eigenvalues of the last tridiag_dc_values of the same matrix, ascending
void tridiag_dc_vectors(Ctx* c, int n, const double* e, int keep, double* Zt, int ldz) {
  DMRG_REQUIRE(c->dc_n == n && keep >= 1 && keep <= n, "tridiag_dc: vectors without their eigenvalues");
  int levels = 0;
  while ((DC_LEAF << levels) < n) ++levels;
  const int blocks = 1 << levels, B = (n + blocks - 1) / blocks, np = B * blocks;
  const size_t nq = (size_t)np * np;
  double* ws = (double*)ws_get(c, WS_TRD_DC, dc_ws_bytes(np));
  double* Q[2] = {ws, ws + nq};
  double* Ut = Q[1] + nq;
  double* arr = Ut + nq + 2 * (size_t)np;
  if (levels == 0) {
    dc_rows_k<<<std::min(1024, (keep * n + 255) / 256), 256, 0, c->stream>>>(Q[0], B, n, B - keep, keep, Zt, ldz);
    DMRG_CHECK_HIP(hipGetLastError());
    return;
  }
  const int cur = (levels - 1) & 1, S = np / 2;
  DcLevel L = dc_level(n, e, S, arr, np);
  dc_vectors_k<<<dim3((keep + 3) / 4, 1), 256, 0, c->stream>>>(L, np - keep, keep, Ut);
  DMRG_CHECK_HIP(hipGetLastError());
  for (int half = 0; half < 2; ++half) {
    GemmDesc g = gdesc(keep, half ? n - S : S, S, S, S, ldz, REAL, 4);
    g.transB = true;
    gemm_f64(c, g, Ut + (size_t)half * keep * S, Q[cur] + (size_t)half * S * S, Zt + (size_t)half * S);
  }
}

}  // namespace dmrg
