// MFMA GEMM for complex products and for products with few output tiles (the
// H_eff, environment and split GEMMs at small and mid bond dimensions): each
// workgroup computes one 16 x 16, 32 x 16 or 32 x 32 tile, its waves split the inner
// dimension, and every wave loads its MFMA fragments straight from global
// memory one k-step ahead, with no LDS staging and no barrier in the k-loop.
// What bounds such a product is the chain of k-steps of the few workgroups it
// has, each a round trip to the L2: splitting the tiles finer and the inner
// dimension over waves shortens the chain (FP64 256 x 64 x 320: 4 workgroups of
// 64 x 64, 22.4 us, now 64 workgroups of 4 waves, 5 us; 1024 x 256 x 1280:
// 80 us, now 24).  Large complex products are bound by the FP64 matrix cores
// and gain from the missing barriers: 2400 x 6400 x 400 1102 us (44 TFLOP/s)
// with LDS tiles, now 763 (64 TFLOP/s of 72).
#include "gemm_kernels.h"
#include "tile_order.h"

#include <type_traits>

namespace dmrg {

template <typename T, bool CX, int WM, int WN, bool TA, bool TB, int TAG, typename CT>
__global__ __launch_bounds__(256) void gemm_direct(const T* __restrict__ A, const T* __restrict__ B,
                                                   CT* __restrict__ C, GemmArgs g) {
  constexpr int TM = 16 * WM, TN = 16 * WN, NP = CX ? 2 : 1;
  constexpr int STG = 2;   // k-steps of fragments per wave: one multiplied, one in flight
  typedef typename Mfma<T>::acc_t acc_t;
  extern __shared__ double smem[];
  T* red = reinterpret_cast<T*>(smem);

  const long long bz = blockIdx.z;
  A += bz * g.sA;
  B += bz * g.sB;
  C += bz * g.sC;
  int tr, tc;
  if (g.lower) {   // Hermitian C: row-major tiles, as every XCD then has an even share below the diagonal
    tr = blockIdx.x / g.nbx;
    tc = blockIdx.x % g.nbx;
    if (tile_above_diagonal(tr, tc, TM, TN)) return;
  } else {
    xcd_tile_of(blockIdx.x, 0, g.nbx, g.nby, tr, tc);
  }
  const int m0 = tr * TM, n0 = tc * TN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), KS = blockDim.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int M = g.M, N = g.N, K = g.K;

  acc_t acc[NP][WM][WN];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
      for (int b = 0; b < WN; ++b) acc[p][a][b] = acc_t{0, 0, 0, 0};

  // Addresses: a wave-uniform base per k-step plus one byte offset per lane
  // and 16-row block.  Rows / columns past the edge repeat the last one;
  // their results are not stored.
  const char* Ab = reinterpret_cast<const char*>(A + (TA ? (long long)m0 : (long long)m0 * g.lda));
  const char* Bb = reinterpret_cast<const char*>(B + (TB ? (long long)n0 * g.ldb : (long long)n0));
  long long oa[WM], ob[WN];
#pragma unroll
  for (int a = 0; a < WM; ++a) {
    const long long m = min(a * 16 + li, M - 1 - m0);
    oa[a] = (TA ? 4LL * lk * g.lda + m : m * g.lda + 4 * lk) * (long long)sizeof(T);
  }
#pragma unroll
  for (int b = 0; b < WN; ++b) {
    const long long n = min(b * 16 + li, N - 1 - n0);
    ob[b] = (TB ? n * g.ldb + 4 * lk : 4LL * lk * g.ldb + n) * (long long)sizeof(T);
  }
  // byte strides of one k and of the imaginary plane
  const long long ka = (TA ? (long long)g.lda : 1LL) * (long long)sizeof(T);
  const long long kb = (TB ? 1LL : (long long)g.ldb) * (long long)sizeof(T);
  const long long ppa = g.pA * (long long)sizeof(T), ppb = g.pB * (long long)sizeof(T);
  auto at = [](const char* base, long long off) { return *reinterpret_cast<const T*>(base + off); };
  const T sgnA = (CX && g.conjA) ? T(-1) : T(1);
  const T sgnB = (CX && g.conjB) ? T(-1) : T(1);

  // this wave's k-steps of 16: lane group lk holds k0 + 4 lk + t for MFMA t.
  // The loads of the main loop carry no branch (a step past the end reloads
  // the last full one), so the waits before an MFMA leave the later stages
  // in flight; a partial last step is masked and done at the end.
  const int steps = (K + 15) >> 4;
  const int per = (steps + KS - 1) / KS;
  const int s0 = min(steps, wave * per), s1 = min(steps, s0 + per);
  const int sf = min(s1, K >> 4);   // full steps: s0 .. sf - 1

  T fa[STG][NP][WM][4], fb[STG][NP][WN][4];
  auto load = [&](int q, int s) {
    const char* as = Ab + (long long)(s << 4) * ka;
    const char* bs = Bb + (long long)(s << 4) * kb;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int a = 0; a < WM; ++a) fa[q][p][a][t] = at(as + p * ppa + t * ka, oa[a]);
#pragma unroll
        for (int b = 0; b < WN; ++b) fb[q][p][b][t] = at(bs + p * ppb + t * kb, ob[b]);
      }
    __builtin_amdgcn_sched_barrier(0);   // keep the stages' loads in order
  };
  auto load_tail = [&](int q, int s) {   // k past the end: the last k's value, zeroed
    const int k0 = s << 4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool ok = k0 + 4 * lk + t < K;
      const long long back = ok ? t : (long long)(K - 1) - (k0 + 4 * lk);   // from the lane's first k
#pragma unroll
      for (int p = 0; p < NP; ++p) {
#pragma unroll
        for (int a = 0; a < WM; ++a) {
          const T x = at(Ab + (k0 + back) * ka + p * ppa, oa[a]);
          fa[q][p][a][t] = ok ? x : T(0);
        }
#pragma unroll
        for (int b = 0; b < WN; ++b) {
          const T x = at(Bb + (k0 + back) * kb + p * ppb, ob[b]);
          fb[q][p][b][t] = ok ? x : T(0);
        }
      }
    }
  };
  auto mma = [&](int q) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (!CX) {
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
          for (int b = 0; b < WN; ++b) acc[0][a][b] = Mfma<T>::op(fa[q][0][a][t], fb[q][0][b][t], acc[0][a][b]);
      } else {
        T ai[WM], na[WM], bi[WN];
#pragma unroll
        for (int a = 0; a < WM; ++a) {
          ai[a] = sgnA * fa[q][NP - 1][a][t];
          na[a] = -ai[a];
        }
#pragma unroll
        for (int b = 0; b < WN; ++b) bi[b] = sgnB * fb[q][NP - 1][b][t];
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
          for (int b = 0; b < WN; ++b) {
            acc[0][a][b] = Mfma<T>::op(fa[q][0][a][t], fb[q][0][b][t], acc[0][a][b]);
            acc[NP - 1][a][b] = Mfma<T>::op(fa[q][0][a][t], bi[b], acc[NP - 1][a][b]);
            acc[0][a][b] = Mfma<T>::op(na[a], bi[b], acc[0][a][b]);
            acc[NP - 1][a][b] = Mfma<T>::op(ai[a], fb[q][0][b][t], acc[NP - 1][a][b]);
          }
      }
    }
  };
  if (sf > s0) {
#pragma unroll
    for (int q = 0; q < STG - 1; ++q) load(q, min(s0 + q, sf - 1));
    for (int s = s0; s < sf; s += STG) {
#pragma unroll
      for (int q = 0; q < STG; ++q) {
        load((q + STG - 1) % STG, min(s + q + STG - 1, sf - 1));
        if (s + q < sf) mma(q);
      }
    }
  }
  if (s1 > sf && s1 > s0) {
    load_tail(0, s1 - 1);
    mma(0);
  }

  // sum over the waves, in halves (a fixed order), through LDS laid out
  // [register][lane]
  for (int h = KS >> 1; h >= 1; h >>= 1) {
    if (wave >= h && wave < 2 * h) {
      T* dst = red + (size_t)(wave - h) * (NP * WM * WN * 4 * 64);
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
          for (int b = 0; b < WN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[(((p * WM + a) * WN + b) * 4 + r) * 64 + lane] = acc[p][a][b][r];
    }
    __syncthreads();
    if (wave < h) {
      const T* src = red + (size_t)wave * (NP * WM * WN * 4 * 64);
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
          for (int b = 0; b < WN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[p][a][b][r] += src[(((p * WM + a) * WN + b) * 4 + r) * 64 + lane];
    }
    if (h > 1) __syncthreads();
  }
  if (wave != 0) return;

  const T alpha = T(g.alpha), beta = T(g.beta);
#pragma unroll
  for (int a = 0; a < WM; ++a)
#pragma unroll
    for (int b = 0; b < WN; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = (sizeof(T) == 8) ? (4 * r + lk) : (lk * 4 + r);
        const int row = m0 + a * 16 + rr, col = n0 + b * 16 + li;
        if (row < M && col < N) {
          const long long off = (long long)row * g.ldc + col;
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            T v = alpha * acc[p][a][b][r];
            if (g.beta != 0.0) v += beta * (T)C[off + p * g.pC];
            C[off + p * g.pC] = (CT)v;
          }
        }
      }
}

template <typename T, bool CX, int WM, int WN, bool TA, bool TB, int TAG, typename CT>
static void launch_direct_as(Ctx* c, const GemmDesc& d, const T* A, const T* B, CT* C, int ks) {
  constexpr int TM = 16 * WM, TN = 16 * WN;
  const GemmArgs g = make_args(d, TM, TN);
  const dim3 grid((unsigned)g.nbx * g.nby, 1, d.batch);
  const size_t lds = (size_t)(ks / 2) * (CX ? 2 : 1) * TM * TN * sizeof(T);
  gemm_direct<T, CX, WM, WN, TA, TB, TAG, CT><<<grid, 64 * ks, lds, c->stream>>>(A, B, C, g);
  DMRG_CHECK_HIP(hipGetLastError());
}

template <typename T, bool CX, int WM, int WN, bool TA, bool TB>
static void launch_direct_tagged(Ctx* c, const GemmDesc& d, const T* A, const T* B, T* C, int ks) {
  switch (d.tag) {
#define CASE(t) \
  case t: launch_direct_as<T, CX, WM, WN, TA, TB, t, T>(c, d, A, B, C, ks); break;
    DMRG_GEMM_TAGS(CASE)
#undef CASE
    default: throw Error("gemm: bad tag");
  }
}

template <typename T, bool CX, int WM, int WN, typename CT>
static void launch_direct_tt(Ctx* c, const GemmDesc& d, const T* A, const T* B, CT* C, int ks) {
  if constexpr (!std::is_same<T, CT>::value) launch_direct_as<T, CX, WM, WN, false, false, 2, CT>(c, d, A, B, C, ks);
  else if (!d.transA && !d.transB) launch_direct_tagged<T, CX, WM, WN, false, false>(c, d, A, B, C, ks);
  else if (d.transA && !d.transB) launch_direct_tagged<T, CX, WM, WN, true, false>(c, d, A, B, C, ks);
  else if (!d.transA && d.transB) launch_direct_tagged<T, CX, WM, WN, false, true>(c, d, A, B, C, ks);
  else launch_direct_tagged<T, CX, WM, WN, true, true>(c, d, A, B, C, ks);
}

// Tile and split.  Four waves share a tile's inner dimension where tiles are
// few or the dimension long (complex 2259 x 256 x 1280: 137 us against 172
// with one wave per tile; 8 waves were no faster anywhere), one wave otherwise
// (complex 2400 x 6400 x 400: 759 against 831, on 32 x 32 tiles).
// Up to 192 tiles of 32 x 32 the time is the latency of one tile's chain, and
// 16 x 16 is shortest (256 x 64 x 320: 5 us against 10; 256 x 256 x 1024: 11
// against 21; 760 x 187 x 935: 18.5 against 20).  Above, four waves fill a
// CU's matrix cores, so the time goes by rounds of the 256 CUs times the
// tile's size; smaller tiles load more per MFMA, 1.1 and 1.25 times the time
// per area.  Measured (us, 32 x 32 / 32 x 16 / 16 x 16):
//   complex  2259 x 256 x 1280  150 / 129 / 131    1620 x 180 x 900  76 / 58 / 54
//            600^3               52 /  41 /  45    3600 x 400 x 2000 404 / 439 / 473
//            256 x 256 x 768 x 5 61 /  52 /  47
//   FP64     1024 x 256 x 1280   22 /  30 /  34    650^3             24 / 28 / 29
//   FP32     2400 x 150 x 900    21 /  18 /  19
template <typename T, bool CX, typename CT>
static void launch_direct(Ctx* c, const GemmDesc& d, const T* A, const T* B, CT* C) {
  auto tiles = [&](int tm, int tn) { return (long long)((d.M + tm - 1) / tm) * ((d.N + tn - 1) / tn) * d.batch; };
  auto rounds = [&](int tm, int tn) { return (double)((tiles(tm, tn) + 255) / 256); };
  const int steps = (d.K + 15) / 16;
  int ks = tiles(32, 32) < 1024 || d.K >= 800 ? 4 : 1;
  const bool one = ks == 1;
  while (ks > 1 && steps < ks) ks >>= 1;
  const double c22 = 2.0 * rounds(32, 32), c21 = 1.1 * rounds(32, 16), c11 = 0.625 * rounds(16, 16);
  if (tiles(32, 32) <= 192) launch_direct_tt<T, CX, 1, 1, CT>(c, d, A, B, C, ks);
  else if (one || (c22 <= c21 && c22 <= c11)) launch_direct_tt<T, CX, 2, 2, CT>(c, d, A, B, C, ks);
  else if (c21 <= c11) launch_direct_tt<T, CX, 2, 1, CT>(c, d, A, B, C, ks);
  else launch_direct_tt<T, CX, 1, 1, CT>(c, d, A, B, C, ks);
}

void gemm_direct_f64(Ctx* c, const GemmDesc& d, const double* A, const double* B, double* C) {
  if (d.field == REAL) launch_direct<double, false, double>(c, d, A, B, C);
  else launch_direct<double, true, double>(c, d, A, B, C);
}
void gemm_direct_f32(Ctx* c, const GemmDesc& d, const float* A, const float* B, float* C) {
  if (d.field == REAL) launch_direct<float, false, float>(c, d, A, B, C);
  else launch_direct<float, true, float>(c, d, A, B, C);
}
void gemm_direct_f32_c64(Ctx* c, const GemmDesc& d, const float* A, const float* B, double* C) {
  launch_direct<float, false, double>(c, d, A, B, C);
}

}  // namespace dmrg
