// MFMA GEMM kernels for gfx950 (CDNA4): FP64 and FP32 via the 16x16x4
// MFMA shapes, split-BF16x3 via the 16x16x32 BF16 MFMA.  256 threads = four
// 64-wide waves in a 2x2 arrangement; every wave owns a (16*TM) x (16*TN)
// patch of the block tile, so a block computes (32*TM) x (32*TN).  Operand
// tiles are staged through LDS with the next tile prefetched into registers
// while the current one is multiplied.
//
// MFMA lane layout (16x16xK shapes): lane l supplies A[i = l%16][k-slot l/16]
// and B[k-slot l/16][j = l%16]; the accumulator element r (0..3) holds
// C[4*(l/16) + r][l%16] for the FP32 and BF16 shapes and C[4*r + l/16][l%16]
// for the FP64 shape.  The k-slots of one instruction may map to any 4 (FP32/FP64) or
// 32 (BF16, 8 per slot) distinct k values as long as A and B agree, so each
// lane reads 4 (resp. 8) consecutive k from LDS in one vector access.
#include "gemm_kernels.h"
#include "tile_order.h"

#include <type_traits>

namespace dmrg {

// ---------------------------------------------------------------------------
// Real FP64 / FP32 kernel for products with enough output tiles to fill the
// chip (the H_eff, environment and Gram GEMMs at large bond dimensions):
// operand tiles in double-buffered LDS, one barrier per k-tile, the next
// k-tile's 16-byte vectors loaded into registers while the current one is
// multiplied, XCD-aware tile order (xcd_tile, tile_order.h).  MFMA bound.
// The loads carry no per-element bounds check (see load_full); with a check
// and a branch around every vector the same loop ran the FP32 products
// 5070 x 3428 x 845 / 3918 x 11696 x 653 / 10448 x 731 x 4386 at 72 / 83 /
// 73 TFLOP/s, now 103 / 115 / 116, and 6144 x 16384 x 1024 at 112, now 130
// (a large library product reaches 148).
// ---------------------------------------------------------------------------

// Tile (row, column) of this workgroup in the XCD-grouped order of
// tile_order.h.
__device__ __forceinline__ void xcd_tile(int nbx, int nby, int& tr, int& tc) {
  xcd_tile_of(blockIdx.x, blockIdx.y, nbx, nby, tr, tc);
}
template <typename T, int TM, int TN, bool TA, bool TB, int TAG, typename CT = T>
__global__ __launch_bounds__(256) void gemm_fast(const T* __restrict__ A, const T* __restrict__ B,
                                                 CT* __restrict__ C, GemmArgs g) {
  // k per tile: 16, or 32 where 16 would not give every thread whole vectors
  constexpr int BM = 32 * TM, BN = 32 * TN;
  constexpr int BK = (BM * 16) % (Vec<T>::W * 256) == 0 && (BN * 16) % (Vec<T>::W * 256) == 0 ? 16 : 32;
  constexpr int PAD = 16 / sizeof(T);     // keeps rows 16-byte aligned
  constexpr int VW = Vec<T>::W;
  typedef typename Vec<T>::type vec_t;
  constexpr int NA = BM * BK / (VW * 256), NB = BN * BK / (VW * 256);
  typedef typename Mfma<T>::acc_t acc_t;

  // Each operand tile keeps the orientation of its global rows, so every
  // 16-byte global vector lands in LDS with one 16-byte store (no transposed
  // scalar stores and their bank conflicts): [m][k] / [n][k] when k is the
  // contiguous global index, [k][m] / [k][n] otherwise.  MFMA fragments read
  // 4 consecutive k either as one vector or as 4 scalars from 4 rows.
  constexpr int AR = TA ? BK : BM, AC = (TA ? BM : BK) + PAD;
  constexpr int BR = TB ? BN : BK, BC = (TB ? BK : BN) + PAD;
  __shared__ __attribute__((aligned(16))) T As[2][AR][AC];
  __shared__ __attribute__((aligned(16))) T Bs[2][BR][BC];

  const long long bz = blockIdx.z;
  A += bz * g.sA;
  B += bz * g.sB;
  C += bz * g.sC;
  int tr, tc;
  if (g.lower) {
    // Hermitian C: row-major tiles (every XCD gets an even share of the
    // lower-triangle tiles), those strictly above the diagonal exit at once
    tr = blockIdx.x / g.nbx;
    tc = blockIdx.x % g.nbx;
    if (tile_above_diagonal(tr, tc, BM, BN)) return;
  } else {
    xcd_tile_of(blockIdx.x, 0, g.nbx, g.nby, tr, tc);
  }
  const int m0 = tr * BM, n0 = tc * BN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lk = lane >> 4;
  const int M = g.M, N = g.N, K = g.K;

  acc_t acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = acc_t{0, 0, 0, 0};

  vec_t ra[NA], rb[NB];

  // Each thread's vectors: a wave-uniform base per k-tile plus one byte
  // offset per vector.  A vector along m / n may run over the edge of its row
  // into the next one (what it picks up there is not stored); in an edge tile
  // the k-tile that holds the last k (for rows shorter than a vector, the
  // last few) is therefore read element by element with a mask, as is a
  // partial k-tile; all others (up to kfull) without.  Rows and columns
  // wholly past the edge repeat the tile's first.
  const char* Ab = reinterpret_cast<const char*>(A + (TA ? (long long)m0 : (long long)m0 * g.lda));
  const char* Bb = reinterpret_cast<const char*>(B + (TB ? (long long)n0 * g.ldb : (long long)n0));
  const bool overA = TA && m0 + BM > M, overB = !TB && n0 + BN > N;
  const int kfull = !(overA || overB) ? K : K - 1 - ((TA && g.lda < VW) || (!TB && g.ldb < VW) ? VW : 0);
  long long oa[NA], ob[NB];
#pragma unroll
  for (int e = 0; e < NA; ++e) {
    const int v = tid + 256 * e;
    int r, c;  // element (m = m0 + r, k = k0 + c) is the first of the vector
    if (!TA) { r = v / (BK / VW); c = (v % (BK / VW)) * VW; } else { c = v / (BM / VW); r = (v % (BM / VW)) * VW; }
    if (m0 + r >= M) r = 0;
    oa[e] = (TA ? (long long)c * g.lda + r : (long long)r * g.lda + c) * (long long)sizeof(T);
  }
#pragma unroll
  for (int e = 0; e < NB; ++e) {
    const int v = tid + 256 * e;
    int r, c;  // element (n = n0 + r, k = k0 + c)
    if (!TB) { c = v / (BN / VW); r = (v % (BN / VW)) * VW; } else { r = v / (BK / VW); c = (v % (BK / VW)) * VW; }
    if (n0 + r >= N) r = 0;
    ob[e] = (TB ? (long long)r * g.ldb + c : (long long)c * g.ldb + r) * (long long)sizeof(T);
  }
  const long long ka = (TA ? (long long)g.lda : 1LL) * (long long)sizeof(T);   // byte stride of one k
  const long long kb = (TB ? 1LL : (long long)g.ldb) * (long long)sizeof(T);

  auto load_full = [&](int k0) {
    const char* pa = Ab + k0 * ka;
    const char* pb = Bb + k0 * kb;
#pragma unroll
    for (int e = 0; e < NA; ++e) __builtin_memcpy(&ra[e], pa + oa[e], sizeof(vec_t));
#pragma unroll
    for (int e = 0; e < NB; ++e) __builtin_memcpy(&rb[e], pb + ob[e], sizeof(vec_t));
  };
  auto load_masked = [&](int k0) {
#pragma unroll
    for (int e = 0; e < NA; ++e) {
      const int v = tid + 256 * e;
      int r, c;
      if (!TA) { r = v / (BK / VW); c = (v % (BK / VW)) * VW; } else { c = v / (BM / VW); r = (v % (BM / VW)) * VW; }
#pragma unroll
      for (int j = 0; j < VW; ++j) {
        const int gm = m0 + r + (TA ? j : 0), gk = k0 + c + (TA ? 0 : j);
        ra[e][j] = (gm < M && gk < K) ? A[TA ? (long long)gk * g.lda + gm : (long long)gm * g.lda + gk] : T(0);
      }
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int v = tid + 256 * e;
      int r, c;
      if (!TB) { c = v / (BN / VW); r = (v % (BN / VW)) * VW; } else { r = v / (BK / VW); c = (v % (BK / VW)) * VW; }
#pragma unroll
      for (int j = 0; j < VW; ++j) {
        const int gn = n0 + r + (TB ? 0 : j), gk = k0 + c + (TB ? j : 0);
        rb[e][j] = (gn < N && gk < K) ? B[TB ? (long long)gn * g.ldb + gk : (long long)gk * g.ldb + gn] : T(0);
      }
    }
  };
  auto load_regs = [&](int k0) {
    if (k0 + BK <= kfull) load_full(k0);
    else load_masked(k0);
  };
  auto store_regs = [&](int buf) {
#pragma unroll
    for (int e = 0; e < NA; ++e) {
      const int v = tid + 256 * e;
      if (!TA) {
        const int r = v / (BK / VW), c = (v % (BK / VW)) * VW;     // As[m][k]
        *reinterpret_cast<vec_t*>(&As[buf][r][c]) = ra[e];
      } else {
        const int c = v / (BM / VW), r = (v % (BM / VW)) * VW;     // As[k][m]
        *reinterpret_cast<vec_t*>(&As[buf][c][r]) = ra[e];
      }
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int v = tid + 256 * e;
      if (!TB) {
        const int c = v / (BN / VW), r = (v % (BN / VW)) * VW;     // Bs[k][n]
        *reinterpret_cast<vec_t*>(&Bs[buf][c][r]) = rb[e];
      } else {
        const int r = v / (BK / VW), c = (v % (BK / VW)) * VW;     // Bs[n][k]
        *reinterpret_cast<vec_t*>(&Bs[buf][r][c]) = rb[e];
      }
    }
  };

  // FP64 tiles with beta != 0 (among them the tridiagonalisation's trailing
  // updates, inner dimension 64): the C tile is loaded before the k-loop, so
  // its read does not wait behind the MFMA work in the epilogue
  constexpr bool CPRE = sizeof(T) == 8 && sizeof(CT) == 8 && TM * TN <= 4;
  CT cpre[CPRE ? TM : 1][CPRE ? TN : 1][4];
  const bool pre = CPRE && g.beta != 0.0;
  if (CPRE && pre) {
#pragma unroll
    for (int a = 0; a < (CPRE ? TM : 1); ++a)
#pragma unroll
      for (int b = 0; b < (CPRE ? TN : 1); ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rr = (sizeof(T) == 8) ? (4 * r + lk) : (lk * 4 + r);
          const int row = m0 + wm * TM * 16 + a * 16 + rr;
          const int col = n0 + wn * TN * 16 + b * 16 + li;
          cpre[a][b][r] = (row < M && col < N) ? C[(long long)row * g.ldc + col] : CT(0);
        }
  }

  load_regs(0);
  store_regs(0);
  __syncthreads();
  int cur = 0;
  for (int k0 = 0; k0 < K; k0 += BK) {
    const bool more = k0 + BK < K;
    if (more) load_regs(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      T fa[TM][4], fb[TN][4];
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        const int row = wm * TM * 16 + a * 16 + li;
#pragma unroll
        for (int t = 0; t < 4; ++t) fa[a][t] = TA ? As[cur][kk + lk * 4 + t][row] : As[cur][row][kk + lk * 4 + t];
      }
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        const int col = wn * TN * 16 + b * 16 + li;
#pragma unroll
        for (int t = 0; t < 4; ++t) fb[b][t] = TB ? Bs[cur][col][kk + lk * 4 + t] : Bs[cur][kk + lk * 4 + t][col];
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int b = 0; b < TN; ++b) acc[a][b] = Mfma<T>::op(fa[a][t], fb[b][t], acc[a][b]);
    }
    if (more) store_regs(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }

  const T alpha = T(g.alpha), beta = T(g.beta);
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = (sizeof(T) == 8) ? (4 * r + lk) : (lk * 4 + r);
        const int row = m0 + wm * TM * 16 + a * 16 + rr;
        const int col = n0 + wn * TN * 16 + b * 16 + li;
        if (row < M && col < N) {
          const long long off = (long long)row * g.ldc + col;
          T v = alpha * acc[a][b][r];
          if (g.beta != 0.0) {
            T cold;
            if constexpr (CPRE) cold = (T)cpre[CPRE ? a : 0][CPRE ? b : 0][r];
            else cold = (T)C[off];
            v += beta * cold;
          }
          C[off] = (CT)v;
        }
      }
}

// ---------------------------------------------------------------------------
// split-BF16x3 kernel: FP32 operands, x = hi + lo with hi = bf16(x) and
// lo = bf16(x - hi); C += Ahi*Bhi + Ahi*Blo + Alo*Bhi with FP32 accumulation.
// The split happens once per element when the tile is written to LDS.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void split_bf16(float x, __bf16& hi, __bf16& lo) {
  hi = (__bf16)x;
  lo = (__bf16)(x - (float)hi);
}

template <bool CX, int TM, int TN, bool TA, bool TB, int TAG>
__global__ __launch_bounds__(256) void gemm_bf16x3_k(const float* __restrict__ A, const float* __restrict__ B,
                                                     float* __restrict__ C, GemmArgs g) {
  constexpr int BM = 32 * TM, BN = 32 * TN, BK = 32;
  constexpr int PAD = 8;
  constexpr int NP = CX ? 2 : 1;
  constexpr int LA = BM * BK / 256, LB = BN * BK / 256;

  __shared__ __bf16 Ah[NP][BM][BK + PAD], Al[NP][BM][BK + PAD];
  __shared__ __bf16 Bh[NP][BN][BK + PAD], Bl[NP][BN][BK + PAD];

  const long long bz = blockIdx.z;
  A += bz * g.sA;
  B += bz * g.sB;
  C += bz * g.sC;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lk = lane >> 4;
  const int M = g.M, N = g.N, K = g.K;

  flt4 acc[NP][TM][TN];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b) acc[p][a][b] = flt4{0, 0, 0, 0};

  float ra[NP][LA], rb[NP][LB];
  const float sgnA = (CX && g.conjA) ? -1.f : 1.f;
  const float sgnB = (CX && g.conjB) ? -1.f : 1.f;

  auto load_regs = [&](int k0) {
#pragma unroll
    for (int e = 0; e < LA; ++e) {
      int idx = tid + 256 * e;
      int r, c;
      if (!TA) { r = idx / BK; c = idx % BK; } else { c = idx / BM; r = idx % BM; }
      int gm = m0 + r, gk = k0 + c;
      bool ok = (gm < M) && (gk < K);
      long long off = TA ? (long long)gk * g.lda + gm : (long long)gm * g.lda + gk;
#pragma unroll
      for (int p = 0; p < NP; ++p) ra[p][e] = ok ? A[off + p * g.pA] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < LB; ++e) {
      int idx = tid + 256 * e;
      int r, c;
      if (!TB) { c = idx / BN; r = idx % BN; } else { r = idx / BK; c = idx % BK; }
      int gn = n0 + r, gk = k0 + c;
      bool ok = (gn < N) && (gk < K);
      long long off = TB ? (long long)gn * g.ldb + gk : (long long)gk * g.ldb + gn;
#pragma unroll
      for (int p = 0; p < NP; ++p) rb[p][e] = ok ? B[off + p * g.pB] : 0.f;
    }
  };
  auto store_regs = [&]() {
#pragma unroll
    for (int e = 0; e < LA; ++e) {
      int idx = tid + 256 * e;
      int r, c;
      if (!TA) { r = idx / BK; c = idx % BK; } else { c = idx / BM; r = idx % BM; }
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        float x = (p == 1) ? sgnA * ra[p][e] : ra[p][e];
        __bf16 h, l;
        split_bf16(x, h, l);
        Ah[p][r][c] = h;
        Al[p][r][c] = l;
      }
    }
#pragma unroll
    for (int e = 0; e < LB; ++e) {
      int idx = tid + 256 * e;
      int r, c;
      if (!TB) { c = idx / BN; r = idx % BN; } else { r = idx / BK; c = idx % BK; }
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        float x = (p == 1) ? sgnB * rb[p][e] : rb[p][e];
        __bf16 h, l;
        split_bf16(x, h, l);
        Bh[p][r][c] = h;
        Bl[p][r][c] = l;
      }
    }
  };

  load_regs(0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    store_regs();
    __syncthreads();
    if (k0 + BK < K) load_regs(k0 + BK);
    bf16x8 ah[NP][TM], al[NP][TM], bh[NP][TN], bl[NP][TN];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        int row = wm * TM * 16 + a * 16 + li;
        ah[p][a] = *reinterpret_cast<const bf16x8*>(&Ah[p][row][lk * 8]);
        al[p][a] = *reinterpret_cast<const bf16x8*>(&Al[p][row][lk * 8]);
      }
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        int row = wn * TN * 16 + b * 16 + li;
        bh[p][b] = *reinterpret_cast<const bf16x8*>(&Bh[p][row][lk * 8]);
        bl[p][b] = *reinterpret_cast<const bf16x8*>(&Bl[p][row][lk * 8]);
      }
    }
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        if (!CX) {
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[0][a], bh[0][b], acc[0][a][b], 0, 0, 0);
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[0][a], bl[0][b], acc[0][a][b], 0, 0, 0);
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[0][a], bh[0][b], acc[0][a][b], 0, 0, 0);
        } else {
          bf16x8 nah = -ah[1][a], nal = -al[1][a];
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[0][a], bh[0][b], acc[0][a][b], 0, 0, 0);
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[0][a], bl[0][b], acc[0][a][b], 0, 0, 0);
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[0][a], bh[0][b], acc[0][a][b], 0, 0, 0);
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(nal, bh[1][b], acc[0][a][b], 0, 0, 0);
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(nah, bl[1][b], acc[0][a][b], 0, 0, 0);
          acc[0][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(nah, bh[1][b], acc[0][a][b], 0, 0, 0);
          acc[1][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[0][a], bh[1][b], acc[1][a][b], 0, 0, 0);
          acc[1][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[0][a], bl[1][b], acc[1][a][b], 0, 0, 0);
          acc[1][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[0][a], bh[1][b], acc[1][a][b], 0, 0, 0);
          acc[1][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[1][a], bh[0][b], acc[1][a][b], 0, 0, 0);
          acc[1][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[1][a], bl[0][b], acc[1][a][b], 0, 0, 0);
          acc[1][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[1][a], bh[0][b], acc[1][a][b], 0, 0, 0);
        }
      }
    __syncthreads();
  }

  const float alpha = (float)g.alpha, beta = (float)g.beta;
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int row = m0 + wm * TM * 16 + a * 16 + lk * 4 + r;
        int col = n0 + wn * TN * 16 + b * 16 + li;
        if (row < M && col < N) {
          long long off = (long long)row * g.ldc + col;
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            float v = alpha * acc[p][a][b][r];
            if (g.beta != 0.0) v += beta * C[off + p * g.pC];
            C[off + p * g.pC] = v;
          }
        }
      }
}

// ---------------------------------------------------------------------------
// split-BF16x3 kernel on pre-split operands: C[m][n] = sum_k A[m][k] B[n][k]
// with A and B each given as a (hi, lo) pair of bf16 arrays whose rows are
// k-contiguous (row pitches multiples of 8 elements, 16-byte aligned), so
// every global load and every LDS store is a 16-byte vector and each MFMA
// operand fragment (8 consecutive k) is one 16-byte LDS read.  The split
// happens once per element outside the GEMM (environments once per bond,
// theta once per apply, the MPO pass writes T2 split).  128x128 block tile,
// BK = 32 (one v_mfma_f32_16x16x32_bf16 k-step), double-buffered LDS with
// one barrier per k-step, XCD-aware tile order; C is FP32.
// ---------------------------------------------------------------------------
struct B3Args {
  int M, N, K, lda, ldb, ldc;
};

template <int TM, int TN, int TAG>
__global__ __launch_bounds__(256) void gemm_b3nt_k(const __bf16* __restrict__ Ah, const __bf16* __restrict__ Al,
                                                   const __bf16* __restrict__ Bh, const __bf16* __restrict__ Bl,
                                                   float* __restrict__ C, B3Args g) {
  constexpr int BM = 32 * TM, BN = 32 * TN, BK = 32, LDK = BK + 8;   // row pitch 80 bytes
  constexpr int NA = BM * BK / (8 * 256), NB = BN * BK / (8 * 256); // 16-byte vectors per thread
  __shared__ __attribute__((aligned(16))) __bf16 sAh[2][BM][LDK], sAl[2][BM][LDK];
  __shared__ __attribute__((aligned(16))) __bf16 sBh[2][BN][LDK], sBl[2][BN][LDK];
  int tr, tc;
  xcd_tile(gridDim.x, gridDim.y, tr, tc);
  const int m0 = tr * BM, n0 = tc * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 15, lk = lane >> 4;
  const int M = g.M, N = g.N, K = g.K;
  flt4 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = flt4{0.f, 0.f, 0.f, 0.f};
  bf16x8 rah[NA], ral[NA], rbh[NB], rbl[NB];
  const bf16x8 zero8 = bf16x8{};
  auto load = [&](int k0) {
#pragma unroll
    for (int e = 0; e < NA; ++e) {
      const int v = tid + 256 * e, r = v / (BK / 8), c = (v % (BK / 8)) * 8;
      const int gm = m0 + r, gk = k0 + c;
      if (gm < M && gk < K) {   // the row pitch covers the vector; k >= K is masked
        const long long off = (long long)gm * g.lda + gk;
        rah[e] = *reinterpret_cast<const bf16x8*>(Ah + off);
        ral[e] = *reinterpret_cast<const bf16x8*>(Al + off);
        if (gk + 8 > K) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (gk + j >= K) { rah[e][j] = (__bf16)0.f; ral[e][j] = (__bf16)0.f; }
        }
      } else {
        rah[e] = zero8;
        ral[e] = zero8;
      }
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int v = tid + 256 * e, r = v / (BK / 8), c = (v % (BK / 8)) * 8;
      const int gn = n0 + r, gk = k0 + c;
      if (gn < N && gk < K) {
        const long long off = (long long)gn * g.ldb + gk;
        rbh[e] = *reinterpret_cast<const bf16x8*>(Bh + off);
        rbl[e] = *reinterpret_cast<const bf16x8*>(Bl + off);
        if (gk + 8 > K) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (gk + j >= K) { rbh[e][j] = (__bf16)0.f; rbl[e][j] = (__bf16)0.f; }
        }
      } else {
        rbh[e] = zero8;
        rbl[e] = zero8;
      }
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int e = 0; e < NA; ++e) {
      const int v = tid + 256 * e, r = v / (BK / 8), c = (v % (BK / 8)) * 8;
      *reinterpret_cast<bf16x8*>(&sAh[buf][r][c]) = rah[e];
      *reinterpret_cast<bf16x8*>(&sAl[buf][r][c]) = ral[e];
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int v = tid + 256 * e, r = v / (BK / 8), c = (v % (BK / 8)) * 8;
      *reinterpret_cast<bf16x8*>(&sBh[buf][r][c]) = rbh[e];
      *reinterpret_cast<bf16x8*>(&sBl[buf][r][c]) = rbl[e];
    }
  };
  load(0);
  store(0);
  __syncthreads();
  int cur = 0;
  for (int k0 = 0; k0 < K; k0 += BK) {
    const bool more = k0 + BK < K;
    if (more) load(k0 + BK);
    bf16x8 ah[TM], al[TM], bh[TN], bl[TN];
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      const int row = wm * TM * 16 + a * 16 + li;
      ah[a] = *reinterpret_cast<const bf16x8*>(&sAh[cur][row][lk * 8]);
      al[a] = *reinterpret_cast<const bf16x8*>(&sAl[cur][row][lk * 8]);
    }
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      const int col = wn * TN * 16 + b * 16 + li;
      bh[b] = *reinterpret_cast<const bf16x8*>(&sBh[cur][col][lk * 8]);
      bl[b] = *reinterpret_cast<const bf16x8*>(&sBl[cur][col][lk * 8]);
    }
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[a], bh[b], acc[a][b], 0, 0, 0);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a], bl[b], acc[a][b], 0, 0, 0);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a], bh[b], acc[a][b], 0, 0, 0);
      }
    if (more) store(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm * TM * 16 + a * 16 + lk * 4 + r;
        const int col = n0 + wn * TN * 16 + b * 16 + li;
        if (row < M && col < N) C[(long long)row * g.ldc + col] = acc[a][b][r];
      }
}

template <int TM, int TN>
static void launch_b3nt(Ctx* c, dim3 grid, int tag, const __bf16* Ah, const __bf16* Al, const __bf16* Bh,
                        const __bf16* Bl, float* C, const B3Args& g) {
  if (tag == 1) gemm_b3nt_k<TM, TN, 1><<<grid, 256, 0, c->stream>>>(Ah, Al, Bh, Bl, C, g);
  else if (tag == 2) gemm_b3nt_k<TM, TN, 2><<<grid, 256, 0, c->stream>>>(Ah, Al, Bh, Bl, C, g);
  else gemm_b3nt_k<TM, TN, 0><<<grid, 256, 0, c->stream>>>(Ah, Al, Bh, Bl, C, g);
}

void gemm_b3nt(Ctx* c, int M, int N, int K, const __bf16* Ah, const __bf16* Al, int lda, const __bf16* Bh,
               const __bf16* Bl, int ldb, float* C, int ldc, int tag) {
  DMRG_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_b3nt: bad sizes");
  DMRG_REQUIRE(lda % 8 == 0 && ldb % 8 == 0 && lda >= K && ldb >= K, "gemm_b3nt: pitches must be multiples of 8");
  auto al = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  DMRG_REQUIRE(al(Ah) && al(Al) && al(Bh) && al(Bl), "gemm_b3nt: operands must be 16-byte aligned");
  B3Args g{M, N, K, lda, ldb, ldc};
  const long long tiles128 = (long long)((M + 127) / 128) * ((N + 127) / 128);
  if (tiles128 >= 256) {
    dim3 grid((N + 127) / 128, (M + 127) / 128);
    DMRG_REQUIRE(grid.y <= 65535, "gemm_b3nt: M too large");
    launch_b3nt<4, 4>(c, grid, tag, Ah, Al, Bh, Bl, C, g);
  } else {
    dim3 grid((N + 63) / 64, (M + 63) / 64);
    DMRG_REQUIRE(grid.y <= 65535, "gemm_b3nt: M too large");
    launch_b3nt<2, 2>(c, grid, tag, Ah, Al, Bh, Bl, C, g);
  }
  DMRG_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// host dispatch
// ---------------------------------------------------------------------------
static void check_desc(const GemmDesc& d) {
  DMRG_REQUIRE(d.M >= 0 && d.N >= 0 && d.K >= 0 && d.batch >= 1, "gemm: negative size");
  DMRG_REQUIRE(d.batch <= 65535, "gemm: batch too large");
  DMRG_REQUIRE(d.M <= 65535 * (d.field == CPLX ? 64 : 128), "gemm: M too large for one launch");
  DMRG_REQUIRE(d.ldc >= d.N || d.M <= 1, "gemm: ldc < N");
  DMRG_REQUIRE(d.transA ? (d.lda >= d.M || d.K <= 1) : (d.lda >= d.K || d.M <= 1), "gemm: bad lda");
  DMRG_REQUIRE(d.transB ? (d.ldb >= d.K || d.N <= 1) : (d.ldb >= d.N || d.K <= 1), "gemm: bad ldb");
}

// Launch helpers: pick the instantiation for (transA, transB, tag).
template <typename T, int TM, int TN, bool TA, bool TB>
static void launch_fast_tagged(Ctx* c, const GemmDesc& d, const T* A, const T* B, T* C) {
  const GemmArgs g = make_args(d, 32 * TM, 32 * TN);
  const dim3 grid((unsigned)g.nbx * g.nby, 1, d.batch);
  switch (d.tag) {
#define CASE(t) \
  case t: gemm_fast<T, TM, TN, TA, TB, t><<<grid, 256, 0, c->stream>>>(A, B, C, g); break;
    DMRG_GEMM_TAGS(CASE)
#undef CASE
    default: throw Error("gemm: bad tag");
  }
  DMRG_CHECK_HIP(hipGetLastError());
}

template <typename T, int TM, int TN, typename CT = T>
static void launch_fast(Ctx* c, const GemmDesc& d, const T* A, const T* B, CT* C) {
  if constexpr (!std::is_same<T, CT>::value) {   // gemm_f32_c64
    const GemmArgs g = make_args(d, 32 * TM, 32 * TN);
    gemm_fast<T, TM, TN, false, false, 2, CT><<<dim3((unsigned)g.nbx * g.nby, 1, d.batch), 256, 0, c->stream>>>(A, B, C, g);
    DMRG_CHECK_HIP(hipGetLastError());
  } else if (!d.transA && !d.transB) launch_fast_tagged<T, TM, TN, false, false>(c, d, A, B, C);
  else if (d.transA && !d.transB) launch_fast_tagged<T, TM, TN, true, false>(c, d, A, B, C);
  else if (!d.transA && d.transB) launch_fast_tagged<T, TM, TN, false, true>(c, d, A, B, C);
  else launch_fast_tagged<T, TM, TN, true, true>(c, d, A, B, C);
}

// Which kernel a real product takes.  The LDS kernel runs square tiles
// of 64 (FP32 also 96 and 128); products whose 64 x 64 tiles would leave the 256 CUs idle
// or badly balanced go to the direct-load kernel (gemm_direct.hip), which
// spreads 16 x 16 / 32 x 32 tiles and splits the inner dimension.  Measured
// (LDS 64 x 64 / direct, us):
//   FP64  760 x 187 x 935 (36 tiles) 54 / 18;  1024 x 256 x 1280 (64) 70 / 24;
//         650^3 (121) 40 / 24;  950 x 748 x 190 (180) 15.0 / 15.7;
//         650 x 2000 x 128 (352) 15.4 / 16.5;  1280 x 1024 x 256 (320) 25.9 / 24.7;
//         650 x 2588 x 2612 (451) 215 / 203;  6400 x 400 x 2400 (700) 285 / 293;
//         3000 x 3000 x 512 (2209) 184 / 213
//   FP32  4800 x 300 x 1800 (375) 80 / 93;  131 x 1 x 200 (3) 8.6 / 5.1
// so FP64 changes at 512 tiles (160 for short inner dimensions, where a
// workgroup has little to hide), FP32 at 200.
static bool use_direct(const GemmDesc& d, bool f64) {
  const long long tiles64 = (long long)((d.M + 63) / 64) * ((d.N + 63) / 64) * d.batch;
  return tiles64 < (f64 ? (d.K <= 200 ? 160 : 512) : 200);
}

// FP32 tile of the LDS kernel: 128, 96 or 64 square, whichever is estimated
// fastest: rounds of the 256 CUs x tile area x the time per area and k, which
// measured 4.2 / 4.45 / 4.75 e-6 us (smaller tiles read LDS more per MFMA);
// a single round (two of 64 x 64) has too few workgroups per CU to hide its
// loads and measured 1.1 / 1.25 / 1.17 times that.  Measured (us, 128 / 96 / 64):
//   857 x 857 x 3380 x 6     464 / 280 / 323     1500^3               114 / 75 / 92
//   5070 x 3428 x 845        291 / 273 / 279     2200 x 2200 x 1100   150 / 135 / 110
//   10448 x 731 x 4386       579 / 685 / 662     700 x 700 x 2800 x 6 224 / 231 / 166
//   6144 x 16384 x 1024     1581 / 1663 / 1837   4800 x 300 x 1800    136 / 90 / 82
static int fast_tile(const GemmDesc& d) {
  auto cost = [&](int tile, double per_area, int few, double penalty) {
    const long long t = (long long)((d.M + tile - 1) / tile) * ((d.N + tile - 1) / tile) * d.batch;
    const long long rounds = (t + 255) / 256;
    return (double)rounds * tile * tile * per_area * (rounds <= few ? penalty : 1.0);
  };
  const double c128 = cost(128, 1.0, 1, 1.1), c96 = cost(96, 1.07, 1, 1.25), c64 = cost(64, 1.14, 2, 1.17);
  return c128 <= c96 && c128 <= c64 ? 128 : (c96 <= c64 ? 96 : 64);
}

template <typename CT>
static void launch_fast_f32(Ctx* c, const GemmDesc& d, const float* A, const float* B, CT* C) {
  switch (fast_tile(d)) {
    case 128: launch_fast<float, 4, 4, CT>(c, d, A, B, C); break;
    case 96: launch_fast<float, 3, 3, CT>(c, d, A, B, C); break;
    default: launch_fast<float, 2, 2, CT>(c, d, A, B, C);
  }
}

// Real FP32 GEMM writing an FP64 result: the R-step of the FP32 H_eff apply
// writes y straight into the FP64 Krylov vector, with no conversion pass.
// Built for that caller only (no transposes, tag 2).
void gemm_f32_c64(Ctx* c, const GemmDesc& d, const float* A, const float* B, double* C) {
  DMRG_REQUIRE(d.field == REAL && d.beta == 0.0 && !d.transA && !d.transB && d.tag == 2,
               "gemm_f32_c64: real field, beta = 0, no transposes and tag 2 only");
  check_desc(d);
  if (d.M == 0 || d.N == 0) return;
  if (use_direct(d, false)) gemm_direct_f32_c64(c, d, A, B, C);
  else launch_fast_f32(c, d, A, B, C);
}

void gemm_f64(Ctx* c, const GemmDesc& d, const double* A, const double* B, double* C) {
  check_desc(d);
  if (d.M == 0 || d.N == 0) return;
  if (d.field == CPLX || use_direct(d, true)) gemm_direct_f64(c, d, A, B, C);
  else launch_fast<double, 2, 2>(c, d, A, B, C);
}

void gemm_f32(Ctx* c, const GemmDesc& d, const float* A, const float* B, float* C) {
  check_desc(d);
  if (d.M == 0 || d.N == 0) return;
  if (d.field == CPLX || use_direct(d, false)) gemm_direct_f32(c, d, A, B, C);
  else launch_fast_f32(c, d, A, B, C);
}

// C[i][j] = conj(C[j][i]) for j > i (n x n, row pitch ld, imaginary plane at
// +plane when cx): the strict upper triangle of a Hermitian product computed
// with GemmDesc::lower.  One 32 x 32 tile pair per block: the lower tile
// (J, I) is read coalesced, transposed through LDS and written as (I, J).
__global__ __launch_bounds__(256) void mirror_lower_k(double* __restrict__ C, int n, int ld, long long plane,
                                                      int cx) {
  __shared__ double t[32][33];
  const int I = blockIdx.y, J = blockIdx.x;   // destination tile (I, J), I <= J
  if (I > J) return;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
  for (int pl = 0; pl < (cx ? 2 : 1); ++pl) {
    double* P = C + pl * plane;
    for (int r = ty; r < 32; r += 8) {   // source rows J*32 + r, columns I*32 + tx
      const int sr = J * 32 + r, sc = I * 32 + tx;
      t[r][tx] = (sr < n && sc < n) ? P[(size_t)sr * ld + sc] : 0.0;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {   // destination rows I*32 + r, columns J*32 + tx
      const int dr = I * 32 + r, dc = J * 32 + tx;
      if (dr < n && dc < n && dc > dr) P[(size_t)dr * ld + dc] = pl ? -t[tx][r] : t[tx][r];
    }
    __syncthreads();
  }
}

void mirror_lower(Ctx* c, double* C, int n, int ld, long long plane, int field) {
  if (n <= 1) return;
  const int nt = (n + 31) / 32;
  mirror_lower_k<<<dim3(nt, nt), 256, 0, c->stream>>>(C, n, ld, plane, field == CPLX ? 1 : 0);
  DMRG_CHECK_HIP(hipGetLastError());
}

template <bool CX, int TM, int TN, bool TA, bool TB>
static void launch_b3_tagged(Ctx* c, const GemmDesc& d, const float* A, const float* B, float* C) {
  GemmArgs g = make_args(d, 32 * TM, 32 * TN);
  dim3 grid((d.N + 32 * TN - 1) / (32 * TN), (d.M + 32 * TM - 1) / (32 * TM), d.batch);
  DMRG_REQUIRE(grid.y <= 65535, "gemm: M too large for one launch");
  switch (d.tag) {
#define CASE(t) \
  case t: gemm_bf16x3_k<CX, TM, TN, TA, TB, t><<<grid, 256, 0, c->stream>>>(A, B, C, g); break;
    DMRG_GEMM_TAGS(CASE)
#undef CASE
    default: throw Error("gemm: bad tag");
  }
  DMRG_CHECK_HIP(hipGetLastError());
}

template <bool CX, int TM, int TN>
static void launch_b3_tt(Ctx* c, const GemmDesc& d, const float* A, const float* B, float* C) {
  if (!d.transA && !d.transB) launch_b3_tagged<CX, TM, TN, false, false>(c, d, A, B, C);
  else if (d.transA && !d.transB) launch_b3_tagged<CX, TM, TN, true, false>(c, d, A, B, C);
  else if (!d.transA && d.transB) launch_b3_tagged<CX, TM, TN, false, true>(c, d, A, B, C);
  else launch_b3_tagged<CX, TM, TN, true, true>(c, d, A, B, C);
}

void gemm_bf16x3(Ctx* c, const GemmDesc& d, const float* A, const float* B, float* C) {
  check_desc(d);
  if (d.M == 0 || d.N == 0) return;
  long long tiles128 = (long long)((d.M + 127) / 128) * ((d.N + 127) / 128) * d.batch;
  if (d.field == CPLX) {
    long long tiles64 = (long long)((d.M + 63) / 64) * ((d.N + 63) / 64) * d.batch;
    if (tiles64 >= 512) launch_b3_tt<true, 2, 2>(c, d, A, B, C);
    else launch_b3_tt<true, 1, 1>(c, d, A, B, C);
  } else {
    if (tiles128 >= 256) launch_b3_tt<false, 4, 4>(c, d, A, B, C);
    else launch_b3_tt<false, 2, 2>(c, d, A, B, C);
  }
}

}  // namespace dmrg
