// Shared by the GEMM translation units: MFMA wrappers, kernel arguments and
// the launchers of the direct-load kernel (gemm_direct.hip).
#pragma once

#include "dmrg_common.h"

namespace dmrg {

typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <typename T> struct Mfma;
template <> struct Mfma<double> {
  typedef dbl4 acc_t;
  static __device__ __forceinline__ acc_t op(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma<float> {
  typedef flt4 acc_t;
  static __device__ __forceinline__ acc_t op(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// 16-byte vector of T
template <typename T> struct Vec;
template <> struct Vec<float> { typedef flt4 type; static constexpr int W = 4; };
template <> struct Vec<double> { typedef dbl2 type; static constexpr int W = 2; };

struct GemmArgs {
  int M, N, K, lda, ldb, ldc;
  long long sA, sB, sC, pA, pB, pC;
  double alpha, beta;
  int conjA, conjB;
  int lower;   // skip tiles strictly above the diagonal (Hermitian C)
  int nbx, nby;   // output tiles along N and M (the grid is nbx * nby x 1 x batch)
};

inline GemmArgs make_args(const GemmDesc& d, int tm, int tn) {   // tm x tn output tiles
  GemmArgs g;
  g.nbx = (d.N + tn - 1) / tn;
  g.nby = (d.M + tm - 1) / tm;
  g.M = d.M; g.N = d.N; g.K = d.K;
  g.lda = d.lda; g.ldb = d.ldb; g.ldc = d.ldc;
  g.sA = d.sA; g.sB = d.sB; g.sC = d.sC;
  g.pA = d.pA; g.pB = d.pB; g.pC = d.pC;
  g.alpha = d.alpha; g.beta = d.beta;
  g.conjA = d.conjA; g.conjB = d.conjB;
  g.lower = d.lower ? 1 : 0;
  return g;
}

// instantiations per profile tag (GemmDesc::tag)
#define DMRG_GEMM_TAGS(X) X(0) X(1) X(2) X(3) X(4) X(5)

void gemm_direct_f64(Ctx* c, const GemmDesc& d, const double* A, const double* B, double* C);
void gemm_direct_f32(Ctx* c, const GemmDesc& d, const float* A, const float* B, float* C);
void gemm_direct_f32_c64(Ctx* c, const GemmDesc& d, const float* A, const float* B, double* C);

}  // namespace dmrg
