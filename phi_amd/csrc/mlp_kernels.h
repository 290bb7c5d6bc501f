// Launchers of the closure-network kernels (mlp_kernels.hip).
#ifndef PHI_AMD_MLP_KERNELS_H_
#define PHI_AMD_MLP_KERNELS_H_

#include <hip/hip_runtime.h>

namespace phi {
namespace mlp {

// What a product's epilogue does with acc(i, j) = sum_k A(i, k) B(k, j).
enum Epilogue {
  kBias = 0,      // C = acc + bias[j]
  kGelu,          // Z = acc + bias[j], C = GELU(Z)
  kMseGrad,       // d = acc + bias[j] - T(row i, j): C = scale d, loss partials of d^2
  kGeluGrad,      // C = acc GELU'(Z)
  kWeight         // gradient: stored in C, or (p non-null) taken by an Adam step of p
};

struct AdamArgs {
  float lr_t, beta1, beta2, eps_t;  // bias-corrected step sizes
};

// Operands: A(i, k) = A[row(i) * lda + k] (layers and input gradients) or
// A[k * lda + i] (kWeight); B(k, j) = B[j * ldb + k] (layers) or
// B[row(k) * ldb + j] (gradients).  rows (or null for the identity) gathers
// minibatch rows out of a data set: of A for a layer, of B for kWeight, of T
// for kMseGrad.
struct GemmArgs {
  int M, N, K;
  const float* A;
  long long lda;
  const float* B;
  long long ldb;
  float* C;
  long long ldc;
  const int* rows;
  const float* bias;
  float* Z;             // ldc apart
  const float* T;       // kMseGrad: N apart
  float scale;
  double* partial;      // kMseGrad: one sum per block
  float* bias_out;      // kWeight: the bias gradient, sums of A(i, k) over k
  float *p, *m, *v;     // kWeight with Adam: parameters and moments (ldc = N apart)
  float *bp, *bm, *bv;  // the bias'
};

}  // namespace mlp

// Blocks of a layer (one loss partial each for kMseGrad).
int LayerBlocks(int M, int N);
// Layers: kBias, kGelu, kMseGrad.
hipError_t LaunchLayer(const mlp::GemmArgs& g, mlp::Epilogue e, hipStream_t s);
// kGeluGrad: input gradient dZ W through the previous layer's GELU.
hipError_t LaunchInputGrad(const mlp::GemmArgs& g, hipStream_t s);
// kWeight: up to three layers' weight and bias gradients in one launch.
hipError_t LaunchWeightGrads(const mlp::GemmArgs* g, int count, const mlp::AdamArgs& adam,
                             hipStream_t s);

}  // namespace phi

#endif  // PHI_AMD_MLP_KERNELS_H_
