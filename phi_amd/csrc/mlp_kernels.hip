// Kernels of the truncation-closure network (gfx950): bfloat16 matrix-core
// products with float32 accumulation whose epilogues are GELU, the
// squared-error loss, the gradients and Adam.
//
// Storage: float32 everywhere in HBM (weights (out, in) row-major,
// activations (batch, features) row-major); operands are rounded to bfloat16
// (nearest even) when loaded, products accumulate in float32.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mlp_act.h"
#include "mlp_kernels.h"

namespace phi {
namespace mlp {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

using act::gelu;
using act::gelu_grad;

// --- Products ----------------------------------------------------------------------
// The network's products are small (512 x 256 x 105 up to 686 x 256 x 512):
// what bounds them is latency and launches, not the matrix cores (a training
// step's 0.8 GFLOP is under 1 us of them) or bytes (all operands stay in L2).
// So a wave takes a 32 x 32 tile straight from global memory into MFMA
// fragments, with no LDS and no barrier in the loop.  The layers accumulate
// over K in order (the fused closure pass does, and evaluates the same
// function to the bit): a block's four waves own four tiles.  The gradients'
// longer sums (K = outputs or batch rows) are split: the four waves take the
// K steps w, w + 4, ... of one tile and are added through LDS in wave order
// (deterministic).  The epilogue does what would be further launches: bias,
// GELU, the loss and its gradient, GELU', the bias gradient (row sums of the
// FP32 A operand) and Adam.  A training step of batch 512 is 6 launches
// instead of 17.
//
// v_mfma_f32_16x16x32_bf16: lane l holds A[l%16][8(l/16) .. +7] and
// B[8(l/16) .. +7][l%16]; output register r holds D[4(l/16) + r][l%16].
// Operands are rounded to bfloat16 (nearest even) as they are loaded.
constexpr int kTile = 32, kStep = 32;

typedef float F4u __attribute__((ext_vector_type(4), aligned(4)));

// Eight consecutive k of one row r (k contiguous): two 16-byte loads where
// the whole step is inside K, else masked elements.
__device__ __forceinline__ void load_rowk(const float* p, int k, int K, bool whole, float* v) {
  if (whole) {
    const F4u a = *reinterpret_cast<const F4u*>(p + k);
    const F4u b = *reinterpret_cast<const F4u*>(p + k + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = p[min(k + e, K - 1)];
      v[e] = k + e < K ? x : 0.f;
    }
  }
}

// Eight consecutive k of one column c (k strided by ld; rows gathers them).
__device__ __forceinline__ void load_colk(const float* base, long long ld, const int* rows,
                                          int c, int k, int K, float* v) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int kk = min(k + e, K - 1);
    const float x = base[(long long)(rows ? rows[kk] : kk) * ld + c];
    v[e] = k + e < K ? x : 0.f;
  }
}

__device__ __forceinline__ bf16x8 pack8(const float* v) {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (__bf16)v[e];
  return r;
}

__device__ __forceinline__ void adam_one(float* p, float* m, float* v, long long o, float g,
                                         const AdamArgs& a) {
  const float mi = a.beta1 * m[o] + (1.f - a.beta1) * g;
  const float vi = a.beta2 * v[o] + (1.f - a.beta2) * g * g;
  m[o] = mi;
  v[o] = vi;
  p[o] -= a.lr_t * mi / (sqrtf(vi) + a.eps_t);
}

template <int EPI>
__device__ __forceinline__ void product(const GemmArgs& g, int block, const AdamArgs& adam) {
  __shared__ float part[4][kTile][kTile + 1];
  __shared__ float bsum[4][4][kTile];
  constexpr bool kAk = EPI != kWeight;                 // A rows contiguous along k
  constexpr bool kBk = EPI <= kMseGrad;                // B columns contiguous along k
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, c = lane & 15;
  constexpr bool kSplit = EPI > kMseGrad;
  const int tj = (g.N + kTile - 1) / kTile, tiles = (g.M + kTile - 1) / kTile * tj;
  const int tile = kSplit ? block : min(4 * block + wave, tiles - 1);
  const bool live = kSplit || 4 * block + wave < tiles;
  const int i0 = tile / tj * kTile, j0 = tile % tj * kTile;
  int ri[2], cj[2];
  const float *pa[2], *pb[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    // (rows and columns past the matrices repeat the last one; unused)
    ri[t] = min(i0 + 16 * t + c, g.M - 1);
    cj[t] = min(j0 + 16 * t + c, g.N - 1);
    pa[t] = nullptr;
    pb[t] = nullptr;
    if constexpr (kAk) {
      const bool gather = EPI <= kMseGrad && EPI != kMseGrad && g.rows;
      pa[t] = g.A + (long long)(gather ? g.rows[ri[t]] : ri[t]) * g.lda;
    }
    if constexpr (kBk) pb[t] = g.B + (long long)cj[t] * g.ldb;
  }
  floatx4 acc[2][2];
  float rs[2] = {0.f, 0.f};
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = (floatx4){0.f, 0.f, 0.f, 0.f};
  const int nsteps = (g.K + kStep - 1) / kStep;
#pragma unroll 2
  for (int st = kSplit ? wave : 0; st < nsteps; st += kSplit ? 4 : 1) {
    const int k = st * kStep + 8 * q;
    const bool whole = (st + 1) * kStep <= g.K;
    float va[2][8], vb[2][8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if constexpr (kAk) load_rowk(pa[t], k, g.K, whole, va[t]);
      else load_colk(g.A, g.lda, nullptr, ri[t], k, g.K, va[t]);
      if constexpr (kBk) load_rowk(pb[t], k, g.K, whole, vb[t]);
      else load_colk(g.B, g.ldb, EPI == kWeight ? g.rows : nullptr, cj[t], k, g.K, vb[t]);
    }
    bf16x8 fa[2], fb[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if constexpr (EPI == kWeight) {
#pragma unroll
        for (int e = 0; e < 8; ++e) rs[t] += va[t][e];
      }
      fa[t] = pack8(va[t]);
      fb[t] = pack8(vb[t]);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][16 * a + 4 * q + r][16 * b + c] = acc[a][b][r];
  if constexpr (EPI == kWeight) {
    bsum[wave][q][c] = rs[0];
    bsum[wave][q][16 + c] = rs[1];
  }
  __syncthreads();
  // Epilogue: thread t takes column t % 32 of rows t / 32, + 8, ... (its
  // wave's own tile: lane / 32, + 2, ...)
  const int col = tid & 31, j = j0 + col;
  double loss = 0;
#pragma unroll
  for (int r = 0; r < (kSplit ? 4 : 16); ++r) {
    const int row = kSplit ? (tid >> 5) + 8 * r : (lane >> 5) + 2 * r, i = i0 + row;
    if (!live || i >= g.M || j >= g.N) continue;
    float x = kSplit ? ((part[0][row][col] + part[1][row][col]) + part[2][row][col]) +
                           part[3][row][col]
                     : part[wave][row][col];
    const long long o = (long long)i * g.ldc + j;
    if constexpr (EPI == kBias) {
      g.C[o] = x + g.bias[j];
    } else if constexpr (EPI == kGelu) {
      x += g.bias[j];
      g.Z[o] = x;
      g.C[o] = gelu(x);
    } else if constexpr (EPI == kMseGrad) {
      const float d = x + g.bias[j] - g.T[(long long)(g.rows ? g.rows[i] : i) * g.N + j];
      g.C[o] = g.scale * d;
      loss += (double)d * d;
    } else if constexpr (EPI == kGeluGrad) {
      g.C[o] = x * gelu_grad(g.Z[o]);
    } else {
      if (g.p) adam_one(g.p, g.m, g.v, o, x, adam);
      else g.C[o] = x;
    }
  }
  if constexpr (EPI == kWeight) {
    if (j0 == 0 && tid < kTile && i0 + tid < g.M) {
      float x = 0.f;
      for (int w = 0; w < 4; ++w)
        for (int u = 0; u < 4; ++u) x += bsum[w][u][tid];
      if (g.bp) adam_one(g.bp, g.bm, g.bv, i0 + tid, x, adam);
      else g.bias_out[i0 + tid] = x;
    }
  }
  if constexpr (EPI == kMseGrad) {
    __shared__ double red[4];
    for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
    if (lane == 0) red[wave] = loss;
    __syncthreads();
    if (tid == 0) g.partial[block] = ((red[0] + red[1]) + red[2]) + red[3];
  }
}

template <int EPI>
__global__ void __launch_bounds__(256) gemm_bf16(GemmArgs g) {
  product<EPI>(g, blockIdx.x, AdamArgs{});
}

// Layers' weight gradients, one after the other in the grid.
struct WeightArgs {
  GemmArgs g[3];
  int first[4];
  AdamArgs adam;
};

__global__ void __launch_bounds__(256) weight_grads(WeightArgs w) {
  const int b = blockIdx.x;
  if (b < w.first[1]) product<kWeight>(w.g[0], b, w.adam);
  else if (b < w.first[2]) product<kWeight>(w.g[1], b - w.first[1], w.adam);
  else product<kWeight>(w.g[2], b - w.first[2], w.adam);
}

}  // namespace mlp

// --- Host launchers ---------------------------------------------------------------

static int Tiles(int M, int N) {
  return (M + mlp::kTile - 1) / mlp::kTile * ((N + mlp::kTile - 1) / mlp::kTile);
}

int LayerBlocks(int M, int N) { return (Tiles(M, N) + 3) / 4; }

hipError_t LaunchLayer(const mlp::GemmArgs& g, mlp::Epilogue e, hipStream_t s) {
  const dim3 grid(LayerBlocks(g.M, g.N)), block(256);
  if (e == mlp::kBias)
    hipLaunchKernelGGL(mlp::gemm_bf16<mlp::kBias>, grid, block, 0, s, g);
  else if (e == mlp::kGelu)
    hipLaunchKernelGGL(mlp::gemm_bf16<mlp::kGelu>, grid, block, 0, s, g);
  else if (e == mlp::kMseGrad)
    hipLaunchKernelGGL(mlp::gemm_bf16<mlp::kMseGrad>, grid, block, 0, s, g);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t LaunchInputGrad(const mlp::GemmArgs& g, hipStream_t s) {
  hipLaunchKernelGGL(mlp::gemm_bf16<mlp::kGeluGrad>, dim3(Tiles(g.M, g.N)), dim3(256), 0, s,
                     g);
  return hipGetLastError();
}

hipError_t LaunchWeightGrads(const mlp::GemmArgs* g, int count, const mlp::AdamArgs& adam,
                             hipStream_t s) {
  if (count != 3) return hipErrorInvalidValue;
  mlp::WeightArgs w{};
  w.adam = adam;
  for (int i = 0; i < 3; ++i) {
    w.g[i] = g[i];
    w.first[i + 1] = w.first[i] + Tiles(g[i].M, g[i].N);
  }
  hipLaunchKernelGGL(mlp::weight_grads, dim3(w.first[3]), dim3(256), 0, s, w);
  return hipGetLastError();
}

}  // namespace phi
