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
// function to the bit), one wave a block so that 128 tiles reach 128 CUs.  The
// gradients' longer sums (K = outputs or batch rows) are split: a block's
// four waves take the K steps w, w + 4, ... of one tile and are added through
// LDS in wave order (deterministic).  The epilogue does what would be further launches: bias,
// GELU, the loss and its gradient, GELU', the bias gradient (row sums of the
// FP32 A operand) and Adam.  A training step of batch 512 is 6 launches
// instead of 17.
//
// v_mfma_f32_16x16x32_bf16: lane l holds A[l%16][8(l/16) .. +7] and
// B[8(l/16) .. +7][l%16]; output register r holds D[4(l/16) + r][l%16].
// Operands are rounded to bfloat16 (nearest even) as they are loaded.
constexpr int kTile = 32, kStep = 32;

template <int V>
struct Int {
  static constexpr int value = V;
};

typedef float F4u __attribute__((ext_vector_type(4), aligned(4)));

// Eight consecutive k of one row r (k contiguous): two 16-byte loads where
// the whole step is inside K, else masked elements.
template <bool WHOLE>
__device__ __forceinline__ void load_rowk(const float* p, int k, int K, float* v) {
  if constexpr (WHOLE) {
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
template <bool WHOLE>
__device__ __forceinline__ void load_colk(const float* base, long long ld, const int* rows,
                                          int c, int k, int K, float* v) {
  int kk[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) kk[e] = WHOLE ? k + e : min(k + e, K - 1);
  if (rows) {
#pragma unroll
    for (int e = 0; e < 8; ++e) kk[e] = rows[kk[e]];
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = base[(long long)kk[e] * ld + c];
    v[e] = WHOLE || k + e < K ? x : 0.f;
  }
}

__device__ __forceinline__ bf16x8 pack8(const float* v) {
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (__bf16)v[e];
  return r;
}

struct AdamIn {
  float p, m, v;
};
__device__ __forceinline__ AdamIn adam_load(const float* p, const float* m, const float* v,
                                            long long o) {
  return AdamIn{p[o], m[o], v[o]};
}
__device__ __forceinline__ void adam_one(float* p, float* m, float* v, long long o, float g,
                                         const AdamIn& x, const AdamArgs& a) {
  const float mi = a.beta1 * x.m + (1.f - a.beta1) * g;
  const float vi = a.beta2 * x.v + (1.f - a.beta2) * g * g;
  m[o] = mi;
  v[o] = vi;
  p[o] = x.p - a.lr_t * mi / (sqrtf(vi) + a.eps_t);
}

template <int EPI>
__device__ __forceinline__ void product(const GemmArgs& g, int block, const AdamArgs& adam) {
  constexpr bool kSplit = EPI > kMseGrad;
  constexpr int kWaves = kSplit ? 4 : 1;
  __shared__ float part[kWaves][kTile][kTile + 1];
  __shared__ float bsum[kWaves][4][kTile];
  constexpr bool kAk = EPI != kWeight;                 // A rows contiguous along k
  constexpr bool kBk = EPI <= kMseGrad;                // B columns contiguous along k
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, c = lane & 15;
  const int tj = (g.N + kTile - 1) / kTile;
  const int i0 = block / tj * kTile, j0 = block % tj * kTile;
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
  // Epilogue: thread t takes column t % 32 of rows t / 32, + 8, ... (its
  // wave's own tile: lane / 32, + 2, ...).  Its operands are loaded before
  // the K loop (clamped inside the matrices, unused there).
  constexpr int kRows = kSplit ? 4 : 16;
  const int col = tid & 31, j = j0 + col, jc = min(j, g.N - 1);
  int ie[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r)
    ie[r] = min(i0 + (kSplit ? (tid >> 5) + 8 * r : (lane >> 5) + 2 * r), g.M - 1);
  float in[kRows], bias = 0.f;
  AdamIn ad[kRows], adb{0.f, 0.f, 0.f};
  if constexpr (EPI <= kMseGrad) bias = g.bias[jc];
  if constexpr (EPI == kMseGrad) {
    int row[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) row[r] = g.rows ? g.rows[ie[r]] : ie[r];
#pragma unroll
    for (int r = 0; r < kRows; ++r) in[r] = g.T[(long long)row[r] * g.N + jc];
  }
  if constexpr (EPI == kGeluGrad) {
#pragma unroll
    for (int r = 0; r < kRows; ++r) in[r] = g.Z[(long long)ie[r] * g.ldc + jc];
  }
  if constexpr (EPI == kWeight) {
    if (g.p) {
#pragma unroll
      for (int r = 0; r < kRows; ++r)
        ad[r] = adam_load(g.p, g.m, g.v, (long long)ie[r] * g.ldc + jc);
      adb = adam_load(g.bp, g.bm, g.bv, min(i0 + (tid & 31), g.M - 1));
    }
  }
  floatx4 acc[2][2];
  float rs[2] = {0.f, 0.f};
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = (floatx4){0.f, 0.f, 0.f, 0.f};
  // `count` K steps from st, all their loads in flight before the first use.
  constexpr int kInc = kSplit ? 4 : 1;
  auto steps = [&](int st, auto count, auto whole) {
    constexpr int kCount = decltype(count)::value;
    constexpr bool kWhole = decltype(whole)::value;
    float va[kCount][2][8], vb[kCount][2][8];
#pragma unroll
    for (int u = 0; u < kCount; ++u) {
      const int k = (st + u * kInc) * kStep + 8 * q;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if constexpr (kAk) load_rowk<kWhole>(pa[t], k, g.K, va[u][t]);
        else load_colk<kWhole>(g.A, g.lda, nullptr, ri[t], k, g.K, va[u][t]);
        if constexpr (kBk) load_rowk<kWhole>(pb[t], k, g.K, vb[u][t]);
        else load_colk<kWhole>(g.B, g.ldb, EPI == kWeight ? g.rows : nullptr, cj[t], k, g.K,
                               vb[u][t]);
      }
    }
#pragma unroll
    for (int u = 0; u < kCount; ++u) {
      bf16x8 fa[2], fb[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if constexpr (EPI == kWeight) {
#pragma unroll
          for (int e = 0; e < 8; ++e) rs[t] += va[u][t][e];
        }
        fa[t] = pack8(va[u][t]);
        fb[t] = pack8(vb[u][t]);
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
    }
  };
  const int nwhole = g.K / kStep;
  int st = kSplit ? wave : 0;
  for (; st + 3 * kInc < nwhole; st += 4 * kInc) steps(st, Int<4>{}, Int<1>{});
  if (st + kInc < nwhole) {
    steps(st, Int<2>{}, Int<1>{});
    st += 2 * kInc;
  }
  if (st < nwhole) {
    steps(st, Int<1>{}, Int<1>{});
    st += kInc;
  }
  if (g.K % kStep != 0 && st == nwhole) steps(st, Int<1>{}, Int<0>{});
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
  double loss = 0;
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const int row = kSplit ? (tid >> 5) + 8 * r : (lane >> 5) + 2 * r;
    float x = part[0][row][col];
    if constexpr (kSplit)
      x = ((x + part[1][row][col]) + part[2][row][col]) + part[3][row][col];
    const long long o = (long long)ie[r] * g.ldc + jc;
    const bool ok = i0 + row < g.M && j < g.N;
    if constexpr (EPI == kBias) {
      if (ok) g.C[o] = x + bias;
    } else if constexpr (EPI == kGelu) {
      x += bias;
      const float h = gelu(x);
      if (ok) {
        g.Z[o] = x;
        g.C[o] = h;
      }
    } else if constexpr (EPI == kMseGrad) {
      const float d = x + bias - in[r];
      if (ok) {
        g.C[o] = g.scale * d;
        loss += (double)d * d;
      }
    } else if constexpr (EPI == kGeluGrad) {
      const float d = x * gelu_grad(in[r]);
      if (ok) g.C[o] = d;
    } else {
      if (ok) {
        if (g.p) adam_one(g.p, g.m, g.v, o, x, ad[r], adam);
        else g.C[o] = x;
      }
    }
  }
  if constexpr (EPI == kWeight) {
    if (j0 == 0 && tid < kTile && i0 + tid < g.M) {
      float x = 0.f;
      for (int w = 0; w < 4; ++w)
        for (int u = 0; u < 4; ++u) x += bsum[w][u][tid];
      if (g.bp) adam_one(g.bp, g.bm, g.bv, i0 + tid, x, adb, adam);
      else g.bias_out[i0 + tid] = x;
    }
  }
  if constexpr (EPI == kMseGrad) {
    for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
    if (lane == 0) g.partial[block] = loss;
  }
}

template <int EPI>
__global__ void __launch_bounds__(EPI > kMseGrad ? 256 : 64) gemm_bf16(GemmArgs g) {
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

int LayerBlocks(int M, int N) { return Tiles(M, N); }

hipError_t LaunchLayer(const mlp::GemmArgs& g, mlp::Epilogue e, hipStream_t s) {
  const dim3 grid(LayerBlocks(g.M, g.N)), block(64);
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
