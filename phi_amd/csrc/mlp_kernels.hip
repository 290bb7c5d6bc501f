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
// So (but for large batches or layers: gemm_big) a wave takes a 32 x 32 tile straight from global memory into MFMA
// fragments, with no LDS and no barrier in the loop.  Every product
// accumulates over K in order, whatever the tile (the fused closure pass does,
// and evaluates the same function to the bit; a training run carries each
// bfloat16 rounding on, so another order of the gradients' sums ends 1e-4
// away).  A layer is one wave a block so that 128 tiles reach 128 CUs.  The
// gradients' longer sums (K = outputs or batch rows) take four waves a tile:
// the loads and roundings of 16 K steps are split over the waves, the
// fragments meet in LDS, and each wave accumulates one 16 x 16 quarter over
// all K.  The epilogue does what would be further launches: bias, GELU, the
// loss and its gradient, GELU' and Adam; the bias gradients are blocks of the
// weight gradients' launch.  A training step of batch 512 (105, 256, 256, 686)
// is 6 launches and 50 us of kernels instead of 14 and 171 with a 64 x 64 LDS
// tile and separate epilogues (17 with Adam and the gathers); the gradients'
// split by partial sums instead of loads took the same time.
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
  // (the rounding of the sums written out: left to the compiler, it depends on
  // the code around them)
  const float mi = fmaf(1.f - a.beta1, g, a.beta1 * x.m);
  const float vi = fmaf((1.f - a.beta2) * g, g, a.beta2 * x.v);
  m[o] = mi;
  v[o] = vi;
  p[o] = x.p - a.lr_t * mi / (sqrtf(vi) + a.eps_t);
}

// LDS of a block, 16 bytes each: with four waves the fragments of kChunk K
// steps (A's rows, then B's columns), then the tile's sums.
constexpr int kChunk = 16;
constexpr int kTileLds = (kTile * (kTile + 1) * sizeof(float) + 15) / 16;
constexpr int ProductLds(int epi) { return epi > kMseGrad ? kChunk * 2 * 2 * 64 : kTileLds; }

template <int EPI>
__device__ __forceinline__ void product(const GemmArgs& g, int block, const AdamArgs& adam,
                                        bf16x8* lds) {
  constexpr bool kSplit = EPI > kMseGrad;
  bf16x8 (*frag)[2][2][64] = reinterpret_cast<bf16x8 (*)[2][2][64]>(lds);
  float (*part)[kTile + 1] = reinterpret_cast<float (*)[kTile + 1]>(lds);
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
  AdamIn ad[kRows];
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
    }
  }
  // One K step's operands of rows ri and columns cj.
  auto load = [&](int st, auto whole, float va[2][8], float vb[2][8]) {
    constexpr bool kWhole = decltype(whole)::value;
    const int k = st * kStep + 8 * q;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if constexpr (kAk) load_rowk<kWhole>(pa[t], k, g.K, va[t]);
      else load_colk<kWhole>(g.A, g.lda, nullptr, ri[t], k, g.K, va[t]);
      if constexpr (kBk) load_rowk<kWhole>(pb[t], k, g.K, vb[t]);
      else load_colk<kWhole>(g.B, g.ldb, EPI == kWeight ? g.rows : nullptr, cj[t], k, g.K, vb[t]);
    }
  };
  const int nwhole = g.K / kStep, nsteps = (g.K + kStep - 1) / kStep;
  if constexpr (kSplit) {
    floatx4 acc = (floatx4){0.f, 0.f, 0.f, 0.f};
    const int ta = wave >> 1, tb = wave & 1;  // this wave's quarter
    for (int s0 = 0; s0 < nsteps; s0 += kChunk) {
      // this wave's steps of the chunk, all their loads in flight
      float va[4][2][8], vb[4][2][8];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int st = s0 + wave + 4 * u;
        if (st < nwhole) load(st, Int<1>{}, va[u], vb[u]);
        else if (st < nsteps) load(st, Int<0>{}, va[u], vb[u]);
      }
      if (s0 > 0) __syncthreads();
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (s0 + wave + 4 * u < nsteps)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            frag[wave + 4 * u][0][t][lane] = pack8(va[u][t]);
            frag[wave + 4 * u][1][t][lane] = pack8(vb[u][t]);
          }
      __syncthreads();
      const int n = min(kChunk, nsteps - s0);
#pragma unroll 4
      for (int u = 0; u < n; ++u)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag[u][0][ta][lane], frag[u][1][tb][lane],
                                                      acc, 0, 0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) part[16 * ta + 4 * q + r][16 * tb + c] = acc[r];
  } else {
    floatx4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = (floatx4){0.f, 0.f, 0.f, 0.f};
    // `count` K steps from st, all their loads in flight before the first use.
    auto steps = [&](int st, auto count, auto whole) {
      constexpr int kCount = decltype(count)::value;
      float va[kCount][2][8], vb[kCount][2][8];
#pragma unroll
      for (int u = 0; u < kCount; ++u) load(st + u, whole, va[u], vb[u]);
#pragma unroll
      for (int u = 0; u < kCount; ++u) {
        bf16x8 fa[2], fb[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
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
    int st = 0;
    for (; st + 3 < nwhole; st += 4) steps(st, Int<4>{}, Int<1>{});
    if (st + 1 < nwhole) {
      steps(st, Int<2>{}, Int<1>{});
      st += 2;
    }
    if (st < nwhole) {
      steps(st, Int<1>{}, Int<1>{});
      ++st;
    }
    if (st < nsteps) steps(st, Int<1>{}, Int<0>{});
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[16 * a + 4 * q + r][16 * b + c] = acc[a][b][r];
  }
  __syncthreads();
  double loss = 0;
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const int row = kSplit ? (tid >> 5) + 8 * r : (lane >> 5) + 2 * r;
    float x = part[row][col];
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
  if constexpr (EPI == kMseGrad) {
    for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
    if (lane == 0) g.partial[block] = loss;
  }
}

// Bias gradients: the sums over the rows k of A(i, k), 16 columns a block, in
// a fixed order: thread (grp, c) sums rows grp, grp + 16, ... (8 loads in
// flight), then the 16 groups' sums are added in group order.
constexpr int kSumCols = 16, kSumGroups = 16;

__device__ __forceinline__ void bias_grad(const GemmArgs& g, int block, const AdamArgs& adam,
                                          bf16x8* lds) {
  float (*part)[kSumCols] = reinterpret_cast<float (*)[kSumCols]>(lds);
  const int c = threadIdx.x % kSumCols, grp = threadIdx.x / kSumCols;
  const int i = block * kSumCols + c, ic = min(i, g.M - 1);
  AdamIn ad{0.f, 0.f, 0.f};
  if (g.bp) ad = adam_load(g.bp, g.bm, g.bv, ic);
  float s = 0.f;
  int k = grp;
  for (; k + 7 * kSumGroups < g.K; k += 8 * kSumGroups) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = g.A[(long long)(k + u * kSumGroups) * g.lda + ic];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; k < g.K; k += kSumGroups) s += g.A[(long long)k * g.lda + ic];
  part[grp][c] = s;
  __syncthreads();
  if (grp == 0 && i < g.M) {
    float x = part[0][c];
    for (int u = 1; u < kSumGroups; ++u) x += part[u][c];
    if (g.bp) adam_one(g.bp, g.bm, g.bv, i, x, ad, adam);
    else g.bias_out[i] = x;
  }
}

// The same products (all but kWeight) from 64 x 64 tiles, for operands that no
// longer come for free: four waves of 32 x 32, each operand element loaded and
// rounded once a block into LDS, the next K step's loads in flight while the
// current one is multiplied (two buffers, one barrier a step).  The same order
// over K, so the same results to the bit.
constexpr int kBig = 64, kPad = 8, kPer = kBig * kStep / 256;

template <int EPI>
__global__ void __launch_bounds__(256) gemm_big(GemmArgs g) {
  static_assert(EPI != kWeight, "layers and input gradients");
  __shared__ __align__(16) unsigned short As[2][kBig][kStep + kPad];
  __shared__ __align__(16) unsigned short Bs[2][kBig][kStep + kPad];  // Bs[j][k]
  constexpr bool kBk = EPI <= kMseGrad;  // B columns contiguous along k
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave >> 1, wn = wave & 1, q = lane >> 4, c = lane & 15;
  const int tj = (g.N + kBig - 1) / kBig;
  const int i0 = blockIdx.x / tj * kBig, j0 = blockIdx.x % tj * kBig;
  // This thread's elements of a step: (tile row, k) = (tid / 32 + 8 t, tid % 32)
  // where the operand is contiguous along k, else (tid % 64, tid / 64 + 4 t).
  // (Rows and columns past the matrices repeat the last one; unused.)
  const int ak = tid & (kStep - 1);
  const float *pa[kPer], *pb[kPer];
  int br[kPer], bk[kPer];
#pragma unroll
  for (int t = 0; t < kPer; ++t) {
    const int i = min(i0 + (tid >> 5) + 8 * t, g.M - 1);
    const bool gather = (EPI == kBias || EPI == kGelu) && g.rows;
    pa[t] = g.A + (long long)(gather ? g.rows[i] : i) * g.lda;
    br[t] = kBk ? (tid >> 5) + 8 * t : (tid & 63);
    bk[t] = kBk ? ak : (tid >> 6) + 4 * t;
    const int j = min(j0 + br[t], g.N - 1);
    pb[t] = kBk ? g.B + (long long)j * g.ldb : g.B + j;
  }
  float ra[kPer], rb[kPer];
  auto load = [&](int k0) {
#pragma unroll
    for (int t = 0; t < kPer; ++t) {
      const int ka = k0 + ak, kb = k0 + bk[t], kac = min(ka, g.K - 1), kbc = min(kb, g.K - 1);
      const float va = pa[t][kac];
      const float vb = kBk ? pb[t][kbc] : pb[t][(long long)kbc * g.ldb];
      ra[t] = ka < g.K ? va : 0.f;
      rb[t] = kb < g.K ? vb : 0.f;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int t = 0; t < kPer; ++t) {
      As[buf][(tid >> 5) + 8 * t][ak] = act::to_bf16(ra[t]);
      Bs[buf][br[t]][bk[t]] = act::to_bf16(rb[t]);
    }
  };
  floatx4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = (floatx4){0.f, 0.f, 0.f, 0.f};
  load(0);
  put(0);
  __syncthreads();
  const int nsteps = (g.K + kStep - 1) / kStep;
  for (int st = 0; st < nsteps; ++st) {
    const int cur = st & 1;
    load((st + 1) * kStep);  // past the end: the last element, then zero
    bf16x8 fa[2], fb[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      fa[a] = *reinterpret_cast<const bf16x8*>(&As[cur][wm * 32 + a * 16 + c][8 * q]);
      fb[a] = *reinterpret_cast<const bf16x8*>(&Bs[cur][wn * 32 + a * 16 + c][8 * q]);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
    if (st + 1 < nsteps) put(cur ^ 1);
    __syncthreads();
  }
  double loss = 0;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + wm * 32 + a * 16 + 4 * q + r, ic = min(i, g.M - 1);
      const long long trow = EPI == kMseGrad ? (g.rows ? g.rows[ic] : ic) : 0;
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int j = j0 + wn * 32 + b * 16 + c;
        if (i >= g.M || j >= g.N) continue;
        const long long o = (long long)i * g.ldc + j;
        float x = acc[a][b][r];
        if constexpr (EPI == kBias) {
          g.C[o] = x + g.bias[j];
        } else if constexpr (EPI == kGelu) {
          x += g.bias[j];
          g.Z[o] = x;
          g.C[o] = gelu(x);
        } else if constexpr (EPI == kMseGrad) {
          const float d = x + g.bias[j] - g.T[trow * g.N + j];
          g.C[o] = g.scale * d;
          loss += (double)d * d;
        } else {
          g.C[o] = x * gelu_grad(g.Z[o]);
        }
      }
    }
  if constexpr (EPI == kMseGrad) {
    __shared__ double red[4];
    for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
    if (lane == 0) red[wave] = loss;
    __syncthreads();
    if (tid == 0) g.partial[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
  }
}

template <int EPI>
__global__ void __launch_bounds__(EPI > kMseGrad ? 256 : 64) gemm_bf16(GemmArgs g) {
  __shared__ bf16x8 lds[ProductLds(EPI)];
  product<EPI>(g, blockIdx.x, AdamArgs{}, lds);
}

// Layers' weight gradients, one after the other in the grid, then their bias
// gradients.
struct WeightArgs {
  GemmArgs g[3];
  int first[7];
  AdamArgs adam;
};

__global__ void __launch_bounds__(256) weight_grads(WeightArgs w) {
  __shared__ bf16x8 lds[ProductLds(kWeight)];
  const int b = blockIdx.x;
  int l = 0;
  while (l < 5 && b >= w.first[l + 1]) ++l;
  const int i = b - w.first[l];
  if (l < 3) product<kWeight>(w.g[l], i, w.adam, lds);
  else bias_grad(w.g[l - 3], i, w.adam, lds);
}

}  // namespace mlp

// --- Host launchers ---------------------------------------------------------------

static int Tiles(int M, int N, int tile) {
  return (M + tile - 1) / tile * ((N + tile - 1) / tile);
}

// 64 x 64 tiles where they fill the chip, else the 32 x 32 ones that spread a
// small product over more CUs.  The line in 64 x 64 tiles, us of one launch,
// small / big tiles: layers at 176 (1024 x 686, K 256) 10.2 / 10.8 and (K
// 1024) 27.7 / 30.2, at 256 (1024 x 1024, K 1024) 36.1 / 31.1, at 512 (8192 x
// 256, K 256) 21.8 / 15.0, at 1408 (8192 x 686, K 256) 49.7 / 26.3 and (K
// 2048) 347 / 139; input gradients, whose B is strided in either, at 256
// (4096 x 256, K 256) 11.9 / 13.8, at 512 (8192 x 256) 22.3 / 16.0.
static bool UseBig(int M, int N, bool input_grad) {
  return Tiles(M, N, mlp::kBig) >= (input_grad ? 512 : 256);
}

int LayerBlocks(int M, int N) {
  return Tiles(M, N, UseBig(M, N, false) ? mlp::kBig : mlp::kTile);
}

template <int EPI>
static hipError_t LaunchProduct(const mlp::GemmArgs& g, hipStream_t s) {
  constexpr bool kGrad = EPI == mlp::kGeluGrad;
  if (UseBig(g.M, g.N, kGrad))
    hipLaunchKernelGGL(mlp::gemm_big<EPI>, dim3(Tiles(g.M, g.N, mlp::kBig)), dim3(256), 0, s, g);
  else
    hipLaunchKernelGGL(mlp::gemm_bf16<EPI>, dim3(Tiles(g.M, g.N, mlp::kTile)),
                       dim3(kGrad ? 256 : 64), 0, s, g);
  return hipGetLastError();
}

hipError_t LaunchLayer(const mlp::GemmArgs& g, mlp::Epilogue e, hipStream_t s) {
  if (e == mlp::kBias) return LaunchProduct<mlp::kBias>(g, s);
  if (e == mlp::kGelu) return LaunchProduct<mlp::kGelu>(g, s);
  if (e == mlp::kMseGrad) return LaunchProduct<mlp::kMseGrad>(g, s);
  return hipErrorInvalidValue;
}

hipError_t LaunchInputGrad(const mlp::GemmArgs& g, hipStream_t s) {
  return LaunchProduct<mlp::kGeluGrad>(g, s);
}

hipError_t LaunchWeightGrads(const mlp::GemmArgs* g, int count, const mlp::AdamArgs& adam,
                             hipStream_t s) {
  if (count != 3) return hipErrorInvalidValue;
  mlp::WeightArgs w{};
  w.adam = adam;
  for (int i = 0; i < 3; ++i) {
    w.g[i] = g[i];
    w.first[i + 1] = w.first[i] + Tiles(g[i].M, g[i].N, mlp::kTile);
  }
  for (int i = 0; i < 3; ++i)
    w.first[i + 4] = w.first[i + 3] + (g[i].M + mlp::kSumCols - 1) / mlp::kSumCols;
  hipLaunchKernelGGL(mlp::weight_grads, dim3(w.first[6]), dim3(256), 0, s, w);
  return hipGetLastError();
}

}  // namespace phi
