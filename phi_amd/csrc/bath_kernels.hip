// RHS of the diagonal and full coupling models (formulas in bath_kernels.h).
// FP64 throughout.
#include "bath_kernels.h"

#include "heom_device.h"

namespace phi {
namespace dev {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cscale(double s, double2 a) {
  return make_double2(s * a.x, s * a.y);
}
// -i z
__device__ __forceinline__ double2 mul_negi(double2 z) { return make_double2(z.y, -z.x); }

constexpr int kMaxPerThread = 4;  // N <= 32 with 256 threads

// Diagonal operators: one block per node (grid-stride).
__global__ void __launch_bounds__(256) rhs_bath(RhsArgs A, BathArgs B,
                                                const double2* __restrict__ x,
                                                double2* __restrict__ y) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int N = A.N, NE = A.NE, D = A.D;
  double2* xs = reinterpret_cast<double2*>(smem);
  for (int n = blockIdx.x; n < A.num_nodes; n += gridDim.x) {
    __syncthreads();
    for (int e = threadIdx.x; e < NE; e += blockDim.x) xs[e] = x[(size_t)n * NE + e];
    __syncthreads();
    for (int e = threadIdx.x; e < NE; e += blockDim.x) {
      const int a = e % N, b = e / N;  // element (a, b)
      // -(i/hbar)(H x - x H^dagger)
      double2 u = make_double2(0., 0.);
      for (int c = 0; c < N; ++c) {
        u = cadd(u, cmul(A.Hraw[a + c * N], xs[c + b * N]));
        u = csub(u, cmul(xs[a + c * N], A.Hadj[c + b * N]));
      }
      double2 o = cscale(A.inv_hbar, mul_negi(u));
      if (!A.vacuum) {
        o = csub(o, cscale(A.mu[n], xs[e]));
        for (int j = 0; j < D; ++j) {
          const int m = j / B.K;
          const int k = A.occ[(size_t)n * D + j];
          const int nx = A.next[(size_t)n * D + j];
          const int pv = A.prev[(size_t)n * D + j];
          const double2 ba = B.ops[m * N + a], bb = B.ops[m * N + b];
          if (nx >= 0) o = cadd(o, cmul(mul_negi(csub(ba, bb)), x[(size_t)nx * NE + e]));
          if (pv >= 0) {
            const double2 c = B.corr[j];
            const double2 op = mul_negi(csub(cmul(ba, c), cmul(bb, cconj(c))));
            o = cadd(o, cscale((double)k, cmul(op, x[(size_t)pv * NE + e])));
          }
        }
        for (int m = 0; m < B.M; ++m) {
          const double2 d = csub(B.ops[m * N + a], B.ops[m * N + b]);
          o = csub(o, cscale(B.alpha[m], cmul(cmul(d, d), xs[e])));
        }
      }
      y[(size_t)n * NE + e] = o;
    }
  }
}

// Full operators.  All terms of bath m are products with the one matrix F_m,
//   F_m L_m + R_m F_m,  C = F_m x - x F_m,
//   L_m = -alpha_m C + sum_j (-i s_j x_{n+e_j} - row_j x_{n-e_j}),
//   R_m = +alpha_m C + sum_j (+i s_j x_{n+e_j} - col_j x_{n-e_j}),
// so the neighbours enter elementwise and a bath costs four N^3 products
// instead of four per mode and four more.  A block takes T nodes (as many as
// fill its threads) with x, L, R, F (and H) in LDS; what bounds it is the
// LDS reads, 8 N per element and bath.  With ALL the operators of every bath
// and H stay in LDS, else F_m is staged bath by bath.  792 7-site nodes: one
// launch 13.4 us (40.6 with a commutator per mode from global memory and 49
// of 256 threads working; 16.1 with N a run-time value).
template <int EPT, bool ALL, int NT>
__global__ void __launch_bounds__(256) rhs_full(RhsArgs A, BathArgs B, int T,
                                                const double2* __restrict__ x,
                                                double2* __restrict__ y) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int N = NT > 0 ? NT : A.N, NE = N * N, D = A.D, L = A.L, K = B.K, TE = T * NE;
  double2* xs = reinterpret_cast<double2*>(smem);
  double2* ls = xs + TE;
  double2* rs = ls + TE;
  double2* fs = rs + TE;
  double2* hs = fs + (size_t)B.M * NE;   // (ALL)
  const int tid = threadIdx.x, nth = blockDim.x;
  if (ALL) {
    for (int e = tid; e < B.M * NE; e += nth) fs[e] = B.ops[e];
    for (int e = tid; e < NE; e += nth) {
      hs[e] = A.Hraw[e];
      hs[NE + e] = A.Hadj[e];
    }
  }
  const double2* H = ALL ? hs : A.Hraw;
  const double2* Hd = ALL ? hs + NE : A.Hadj;
  for (int n0 = blockIdx.x * T; n0 < A.num_nodes; n0 += gridDim.x * T) {
    const int tot = min(T, A.num_nodes - n0) * NE;
    __syncthreads();
    for (int e = tid; e < tot; e += nth) xs[e] = x[(size_t)n0 * NE + e];
    // Element i of this thread: node base in LDS, row, column, node id.
    int nb[EPT], ra[EPT], cb[EPT], id[EPT];
    bool ok[EPT];
    double2 out[EPT], un[EPT], wn[EPT];
    int kn[EPT], pn[EPT], xn[EPT];
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int e = tid + i * nth;
      ok[i] = e < tot;
      const int t = ok[i] ? e / NE : 0, r = ok[i] ? e - t * NE : 0;
      nb[i] = t * NE;
      cb[i] = r / N;
      ra[i] = r - cb[i] * N;
      id[i] = n0 + t;
    }
    // The neighbours of mode j (absent: the node itself with zero weight).
    auto fetch = [&](int j) {
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const size_t o = (size_t)id[i] * D + j;
        xn[i] = A.next[o];
        pn[i] = A.prev[o];
        kn[i] = A.occ[o];
      }
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const int r = cb[i] * N + ra[i];
        un[i] = x[(size_t)(xn[i] >= 0 ? xn[i] : id[i]) * NE + r];
        wn[i] = x[(size_t)(pn[i] >= 0 ? pn[i] : id[i]) * NE + r];
      }
    };
    if (!A.vacuum && D > 0) fetch(0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int a = ra[i], b = cb[i];
      const double2* xv = xs + nb[i];
      double2 u = make_double2(0., 0.);
      for (int c = 0; c < N; ++c) {
        u = cadd(u, cmul(H[a + c * N], xv[c + b * N]));
        u = csub(u, cmul(xv[a + c * N], Hd[c + b * N]));
      }
      out[i] = cscale(A.inv_hbar, mul_negi(u));
      if (!A.vacuum) out[i] = csub(out[i], cscale(A.mu[id[i]], xv[a + b * N]));
    }
    if (!A.vacuum) {
      for (int m = 0; m < B.M; ++m) {
        const double2* F = fs + (ALL ? (size_t)m * NE : 0);
        if (!ALL) {
          __syncthreads();
          for (int e = tid; e < NE; e += nth) fs[e] = B.ops[(size_t)m * NE + e];
          __syncthreads();
        }
        double2 lv[EPT], rv[EPT];
        const double al = B.alpha[m];
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
          const int a = ra[i], b = cb[i];
          const double2* xv = xs + nb[i];
          double2 c2 = make_double2(0., 0.);
          for (int c = 0; c < N; ++c) {
            c2 = cadd(c2, cmul(F[a + c * N], xv[c + b * N]));
            c2 = csub(c2, cmul(xv[a + c * N], F[c + b * N]));
          }
          lv[i] = cscale(-al, c2);
          rv[i] = cscale(al, c2);
        }
        for (int q = 0; q < K; ++q) {
          const int j = m * K + q;
#pragma unroll
          for (int i = 0; i < EPT; ++i) {
            if (xn[i] >= 0) {
              const double2 v = cscale(A.next_s[j * L + kn[i]], mul_negi(un[i]));
              lv[i] = cadd(lv[i], v);
              rv[i] = csub(rv[i], v);
            }
            if (pn[i] >= 0) {
              lv[i] = csub(lv[i], cmul(A.prev_row[j * L + kn[i]], wn[i]));
              rv[i] = csub(rv[i], cmul(A.prev_col[j * L + kn[i]], wn[i]));
            }
          }
          if (j + 1 < D) fetch(j + 1);
        }
#pragma unroll
        for (int i = 0; i < EPT; ++i)
          if (ok[i]) {
            ls[nb[i] + ra[i] + cb[i] * N] = lv[i];
            rs[nb[i] + ra[i] + cb[i] * N] = rv[i];
          }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
          const int a = ra[i], b = cb[i];
          const double2 *lm = ls + nb[i], *rm = rs + nb[i];
          double2 o = out[i];
          for (int c = 0; c < N; ++c) {
            o = cadd(o, cmul(F[a + c * N], lm[c + b * N]));
            o = cadd(o, cmul(rm[a + c * N], F[c + b * N]));
          }
          out[i] = o;
        }
        __syncthreads();
      }
    }
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (ok[i]) y[(size_t)n0 * NE + tid + i * nth] = out[i];
  }
}

// One block per node of the range; x_n, Q_m, X_m (and F_m) in LDS.
__global__ void __launch_bounds__(256) timelocal_term(int N, TimeLocalArgs T,
                                                      const double2* __restrict__ x,
                                                      double2* __restrict__ y) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int NE = N * N;
  double2* xs = reinterpret_cast<double2*>(smem);
  double2* qs = xs + NE;
  double2* Xs = qs + NE;
  double2* fs = Xs + NE;
  for (int b = blockIdx.x; b < T.count; b += gridDim.x) {
    const size_t n = (size_t)T.first + b;
    __syncthreads();
    for (int e = threadIdx.x; e < NE; e += blockDim.x) xs[e] = x[n * NE + e];
    double2 out[kMaxPerThread];
#pragma unroll
    for (int i = 0; i < kMaxPerThread; ++i) out[i] = make_double2(0, 0);
    for (int m = 0; m < T.M; ++m) {
      __syncthreads();
      for (int e = threadIdx.x; e < NE; e += blockDim.x) {
        qs[e] = T.Q[(size_t)m * NE + e];
        if (T.model == 2) fs[e] = T.ops[(size_t)m * NE + e];
      }
      __syncthreads();
      for (int e = threadIdx.x; e < NE; e += blockDim.x) {
        const int r = e % N, c = e / N;
        double2 s = make_double2(0, 0);
        for (int k = 0; k < N; ++k) {
          s = cadd(s, cmul(qs[r + k * N], xs[k + c * N]));
          s = csub(s, cmul(xs[r + k * N], cconj(qs[c + k * N])));
        }
        Xs[e] = s;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kMaxPerThread; ++i) {
        const int e = threadIdx.x + i * blockDim.x;
        if (e >= NE) continue;
        const int r = e % N, c = e / N;
        if (T.model == 0) {
          const int st = T.site[m];
          if (c == st) out[i] = cadd(out[i], Xs[e]);
          if (r == st) out[i] = csub(out[i], Xs[e]);
        } else if (T.model == 1) {
          const double2 d = csub(T.ops[(size_t)m * N + r], T.ops[(size_t)m * N + c]);
          out[i] = csub(out[i], cmul(d, Xs[e]));
        } else {
          double2 s = make_double2(0, 0);
          for (int k = 0; k < N; ++k) {
            s = cadd(s, cmul(fs[r + k * N], Xs[k + c * N]));
            s = csub(s, cmul(Xs[r + k * N], fs[k + c * N]));
          }
          out[i] = csub(out[i], s);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kMaxPerThread; ++i) {
      const int e = threadIdx.x + i * blockDim.x;
      if (e < NE) y[n * NE + e] = cadd(y[n * NE + e], out[i]);
    }
  }
}

}  // namespace dev

hipError_t LaunchTimeLocal(int N, const TimeLocalArgs& t, const double* x, double* y,
                           hipStream_t s) {
  if (N < 1 || N * N > 256 * dev::kMaxPerThread || t.model < 0 || t.model > 2 || t.M < 1 ||
      !t.Q || (t.model != 0 && !t.ops) || (t.model == 0 && !t.site))
    return hipErrorInvalidValue;
  if (t.count <= 0) return hipSuccess;
  const size_t sh = 4 * (size_t)N * N * sizeof(double2);
  const int grid = t.count < 65535 ? t.count : 65535;
  hipLaunchKernelGGL(dev::timelocal_term, dim3(grid), dim3(256), sh, s, N, t, (const double2*)x,
                     (double2*)y);
  return hipGetLastError();
}

hipError_t LaunchRhsBath(const RhsArgs& a, const BathArgs& b, const double* x, double* y,
                         hipStream_t s) {
  if (a.N < 1 || a.NE > 256 * dev::kMaxPerThread || (b.model != 1 && b.model != 2))
    return hipErrorInvalidValue;
  if (b.model == 1) {
    const int grid = a.num_nodes < 65535 ? a.num_nodes : 65535;
    hipLaunchKernelGGL(dev::rhs_bath, dim3(grid), dim3(256), (size_t)a.NE * sizeof(double2), s, a,
                       b, (const double2*)x, (double2*)y);
    return hipGetLastError();
  }
  // A wave per node up to 8 x 8 (more nodes for smaller ones), else up to
  // 256 threads of 1, 2 or 4 elements.
  const int T = a.NE <= 64 ? 64 / a.NE : 1;
  const int threads = a.NE <= 64 ? 64 : (a.NE >= 256 ? 256 : (a.NE + 63) / 64 * 64);
  const int ept = (T * a.NE + threads - 1) / threads;
  const size_t elem = (size_t)a.NE * sizeof(double2);
  const size_t all = (3 * T + b.M + 2) * elem;
  const int blocks = (a.num_nodes + T - 1) / T;
  const dim3 grid(blocks < 65535 ? blocks : 65535), block(threads);
  const double2* xp = (const double2*)x;
  double2* yp = (double2*)y;
  // (all operators in LDS while several blocks still share a CU's)
  if (all <= 24 * 1024 && ept == 1) {
    // (sizes a wave holds whole nodes of: N known, loops unrolled)
    switch (a.N) {
#define PHI_FULL(n)                                                                            \
  case n:                                                                                      \
    hipLaunchKernelGGL((dev::rhs_full<1, true, n>), grid, block, all, s, a, b, T, xp, yp);     \
    break;
      PHI_FULL(2) PHI_FULL(3) PHI_FULL(4) PHI_FULL(5) PHI_FULL(6) PHI_FULL(7) PHI_FULL(8)
#undef PHI_FULL
      default:
        hipLaunchKernelGGL((dev::rhs_full<1, true, 0>), grid, block, all, s, a, b, T, xp, yp);
    }
  } else {
    const size_t sh = (3 * T + 1) * elem;
    if (ept <= 1)
      hipLaunchKernelGGL((dev::rhs_full<1, false, 0>), grid, block, sh, s, a, b, T, xp, yp);
    else if (ept == 2)
      hipLaunchKernelGGL((dev::rhs_full<2, false, 0>), grid, block, sh, s, a, b, T, xp, yp);
    else
      hipLaunchKernelGGL((dev::rhs_full<4, false, 0>), grid, block, sh, s, a, b, T, xp, yp);
  }
  return hipGetLastError();
}

}  // namespace phi
