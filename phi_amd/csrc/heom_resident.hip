// RK4 of a small Hermitian hierarchy inside one workgroup: the whole state in
// registers and LDS, any number of steps in one launch.
//
// What bounds the stage kernels on a hierarchy of a few hundred small ADOs
// is the launch itself (about 5 us each, four a step, for 30 KB of data).
// Here a thread owns up to EPT elements (a, b), a <= b, of the packed state
// (heom_packed.h): its FP64 state, its K, the LDS offsets of its neighbours
// and their coefficients stay in registers over all steps; the stage vector
// goes through LDS, full matrices (both triangles), so a stage is 4 gathers
// per mode slot and 2 N matrix elements of LDS per element, and one barrier
// (two where only one stage vector fits).  Elements are dealt element-major
// (all nodes of (0,0), then of (0,1), ...), so a wavefront's lanes share
// (a, b): no divergence, broadcast reads of H; the odd node stride spreads
// them over the banks.  The same increment form and arithmetic as PkIncr.
#include "heom_packed.h"

namespace phi {
namespace dev {

struct ResidentArgs {
  double* rho;          // packed state
  long long nsteps, step_offset;
  int snap_every;       // 0: none
  double* hist;
  int* counter;
  int capacity;
  int bufs;             // stage vectors in LDS (1 or 2)
  double dt;
};

template <typename TB, int EPT, int MPS, int MAXT>
__global__ void __launch_bounds__(MAXT) resident_rk4(RhsArgs A, ResidentArgs R) {
  typedef typename C2<TB>::type V;
  extern __shared__ __align__(16) unsigned char smem[];
  const int N = A.N, NE = A.NE, NP = NE | 1, nodes = A.num_nodes;
  const int tid = threadIdx.x, nth = blockDim.x;
  V* sH = reinterpret_cast<V*>(smem);
  V* sY = sH + NE;
  const int other = R.bufs == 2 ? nodes * NP : 0;
  for (int e = tid; e < NE; e += nth) {
    const double2 h = A.H[e];
    sH[e] = mk<TB>((TB)(h.x * A.inv_hbar), (TB)(h.y * A.inv_hbar));
  }
  // Per element: LDS offset of its node | a << 16 | b << 24; offsets of the
  // neighbours n + e_j | n - e_j << 16.
  bool own[EPT], diag[EPT], first[EPT];
  unsigned where[EPT], nb[EPT][2][MPS];
  TB fs[EPT], cs[EPT][2][MPS], cx[EPT][2][MPS], cy[EPT][2][MPS];
  double2 rho[EPT];
  V kk[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int e = tid + i * nth;
    own[i] = e < nodes * A.PE;
    const int t = own[i] ? e / nodes : 0, n = own[i] ? e - t * nodes : 0;
    const int4 el = A.elem[t];
    const int a = el.x, b = el.y;
    diag[i] = a == b;
    where[i] = (unsigned)(n * NP) | (unsigned)a << 16 | (unsigned)b << 24;
    first[i] = n == 0 && own[i];
    const double* src = R.rho + (size_t)n * NE + el.z;
    rho[i] = make_double2(src[0], diag[i] ? 0. : src[1]);
    fs[i] = (TB)A.mu[n] + (diag[i] ? (TB)0 : (TB)A.delta[a] + (TB)A.delta[b]);
#pragma unroll
    for (int side = 0; side < 2; ++side)
#pragma unroll
      for (int q = 0; q < MPS; ++q) {
        const int4 c = A.edge[((size_t)n * N + (side == 0 ? b : a)) * A.mps + q];
        const int z = max(c.z, 0);
        const double2 pc = A.prev_col[z];
        nb[i][side][q] = (unsigned)((c.x >= 0 ? c.x : n) * NP) |
                         (unsigned)((c.y >= 0 ? c.y : n) * NP) << 16;
        cs[i][side][q] = c.x >= 0 ? (TB)A.next_s[z] : (TB)0;
        cx[i][side][q] = c.y >= 0 ? (TB)pc.x : (TB)0;
        cy[i][side][q] = c.y >= 0 ? (TB)pc.y : (TB)0;
      }
  }
  auto put = [&](V* y, int i, TB x, TB w) {
    if (own[i]) {
      const unsigned o = pk_opaque(where[i]), b = o >> 24, a = o >> 16 & 255, base = o & 0xffff;
      y[base + b * N + a] = mk<TB>(x, w);
      if (!diag[i]) y[base + a * N + b] = mk<TB>(x, -w);
    }
  };
#pragma unroll
  for (int i = 0; i < EPT; ++i) put(sY, i, (TB)rho[i].x, (TB)rho[i].y);
  int slot = *R.counter;
  __syncthreads();
  const bool realh = A.real_h != 0;
  // (L y)(a, b) of element i
  auto rhs = [&](const V* y, int i) {
    const unsigned w0 = pk_opaque(where[i]), b = w0 >> 24, a = w0 >> 16 & 255;
    const unsigned base = w0 & 0xffff;
    const V* yo = y + (b * N + a);
    const V v = yo[base];
    TB ax = -fs[i] * v.x, ay = -fs[i] * v.y;
#pragma unroll
    for (int q = 0; q < MPS; ++q) {
      const unsigned nb0 = pk_opaque(nb[i][0][q]), nb1 = pk_opaque(nb[i][1][q]);
      const V g1 = yo[nb0 & 0xffff], g3 = yo[nb0 >> 16];
      const V g2 = yo[nb1 & 0xffff], g4 = yo[nb1 >> 16];
      ax -= cs[i][0][q] * g1.y + (cx[i][0][q] * g3.x - cy[i][0][q] * g3.y);
      ay += cs[i][0][q] * g1.x - (cx[i][0][q] * g3.y + cy[i][0][q] * g3.x);
      ax += cs[i][1][q] * g2.y - (cx[i][1][q] * g4.x + cy[i][1][q] * g4.y);
      ay -= cs[i][1][q] * g2.x + (cx[i][1][q] * g4.y - cy[i][1][q] * g4.x);
      if (MPS > 1) __builtin_amdgcn_sched_barrier(0);
    }
    // -(i/hbar) (H y - y H^dagger): y Hermitian, so the second product is the
    // conjugate transpose of the first
    TB hr = 0, hi = 0;
    const V* col = y + base + b * N;
    const V* row = y + base + a;
    if (realh) {
#pragma unroll 1
      for (int c = 0; c < N; ++c) {
        const TB p = sH[a + c * N].x, q = sH[b + c * N].x;
        const V u = col[c], w = row[c * N];
        hr += p * u.x - q * w.x;
        hi += p * u.y - q * w.y;
      }
    } else {
      for (int c = 0; c < N; ++c) {
        const V p = sH[a + c * N], q = sH[b + c * N];
        const V u = col[c], w = row[c * N];
        hr += p.x * u.x - p.y * u.y - (q.x * w.x + q.y * w.y);
        hi += p.x * u.y + p.y * u.x - (q.x * w.y - q.y * w.x);
      }
    }
    // (one element after the other: interleaving them costs registers)
    __builtin_amdgcn_sched_barrier(0);
    return mk<TB>(ax + hi, diag[i] ? (TB)0 : ay - hr);
  };
  const double dt = R.dt;
  const TB c0 = (TB)(dt / 4), c1 = (TB)(dt / 3), c2 = (TB)(dt / 2);
  int cur = 0;
  for (long long s = 0; s < R.nsteps; ++s) {
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      V out[EPT];
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const V k = rhs(sY + cur, i);
        if (st == 0) {
          kk[i] = k;
          out[i] = k;
        } else if (st == 1) {
          out[i] = mk<TB>(c1 * (kk[i].x + c0 * k.x), c1 * (kk[i].y + c0 * k.y));
        } else if (st == 2) {
          out[i] = mk<TB>(c2 * (kk[i].x + k.x), c2 * (kk[i].y + k.y));
        } else {
          rho[i].x += dt * ((double)kk[i].x + (double)k.x);
          rho[i].y += dt * ((double)kk[i].y + (double)k.y);
          out[i] = mk<TB>((TB)rho[i].x, (TB)rho[i].y);
        }
      }
      if (other == 0) __syncthreads();
      else cur = other - cur;
#pragma unroll
      for (int i = 0; i < EPT; ++i) put(sY + cur, i, out[i].x, out[i].y);
      __syncthreads();
    }
    if (R.snap_every > 0 && (R.step_offset + s) % R.snap_every == 0) {
      if (slot < R.capacity) {
        double2* h = reinterpret_cast<double2*>(R.hist) + (size_t)slot * NE;
#pragma unroll
        for (int i = 0; i < EPT; ++i)
          if (first[i]) {
            const int a = where[i] >> 16 & 255, b = where[i] >> 24;
            h[b * N + a] = rho[i];
            if (!diag[i]) h[a * N + b] = make_double2(rho[i].x, -rho[i].y);
          }
      }
      ++slot;
    }
  }
#pragma unroll
  for (int i = 0; i < EPT; ++i)
    if (own[i]) {
      const int e = tid + i * nth, t = e / nodes, n = e - t * nodes;
      double* dst = R.rho + (size_t)n * NE + A.elem[t].z;
      dst[0] = rho[i].x;
      if (!diag[i]) dst[1] = rho[i].y;
    }
  if (tid == 0) *R.counter = slot;
}

}  // namespace dev

namespace {

constexpr size_t kResidentLds = 150 * 1024;

size_t StageBytes(const RhsArgs& a, bool fp32) {
  return (size_t)a.num_nodes * (a.NE | 1) * (fp32 ? sizeof(float2) : sizeof(double2));
}

// Threads a block of EPT elements per thread may have so that their
// coefficients stay in registers (512 registers over the waves of a SIMD):
// the 495-node dimer, 2 FP64 elements of two modes per site each, 24.6 us a
// step on 1024 threads (380 bytes spilled) and 8.8 on 768.
constexpr int ResidentThreads(bool fp32, int ept, int mps) {
  return (mps == 2 && ept == 2 && !fp32) || ept == 4 ? 768 : 1024;
}

// Elements per thread: 1, 2 or (FP32, one mode per site, whose threads hold
// the fewest coefficients) 4; 0 when there are too many.  (FP64 with 4: 19.9
// us a step of 364 3-site nodes, 16.1 on the stage kernels.)
int ResidentEpt(const RhsArgs& a, bool fp32) {
  const long long tot = (long long)a.num_nodes * a.PE;
  const int most = a.mps <= 1 && fp32 ? 4 : 2;
  for (int ept = 1; ept <= most; ept *= 2)
    if (tot <= (long long)ResidentThreads(fp32, ept, a.mps <= 1 ? 1 : 2) * ept) return ept;
  return 0;
}

template <typename TB, int EPT, int MPS>
hipError_t LaunchResidentK(const RhsArgs& a, const dev::ResidentArgs& r, hipStream_t s) {
  constexpr int kMax = ResidentThreads(sizeof(TB) == 4, EPT, MPS);
  const size_t sh = (size_t)a.NE * 2 * sizeof(TB) +
                    r.bufs * StageBytes(a, sizeof(TB) == 4);
  const void* k = reinterpret_cast<const void*>(&dev::resident_rk4<TB, EPT, MPS, kMax>);
  if (sh > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)sh);
    if (e != hipSuccess) return e;
  }
  const int tot = a.num_nodes * a.PE;
  const int threads = ((tot + EPT - 1) / EPT + 63) / 64 * 64;
  hipLaunchKernelGGL((dev::resident_rk4<TB, EPT, MPS, kMax>), dim3(1), dim3(threads), sh, s, a, r);
  return hipGetLastError();
}

template <typename TB>
hipError_t LaunchResidentT(const RhsArgs& a, const dev::ResidentArgs& r, hipStream_t s) {
  const int ept = ResidentEpt(a, sizeof(TB) == 4);
  if (a.mps <= 1) {
    if (ept == 1) return LaunchResidentK<TB, 1, 1>(a, r, s);
    if constexpr (sizeof(TB) == 4)
      if (ept == 4) return LaunchResidentK<TB, 4, 1>(a, r, s);
    return LaunchResidentK<TB, 2, 1>(a, r, s);
  }
  if (ept == 1) return LaunchResidentK<TB, 1, 2>(a, r, s);
  return LaunchResidentK<TB, 2, 2>(a, r, s);
}

}  // namespace

bool ResidentFits(const RhsArgs& a, bool fp32) {
  if (a.N > 32 || a.mps > 2 || !a.elem || !a.edge || ResidentEpt(a, fp32) == 0) return false;
  return StageBytes(a, fp32) + (size_t)a.NE * sizeof(double2) <= kResidentLds;
}

hipError_t LaunchResidentRk4(const RhsArgs& a, bool fp32, double* rho, long long nsteps,
                             double dt, long long step_offset, int snap_every, double* hist,
                             int* counter, int capacity, hipStream_t s) {
  if (!ResidentFits(a, fp32)) return hipErrorInvalidConfiguration;
  const int bufs =
      2 * StageBytes(a, fp32) + (size_t)a.NE * sizeof(double2) <= kResidentLds ? 2 : 1;
  const dev::ResidentArgs r{rho,     nsteps,   step_offset, snap_every, hist,
                            counter, capacity, bufs,        dt};
  return fp32 ? LaunchResidentT<float>(a, r, s) : LaunchResidentT<double>(a, r, s);
}

}  // namespace phi
