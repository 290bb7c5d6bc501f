// Persistent stage kernels on packed Hermitian ADOs (N <= 32, at most two
// bath modes per site): the RK4 increment form and RKF45 of a Hermitian
// state.
//
// A Hermitian N x N ADO has N^2 independent real values, half of what the
// full layout (heom_device.h) stores.  A packed node is N^2 reals: the
// diagonal as reals and the upper triangle as (re, im) pairs, in 4 x 4 blocks
// of the matrix (block column by block column; within a block, column by
// column; within a diagonal block its pairs, then its reals), so that the
// elements (i, j), i = 0..N-1, which a neighbour's RHS gathers for site j,
// lie in few cache lines.  elem[e] = {a, b, o, 0} lists the PE = N (N + 1) / 2
// elements in storage order: element (a, b), a <= b, at real offset o.
//
// One thread owns element (a, b) of a node, for both (a, b) and (b, a):
//   k(a,b) = E(a,b) + G(a,b) + conj(G(b,a)),   G = -(i/hbar) H Y,
//   E = -(mu + (Delta_a + Delta_b)[a != b]) Y(a,b)
//       + sum over the modes j of site b: i s_j Y_{n+e_j}(a,b) - c_j Y_{n-e_j}(a,b)
//       - sum over the modes j of site a: i s_j Y_{n+e_j}(a,b) + conj(c_j) Y_{n-e_j}(a,b),
// the same RHS as heom_stream.h's W + W^dagger with the two halves summed in
// registers.  On the diagonal the imaginary part is dropped (it is zero).
//
// What bounds it: HBM and L2 bytes for large slabs, the chain record ->
// gather -> product for small ones.  A block works through its tiles with
// every load of tile i+1 (elements, gathers) issued before the product of
// tile i, and the edge records two tiles ahead, resolved once per (node,
// site) into LDS as byte offsets and coefficients.  E stays in registers, so
// the tile's Y and G need one LDS buffer each.
#ifndef PHI_AMD_HEOM_PACKED_H_
#define PHI_AMD_HEOM_PACKED_H_

#include <type_traits>

#include "heom_stream.h"

namespace phi {
namespace dev {

// Packed pairs start at any real offset (N^2 is odd for odd N), so their
// vector accesses only assume the alignment of one real.  (Padding nodes to
// an even size and picking diagonal reals out of aligned pairs moved the
// 512 x 7-site FP32 step from 1.58 to 1.66 ms: the bytes and selects cost
// more than the alignment saves.)
typedef float PkF2 __attribute__((ext_vector_type(2), aligned(4)));
typedef double PkD2 __attribute__((ext_vector_type(2), aligned(8)));
template <typename T> struct PkV;
template <> struct PkV<float> { typedef PkF2 type; };
template <> struct PkV<double> { typedef PkD2 type; };

// The reals o and o + 1 of a packed slab (a diagonal element's second value
// is its successor's and not used; slabs are padded by at least one real).
// Offsets are 32-bit bytes from a uniform base: no 64-bit lane arithmetic.
template <typename T>
__device__ __forceinline__ const T* pk_at(const T* p, unsigned o) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + o * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T* pk_at(T* p, unsigned o) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(p) + o * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ typename C2<T>::type pk_ld(const T* p, unsigned o) {
  const typename PkV<T>::type v =
      *reinterpret_cast<const typename PkV<T>::type*>(pk_at(p, o));
  return mk<T>(v.x, v.y);
}
template <typename T>
__device__ __forceinline__ typename C2<T>::type pk_ld_nt(const T* p, unsigned o) {
  const typename PkV<T>::type v =
      __builtin_nontemporal_load(reinterpret_cast<const typename PkV<T>::type*>(pk_at(p, o)));
  return mk<T>(v.x, v.y);
}
template <typename T>
__device__ __forceinline__ void pk_st_nt(T* p, unsigned o, typename C2<T>::type w, bool diag) {
  T* q = pk_at(p, o);
  if (diag) {
    __builtin_nontemporal_store(w.x, q);
  } else {
    typename PkV<T>::type v;
    v.x = w.x;
    v.y = w.y;
    __builtin_nontemporal_store(v, reinterpret_cast<typename PkV<T>::type*>(q));
  }
}
template <typename T>
__device__ __forceinline__ void pk_st(T* p, unsigned o, typename C2<T>::type w, bool diag) {
  T* q = pk_at(p, o);
  if (diag) {
    *q = w.x;
  } else {
    typename PkV<T>::type v;
    v.x = w.x;
    v.y = w.y;
    *reinterpret_cast<typename PkV<T>::type*>(q) = v;
  }
}

// Resolved edge record of one (node, site, mode slot) in LDS: byte offsets
// of n + e_j and n - e_j from the member's slab (the node itself where the
// neighbour does not exist, with zero coefficients).
template <typename TB>
struct __attribute__((aligned(16))) PkRec {
  unsigned offn, offp;
  TB s, cx, cy;
};

// LDS column stride of Y and G in complex elements: the 4 ceil(N/4) rows the
// matrix cores read (rows past N stay zero), plus 2, which keeps columns 16
// bytes aligned and spreads 16 neighbouring columns over the banks.
__host__ __device__ inline int PkStride(int N) { return 4 * ((N + 3) >> 2) + 2; }
__host__ __device__ inline int PkCols(int N, int T) { return (T * N + 15) & ~15; }

__host__ __device__ inline size_t PackedLdsBytes(int N, int D, int L, int mps, int T,
                                                 size_t real) {
  const size_t V = 2 * real;
  size_t b = V * 2 * (size_t)PkCols(N, T) * PkStride(N);                       // Y, G
  b += 2 * (size_t)T * N * mps * 32;                                   // records
  b += V * (size_t)D * L;                                                      // pcol
  b += real * ((size_t)D * L + N + 2 * (size_t)T + 2 * (size_t)StreamFragCount(N));
  return Align16(b);
}

template <typename TB>
struct PackedLds {
  typedef typename C2<TB>::type V;
  V* Y;
  V* G;
  PkRec<TB>* rec;   // two tiles of T*N*mps
  V* pcol;
  TB* hfr;
  TB* hfi;
  TB* ns;
  TB* delta;
  TB* mu;           // two tiles of T
};

template <typename TB>
__device__ __forceinline__ PackedLds<TB> packed_carve(unsigned char* smem, const RhsArgs& A,
                                                      int T) {
  typedef typename C2<TB>::type V;
  static_assert(sizeof(PkRec<TB>) == 32, "record size");
  PackedLds<TB> s;
  const int cols = PkCols(A.N, T) * PkStride(A.N);
  s.Y = reinterpret_cast<V*>(smem);
  s.G = s.Y + cols;
  s.rec = reinterpret_cast<PkRec<TB>*>(s.G + cols);
  s.pcol = reinterpret_cast<V*>(s.rec + 2 * T * A.N * A.mps);
  s.hfr = reinterpret_cast<TB*>(s.pcol + A.D * A.L);
  s.hfi = s.hfr + StreamFragCount(A.N);
  s.ns = s.hfi + StreamFragCount(A.N);
  s.delta = s.ns + A.D * A.L;
  s.mu = s.delta + A.N;
  return s;
}

// The same value, opaque to the compiler: what is derived from it is
// computed where it is used instead of being kept in registers over the loop
// (occupancy is worth more than the few integer operations).
__device__ __forceinline__ unsigned pk_opaque(unsigned v) {
  asm volatile("" : "+v"(v));
  return v;
}

// G = (H / hbar scaled) product of the tile's columns: work items are
// (16-column slice, 16-row tile of H) pairs dealt to the waves.  The
// fragments hold H / hbar, so G = -i (frag Y): re = im part of the product,
// im = -re part.  Columns past the tile hold stale values; their results
// are never read.
__device__ __forceinline__ void pk_put_g(float2* col, int mt, int g, int N, int KS,
                                         const floatx4& xr, const floatx4& xi) {
  const int row0 = 16 * mt + 4 * g;
  if (row0 < N) {  // rows row0 .. row0 + 3 < 4 KS
    float4* w = reinterpret_cast<float4*>(col + row0);
    w[0] = make_float4(xi[0], -xr[0], xi[1], -xr[1]);
    w[1] = make_float4(xi[2], -xr[2], xi[3], -xr[3]);
  }
}
__device__ __forceinline__ void pk_put_g(double2* col, int mt, int g, int N, int KS,
                                         const doublex4& xr, const doublex4& xi) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * mt + r < KS) col[16 * mt + 4 * r + g] = make_double2(xi[r], -xr[r]);
}

template <typename TB>
__device__ __forceinline__ void packed_gemm(const RhsArgs& A, const PackedLds<TB>& s, int ncols) {
  typedef typename C2<TB>::type V;
  typedef Mfma<TB> M;
  const int N = A.N, KS = (N + 3) >> 2, S = PkStride(N);
  const int two = N > 16 ? 1 : 0;  // row tiles - 1
  const unsigned tid = pk_opaque(threadIdx.x);
  const int lane = tid & 63, g = lane >> 4, c16 = lane & 15;
  const int nwaves = blockDim.x >> 6;
  const int nitems = ((ncols + 15) >> 4) << two;
  const bool realh = A.real_h != 0;
  for (int item = __builtin_amdgcn_readfirstlane(tid >> 6); item < nitems; item += nwaves) {
    const int mt = item & two, j = (item >> two) * 16 + c16;
    const V* y = s.Y + j * S + g * KS;
    const TB* hr = s.hfr + mt * KS * 64 + lane;
    typename M::acc xr = M::zero(), xi = M::zero();
    if (realh) {
#pragma unroll 2
      for (int st = 0; st < KS; ++st) {
        const V v = y[st];
        const TB h = hr[st * 64];
        xr = M::mac(h, v.x, xr);
        xi = M::mac(h, v.y, xi);
      }
    } else {
      const TB* hi = s.hfi + mt * KS * 64 + lane;
      for (int st = 0; st < KS; ++st) {
        const V v = y[st];
        const TB h = hr[st * 64], q = hi[st * 64];
        xr = M::mac(h, v.x, xr);
        xi = M::mac(h, v.y, xi);
        xr = M::mac(-q, v.y, xr);
        xi = M::mac(q, v.x, xi);
      }
    }
    pk_put_g(s.G + j * S, mt, g, N, KS, xr, xi);
  }
}

// The owned elements of a thread, the same in every tile.
template <int EPT>
struct PkElems {
  int te[EPT];           // node of the tile (T: no element)
  unsigned off[EPT];     // real offset from the tile's first node
  unsigned goff[EPT];    // byte offset within the node of the input
  unsigned rec[EPT];     // record indices (slot 0) of site b, and of site a << 16
  unsigned lds[EPT];     // LDS offsets of (a, b), and of (b, a) << 16
  bool diag[EPT];
};

// ENS: an ensemble's tile list, as in stream_stage (same tile order).
//
// The vector-memory counter is in order, so the order of issue within an
// iteration is the order of use: the records of tile i+2 (needed before the
// second barrier), the epilogue operands of tile i, the loads of tile i+1;
// and the stores of tile i-1 wait in registers until the loads of tile i
// have arrived (a wait for loads issued before a store under a branch would
// otherwise drain the store as well).
template <typename TB, typename TI, int EPT, int MPS, bool ENS, class EPI>
__global__ void __launch_bounds__(512)
    packed_stage(RhsArgs A, const TI* __restrict__ in, EPI epi) {
  typedef typename C2<TB>::type V;
  typedef typename C2<TI>::type VI;
  typedef typename EPI::Pre Pre;
  typedef typename EPI::Out Out;
  // Records per thread: T N MPS records against T PE = T N (N + 1) / 2
  // elements at EPT per thread.
  constexpr int RPT = EPT * MPS;
  extern __shared__ __align__(16) unsigned char smem[];
  const int N = A.N, NE = A.NE, T = A.tile;
  const PackedLds<TB> s = packed_carve<TB>(smem, A, T);
  const int ntiles = ENS ? A.ntiles : (A.num_nodes + T - 1) / T;
  int tile, tile_end, step;
  int* ctr = nullptr;
  if constexpr (ENS) {
    const int G = gridDim.x, X = G < 8 ? G : 8;
    const int x = blockIdx.x % X;
    // (the first runs one longer, as the first ones have one block more: with
    // a block a tile every block has one.  Runs of rounded eighths gave some
    // blocks two: 8 members of 6 sites, 228 FP64 tiles, 7.3 us a stage, 5.6
    // this way)
    const int q = ntiles / X, r = ntiles % X, first = x * q + min(x, r);
    tile = first + (int)(blockIdx.x / X);
    tile_end = first + q + (x < r ? 1 : 0);
    step = G / X + (x < G % X ? 1 : 0);
    ctr = A.tile_ctr + 16 * (8 * A.ctr_set + x);
  } else {
    const int G = gridDim.x, x = blockIdx.x & 7, base = G >> 3, r = G & 7;
    tile = x * base + min(x, r) + (int)(blockIdx.x >> 3);
    tile_end = ntiles;
    step = G;
  }
  const int tid = threadIdx.x, nth = blockDim.x;
  __shared__ int fetched;
  // An ensemble block takes its tiles in claims of kClaim, the tiles step
  // apart of one round; the first claim is its slot, later ones come from its
  // run's counter.  So the run's blocks stay within a few rounds of each
  // other: with fixed strides they drift apart by several members and evict
  // the input their neighbours still gather from (512 x 7-site FP32 stage 1:
  // 8.8 M instead of 2.4 M L2 line fetches for 2.1 M lines).  One claim per
  // tile would be bound by the counter (22 ns an atomic).  Each launch
  // clears the other counter set for the next launch.
  constexpr int kClaim = 4;
  const int start = tile - (ENS ? (int)(blockIdx.x / (gridDim.x < 8 ? gridDim.x : 8)) : 0);
  const bool claims = ENS && (long long)step * kClaim < tile_end - start;
  if (ENS && blockIdx.x == 0 && tid < 8)
    A.tile_ctr[16 * (8 * (A.ctr_set ^ 1) + tid)] = 0;
  if (tile >= tile_end) return;
  auto claim_tile = [&](int m) { return start + m / step * kClaim * step + m % step; };
  const int nrec = T * N * MPS;

  // Records and mu of a tile: issued here, resolved into LDS by put_rec.
  // Tables are padded by a tile, so a short tile's loads stay inside them.
  int4 rr[RPT];
  double mr[EPT];
  auto load_rec = [&](const TileInfo& t) {
    const int4* e = A.edge + (size_t)t.local * N * MPS;
    const double* m = A.mu + t.local;
    const int tid = (int)pk_opaque(threadIdx.x);
#pragma unroll
    for (int i = 0; i < RPT; ++i)
      rr[i] = *reinterpret_cast<const int4*>(reinterpret_cast<const char*>(e) +
                                             (unsigned)min(tid + i * nth, nrec - 1) * 16u);
#pragma unroll
    for (int i = 0; i < EPT; ++i) mr[i] = *pk_at(m, (unsigned)min(tid + i * nth, T - 1));
  };
  auto put_rec = [&](const TileInfo& t, int buf) {
    PkRec<TB>* dst = s.rec + buf * nrec;
    const int tid = (int)pk_opaque(threadIdx.x);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int q = tid + i * nth;
      if (q < nrec) {
        const int4 c = rr[i];
        // (a node past a short tile's end resolves to the tile's last one)
        const int self = t.local + min(fdiv(q, A.mNM), t.nt - 1);
        const bool hn = (unsigned)c.x < (unsigned)t.count, hp = (unsigned)c.y < (unsigned)t.count;
        const int z = max(c.z, 0);
        const V pc = s.pcol[z];
        PkRec<TB> r;
        r.offn = (unsigned)(hn ? c.x : self) * (unsigned)(NE * sizeof(TI));
        r.offp = (unsigned)(hp ? c.y : self) * (unsigned)(NE * sizeof(TI));
        r.s = hn ? s.ns[z] : (TB)0;
        r.cx = hp ? pc.x : (TB)0;
        r.cy = hp ? pc.y : (TB)0;
        dst[q] = r;
      }
    }
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (tid + i * nth < T) s.mu[buf * T + tid + i * nth] = (TB)mr[i];
  };

  // Prologue: per-block constants, the first tile's records and loads.
  TileInfo t0 = stream_tile<ENS>(A, tile), t1 = t0, t2 = t0;
  load_rec(t0);
  int hmember = t0.member;
  const int DL = A.D * A.L, nf = StreamFragCount(N);
  const V* frag = reinterpret_cast<const V*>(A.hfrag);
  PkElems<EPT> C;
  int eb[EPT], ea[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int e = tid + i * nth;
    const bool ok = e < T * A.PE;
    const int te = ok ? fdiv(e, A.mPE) : 0;
    const int4 el = A.elem[ok ? e - te * A.PE : 0];
    C.te[i] = ok ? te : T;  // never below a tile's node count
    ea[i] = el.x;
    eb[i] = el.y;
    C.goff[i] = (unsigned)el.z * (unsigned)sizeof(TI);
    C.off[i] = (unsigned)(te * NE + el.z);
    C.rec[i] = (unsigned)((te * N + el.y) * MPS) | (unsigned)((te * N + el.x) * MPS) << 16;
    C.lds[i] = (unsigned)((te * N + el.y) * PkStride(N) + el.x) |
               (unsigned)((te * N + el.x) * PkStride(N) + el.y) << 16;
    C.diag[i] = el.x == el.y;
  }
  for (int e = tid; e < DL; e += nth) {
    s.pcol[e] = ld<TB, double>(reinterpret_cast<const double*>(A.prev_col), e);
    s.ns[e] = (TB)A.next_s[e];
  }
  for (int e = tid; e < N; e += nth) s.delta[e] = (TB)A.delta[e];
  for (int f = tid; f < nf; f += nth) {
    const V h = frag[(size_t)hmember * nf + f];
    s.hfr[f] = h.x;
    s.hfi[f] = h.y;
  }
  {
    // rows N .. 4 KS - 1 and columns past the tile are multiplied by zero
    const int cols = PkCols(N, T) * PkStride(N);
    for (int e = tid; e < cols; e += nth) s.Y[e] = mk<TB>((TB)0, (TB)0);
  }
  __syncthreads();
  put_rec(t0, 0);
  int i1 = tile + step, i2 = i1 + step;  // the next two tiles (past the end: none)
  int taken = 3;                         // tiles of the current claim handed out
  if (i1 < tile_end) {
    t1 = stream_tile<ENS>(A, i1);
    load_rec(t1);
  }
  t2 = i2 < tile_end ? stream_tile<ENS>(A, i2) : t1;
  __syncthreads();
  TB fd[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i)
    fd[i] = ea[i] != eb[i] ? s.delta[ea[i]] + s.delta[eb[i]] : (TB)0;
  // Elements and gathers of a tile whose records are in LDS buffer buf.
  VI y[EPT], gn[EPT][2][MPS], gp[EPT][2][MPS];
  auto load_tile = [&](const TileInfo& t, int buf) {
    const TI* own = in + (size_t)t.base * NE;
    const char* slab = reinterpret_cast<const char*>(in + (size_t)(t.base - t.local) * NE);
    auto at = [&](unsigned o) {
      const typename PkV<TI>::type v = *reinterpret_cast<const typename PkV<TI>::type*>(slab + o);
      return mk<TI>(v.x, v.y);
    };
    const PkRec<TB>* R = s.rec + buf * nrec;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      y[i] = pk_ld(own, pk_opaque(C.off[i]));
      const unsigned o = C.goff[i], w = pk_opaque(C.rec[i]);
      const PkRec<TB>*rb = R + (w & 0xffffu), *ra = R + (w >> 16);
#pragma unroll
      for (int q = 0; q < MPS; ++q) {
        gn[i][0][q] = at(rb[q].offn + o);
        gp[i][0][q] = at(rb[q].offp + o);
        gn[i][1][q] = at(ra[q].offn + o);
        gp[i][1][q] = at(ra[q].offp + o);
      }
    }
  };
  load_tile(t0, 0);
  if (i1 < tile_end) put_rec(t1, 1);
  V hp[2] = {mk<TB>((TB)0, (TB)0), mk<TB>((TB)0, (TB)0)};
  double emax = 0;
  Out out[EPT];
  unsigned have = 0;   // bit i: out[i] is tile tb0's, to be stored
  size_t tb0 = 0;
  __syncthreads();

  auto flush = [&]() {
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (have >> i & 1) epi.store(tb0, pk_opaque(C.off[i]), C.diag[i], out[i]);
  };
  int buf = 0;
  // One tile; with `more`, the loads of the tiles after it.
  auto work = [&](auto more) {
    constexpr bool kMore = decltype(more)::value;
    // H of a new member, from the registers the previous tile loaded.
    if (ENS && t0.member != hmember) {
      hmember = t0.member;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int f = (int)pk_opaque(tid) + j * nth;
        if (f < nf) {
          s.hfr[f] = hp[j].x;
          s.hfi[f] = hp[j].y;
        }
      }
    }
    // (1) E of this tile; its Y (both triangles) -> LDS
    TB ex[EPT], ey[EPT];
    Pre pre[EPT];
    const PkRec<TB>* R = s.rec + buf * nrec;
    const size_t tb = (size_t)t0.base * NE;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const bool dg = C.diag[i];
      const TB yx = (TB)y[i].x, yy = dg ? (TB)0 : (TB)y[i].y;
      const TB f = s.mu[buf * T + min(C.te[i], T - 1)] + fd[i];
      if (EPI::kInIsState) pre[i] = epi.from_state((double)y[i].x, dg ? 0. : (double)y[i].y);
      TB ax = -f * yx, ay = -f * yy;
      const unsigned w = pk_opaque(C.rec[i]), l = pk_opaque(C.lds[i]);
#pragma unroll
      for (int q = 0; q < MPS; ++q) {
        const PkRec<TB> rb = R[(w & 0xffffu) + q], ra = R[(w >> 16) + q];
        const TB g1x = (TB)gn[i][0][q].x, g1y = dg ? (TB)0 : (TB)gn[i][0][q].y;
        const TB g2x = (TB)gn[i][1][q].x, g2y = dg ? (TB)0 : (TB)gn[i][1][q].y;
        const TB g3x = (TB)gp[i][0][q].x, g3y = dg ? (TB)0 : (TB)gp[i][0][q].y;
        const TB g4x = (TB)gp[i][1][q].x, g4y = dg ? (TB)0 : (TB)gp[i][1][q].y;
        ax -= rb.s * g1y + (rb.cx * g3x - rb.cy * g3y);
        ay += rb.s * g1x - (rb.cx * g3y + rb.cy * g3x);
        ax += ra.s * g2y - (ra.cx * g4x + ra.cy * g4y);
        ay -= ra.s * g2x + (ra.cx * g4y - ra.cy * g4x);
      }
      // (computed here: the gathers' registers are loaded again below)
      asm volatile("" : "+v"(ax), "+v"(ay));
      ex[i] = ax;
      ey[i] = ay;
      if (C.te[i] < T) {
        s.Y[l & 0xffffu] = mk<TB>(yx, yy);
        if (!dg) s.Y[l >> 16] = mk<TB>(yx, -yy);
      }
    }
    // (2) the previous tile's stores, then this iteration's loads
    flush();
    int got = 0;
    // (a claim is left at the first of its tiles past the end, so that no such
    // tile stands in the pipeline before one of the next claim: claims of one
    // round interleave, and the loop ends at the first tile past the end)
    const bool fetch = claims && (taken == kClaim || i2 + step >= tile_end);
    if constexpr (kMore) {
      if (ENS && fetch && tid == 0)
        got = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      load_rec(t2);
      if constexpr (ENS) {
        const V* Hn = frag + (size_t)t1.member * nf;
#pragma unroll
        for (int j = 0; j < 2; ++j)
          hp[j] = *reinterpret_cast<const V*>(
              reinterpret_cast<const char*>(Hn) +
              (unsigned)min((int)pk_opaque(tid) + j * nth, nf - 1) * (unsigned)sizeof(V));
      }
    }
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (!EPI::kInIsState) pre[i] = epi.pre(tb, pk_opaque(C.off[i]));
    if constexpr (kMore) load_tile(t1, buf ^ 1);
    __syncthreads();
    // (3) matrix-core product; the records of the tile after the next
    packed_gemm<TB>(A, s, t0.nt * N);
    if constexpr (kMore) {
      put_rec(t2, buf);
      if (ENS && fetch && tid == 0) fetched = got;
    }
    __syncthreads();
    // (4) the tile after those in flight; epilogue of this tile
    TileInfo t3 = t2;
    int i3 = i2;
    if constexpr (kMore) {
      i3 = i2 + step;
      if (ENS && fetch) {
        i3 = claim_tile(step + __builtin_amdgcn_readfirstlane(fetched));
        taken = 0;
      }
      ++taken;
      if (i3 < tile_end) t3 = stream_tile<ENS>(A, i3);
    }
    have = 0;
    tb0 = tb;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      if (C.te[i] < t0.nt) {
        const unsigned l = pk_opaque(C.lds[i]);
        const V p = s.G[l & 0xffffu], q = s.G[l >> 16];
        out[i] = epi.apply(ex[i] + (p.x + q.x), ey[i] + (p.y - q.y), C.diag[i], pre[i], &emax);
        have |= 1u << i;
      }
    }
    t0 = t1;
    t1 = t2;
    t2 = t3;
    i1 = i2;
    i2 = i3;
    buf ^= 1;
  };
  while (i1 < tile_end) work(std::true_type{});
  work(std::false_type{});
  flush();
  if constexpr (EPI::kReduce) {
    __shared__ double red[16];
    for (int o = 32; o > 0; o >>= 1) {
      const double v = __shfl_xor(emax, o, 64);
      emax = v > emax ? v : emax;
    }
    if ((tid & 63) == 0) red[tid >> 6] = emax;
    __syncthreads();
    if (tid == 0) {
      double m = red[0];
      for (int w = 1; w < (int)(nth >> 6); ++w) m = red[w] > m ? red[w] : m;
      epi.finalize(m);
    }
  }
}

// H / hbar of every member as MFMA A-fragments (re, im), zero outside N x N.
template <typename TB>
__global__ void __launch_bounds__(256) build_hfrag(RhsArgs A, int members,
                                                   typename C2<TB>::type* __restrict__ out) {
  const int nf = StreamFragCount(A.N);
  const long long tot = (long long)members * nf;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < tot;
       i += (long long)gridDim.x * blockDim.x) {
    const int m = (int)(i / nf);
    const double2 h = stream_h_frag(A, A.H + (size_t)m * A.NE, (int)(i - (long long)m * nf));
    out[i] = mk<TB>((TB)(h.x * A.inv_hbar), (TB)(h.y * A.inv_hbar));
  }
}

// EpiIncr (heom_stream.h) on packed slabs.
template <typename TB, int STAGE>
struct PkIncr {
  typedef typename C2<TB>::type V;
  struct Pre { double2 x; V q; };
  typedef typename C2<typename std::conditional<STAGE == 3, double, TB>::type>::type Out;
  static constexpr bool kInIsState = STAGE <= 1;
  static constexpr bool kReduce = false;
  double* rho;
  const TB* kk;   // K (stages 2 and 3)
  TB* yout;
  double dt;
  __device__ __forceinline__ Pre pre(size_t tb, unsigned o) const {
    Pre p;
    p.q = pk_ld_nt(kk + tb, o);
    if (STAGE == 3) p.x = pk_ld_nt(rho + tb, o);
    return p;
  }
  __device__ __forceinline__ Pre from_state(double x, double y) const {
    Pre p;
    p.x = make_double2(x, y);
    return p;
  }
  __device__ __forceinline__ Out apply(TB kx, TB ky, bool, const Pre& p, double*) const {
    if constexpr (STAGE == 0) {
      return mk<TB>(kx, ky);
    } else if constexpr (STAGE == 1) {
      const TB c1 = (TB)(dt / 3), c0 = (TB)(dt / 4);
      return mk<TB>(c1 * ((TB)p.x.x + c0 * kx), c1 * ((TB)p.x.y + c0 * ky));
    } else if constexpr (STAGE == 2) {
      const TB c2 = (TB)(dt / 2);
      return mk<TB>(c2 * (p.q.x + kx), c2 * (p.q.y + ky));
    } else {
      return make_double2(p.x.x + dt * ((double)p.q.x + (double)kx),
                          p.x.y + dt * ((double)p.q.y + (double)ky));
    }
  }
  __device__ __forceinline__ void store(size_t tb, unsigned o, bool diag, const Out& v) const {
    if constexpr (STAGE == 3) pk_st_nt<double>(rho + tb, o, v, diag);
    else pk_st_nt<TB>(yout + tb, o, v, diag);
  }
  __device__ __forceinline__ void finalize(double) const {}
};

// EpiRkf45 (heom_stream.h) on packed slabs.
template <typename TB, int STAGE>
struct PkRkf45 {
  typedef typename C2<TB>::type V;
  struct Pre {
    double2 x;
    V k[5];
  };
  struct Out {
    V k;        // k_STAGE (stages 0..4)
    V tmp;      // the next stage's input
    double2 y;  // y5 (stage 5)
  };
  static constexpr bool kInIsState = STAGE == 0;
  static constexpr bool kReduce = STAGE == 5;
  Rkf45Bufs<TB> B;
  const double* rho;
  Rkf45Coefs cf;
  __device__ __forceinline__ Pre pre(size_t tb, unsigned o) const {
    Pre p;
    p.x = pk_ld(rho + tb, o);
#pragma unroll
    for (int j = 0; j < 5; ++j)
      if (j < STAGE && !(STAGE == 5 && j == 1)) p.k[j] = pk_ld(B.k[j] + tb, o);
    return p;
  }
  __device__ __forceinline__ Pre from_state(double x, double y) const {
    Pre p;
    p.x = make_double2(x, y);
    return p;
  }
  __device__ __forceinline__ Out apply(TB kx, TB ky, bool diag, const Pre& p,
                                       double* emax) const {
    Out r;
    const double ksx = (double)kx, ksy = (double)ky;
    if constexpr (STAGE < 5) {
      double sx = p.x.x, sy = p.x.y;
#pragma unroll
      for (int j = 0; j < 5; ++j)
        if (j < STAGE) {
          sx += (double)p.k[j].x * cf.b[STAGE][j];
          sy += (double)p.k[j].y * cf.b[STAGE][j];
        }
      sx += ksx * cf.b[STAGE][STAGE];
      sy += ksy * cf.b[STAGE][STAGE];
      r.k = mk<TB>(kx, ky);
      r.tmp = mk<TB>((TB)sx, (TB)sy);
    } else {
      const V k0 = p.k[0], k2 = p.k[2], k3 = p.k[3], k4 = p.k[4];
      const double y4x = p.x.x + (double)k0.x * cf.c4[0] + (double)k2.x * cf.c4[1] +
                         (double)k3.x * cf.c4[2] + (double)k4.x * cf.c4[3];
      const double y4y = p.x.y + (double)k0.y * cf.c4[0] + (double)k2.y * cf.c4[1] +
                         (double)k3.y * cf.c4[2] + (double)k4.y * cf.c4[3];
      const double y5x = p.x.x + (double)k0.x * cf.c5[0] + (double)k2.x * cf.c5[1] +
                         (double)k3.x * cf.c5[2] + (double)k4.x * cf.c5[3] + ksx * cf.c5[4];
      const double y5y = p.x.y + (double)k0.y * cf.c5[0] + (double)k2.y * cf.c5[1] +
                         (double)k3.y * cf.c5[2] + (double)k4.y * cf.c5[3] + ksy * cf.c5[4];
      r.y = make_double2(y5x, y5y);
      // (a diagonal element's second value belongs to its successor)
      const double d = diag ? fabs(y4x - y5x) : hypot(y4x - y5x, y4y - y5y);
      *emax = d > *emax ? d : *emax;
    }
    return r;
  }
  __device__ __forceinline__ void store(size_t tb, unsigned o, bool diag, const Out& v) const {
    if constexpr (STAGE < 5) {
      pk_st<TB>(B.k[STAGE] + tb, o, v.k, diag);
      pk_st<TB>(B.tmp_out + tb, o, v.tmp, diag);
    } else {
      pk_st<double>(B.rho_new + tb, o, v.y, diag);
    }
  }
  __device__ __forceinline__ void finalize(double m) const { atomic_max_nonneg(B.err, m); }
};

}  // namespace dev

// --- Launch -------------------------------------------------------------------------

int ResidentBlocks(const void* kernel, int threads, size_t lds);

// Threads of a packed block: the elements per thread `ept` of the
// requested shape, rounded up to whole wavefronts; an ensemble block also
// prefetches a member's H fragments two per thread.
inline int PackedThreads(const RhsArgs& a, int ept, bool ens) {
  int th = ((a.tile * a.PE + ept - 1) / ept + 63) / 64 * 64;
  // (17 to 19 sites: a wave more than the elements need, so that the four
  // items of a node's product are one round: 18 17-site nodes, FP64, 6.0 us
  // a stage without, 5.1 with)
  if (a.N > 16 && ept == 1 && th < 256) th = 256;
  if (ens) th = th > (dev::StreamFragCount(a.N) / 2 + 63) / 64 * 64
                    ? th : (dev::StreamFragCount(a.N) / 2 + 63) / 64 * 64;
  return th;
}

template <typename TB, typename TI, int EPT, int MPS, bool ENS, class EPI>
inline hipError_t LaunchPackedKE(const RhsArgs& a, const TI* in, const EPI& epi, int grid,
                                 hipStream_t s) {
  const int threads = PackedThreads(a, EPT, ENS);
  const size_t sh = dev::PackedLdsBytes(a.N, a.D, a.L, MPS, a.tile, sizeof(TB));
  const void* k = reinterpret_cast<const void*>(&dev::packed_stage<TB, TI, EPT, MPS, ENS, EPI>);
  const int ntiles = ENS ? a.ntiles : (a.num_nodes + a.tile - 1) / a.tile;
  if (threads > 512) return hipErrorInvalidConfiguration;
  int g = grid > 0 ? grid : ResidentBlocks(k, threads, sh);
  if (g > ntiles) g = ntiles;
  if (g < 1) g = 1;
  hipLaunchKernelGGL((dev::packed_stage<TB, TI, EPT, MPS, ENS, EPI>), dim3(g), dim3(threads), sh,
                     s, a, in, epi);
  return hipGetLastError();
}

template <typename TB, typename TI, int EPT, int MPS, class EPI>
inline hipError_t LaunchPackedK(const RhsArgs& a, const TI* in, const EPI& epi, int grid,
                                hipStream_t s) {
  if (a.tiles) return LaunchPackedKE<TB, TI, EPT, MPS, true, EPI>(a, in, epi, grid, s);
  return LaunchPackedKE<TB, TI, EPT, MPS, false, EPI>(a, in, epi, grid, s);
}

// The shape of a precision: pk_tile nodes per block; the requested threads
// give the elements per thread they would have with full nodes (1..4).
template <typename TB, typename TI, class EPI>
inline hipError_t LaunchPacked(const RhsArgs& a0, const TI* in, const EPI& epi, hipStream_t s) {
  const int f = sizeof(TB) == 4 ? 1 : 0;
  RhsArgs a = a0;
  a.tile = a0.pk_tile[f];
  int full = (a0.col_tile[f] * a0.NE + a0.col_threads[f] - 1) / a0.col_threads[f];
  if (full == 1 && a.tile * a.PE > 512) full = 2;
  const int grid = a0.col_grid[f];
  if (a.mps <= 1) {
    switch (full) {
      case 1: return LaunchPackedK<TB, TI, 1, 1, EPI>(a, in, epi, grid, s);
      case 2: return LaunchPackedK<TB, TI, 2, 1, EPI>(a, in, epi, grid, s);
      default: return LaunchPackedK<TB, TI, 4, 1, EPI>(a, in, epi, grid, s);
    }
  }
  switch (full) {
    case 1: return LaunchPackedK<TB, TI, 1, 2, EPI>(a, in, epi, grid, s);
    case 2: return LaunchPackedK<TB, TI, 2, 2, EPI>(a, in, epi, grid, s);
    default: return LaunchPackedK<TB, TI, 4, 2, EPI>(a, in, epi, grid, s);
  }
}

}  // namespace phi

#endif  // PHI_AMD_HEOM_PACKED_H_
