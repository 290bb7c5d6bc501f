// Device argument blocks and launchers of the HEOM kernels (heom_kernels.hip).
#ifndef PHI_AMD_HEOM_KERNELS_H_
#define PHI_AMD_HEOM_KERNELS_H_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace phi {

// Tile of an ensemble slab: slab nodes base .. base + nt - 1 are the local
// nodes local .. local + nt - 1 of `member`, which has `count` nodes.
// 32 bytes, so a block reads one with a single scalar load.
struct __attribute__((aligned(32))) TileDesc {
  int base, local, nt, member, count, pad0, pad1, pad2;
};

// Everything the RHS of one hierarchy needs, as device pointers.
struct RhsArgs {
  int N, NE, D, L, num_nodes, tile, vacuum;
  // Form of the stage kernels: col_nm = 0 element path (H from LDS),
  // 1 matrix-core path (v_mfma 16x16x4, N <= 32), 2 persistent pipelined
  // matrix-core kernels (heom_stream.h; N <= 32, at most 2 modes per
  // site).  Nodes, threads and blocks (0 = as many as fit) per launch, per
  // precision ([0] FP64, [1] FP32).
  int col_nm;
  int col_tile[2];
  int col_threads[2];
  int col_grid[2];
  // Tile of the one-shot kernels when col_nm == 2 (their block is 256
  // threads): RKF45 stages, which have no persistent form.
  int v1_tile[2];
  // Edge records of the persistent kernels: edge[(n*N + b)*mps + q] =
  // {id of n + e_j, id of n - e_j, j*L + n_j, 0} for the q-th mode j of
  // site b ({-1, -1, -1, 0} when absent).
  const int4* edge;
  int mps;
  // Packed Hermitian kernels (heom_packed.h): PE = N (N + 1) / 2 elements per
  // node, elem[e] = {row, column, real offset, 0} in storage order; nodes per
  // block per precision.
  int PE;
  int pk_tile[2];
  const int4* elem;
  const void* hfrag;           // H / hbar fragments in the bulk precision, per member
  unsigned long long mPE, mNM; // ceil(2^32 / PE), ceil(2^32 / (N mps))
  // Ensembles (persistent kernels only): slab of several members of one
  // bath model sharing the tables of the deepest member.  tiles[t] describes
  // tile t (TileDesc) and H holds every member's shifted H (stride N*N).
  // tiles is nullptr for a single hierarchy.
  const TileDesc* tiles;
  int ntiles;
  // Packed kernels: two sets of the 8 runs' claim counters, 64 bytes apart;
  // a launch uses set ctr_set and clears the other for the next launch.
  int* tile_ctr;
  int ctr_set;
  int real_h;                 // imag(H) == 0 everywhere
  unsigned long long mN, mNE; // ceil(2^32 / N), ceil(2^32 / N^2)
  double inv_hbar;
  const int* next;          // [num_nodes * D]
  const int* prev;          // [num_nodes * D]
  const uint8_t* occ;       // [num_nodes * D]
  const double* mu;         // [num_nodes]
  const int* site_ptr;      // [N + 1]
  const int* site_modes;    // [D]
  const double* next_s;     // [D * L]
  const double2* prev_col;  // [D * L]
  const double2* prev_row;  // [D * L]
  const double* delta;      // [N]
  const double2* H;         // N*N, shifted by mean(diag H) (Hermitian path)
  const double2* Hraw;      // N*N, as given (general path)
  const double2* Hadj;      // N*N, conjugate transpose of Hraw
};

template <typename TB>
struct Rkf45Bufs {
  TB* k[5];                  // k0..k4 (bulk precision)
  TB* tmp_out;               // next stage input
  double* rho_new;           // y5 (FP64)
  unsigned long long* err;   // max |y4 - y5| as the bits of a double
};

// RKF45 weights already multiplied by the current dt (host keeps PHI's
// in-place rescaling).  b[s][i]: stage-(s+1) input weights; c4: weights of
// k0,k2,k3,k4 in y4; c5: weights of k0,k2,k3,k4,k5 in y5.
struct Rkf45Coefs {
  double b[5][5];
  double c4[4];
  double c5[5];
};

// Dynamic LDS of one block; `a.tile` must already be the launch's tile.
size_t RhsSharedBytes(const RhsArgs& a, bool fp32);
// LDS bytes of a tile of `tile` nodes (with_h: H staged in LDS, i.e. every
// GEMM form except the matrix-core one).
size_t TileLdsBytes(int N, int D, int L, int tile, bool fp32, bool with_h);
// LDS bytes of a block of the persistent kernels (two tiles in flight).
size_t StreamTileLdsBytes(int N, int D, int L, int tile, bool fp32);

// Stage orders of an RK4 step: PHI's classic order (FP64 accumulator), the
// nested (Horner) order and its increment form (heom_stream.h; persistent
// kernels only).
// kRk4ClassicBulk: PHI's classic order with a bulk-precision accumulator and
// a bulk copy of rho (internal: the learned closure's FP32 runs, whose RHS
// is not linear; persistent kernels only).
enum { kRk4Classic = 0, kRk4Nested = 1, kRk4Increment = 2, kRk4ClassicBulk = 3 };
// One RK4 stage.  aux: the classic form's FP64 accumulator, or the
// increment form's K (bulk precision); unused by the nested form.
hipError_t LaunchRk4Stage(const RhsArgs& a, bool fp32, int stage, int form, const void* in,
                          double* rho, void* aux, void* yout, double dt, hipStream_t s);
hipError_t LaunchRkf45Stage(const RhsArgs& a, bool fp32, int stage, const void* in,
                            const double* rho, const Rkf45Bufs<float>& bf,
                            const Rkf45Bufs<double>& bd, const Rkf45Coefs& c, hipStream_t s);

// Packed Hermitian slabs (heom_packed.h).  LDS bytes of a block.
size_t PackedTileLdsBytes(int N, int D, int L, int mps, int tile, bool fp32);
// Reals past a slab's end that a short tile's loads touch (a tile is at most
// 1024 reals): every buffer a packed stage reads is this much longer, and the
// tables by the nodes that hold as many.
constexpr int kPackedPad = 1024 + 64;
// The increment form's stage and RKF45's on packed slabs (rho, K, yout and
// the RKF45 buffers all packed).
hipError_t LaunchRk4Packed(const RhsArgs& a, bool fp32, int stage, const void* in, double* rho,
                           const void* kk, void* yout, double dt, hipStream_t s);
hipError_t LaunchRkf45Packed(const RhsArgs& a, bool fp32, int stage, const void* in,
                             const double* rho, const Rkf45Bufs<float>& bf,
                             const Rkf45Bufs<double>& bd, const Rkf45Coefs& c, hipStream_t s);
// hfrag (members x fragment elements, complex of the bulk precision) from a.H.
size_t PackedFragElems(int N);
hipError_t LaunchBuildFrag(const RhsArgs& a, bool fp32, int members, void* out, hipStream_t s);
// A small hierarchy's steps inside one workgroup (heom_resident.hip): whether
// it fits, and nsteps steps of the packed state rho in one launch, recording
// node 0 after every step i with (step_offset + i) % snap_every == 0.
bool ResidentFits(const RhsArgs& a, bool fp32);
hipError_t LaunchResidentRk4(const RhsArgs& a, bool fp32, double* rho, long long nsteps,
                             double dt, long long step_offset, int snap_every, double* hist,
                             int* counter, int capacity, hipStream_t s);
// packed <- full; *flag (zeroed before; device or pinned host memory) = 1
// unless every ADO equals its conjugate transpose exactly.
hipError_t LaunchPack(const RhsArgs& a, int nodes, const double* full, double* packed, int* flag,
                      hipStream_t s);
// full <- packed for `nodes` nodes.
hipError_t LaunchUnpack(const RhsArgs& a, int nodes, const double* packed, double* full,
                        hipStream_t s);
// LaunchSnapshot, LaunchSnapshotMean and LaunchGatherNode0 from a packed
// slab; place[e] = 4 * offset + (0 diagonal, 1 upper, 2 lower triangle) of
// column-major element e.
hipError_t LaunchSnapshotPacked(const double* src, const int* place, double* hist, int* counter,
                                int ne, int capacity, hipStream_t s);
hipError_t LaunchSnapshotMeanPacked(const double* src, const int* place,
                                    const int* member_offsets, int members, double* hist,
                                    int* counter, int ne, int capacity, hipStream_t s);
hipError_t LaunchGatherNode0Packed(const double* src, const int* place, const int* member_offsets,
                                   int members, int ne, double* dst, hipStream_t s);
// PHI's Get on any complex input, FP64.  active: the adaptive truncation's
// node flags (inactive neighbours' terms skipped), or null.
hipError_t LaunchRhsGeneral(const RhsArgs& a, const double* x, double* y, int trace_row,
                            hipStream_t s, const unsigned char* active = nullptr);
// Blocks of LaunchRhsGeneralDot (one partial record each), 0 when its LDS
// form does not fit (then it returns hipErrorInvalidValue).
int RhsGeneralDotBlocks(const RhsArgs& a);
// LaunchRhsGeneral (no active flags) fused with the next reductions of the
// steady-state solver, per block: dot 1 = sum conj(w) y (2 doubles), dot 2 =
// |w|^2, 0, conj(w) w2 and conj(w) y (6 doubles), dot 3 = sums of conj(y) w,
// |y|^2, conj(w2) y and conj(w2) w (7 doubles).
hipError_t LaunchRhsGeneralDot(const RhsArgs& a, const double* x, double* y, int trace_row,
                               int dot, const double* w, const double* w2, double* partial,
                               hipStream_t s);
hipError_t LaunchSnapshot(const double* src, double* hist, int* counter, int ne, int capacity,
                          hipStream_t s);
// hist[slot] = mean over the members of their node 0 (fixed summation order).
hipError_t LaunchSnapshotMean(const double* src, const int* member_offsets, int members,
                              double* hist, int* counter, int ne, int capacity, hipStream_t s);
// dst (members x ne complex) = node 0 of every member.
hipError_t LaunchGatherNode0(const double* src, const int* member_offsets, int members, int ne,
                             double* dst, hipStream_t s);
hipError_t LaunchFillU64(unsigned long long* p, unsigned long long v, int n, hipStream_t s);
hipError_t LaunchCastToFloat(const double* src, float* dst, size_t n, hipStream_t s);
// Basis change of every ADO of a slab: a_n <- R a_n R^dagger (R N x N,
// column-major, on the device), in FP64 arithmetic; buf holds FP64 or FP32
// interleaved complex ADOs.
hipError_t LaunchRotateNodes(void* buf, bool fp32, const double2* R, int N, int nodes,
                             hipStream_t s);
hipError_t LaunchDot(const double* u, const double* v, size_t n, int mode, double* partial,
                     int nblocks, double* out, hipStream_t s);
hipError_t LaunchLincomb(double* y, size_t n, int nv, const double* const* x, const double2* c,
                         hipStream_t s);

// BiCGSTAB with its scalars on the device (no host round trip inside an
// iteration).  An iteration is four kernels: v = A p (with the partials of
// rhat . v), the s update (which first closes the previous iteration), t =
// A s (with the partials of t . s, |t|^2, rhat . t, rhat . s) and the
// x/r/p update (with the partials of |r|^2).  The dot products land in this
// struct; the update kernels derive their coefficients from it; the finish
// kernel closes the last iteration of a batch.
struct BicgScalars {
  double2 rho_old, alpha, omega;  // from the previous iteration (1, 1, 1 at start)
  double2 rho_new, rv, ts, tt, rn2;  // dot products of the current iteration
  double2 rho_next;               // rhat . r of the new r (the next rho_new)
  double res;                     // |r| after the last finished iteration
  int done;                       // converged, breakdown (omega = 0) or max_iter
  int it;                         // finished iterations
};
// Reductions are two-pass with a fixed order: a kernel writes one partial
// per block, and the kernel that needs the value sums the partials itself
// (every block the same way), so no single-block reduction kernel runs.
//
// Partials of conj(u) . v (2 doubles per block).
hipError_t LaunchDotPartial(const double* u, const double* v, size_t n, double* partial,
                            int nblocks, hipStream_t s);
// s = r - alpha v for record cur (rv = sum of the nb partials of rhat . v,
// kept in cur, alpha = rho_new / rv); close = true first closes the
// previous iteration (record prev, its nbx |r|^2 partials) into cur, as
// LaunchBicgFinish does.  Nothing once the (closed) record is done.
hipError_t LaunchBicgS(bool close, double* y, size_t n, const double* r, const double* v,
                       const BicgScalars* prev, BicgScalars* cur, const double* rv_part, int nb,
                       const double* xr_part, int nbx, double* hist, double tol, int max_iter,
                       hipStream_t s);
// Partials of conj(t) s, |t|^2, conj(rhat) t, conj(rhat) s (7 doubles per
// block): the matvec's dot 3 on its own.
hipError_t LaunchBicgDots(const double* t, const double* sv, const double* rhat, size_t n,
                          double* partial7, int nblocks, hipStream_t s);
// From those partials: omega = ts / tt (0 if tt = 0), rho_next = rhat . s -
// omega rhat . t (= rhat . r_new), beta; x += alpha p + omega s, r = s -
// omega t, p = r + beta (p - omega v), partials of |r|^2 (1 double per
// block); ts, tt, rho_next kept in st.  Nothing once st->done.
hipError_t LaunchBicgXRP(double* x, double* r, double* p, const double* sv, const double* t,
                         const double* v, size_t n, BicgScalars* st, const double* ts_part,
                         int nb_ts, double* partial, int nblocks, hipStream_t s);
// Closing an iteration: from record prev and the |r|^2 partials, the record
// next of the following iteration (rn2; alpha, omega, rho_old <- this
// iteration's, rho_new <- rho_next; res = |r|; hist[it] = res; done when
// !(res > tol), omega = 0 or it = max_iter).  One block.
hipError_t LaunchBicgFinish(const BicgScalars* prev, BicgScalars* next, const double* xr_part,
                            int nblocks, double* hist, double tol, int max_iter, hipStream_t s);

// BiCGSTAB(ell) with its scalars on the device (Sleijpen and Fokkema 1993,
// Algorithm 3.1).  Dot products land in dot[0..3], and a scalar step on one
// thread derives the scalars from them; the vector updates take their
// coefficient from this record.  stop (breakdown,
// convergence or the step cap) turns every later step and update into a
// no-op, so whole cycles can be enqueued ahead of the host's check.
constexpr int kBicglMaxEll = 8;
struct BicglScalars {
  double2 dot[4];
  double2 rho0, alpha, omega, beta;
  double2 tau[kBicglMaxEll + 1][kBicglMaxEll + 1];
  double2 gp[kBicglMaxEll + 1], g[kBicglMaxEll + 1], gpp[kBicglMaxEll + 1];
  double sigma[kBicglMaxEll + 1];
  double res;   // |r_0| after the last finished cycle
  int stop;     // broke || converged || it >= max_iter
  int broke;
  int it;       // BiCG steps of the finished cycles
  int cycles;   // finished cycles
};
// Scalar steps (one thread):
//   kBlInit   res = sqrt(dot[2]), rho0 = 1, alpha = 0, omega = 1, hist[0];
//             then the first cycle's start
//   kBlBeta   rho1 = dot[0]: beta = alpha rho1 / rho0, rho0 = rho1
//   kBlAlpha  alpha = rho0 / dot[0]
//   kBlTau    tau[i][j] = dot[0] / sigma[i]
//   kBlSigma  sigma[j] = dot[0], gp[j] = dot[1] / sigma[j]; for j = i
//             (= ell) also g, gpp from tau and gp, omega = g[ell]
//   kBlEnd    res = sqrt(dot[2]), it += ell (= i), hist[cycles]; stop; then
//             the next cycle's start
// A cycle's start is rho0 = -omega rho0 and its first BiCG step's beta with
// rho1 = dot[3] = (rtilde, r_0).  A zero rho0 or dot[0] (alpha) or a
// non-positive sigma, or omega = 0 at the end, is a breakdown.
enum { kBlInit = 0, kBlBeta, kBlAlpha, kBlTau, kBlSigma, kBlEnd };
// Two dot products in one pass, conj(a) . b into S->dot[k] and conj(c) . d
// into S->dot[k + 1] (k = 0..2), then the scalar step op, by a kernel of one
// block; partial holds 4 doubles per block (nblocks blocks).
hipError_t LaunchBicglDot2Step(const double* a, const double* b, const double* c,
                               const double* d, size_t n, double* partial, int nblocks,
                               BicglScalars* S, int k, int op, int i, int j, double tol,
                               int max_iter, double* hist, int hist_cap, hipStream_t s);
// Inside a batch of cycles no kernel runs only to reduce: the pass that needs
// a scalar sums the nb partials of the pass before it and takes the scalar
// step in every block alike; block 0 writes the record for the next pass to
// out, which is not in (the other blocks still read that).  op kBlSigma takes
// 6 doubles a block (|r_j|^2, 0, conj(r_j) r_0, conj(r_1) r_{j+1}) and, for
// j < i, is followed by kBlTau (1, j + 1); kBlEnd takes 4, kBlNone nothing
// (in is final), the others 2.  A cycle of ell = 2 over 6435 7-site nodes
// took 22 launches and 130 us with a reduction kernel (4 us) per scalar and
// a pass per update, 10 and about 105 us this way; the passes now run at the rate of
// their 5 MB vectors (4.6 TB/s in the end of a cycle) plus 3 us a step.
// Loads issued behind the partials' ahead of the step: slower (15.6 against
// 14.0 ms a solution), half the blocks in the Gram-Schmidt pass: 14.2.
constexpr int kBlNone = -1;
constexpr int kBicglBlocks = 1024;  // most blocks of the passes below
struct BicglTake {
  const BicglScalars* in;
  BicglScalars* out;
  const double* part;
  int nb, op, i, j;
  double tol;
  int max_iter;
  double* hist;
  int hist_cap;
};
// Several updates with one coefficient, one pass: y_p = a_p + sign_p *
// c * b_p for p < count (count <= kBicglMaxEll + 1; no y_p may be an
// input of another pair), c = alpha or beta; nothing once stopped.
struct ZPairs {
  double* y[kBicglMaxEll + 1];
  const double* a[kBicglMaxEll + 1];
  const double* b[kBicglMaxEll + 1];
  double sign[kBicglMaxEll + 1];
  int count;
};
hipError_t LaunchBicglPairs(const ZPairs& pr, size_t n, const BicglTake& t, bool alpha,
                            hipStream_t s);
// y -= tau[ti][tj] b (b null: no update and no step), then the partials of
// conj(a) y (2 doubles a block), or with norm |y|^2, 0, conj(y) a and, c
// non-null, conj(c) d (6 doubles); *blocks = the blocks.  c and d are not y.
hipError_t LaunchBicglGram(double* y, const double* b, const double* a, const double* c,
                           const double* d, bool norm, size_t n, const BicglTake& t, int ti,
                           int tj, double* partial, int* blocks, hipStream_t s);
// x += g_1 r_0 + sum gpp_j r_j, then r_0 -= gp_ell r_ell + sum gp_j r_j and
// u_0 -= g_ell u_ell + sum g_j u_j, and the partials of |r_0|^2 and (rt, r_0).
struct BicglVectors {
  double* r[kBicglMaxEll + 1];
  double* u[kBicglMaxEll + 1];
};
hipError_t LaunchBicglEnd(double* x, const BicglVectors& v, int ell, const double* rt, size_t n,
                          const BicglTake& t, double* partial, int* blocks, hipStream_t s);
// The step alone, one block (out may be in).
hipError_t LaunchBicglFinish(const BicglTake& t, hipStream_t s);

}  // namespace phi

#endif  // PHI_AMD_HEOM_KERNELS_H_
