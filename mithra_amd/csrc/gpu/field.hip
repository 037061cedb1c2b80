// Field kernels: interior NSFD/FD update, TF/SF seed injection, Mur absorbing boundaries
// and the E/B evaluation, for one domain resident in HBM.
//
// All arithmetic keeps the reference's source order and the library is built with
// -ffp-contract=off, so on identical inputs the FP64 path reproduces the reference's
// potentials bit for bit.
#include <algorithm>
#include <cmath>
#include <initializer_list>
#include <utility>
#include <vector>

#include "common.h"

namespace mithra {

namespace {

constexpr int kTileJ = 64;      // one wavefront along y (contiguous in memory)
constexpr int kNumXcd = 8;      // MI355X: 8 accelerator complex dies, each with its own L2

// Workgroups are dispatched round-robin over the XCDs (workgroup b runs on XCD b % 8).
// Returns the logical tile of workgroup b such that every XCD receives one contiguous range
// of logical tiles: neighbouring tiles, which share their halo rows, then meet in one L2.
__device__ inline int xcd_logical_block(int b, int nblk) {
  int q = nblk / kNumXcd, r = nblk % kNumXcd;
  int xcd = b % kNumXcd, local = b / kNumXcd;
  int base = (xcd < r) ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q;
  return base + local;
}

template <typename PT>
__device__ inline double rd(PT p, long m) { return (double)p[m]; }

struct Plane5 {  // one z plane of a column and its four transverse neighbours
  double c, xp, xm, yp, ym;
};

template <typename PT>
__device__ inline Plane5 load_plane(PT a, long m, long N1) {
  Plane5 p;
  p.c = (double)a[m];
  p.xp = (double)a[m + N1];
  p.xm = (double)a[m - N1];
  p.yp = (double)a[m + 1];
  p.ym = (double)a[m - 1];
  return p;
}

// Interior update (AdvanceField::advance*PotentialNSFD / FD, reference src/database.cpp:44-134,
// loops src/fdtd.cpp:270-303 and src/fdtdSC.cpp:317-366).  Each thread owns one (i, j) column
// and marches kChunkK planes along z with the three planes it needs held in registers; the
// x/y neighbours it reads are the centres of neighbouring lanes and rows, served by L1/L2.
// J (or rho) lives in the A^{n+1} buffer and is overwritten in place, as in the reference.
template <typename R, bool NSFD, int TI, int K, bool FACES = false>
__device__ inline void interior_body(FieldSet an_set, FieldSet anm1_set, FieldSet anp1_set, int ncomp, int N0,
                                     int N1, int N2, int tilesJ, int tilesI, int chunks, double a0, double a1,
                                     double a2, double a3, double a4, double a5, double alpha, double beta, int lb,
                                     const MurYFace& yf = MurYFace{}) {
  const int tj = lb % tilesJ;
  lb /= tilesJ;
  const int ti = lb % tilesI;
  lb /= tilesI;
  const int kc = lb % chunks;
  const int comp = lb / chunks;
  const int lane = threadIdx.x % kTileJ;
  const int j = tj * kTileJ + lane;
  const int i = 1 + ti * TI + (threadIdx.x / kTileJ);
  const int kb = 1 + kc * K;
  const int ke = min(kb + K, N2 - 1);
  if (comp >= ncomp || kb >= ke) return;  // uniform over the workgroup
  // FACES: as in interior_lds_body, the lanes of the face nodes j = 0 and N1-1 update the Mur y
  // faces in `yf.mask`; they take the inward neighbour's new value, its A^{n-1} and its x
  // neighbours of A^n by lane shuffle, and their own A^n column from their register queue.
  const bool face_tile = FACES && (tj == 0 || tj == (N1 - 1) / kTileJ);
  const bool active = i <= N0 - 2 && j >= 1 && j <= N1 - 2;
  const bool face = FACES && i <= N0 - 2 && (((yf.mask & 1) && j == 0) || ((yf.mask & 2) && j == N1 - 1));
  if (!active && !face_tile) return;
  const bool load = active || face;
  const int fs = j == 0 ? 1 : -1;
  const int nb_lane = max(lane + fs, 0);
  const gptr<const R> an = G((const R*)component(an_set, comp));
  const gptr<const R> anm1 = G((const R*)component(anm1_set, comp));
  const gptr<R> anp1 = G((R*)component(anp1_set, comp));
  const double as = comp < 3 ? a4 : a5;
  const long N1N0 = (long)N1 * N0;
  long m = N1N0 * kb + (long)N1 * i + j;
  Plane5 pm = {}, p0 = {};
  if (load) {
    pm = load_plane(an, m - N1N0, N1);
    p0 = load_plane(an, m, N1);
  }
  for (int k = kb; k < ke; ++k, m += N1N0) {
    Plane5 pp = {};
    double v1 = 0.0, r = 0.0;
    if (load) {
      pp = load_plane(an, m + N1N0, N1);
      v1 = (double)ld_stream(anm1, m);
    }
    if (active) {
      const double src = (double)ld_stream(G((const R*)component(anp1_set, comp)), m);
      if (NSFD) {
        double tx = p0.xp + p0.xm + beta * (pp.xp + pm.xp + pp.xm + pm.xm);
        double ty = p0.yp + p0.ym + beta * (pp.yp + pm.yp + pp.ym + pm.ym);
        r = a0 * p0.c - v1 + alpha * (a1 * tx + a2 * ty) + a3 * (pp.c + pm.c) + as * src;
      } else {
        r = a0 * p0.c - v1 + a1 * (p0.xp + p0.xm) + a2 * (p0.yp + p0.ym) + a3 * (pp.c + pm.c) + as * src;
      }
      st_stream(anp1, m, (R)r);
    }
    if (face_tile) {
      const double pn = __shfl((double)(R)r, nb_lane);
      const double mn = __shfl(v1, nb_lane);
      const double nxp = __shfl(p0.xp, nb_lane), nxm = __shfl(p0.xm, nb_lane);
      if (face) {
        const double* B = yf.B;
        const double ns = fs > 0 ? p0.yp : p0.ym, nsp = fs > 0 ? pp.yp : pp.ym, nsm = fs > 0 ? pm.yp : pm.ym;
        anp1[m] = (R)(B[0] * (v1 + pn) + B[1] * mn + B[2] * (p0.c + ns) + B[3] * (nxp + nxm + p0.xp + p0.xm) +
                      B[4] * (nsp + nsm + pp.c + pm.c));
      }
    }
    pm = p0;
    p0 = pp;
  }
}

template <typename R, bool NSFD, int TI, int K, bool FACES>
__global__ __launch_bounds__(kTileJ* TI) void k_interior(
    FieldSet an_set, FieldSet anm1_set, FieldSet anp1_set, int ncomp, int N0, int N1, int N2,
    int tilesJ, int tilesI, int chunks, double a0, double a1, double a2, double a3, double a4, double a5,
    double alpha, double beta, MurYFace yf) {
  interior_body<R, NSFD, TI, K, FACES>(an_set, anm1_set, anp1_set, ncomp, N0, N1, N2, tilesJ, tilesI, chunks, a0,
                                       a1, a2, a3, a4, a5, alpha, beta, xcd_logical_block(blockIdx.x, gridDim.x), yf);
}

// The interior update with the A^n planes staged in LDS (2.5-D blocking).  The workgroup (TI
// wavefronts, one x-row of 64 y-nodes each) marches its K planes in lockstep: plane k+1 of its
// tile plus a one-node halo ring is fetched once, coalesced, into a three-plane LDS ring, and
// every neighbour of the stencil is read from LDS.  Same arithmetic, in the same order, as
// k_interior.
//
// FACES: the workgroups of the first and last tile columns also update the Mur y faces in
// `yf.mask` (mur_face below with s = +-1 along y, t along x, u along z): the lane of face node
// j = 0 (N1-1) takes the new value and the A^{n-1} value of node j = 1 (N1-2) from the
// neighbouring lane and the A^n values from the LDS ring, so the faces cost no extra HBM pass.
// Valid only when nothing writes A^{n+1} between the interior update and the boundaries.
template <typename R, bool NSFD, int TI, int K, bool FACES = false>
__device__ inline void interior_lds_body(FieldSet an_set, FieldSet anm1_set, FieldSet anp1_set, int ncomp, int N0,
                                         int N1, int N2, int tilesJ, int tilesI, int chunks, double a0, double a1,
                                         double a2, double a3, double a4, double a5, double alpha, double beta,
                                         int lb, const MurYFace& yf = MurYFace{}) {
  constexpr int W = kTileJ + 2;           // LDS row: y-halo, 64 nodes, y-halo
  constexpr int P = (TI + 2) * W;         // one plane of the tile with its halo ring
  __shared__ double L[3 * P];
  const int tj = lb % tilesJ;
  lb /= tilesJ;
  const int ti = lb % tilesI;
  lb /= tilesI;
  const int kc = lb % chunks;
  const int comp = lb / chunks;
  const int kb = 1 + kc * K;
  const int ke = min(kb + K, N2 - 1);
  if (comp >= ncomp || kb >= ke) return;  // uniform over the workgroup
  const int lane = threadIdx.x % kTileJ, w = threadIdx.x / kTileJ;
  const int j0 = tj * kTileJ, i0 = 1 + ti * TI;
  const int j = j0 + lane, i = i0 + w;
  const bool active = i <= N0 - 2 && j >= 1 && j <= N1 - 2;
  const gptr<const R> an = G((const R*)component(an_set, comp));
  const gptr<const R> anm1 = G((const R*)component(anm1_set, comp));
  const gptr<R> anp1 = G((R*)component(anp1_set, comp));
  const double as = comp < 3 ? a4 : a5;
  const long N1N0 = (long)N1 * N0;
  // What this thread stages per plane: its own node, and (wave 0 / wave 1) the halo rows
  // i0-1 / i0+TI, and (lanes < 2 TI of wave 0) the halo columns j0-1 / j0+64 of rows i0..i0+TI-1.
  const bool own_ok = i <= N0 - 1 && j <= N1 - 1;
  const long own_off = (long)N1 * i + j;
  const int own_slot = (w + 1) * W + lane + 1;
  int hrow_i = -1, hrow_slot = 0;
  if (w == 0) { hrow_i = i0 - 1; hrow_slot = lane + 1; }
  if (w == 1) { hrow_i = i0 + TI; hrow_slot = (TI + 1) * W + lane + 1; }
  const bool hrow_ok = hrow_i >= 0 && hrow_i <= N0 - 1 && j <= N1 - 1;
  const long hrow_off = (long)N1 * hrow_i + j;
  int hcol_j = -1, hcol_i = 0, hcol_slot = 0;
  if (w == 0 && lane < TI) { hcol_i = i0 + lane; hcol_j = j0 - 1; hcol_slot = (lane + 1) * W; }
  if (w == 0 && lane >= TI && lane < 2 * TI) {
    hcol_i = i0 + lane - TI; hcol_j = j0 + kTileJ; hcol_slot = (lane - TI + 1) * W + kTileJ + 1;
  }
  const bool hcol_ok = hcol_j >= 0 && hcol_j <= N1 - 1 && hcol_i <= N0 - 1;
  const long hcol_off = (long)N1 * hcol_i + hcol_j;
  // y faces: tile columns that hold a face node (uniform over the workgroup), the face lanes,
  // and the lane each reads its inward neighbour from
  const bool face_tile = FACES && (tj == 0 || tj == (N1 - 1) / kTileJ);
  const int fs = j == 0 ? 1 : -1;
  const bool face = FACES && i <= N0 - 2 && (((yf.mask & 1) && j == 0) || ((yf.mask & 2) && j == N1 - 1));
  const int nb_lane = max(lane + fs, 0);
  // Prefetched values stay in the storage type until they are staged or used: a conversion
  // right after a load would make the wave wait for that load there (FP32-bulk).
  R r_own = 0, r_row = 0, r_col = 0;
  auto fetch = [&](int k) {
    const long b = N1N0 * k;
    if (own_ok) r_own = an[b + own_off];
    if (hrow_ok) r_row = an[b + hrow_off];
    if (hcol_ok) r_col = an[b + hcol_off];
  };
  auto stage = [&](int slot) {
    double* p = L + slot * P;
    if (own_ok) p[own_slot] = (double)r_own;
    if (hrow_ok) p[hrow_slot] = (double)r_row;
    if (hcol_ok) p[hcol_slot] = (double)r_col;
  };
  // A^{n-1} and J of the next plane are loaded one plane ahead, like the A^n planes, so their
  // latency overlaps the current plane's work.
  const gptr<const R> jsrc = G((const R*)component(anp1_set, comp));
  const bool need_m1 = active || face;
  R v1_next = 0, src_next = 0;
  fetch(kb - 1);
  stage(0);
  fetch(kb);
  stage(1);
  fetch(kb + 1);
  long m = N1N0 * kb + own_off;
  if (need_m1) v1_next = anm1[m];
  if (active) src_next = jsrc[m];
  for (int k = kb; k < ke; ++k, m += N1N0) {
    const int s0 = (k - kb + 1) % 3, sp = (k - kb + 2) % 3, sm = (k - kb) % 3;
    const double v1 = (double)v1_next, src = (double)src_next;
    stage(sp);
    __syncthreads();
    if (k + 2 <= ke) fetch(k + 2);
    if (k + 1 < ke) {
      if (need_m1) v1_next = anm1[m + N1N0];
      if (active) src_next = jsrc[m + N1N0];
    }
    const double* c0 = L + s0 * P + own_slot;
    const double* cp = L + sp * P + own_slot;
    const double* cm = L + sm * P + own_slot;
    double r = 0.0;
    if (active) {
      if (NSFD) {
        double tx = c0[W] + c0[-W] + beta * (cp[W] + cm[W] + cp[-W] + cm[-W]);
        double ty = c0[1] + c0[-1] + beta * (cp[1] + cm[1] + cp[-1] + cm[-1]);
        r = a0 * c0[0] - v1 + alpha * (a1 * tx + a2 * ty) + a3 * (cp[0] + cm[0]) + as * src;
      } else {
        r = a0 * c0[0] - v1 + a1 * (c0[W] + c0[-W]) + a2 * (c0[1] + c0[-1]) + a3 * (cp[0] + cm[0]) + as * src;
      }
      anp1[m] = (R)r;
    }
    if (face_tile) {
      // the inward neighbour's A^{n+1} as stored, and its A^{n-1}
      const double pn = __shfl((double)(R)r, nb_lane);
      const double mn = __shfl(v1, nb_lane);
      if (face) {
        const double* B = yf.B;
        anp1[m] = (R)(B[0] * (v1 + pn) + B[1] * mn + B[2] * (c0[0] + c0[fs]) +
                      B[3] * (c0[fs + W] + c0[fs - W] + c0[W] + c0[-W]) +
                      B[4] * (cp[fs] + cm[fs] + cp[0] + cm[0]));
      }
    }
    __syncthreads();
  }
}

template <typename R, bool NSFD, int TI, int K, bool FACES>
__global__ __launch_bounds__(kTileJ* TI) void k_interior_lds(
    FieldSet an_set, FieldSet anm1_set, FieldSet anp1_set, int ncomp, int N0, int N1, int N2,
    int tilesJ, int tilesI, int chunks, double a0, double a1, double a2, double a3, double a4, double a5,
    double alpha, double beta, MurYFace yf) {
  interior_lds_body<R, NSFD, TI, K, FACES>(an_set, anm1_set, anp1_set, ncomp, N0, N1, N2, tilesJ, tilesI, chunks,
                                           a0, a1, a2, a3, a4, a5, alpha, beta,
                                           xcd_logical_block(blockIdx.x, gridDim.x), yf);
}

// ---- flat forms (tile shape 0) ---------------------------------------------------------------
// Lanes run over the nodes of rows 1 .. N0-2 of a plane as one contiguous range (flat index
// p = N1 i + j), so a mesh whose N1 is no multiple of 64 wastes only its two boundary columns of
// lanes, and a workgroup marches only as many planes as leave the GPU its waves (flat_planes).
// The transverse neighbours are other lanes' nodes, served by L1/L2; the z neighbours ride in
// registers.  Same expressions, in the same order, as the tiled forms.
//
// What bounds the tiled forms on all but the largest meshes is the serial march of their 32-128
// planes by too few workgroups, and lanes past N1; here it is HBM (71 x 71 x 397 nodes and up).
// Interior update / E/B evaluation against the 4 x 64 tiles, us: 32 x 32 x 128 with phi, FP32
// 56 / 74 -> 8 / 7; 71 x 71 x 397 FP32 82 / 123 -> 26 / 31, FP64 108 / 114 -> 41 / 45;
// 128 x 128 x 1024 FP32 241 / 223 -> 163 / 218; 211 x 211 x 1531 FP64 1851 / 1610 -> 1528 / 1367.
constexpr int kFlatThreads = 256;

// A plane of a column and its transverse neighbours in the storage type.
template <typename R>
struct RawPlane {
  R c, xp, xm, yp, ym;
  __device__ inline Plane5 wide() const { return {(double)c, (double)xp, (double)xm, (double)yp, (double)ym}; }
};

template <typename R, typename PT>
__device__ inline RawPlane<R> raw_plane(PT a, long m, long N1) {
  return {a[m], a[m + N1], a[m - N1], a[m + 1], a[m - 1]};
}

// Tile, chunk and flat node of a flat workgroup; false for lanes without an interior node.
struct FlatNode {
  int kb, ke;    // planes
  int i, j;
  long m;        // node at plane kb
};

__device__ inline bool flat_node(int tile, int kc, int K, int klo, int khi, int N0, int N1, FlatNode& f) {
  f.kb = klo + kc * K;
  f.ke = min(f.kb + K, khi + 1);
  const int p = N1 + tile * kFlatThreads + (int)threadIdx.x;
  f.i = p / N1;
  f.j = p - f.i * N1;
  f.m = (long)N1 * N0 * f.kb + p;
  return f.kb < f.ke && f.i <= N0 - 2 && f.j >= 1 && f.j <= N1 - 2;
}

// FACES: the threads of nodes j = 1 and j = N1-2 also update the Mur y face node beside them (mur_face
// below with t along x, u along z).  Such a thread holds its own new value and A^{n-1} and all
// of A^n that the face takes but two values; those and the face's A^{n-1} are loaded with the
// prefetch, so that no load of the current plane's waits behind it.  Valid only when nothing writes
// A^{n+1} between the interior update and the boundaries, and with N1 >= 4.
template <typename R, bool NSFD, bool FACES>
__device__ inline void interior_flat_body(FieldSet an_set, FieldSet anm1_set, FieldSet anp1_set, int ncomp, int N0,
                                          int N1, int N2, int tiles, int chunks, int K, double a0, double a1,
                                          double a2, double a3, double a4, double a5, double alpha, double beta,
                                          int lb, const MurYFace& yf) {
  const int tile = lb % tiles;
  lb /= tiles;
  const int kc = lb % chunks;
  const int comp = lb / chunks;
  FlatNode f;
  if (comp >= ncomp || !flat_node(tile, kc, K, 1, N2 - 2, N0, N1, f)) return;
  const bool face = FACES && (f.j == 1 || f.j == N1 - 2);
  const int fs = f.j == 1 ? -1 : 1;  // offset of the face node
  const gptr<const R> an = G((const R*)component(an_set, comp));
  const gptr<const R> anm1 = G((const R*)component(anm1_set, comp));
  const gptr<R> anp1 = G((R*)component(anp1_set, comp));
  const double as = comp < 3 ? a4 : a5;
  const long N1N0 = (long)N1 * N0;
  long m = f.m;
  // in the storage type until used: a conversion right after a load would wait for it there
  RawPlane<R> pm = raw_plane<R>(an, m - N1N0, N1), p0 = raw_plane<R>(an, m, N1), pp = raw_plane<R>(an, m + N1N0, N1);
  R v1 = ld_stream(anm1, m), src = ld_stream((gptr<const R>)anp1, m);
  R fm = 0, fxp = 0, fxm = 0;  // the face node's A^{n-1} and its A^n neighbours along x
  if (face) {
    fm = anm1[m + fs];
    fxp = an[m + fs + N1];
    fxm = an[m + fs - N1];
  }
  for (int k = f.kb; k < f.ke; ++k, m += N1N0) {
    RawPlane<R> pn = {};
    R v1n = 0, srcn = 0, fmn = 0, fxpn = 0, fxmn = 0;
    if (k + 1 < f.ke) {  // the next plane's loads go out before this plane's store
      pn = raw_plane<R>(an, m + 2 * N1N0, N1);
      v1n = ld_stream(anm1, m + N1N0);
      srcn = ld_stream((gptr<const R>)anp1, m + N1N0);
      if (face) {
        fmn = anm1[m + N1N0 + fs];
        fxpn = an[m + N1N0 + fs + N1];
        fxmn = an[m + N1N0 + fs - N1];
      }
    }
    const Plane5 qm = pm.wide(), q0 = p0.wide(), qp = pp.wide();
    double r;
    if (NSFD) {
      const double tx = q0.xp + q0.xm + beta * (qp.xp + qm.xp + qp.xm + qm.xm);
      const double ty = q0.yp + q0.ym + beta * (qp.yp + qm.yp + qp.ym + qm.ym);
      r = a0 * q0.c - (double)v1 + alpha * (a1 * tx + a2 * ty) + a3 * (qp.c + qm.c) + as * (double)src;
    } else {
      r = a0 * q0.c - (double)v1 + a1 * (q0.xp + q0.xm) + a2 * (q0.yp + q0.ym) + a3 * (qp.c + qm.c) + as * (double)src;
    }
    st_stream(anp1, m, (R)r);
    if (face) {
      const double* B = yf.B;
      const bool lo = fs < 0;
      const double c = lo ? q0.ym : q0.yp, cp = lo ? qp.ym : qp.yp, cm = lo ? qm.ym : qm.yp;
      anp1[m + fs] = (R)(B[0] * ((double)fm + (double)(R)r) + B[1] * (double)v1 + B[2] * (c + q0.c) +
                         B[3] * (q0.xp + q0.xm + (double)fxp + (double)fxm) + B[4] * (qp.c + qm.c + cp + cm));
    }
    pm = p0;
    p0 = pp;
    pp = pn;
    v1 = v1n;
    src = srcn;
    fm = fmn;
    fxp = fxpn;
    fxm = fxmn;
  }
}

template <typename R, bool NSFD, bool FACES>
__global__ __launch_bounds__(kFlatThreads) void k_interior_flat(FieldSet an, FieldSet anm1, FieldSet anp1, int ncomp,
                                                                int N0, int N1, int N2, int tiles, int chunks, int K,
                                                                double a0, double a1, double a2, double a3, double a4,
                                                                double a5, double alpha, double beta, MurYFace yf) {
  interior_flat_body<R, NSFD, FACES>(an, anm1, anp1, ncomp, N0, N1, N2, tiles, chunks, K, a0, a1, a2, a3, a4, a5,
                                     alpha, beta, xcd_logical_block(blockIdx.x, gridDim.x), yf);
}

// ---- analytic seed (Signal::self src/classes.cpp:534-575, Seed::fields :740-855) --------

// Plane-wave, truncated plane-wave and Gaussian-beam seeds (the types whose output does not
// depend on the previous call).  Writes the boosted-frame vector potential a[3].
__device__ void seed_fields(const mithra_seed& s, double r0, double r1, double r2, double time, double a[3]) {
  double rv[3];
  rv[0] = r0 - s.position[0];
  rv[1] = r1 - s.position[1];
  rv[2] = s.gamma * (r2 + s.beta * s.c0 * (time + s.dt_shift)) - s.position[2];
  double tl = s.gamma * (time + s.dt_shift + s.beta / s.c0 * r2);
  const double z = rv[0] * s.direction[0] + rv[1] * s.direction[1] + rv[2] * s.direction[2];
  tl -= z / s.c0;
  const double* pol = s.polarization;
  const double* dir = s.direction;
  double amp = 0.0;
  double ts = signal(s, tl, 0.0);
  bool zero = fabs(ts) < 1.0e-6;
  if (s.seed_type == MITHRA_SEED_PLANEWAVE) {
    amp = s.amplitude * ts;
  } else {
    double x = rv[0] * pol[0] + rv[1] * pol[1] + rv[2] * pol[2];
    double yv0 = dir[1] * pol[2] - dir[2] * pol[1];
    double yv1 = dir[2] * pol[0] - dir[0] * pol[2];
    double yv2 = dir[0] * pol[1] - dir[1] * pol[0];
    double y = rv[0] * yv0 + rv[1] * yv1 + rv[2] * yv2;
    if (s.seed_type == MITHRA_SEED_PLANEWAVE_TRUNCATED) {
      zero = zero || fabs(x) > s.radius[0] || fabs(y) > s.radius[1];
      amp = s.amplitude * ts;
    } else if (!zero) {
      const double l = s.c0 / s.f0;
      const double zRp = kPI * s.radius[0] * s.radius[0] / l;
      const double wrp = sqrt(1.0 + z * z / (zRp * zRp));
      const double zRs = kPI * s.radius[1] * s.radius[1] / l;
      const double wrs = sqrt(1.0 + z * z / (zRs * zRs));
      const double p = 0.5 * (atan(z / zRp) + atan(z / zRs) - kPI) -
                       kPI * z / l * (sq(x / (zRp * wrp)) + sq(y / (zRs * wrs)));
      ts = signal(s, tl, p);
      const double t = exp(-sq(x / (s.radius[0] * wrp)) - sq(y / (s.radius[1] * wrs))) / sqrt(wrs * wrp) *
                       s.amplitude;
      amp = t * ts;
    }
  }
  if (zero) {
    a[0] = a[1] = a[2] = 0.0;
  } else {
    a[0] = amp * pol[0];
    a[1] = amp * pol[1];
    a[2] = amp * pol[2];
  }
  a[2] *= s.gamma;
}

// TF/SF injection (src/fdtd.cpp:307-373).  Axis 0 injects into planes i = 1, 2, N0-2, N0-3 at the j, k
// two nodes or more from the mesh's faces, axes 1 and 2 likewise: plane 1 takes minus the seed at
// plane 2, plane 2 plus the seed at plane 1, and so at the other end.  The reference runs the axes, and
// the four planes of an axis, one after the other, and a node where planes cross takes one injection
// of each.  Here a thread owns a node and applies all of its injections in the reference's order, so
// one launch serves the three axes: tfsf_count nodes, those with one injection first, in the plane's
// order, then the rest, so that hardly any wavefront evaluates more than one seed.  On an axis
// of fewer than six nodes planes coincide, and every node of the mesh is asked.
//
// Bound by the latency of one seed evaluation.  Three launches, with the squares by pow(x, 2), took 12 us
// each on 32 x 32 x 128 nodes; the one takes 12.6.
__host__ __device__ inline long tfsf_count(int N0, int N1, int N2) {
  if (N0 < 6 || N1 < 6 || N2 < 6) return (long)N0 * N1 * N2;
  const long a = N0 - 4, b = N1 - 4, c = N2 - 4;
  return 2 * (b * c + a * c + a * b) + 2 * ((b - 2) * (c - 2) + (a - 2) * (c - 2) + (a - 2) * (b - 2)) +
         4 * (c + (b - 2) + (a - 2));
}

// Node t of the list.
__device__ inline void tfsf_node(long t, int N0, int N1, int N2, int ijk[3]) {
  if (N0 < 6 || N1 < 6 || N2 < 6) {
    ijk[1] = (int)(t % N1);
    ijk[0] = (int)(t / N1 % N0);
    ijk[2] = (int)(t / N1 / N0);
    return;
  }
  const int a = N0 - 4, b = N1 - 4, c = N2 - 4;
  // a plane of u x v nodes from node lo on, at both ends (first, last) of an axis
  auto planes = [&](int u, int v, int lo, int first, int last, int& pu, int& pv, int& pw) {
    const long n = (long)u * v;
    if (t < 2 * n) {
      const bool hi = t >= n;
      const int q = (int)(t - (hi ? n : 0));
      pu = lo + q % u;
      pv = lo + q / u;
      pw = hi ? last : first;
      return true;
    }
    t -= 2 * n;
    return false;
  };
  int &i = ijk[0], &j = ijk[1], &k = ijk[2];
  if (planes(b, c, 2, 1, N0 - 2, j, k, i) || planes(a, c, 2, 1, N1 - 2, i, k, j) ||
      planes(b, a, 2, 1, N2 - 2, j, i, k) || planes(b - 2, c - 2, 3, 2, N0 - 3, j, k, i) ||
      planes(a - 2, c - 2, 3, 2, N1 - 3, i, k, j) || planes(b - 2, a - 2, 3, 2, N2 - 3, j, i, k))
    return;
  // the inner planes' crossings: along z with their ends, along y, along x
  auto lines = [&](int n, int lo, int& along, int& p, int& q, int lastp, int lastq) {
    if (t < 4L * n) {
      const int which = (int)(t / n);
      along = lo + (int)(t % n);
      p = which & 1 ? lastp : 2;
      q = which & 2 ? lastq : 2;
      return true;
    }
    t -= 4L * n;
    return false;
  };
  if (lines(c, 2, k, i, j, N0 - 3, N1 - 3) || lines(b - 2, 3, j, i, k, N0 - 3, N2 - 3)) return;
  lines(a - 2, 3, i, j, k, N1 - 3, N2 - 3);
}

template <typename R>
__device__ inline void tfsf_body(FieldSet A, int N0, int N1, int N2, const mithra_grid& g, const mithra_seed& s,
                                 double time, double a1, double a2, double a3, long t) {
  if (t >= tfsf_count(N0, N1, N2)) return;
  int ijk[3];
  tfsf_node(t, N0, N1, N2, ijk);
  const int i = ijk[0], j = ijk[1], k = ijk[2];
  const bool in0 = i >= 2 && i < N0 - 2, in1 = j >= 2 && j < N1 - 2, in2 = k >= 2 && k < N2 - 2;
  const long m = (long)N1 * N0 * k + (long)N1 * i + j;
  R* const p[3] = {(R*)A.c[0], (R*)A.c[1], (R*)A.c[2]};
#pragma unroll 1
  for (int axis = 0; axis < 3; ++axis) {
    const int n = axis == 0 ? N0 : axis == 1 ? N1 : N2, at = axis == 0 ? i : axis == 1 ? j : k;
    if (!(axis == 0 ? in1 && in2 : axis == 1 ? in0 && in2 : in0 && in1)) continue;
    // the axis's four injections: into plane 1 from 2, 2 from 1, n-2 from n-3, n-3 from n-2
    unsigned hits = (at == 1 ? 1u : 0u) | (at == 2 ? 2u : 0u) | (at == n - 2 ? 4u : 0u) | (at == n - 3 ? 8u : 0u);
    for (; hits; hits &= hits - 1) {
      const int q = __builtin_ctz(hits);
      const int from = q == 0 ? 2 : q == 1 ? 1 : q == 2 ? n - 3 : n - 2;
      const double x = g.xmin + (axis == 0 ? from : i) * g.dx, y = g.ymin + (axis == 1 ? from : j) * g.dy,
                   z = g.zmin + (axis == 2 ? from : k) * g.dz;
      const double coef = axis == 0 ? a1 : axis == 1 ? a2 : a3;
      double a[3];
      seed_fields(s, x, y, z, time, a);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double v = (double)p[c][m];
        p[c][m] = (R)(q & 1 ? v + coef * a[c] : v - coef * a[c]);
      }
    }
  }
}

template <typename R>
__global__ __launch_bounds__(256) void k_tfsf(FieldSet A, int N0, int N1, int N2, mithra_grid g, mithra_seed s,
                                              double time, double a1, double a2, double a3) {
  tfsf_body<R>(A, N0, N1, N2, g, s, time, a1, a2, a3, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

// ---- the super-gaussian seed's TF/SF injection ------------------------------------------------
// Seed::fields adds the super-gaussian beam into its output vector instead of overwriting it
// (src/classes.cpp:814-851), and FdTd::fieldUpdate passes the same vector, zeroed once per
// step, to every call of the injection (src/fdtd.cpp:239, :307-373).  Call c therefore injects
// the running result of calls 0..c in the reference's loop order: reset to zero by a call whose
// signal is below the threshold, otherwise the beam's (2 o0 + 1)(2 o1 + 1) equal terms added one
// by one, then the z component times gamma.  The calls are numbered in that loop order:
//   x planes  (j outer, k inner, four planes each), y planes (i outer, k inner, four planes each),
//   z = 1, 2 planes (i outer, j inner, two planes each), z = np-2, np-3 planes (likewise).
struct SgCall {
  long m;            // node that receives the injection
  double r[3];       // point the seed is evaluated at (the neighbour across the TF/SF plane)
  int block;         // 0: x planes, 1: y planes, 2: z = 1, 2, 3: z = np-2, np-3
  bool minus;        // mmv (subtract) or pmv (add)
};

__device__ inline SgCall sg_call(const mithra_grid& g, long c) {
  const int N0 = g.N0, N1 = g.N1, N2 = g.N2;
  const long N1N0 = (long)N1 * N0, ni = N0 - 4, nj = N1 - 4, nk = N2 - 4;
  SgCall q;
  const long cx = 4 * nj * nk, cy = 4 * ni * nk, cz = 2 * ni * nj;
  if (c < cx) {
    const long t = c / 4, s = c % 4, j = 2 + t / nk, k = 2 + t % nk;
    const long i = s == 0 ? 1 : s == 1 ? 2 : s == 2 ? N0 - 2 : N0 - 3;
    const long ip = s == 0 ? 2 : s == 1 ? 1 : s == 2 ? N0 - 3 : N0 - 2;  // i of the evaluated node
    q.m = N1N0 * k + N1 * i + j;
    q.r[0] = g.xmin + ip * g.dx; q.r[1] = g.ymin + j * g.dy; q.r[2] = g.zmin + k * g.dz;
    q.block = 0;
    q.minus = (s % 2) == 0;
  } else if (c < cx + cy) {
    const long u = c - cx, t = u / 4, s = u % 4, i = 2 + t / nk, k = 2 + t % nk;
    const long j = s == 0 ? 1 : s == 1 ? 2 : s == 2 ? N1 - 2 : N1 - 3;
    const long jp = s == 0 ? 2 : s == 1 ? 1 : s == 2 ? N1 - 3 : N1 - 2;
    q.m = N1N0 * k + N1 * i + j;
    q.r[0] = g.xmin + i * g.dx; q.r[1] = g.ymin + jp * g.dy; q.r[2] = g.zmin + k * g.dz;
    q.block = 1;
    q.minus = (s % 2) == 0;
  } else {
    const long u = c - cx - cy, upper = u >= cz, v = upper ? u - cz : u, t = v / 2, s = v % 2;
    const long i = 2 + t / nj, j = 2 + t % nj;
    const long k = upper ? (s == 0 ? N2 - 2 : N2 - 3) : (s == 0 ? 1 : 2);
    const long kp = upper ? (s == 0 ? N2 - 3 : N2 - 2) : (s == 0 ? 2 : 1);
    q.m = N1N0 * k + N1 * i + j;
    q.r[0] = g.xmin + i * g.dx; q.r[1] = g.ymin + j * g.dy; q.r[2] = g.zmin + kp * g.dz;
    q.block = upper ? 3 : 2;
    q.minus = s == 0;
  }
  return q;
}

// One call's beam term t * tsignal at boosted-frame point r (every one of its (2 o0 + 1)(2 o1 + 1)
// terms is the same), or a reset (returns true) when the signal is below the threshold
// (src/classes.cpp:742-755, :816-850).
__device__ bool sg_term(const mithra_seed& s, double r0, double r1, double r2, double time, double* term) {
  const double rl2 = s.gamma * (r2 + s.beta * s.c0 * (time + s.dt_shift));
  double tl = s.gamma * (time + s.dt_shift + s.beta / s.c0 * r2);
  const double rv[3] = {r0 - s.position[0], r1 - s.position[1], rl2 - s.position[2]};
  const double z = rv[0] * s.direction[0] + rv[1] * s.direction[1] + rv[2] * s.direction[2];
  tl -= z / s.c0;
  double ts = signal(s, tl, 0.0);
  if (fabs(ts) < 1.0e-6) {
    *term = 0.0;
    return true;
  }
  const double* pol = s.polarization;
  const double* dir = s.direction;
  const double x = rv[0] * pol[0] + rv[1] * pol[1] + rv[2] * pol[2];
  const double yv0 = dir[1] * pol[2] - dir[2] * pol[1];
  const double yv1 = dir[2] * pol[0] - dir[0] * pol[2];
  const double yv2 = dir[0] * pol[1] - dir[1] * pol[0];
  const double y = rv[0] * yv0 + rv[1] * yv1 + rv[2] * yv2;
  const double l = s.c0 / s.f0;
  const double zRp = kPI * s.radius[0] * s.radius[0] / l;
  const double wrp = sqrt(1.0 + z * z / (zRp * zRp));
  const double zRs = kPI * s.radius[1] * s.radius[1] / l;
  const double wrs = sqrt(1.0 + z * z / (zRs * zRs));
  const double p = 0.5 * (atan(z / zRp) + atan(z / zRs) - kPI) -
                   kPI * z / l * (sq(x / (zRp * wrp)) + sq(y / (zRs * wrs)));
  ts = signal(s, tl, p);
  const double t = exp(-sq(x / (s.radius[0] * wrp)) - sq(y / (s.radius[1] * wrs))) / sqrt(wrs * wrp) *
                   s.amplitude;
  *term = t * ts;
  return false;
}

__global__ void k_sg_terms(mithra_grid g, mithra_seed s, double time, long n, double* __restrict__ term,
                           int* __restrict__ reset) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const SgCall q = sg_call(g, c);
  reset[c] = sg_term(s, q.r[0], q.r[1], q.r[2], time, &term[c]) ? 1 : 0;
}

// The same terms at listed points and times (the point evaluator's call order).
__global__ void k_sg_point_terms(mithra_seed s, const double* __restrict__ r, const double* __restrict__ time,
                                 long n, double* __restrict__ term, int* __restrict__ reset) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  reset[c] = sg_term(s, r[3 * c], r[3 * c + 1], r[3 * c + 2], time[c], &term[c]) ? 1 : 0;
}

// The running vector in call order: strictly sequential, one lane.
__global__ void k_sg_running(mithra_seed s, long n, const double* __restrict__ term, const int* __restrict__ reset,
                             double* __restrict__ out) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  const int reps = (2 * s.order[0] + 1) * (2 * s.order[1] + 1);
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  for (long c = 0; c < n; ++c) {
    if (reset[c]) {
      a0 = a1 = a2 = 0.0;
    } else {
      const double v = term[c];
      for (int r = 0; r < reps; ++r) {
        a0 += v * s.polarization[0];
        a1 += v * s.polarization[1];
        a2 += v * s.polarization[2];
      }
    }
    a2 *= s.gamma;
    out[3 * c] = a0;
    out[3 * c + 1] = a1;
    out[3 * c + 2] = a2;
  }
}

// The injection of one block of calls (nodes are distinct within a block; the blocks run in
// the reference's order, so a node two blocks touch gets its two updates in sequence).
template <typename R>
__global__ void k_sg_apply(FieldSet A, mithra_grid g, long first, long count, const double* __restrict__ run,
                           double coef) {
  const long u = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= count) return;
  const long c = first + u;
  const SgCall q = sg_call(g, c);
  for (int k = 0; k < 3; ++k) {
    R* p = (R*)A.c[k];
    const double v = (double)p[q.m];
    p[q.m] = (R)(q.minus ? v - coef * run[3 * c + k] : v + coef * run[3 * c + k]);
  }
}

// The analytic seed on its own, at listed points: one thread per point.
__global__ void k_signal_eval(mithra_seed s, const double* __restrict__ t, const double* __restrict__ phase, long n,
                              double* __restrict__ out) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) out[q] = signal(s, t[q], phase[q]);
}

__global__ void k_seed_eval(mithra_seed s, const double* __restrict__ r, const double* __restrict__ time, long n,
                            double* __restrict__ a) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  double v[3];
  seed_fields(s, r[3 * q], r[3 * q + 1], r[3 * q + 2], time[q], v);
  a[3 * q] = v[0];
  a[3 * q + 1] = v[1];
  a[3 * q + 2] = v[2];
}

// ---- Mur absorbing boundaries (src/database.cpp:137-288, loops src/fdtd.cpp:377-725) ------
// Offsets are in nodes.  For a face node, s is the offset of its inward neighbour and t, u the
// two tangential axes (B[3] multiplies the t-neighbours, B[4] the u-neighbours).  For an edge
// node, o1 and o2 are the two inward offsets and w the offset along the edge.  For a corner,
// sx, sy, sz are the three inward offsets.

template <typename TP, typename TN>
__device__ inline double mur_face(const double* B, TP P, TN N, TN M, long m, long s, long t, long u) {
  return B[0] * (rd(M, m) + rd(P, m + s)) + B[1] * rd(M, m + s) + B[2] * (rd(N, m) + rd(N, m + s)) +
         B[3] * (rd(N, m + s + t) + rd(N, m + s - t) + rd(N, m + t) + rd(N, m - t)) +
         B[4] * (rd(N, m + s + u) + rd(N, m + s - u) + rd(N, m + u) + rd(N, m - u));
}

template <typename TP, typename TN>
__device__ inline double mur_edge(const double* B, TP P, TN N, TN M, long m, long o1, long o2, long w) {
  const long o3 = o1 + o2;
  return B[0] * (rd(P, m + o1) + rd(M, m + o2)) + B[1] * (rd(M, m + o1) + rd(P, m + o2)) +
         B[2] * (rd(M, m) + rd(P, m + o3)) + B[3] * (rd(N, m) + rd(N, m + o1) + rd(N, m + o2) + rd(N, m + o3)) +
         B[4] * (rd(N, m - w) + rd(N, m - w + o1) + rd(N, m - w + o2) + rd(N, m - w + o3) + rd(N, m + w) +
                 rd(N, m + w + o1) + rd(N, m + w + o2) + rd(N, m + w + o3)) -
         rd(M, m + o3);
}

// All six faces in one launch: x faces (j, k), y faces (i, k), z faces (i, j), each min/max.
// The faces in `mask` (faces_mask) were updated by the interior kernel and are skipped.
template <typename R>
__device__ inline void mur_faces_body(FieldSet P, FieldSet N, FieldSet M, int ncomp, int N0, int N1, int N2,
                                      const MurCoeffs& c, long t, int comp, int mask) {
  const long N1N0 = (long)N1 * N0;
  const long X = N1, Y = 1, Z = N1N0;
  const long nx = (long)(N1 - 2) * (N2 - 2), ny = (long)(N0 - 2) * (N2 - 2), nz = (long)(N0 - 2) * (N1 - 2);
  const long nylo = (mask & 1) ? 0 : ny, nyhi = (mask & 2) ? 0 : ny;
  if (comp >= ncomp) return;
  const gptr<const R> pn = G((const R*)component(N, comp));
  const gptr<const R> pm = G((const R*)component(M, comp));
  const gptr<R> pp = G((R*)component(P, comp));
  long m, s, tt, u;
  int axis;
  if (t < 2 * nx) {
    const bool hi = t >= nx;
    t -= hi ? nx : 0;
    const long j = 1 + t % (N1 - 2), k = 1 + t / (N1 - 2);
    m = N1N0 * k + (hi ? N1N0 - N1 : 0) + j;
    s = hi ? -X : X; tt = Y; u = Z; axis = 0;
  } else if ((t -= 2 * nx) < nylo + nyhi) {
    const bool hi = t >= nylo;
    t -= hi ? nylo : 0;
    const long i = 1 + t % (N0 - 2), k = 1 + t / (N0 - 2);
    m = N1N0 * k + (long)N1 * i + (hi ? N1 - 1 : 0);
    s = hi ? -Y : Y; tt = X; u = Z; axis = 1;
  } else if ((t -= nylo + nyhi) < 2 * nz) {
    const bool hi = t >= nz;
    t -= hi ? nz : 0;
    const long j = 1 + t % (N1 - 2), i = 1 + t / (N1 - 2);
    m = (hi ? N1N0 * (N2 - 1) : 0) + (long)N1 * i + j;
    s = hi ? -Z : Z; tt = X; u = Y; axis = 2;
  } else {
    return;
  }
  // The coefficients by selects into registers: a pointer into the coefficient struct would
  // copy the whole struct to scratch memory in every thread.
  double B[5];
#pragma unroll
  for (int q = 0; q < 5; ++q) B[q] = axis == 0 ? c.bB[q] : axis == 1 ? c.cB[q] : c.dB[q];
  pp[m] = (R)mur_face(B, pp, pn, pm, m, s, tt, u);
}

template <typename R>
__global__ void k_mur_faces(FieldSet P, FieldSet N, FieldSet M, int ncomp, int N0, int N1, int N2, MurCoeffs c,
                           int mask) {
  mur_faces_body<R>(P, N, M, ncomp, N0, N1, N2, c, (long)blockIdx.x * blockDim.x + threadIdx.x, blockIdx.y, mask);
}

// The twelve edges and the eight corners (second-order Mur only) in one launch.  A corner reads the new
// values of three edge nodes, which other threads of the launch store: it computes them again itself,
// as the buffer holds them, one edge to a lane, so nothing waits for another thread.  A launch of
// its own for the corners took 4-5 us of every step.  (Edges and corners that compute the faces again
// too, in the faces' launch, gained 4 us more on 32 x 32 x 128 nodes and lost 4 us at 71 x 71 x 397,
// where the faces' threads then have the edges' registers and index arithmetic.)

// Value of edge node m along axis 2, 0 or 1 (`set`: 0 z, 1 x, 2 y), on the sides h1, h2 of the two axes
// across it: x, y of z; y, z of x; z, x of y.
template <typename R, typename TN, typename TP>
__device__ inline double mur_edge_value(const MurCoeffs& c, TP P, TN N, TN M, long m, int set, bool h1, bool h2,
                                        long X, long Z) {
  double B[5];  // by selects, as in mur_faces_body
#pragma unroll
  for (int q = 0; q < 5; ++q) B[q] = set == 0 ? c.eE[q] : set == 1 ? c.fE[q] : c.gE[q];
  const long s1 = set == 0 ? X : set == 1 ? 1 : Z, s2 = set == 0 ? 1 : set == 1 ? Z : X;
  const long w = set == 0 ? Z : set == 1 ? X : 1;
  return (double)(R)mur_edge(B, P, N, M, m, h1 ? -s1 : s1, h2 ? -s2 : s2, w);
}

// Block b of the pass: edges, 256 nodes each, and in the last one (b = nb - 1) the corners, four lanes
// each: lanes 0-2 of a corner compute its edges along x, y, z, lane 0 the corner.
template <typename R>
__device__ inline void mur_rims_body(FieldSet Ps, FieldSet Ns, FieldSet Ms, int ncomp, int N0, int N1, int N2,
                                     const MurCoeffs& c, int b, int nb, int comp) {
  const long X = N1, Z = (long)N1 * N0;
  if (comp >= ncomp) return;
  const gptr<const R> N = G((const R*)component(Ns, comp));
  const gptr<const R> M = G((const R*)component(Ms, comp));
  const gptr<R> P = G((R*)component(Ps, comp));
  if (b == nb - 1) {
    if (threadIdx.x >= 64) return;  // whole wavefronts: the corners take 32 lanes of the first
    const int t = (threadIdx.x & 31) >> 2, a = (threadIdx.x & 3) < 3 ? threadIdx.x & 3 : 0;
    const bool xh = t & 1, yh = t & 2, zh = t & 4;
    const long m = (xh ? Z - X : 0) + (yh ? N1 - 1 : 0) + (zh ? Z * (N2 - 1) : 0);
    const long sx = xh ? -X : X, sy = yh ? -1 : 1, sz = zh ? -Z : Z;
    // edge along x: set 1, sides y, z; along y: set 2, sides z, x; along z: set 0, sides x, y
    const double v = mur_edge_value<R>(c, P, N, M, m + (a == 0 ? sx : a == 1 ? sy : sz), a == 0 ? 1 : a == 1 ? 2 : 0,
                                       a == 0 ? yh : a == 1 ? zh : xh, a == 0 ? zh : a == 1 ? xh : yh, X, Z);
    const int base = __lane_id() & ~3;
    const long o[7] = {sx, sy, sz, sx + sy, sz + sx, sz + sy, sz + sx + sy};
    const double p[7] = {__shfl(v, base),  __shfl(v, base + 1), __shfl(v, base + 2), rd(P, m + o[3]),
                         rd(P, m + o[4]), rd(P, m + o[5]),     rd(P, m + o[6])};
    const double* h = c.hC;
    double s = rd(N, m) * h[16] + rd(M, m) * h[8];
#pragma unroll
    for (int q = 0; q < 7; ++q) s = s + p[q] * h[1 + q] + rd(N, m + o[q]) * h[16] + rd(M, m + o[q]) * h[9 + q];
    if (threadIdx.x < 32 && (threadIdx.x & 3) == 0) P[m] = (R)(-s / h[0]);
    return;
  }
  long t = (long)b * 256 + threadIdx.x, m;
  const long ez = N2 - 2, ex = N0 - 2, ey = N1 - 2;
  bool h1, h2;
  int set;
  if (t < 4 * ez) {  // along z at the four (x, y) corners
    const int which = t / ez;
    h1 = which & 1; h2 = which & 2;
    m = Z * (1 + t % ez) + (h1 ? X * (N0 - 1) : 0) + (h2 ? N1 - 1 : 0);
    set = 0;
  } else if ((t -= 4 * ez) < 4 * ex) {  // along x at the four (y, z) corners
    const int which = t / ex;
    h1 = which & 1; h2 = which & 2;
    m = X * (1 + t % ex) + (h1 ? N1 - 1 : 0) + (h2 ? Z * (N2 - 1) : 0);
    set = 1;
  } else if ((t -= 4 * ex) < 4 * ey) {  // along y at the four (z, x) corners
    const int which = t / ey;
    h1 = which & 1; h2 = which & 2;
    m = 1 + t % ey + (h1 ? Z * (N2 - 1) : 0) + (h2 ? Z - X : 0);
    set = 2;
  } else {
    return;
  }
  P[m] = (R)mur_edge_value<R>(c, P, N, M, m, set, h1, h2, X, Z);
}

template <typename R>
__global__ __launch_bounds__(256) void k_mur_rims(FieldSet P, FieldSet N, FieldSet M, int ncomp, int N0, int N1,
                                                  int N2, MurCoeffs c) {
  mur_rims_body<R>(P, N, M, ncomp, N0, N1, N2, c, blockIdx.x, gridDim.x, blockIdx.y);
}

// E/B on every interior node (FdTd::fieldEvaluate src/fdtd.cpp:818-845, FdTdSC::fieldEvaluate
// src/fdtdSC.cpp:1110-1145); planes k = 0 and N2-1 take copies of k = 1 and N2-2
// (src/fdtd.cpp:742-774).  E_x and E_y are one double expression rounded once to float and E_z
// keeps the float rounding after each term: that is what the reference computes as compiled by
// g++ -O3 (its vectorised x/y lanes drop the intermediate float round trip of
// FieldVector<float>::dv/mdv, src/fieldvector.h:87-108), and the parity fixtures record it.
// Lazy evaluation (the reference evaluates E/B only where particles and samplers read them,
// src/solver.h:241, src/fdtd.cpp:818-845): planes kb..ke-1 are needed if they meet the nodes the
// bunch reads during the coming push (its cells zr[0]..zr[1] at the start, at most one cell of
// motion per field step, nodes k and k+1 of a cell) or the power planes pb0..pb1.
__device__ inline bool lazy_needed(int kb, int ke, const int* zr, int pb0, int pb1) {
  const int a0 = zr[0] - 2, a1 = zr[1] + 2;
  return (ke - 1 >= a0 && kb <= a1) || (ke - 1 >= pb0 && kb <= pb1);
}


// Each thread owns one (i, j) column and marches K planes; the z neighbours of A_x and A_y (and
// phi) at both time levels ride in a three-plane register queue, the transverse neighbours are
// the centres of neighbouring lanes and rows.  Planes outside [klo, khi] are skipped.
template <typename R, bool SC>
__device__ inline void eval_march(FieldSet An, FieldSet Ap, float* __restrict__ eb, int N0, int N1, int N2, int kb,
                                  int ke, long m, const EvalConst& q) {
  const gptr<f2> ebg = G(reinterpret_cast<f2*>(eb));
  const long N1N0 = (long)N1 * N0;
  const gptr<const R> n0 = G((const R*)An.c[0]);
  const gptr<const R> n1 = G((const R*)An.c[1]);
  const gptr<const R> n2 = G((const R*)An.c[2]);
  const gptr<const R> p0 = G((const R*)Ap.c[0]);
  const gptr<const R> p1 = G((const R*)Ap.c[1]);
  const gptr<const R> p2 = G((const R*)Ap.c[2]);
  const gptr<const R> f = G(SC ? (const R*)An.c[3] : (const R*)nullptr);
  const double mdt = q.mdt, dx2 = q.dx2, dy2 = q.dy2, dz2 = q.dz2;
  auto dt_ = [&](double x) { return div_rn(x, mdt, q.rmdt); };
  auto dx_ = [&](double x) { return div_rn(x, dx2, q.rdx2); };
  auto dy_ = [&](double x) { return div_rn(x, dy2, q.rdy2); };
  auto dz_ = [&](double x) { return div_rn(x, dz2, q.rdz2); };
  // queue: [0] plane k-1, [1] plane k, [2] plane k+1
  double qn0[3], qn1[3], qp0[3], qp1[3], qf[3];
  for (int t = 0; t < 2; ++t) {
    const long mm = m + (t - 1) * N1N0;
    qn0[t] = rd(n0, mm); qn1[t] = rd(n1, mm); qp0[t] = rd(p0, mm); qp1[t] = rd(p1, mm);
    if (SC) qf[t] = rd(f, mm);
  }
  for (int k = kb; k < ke; ++k, m += N1N0) {
    qn0[2] = rd(n0, m + N1N0); qn1[2] = rd(n1, m + N1N0); qp0[2] = rd(p0, m + N1N0); qp1[2] = rd(p1, m + N1N0);
    if (SC) qf[2] = rd(f, m + N1N0);
    double ex = dt_(qp0[1]) - dt_(qn0[1]);
    double ey = dt_(qp1[1]) - dt_(qn1[1]);
    float ez = (float)dt_(rd(p2, m));
    ez = (float)((double)ez - dt_(rd(n2, m)));
    if (SC) {
      ex = ex - dx_(rd(f, m + N1) - rd(f, m - N1));
      ey = ey - dy_(rd(f, m + 1) - rd(f, m - 1));
      ez = (float)((double)ez - dz_(qf[2] - qf[0]));
    }
    const float bx = (float)(0.5 * (dy_(rd(n2, m + 1) - rd(n2, m - 1)) - dz_(qn1[2] - qn1[0]) +
                                    dy_(rd(p2, m + 1) - rd(p2, m - 1)) - dz_(qp1[2] - qp1[0])));
    const float by = (float)(0.5 * (dz_(qn0[2] - qn0[0]) - dx_(rd(n2, m + N1) - rd(n2, m - N1)) +
                                    dz_(qp0[2] - qp0[0]) - dx_(rd(p2, m + N1) - rd(p2, m - N1))));
    const float bz = (float)(0.5 * (dx_(rd(n1, m + N1) - rd(n1, m - N1)) - dy_(rd(n0, m + 1) - rd(n0, m - 1)) +
                                    dx_(rd(p1, m + N1) - rd(p1, m - N1)) - dy_(rd(p0, m + 1) - rd(p0, m - 1))));
    const f2 v0 = {(float)ex, (float)ey}, v1 = {ez, bx}, v2 = {by, bz};
    auto put = [&](long node) {  // E/B is read by later kernels only: stream past L2
      st_stream(ebg, kEBPairs * node, v0);
      st_stream(ebg, kEBPairs * node + 1, v1);
      st_stream(ebg, kEBPairs * node + 2, v2);
    };
    put(m);
    if (k == 1) put(m - N1N0);
    if (k == N2 - 2) put(m + N1N0);
    qn0[0] = qn0[1]; qn1[0] = qn1[1]; qp0[0] = qp0[1]; qp1[0] = qp1[1];
    qn0[1] = qn0[2]; qn1[1] = qn1[2]; qp0[1] = qp0[2]; qp1[1] = qp1[2];
    if (SC) { qf[0] = qf[1]; qf[1] = qf[2]; }
  }
}

template <typename R, bool SC, int TI, int K>
__device__ inline void eval_body(FieldSet An, FieldSet Ap, float* __restrict__ eb, int N0, int N1, int N2,
                                 int tilesJ, int tilesI, int klo, int khi, const EvalConst& q,
                                 const int* __restrict__ zr, int pb0, int pb1, int lb) {
  const int tj = lb % tilesJ;
  lb /= tilesJ;
  const int ti = lb % tilesI;
  const int kc = lb / tilesI;
  const int j = tj * kTileJ + (threadIdx.x % kTileJ);
  const int i = 1 + ti * TI + (threadIdx.x / kTileJ);
  const int kb = klo + kc * K;
  const int ke = min(kb + K, khi + 1);
  if (zr && !lazy_needed(kb, ke, zr, pb0, pb1)) return;
  if (i > N0 - 2 || j < 1 || j > N1 - 2 || kb >= ke) return;
  eval_march<R, SC>(An, Ap, eb, N0, N1, N2, kb, ke, (long)N1 * N0 * kb + (long)N1 * i + j, q);
}

// The flat form (see interior_flat_body).
template <typename R, bool SC>
__device__ inline void eval_flat_body(FieldSet An, FieldSet Ap, float* __restrict__ eb, int N0, int N1, int N2,
                                      int tiles, int K, int klo, int khi, const EvalConst& q,
                                      const int* __restrict__ zr, int pb0, int pb1, int lb) {
  const int tile = lb % tiles, kc = lb / tiles;
  FlatNode f;
  if (!flat_node(tile, kc, K, klo, khi, N0, N1, f)) return;
  if (zr && !lazy_needed(f.kb, f.ke, zr, pb0, pb1)) return;
  eval_march<R, SC>(An, Ap, eb, N0, N1, N2, f.kb, f.ke, f.m, q);
}

template <typename R, bool SC>
__global__ __launch_bounds__(kFlatThreads) void k_eval_flat(FieldSet An, FieldSet Ap, float* __restrict__ eb, int N0,
                                                            int N1, int N2, int tiles, int K, int klo, int khi,
                                                            EvalConst q, const int* __restrict__ zr, int pb0,
                                                            int pb1) {
  eval_flat_body<R, SC>(An, Ap, eb, N0, N1, N2, tiles, K, klo, khi, q, zr, pb0, pb1,
                        xcd_logical_block(blockIdx.x, gridDim.x));
}

template <typename R, bool SC, int TI, int K>
__global__ __launch_bounds__(kTileJ* TI) void k_eval_eb(FieldSet An, FieldSet Ap, float* __restrict__ eb, int N0,
                                                        int N1, int N2, int tilesJ, int tilesI, int klo, int khi,
                                                        EvalConst q, const int* __restrict__ zr, int pb0, int pb1) {
  eval_body<R, SC, TI, K>(An, Ap, eb, N0, N1, N2, tilesJ, tilesI, klo, khi, q, zr, pb0, pb1,
                          xcd_logical_block(blockIdx.x, gridDim.x));
}

// The E/B evaluation with plane k of A^n and A^{n+1} staged in LDS (2.5-D blocking, as
// k_interior_lds): the workgroup marches its planes in lockstep, every transverse neighbour is
// read from LDS, the z neighbours of A_x, A_y (and phi) ride in a register queue, and the
// next plane is fetched while the current one is computed.  Same expressions as k_eval_eb.
template <typename R, bool SC, int TI, int K>
__device__ inline void eval_lds_body(FieldSet An, FieldSet Ap, float* __restrict__ eb, int N0, int N1, int N2,
                                     int tilesJ, int tilesI, int klo, int khi, const EvalConst& q,
                                     const int* __restrict__ zr, int pb0, int pb1, int lb) {
  const gptr<f2> ebg = G(reinterpret_cast<f2*>(eb));
  constexpr int NA = SC ? 7 : 6;      // staged arrays: n0 n1 n2 p0 p1 p2 [phi]
  constexpr int NZ = SC ? 5 : 4;      // arrays with z neighbours: n0 n1 p0 p1 [phi]
  constexpr int W = kTileJ + 2, P = (TI + 2) * W;
  __shared__ double L[NA * P];
  const int tj = lb % tilesJ;
  lb /= tilesJ;
  const int ti = lb % tilesI;
  const int kc = lb / tilesI;
  const int kb = klo + kc * K;
  const int ke = min(kb + K, khi + 1);
  if (kb >= ke) return;  // uniform over the workgroup
  if (zr && !lazy_needed(kb, ke, zr, pb0, pb1)) return;
  const int lane = threadIdx.x % kTileJ, w = threadIdx.x / kTileJ;
  const int j0 = tj * kTileJ, i0 = 1 + ti * TI;
  const int j = j0 + lane, i = i0 + w;
  const bool active = i <= N0 - 2 && j >= 1 && j <= N1 - 2;
  const long N1N0 = (long)N1 * N0;
  const gptr<const R> A[7] = {G((const R*)An.c[0]), G((const R*)An.c[1]), G((const R*)An.c[2]),
                              G((const R*)Ap.c[0]), G((const R*)Ap.c[1]), G((const R*)Ap.c[2]),
                              G(SC ? (const R*)An.c[3] : (const R*)nullptr)};
  constexpr int zarr[5] = {0, 1, 3, 4, 6};  // n0 n1 p0 p1 phi
  const bool own_ok = i <= N0 - 1 && j <= N1 - 1;
  const long own_off = (long)N1 * i + j;
  const int own_slot = (w + 1) * W + lane + 1;
  int hrow_i = -1, hrow_slot = 0;
  if (w == 0) { hrow_i = i0 - 1; hrow_slot = lane + 1; }
  if (w == 1) { hrow_i = i0 + TI; hrow_slot = (TI + 1) * W + lane + 1; }
  const bool hrow_ok = hrow_i >= 0 && hrow_i <= N0 - 1 && j <= N1 - 1;
  const long hrow_off = (long)N1 * hrow_i + j;
  int hcol_j = -1, hcol_i = 0, hcol_slot = 0;
  if (w == 0 && lane < TI) { hcol_i = i0 + lane; hcol_j = j0 - 1; hcol_slot = (lane + 1) * W; }
  if (w == 0 && lane >= TI && lane < 2 * TI) {
    hcol_i = i0 + lane - TI; hcol_j = j0 + kTileJ; hcol_slot = (lane - TI + 1) * W + kTileJ + 1;
  }
  const bool hcol_ok = hcol_j >= 0 && hcol_j <= N1 - 1 && hcol_i <= N0 - 1;
  const long hcol_off = (long)N1 * hcol_i + hcol_j;
  // qz[a][s]: own value of z-array a at planes k-1, k, k+1, k+2 (s = 0..3) of iteration k.
  // Prefetched values stay in the storage type until they are staged or used: a conversion
  // right after a load would make the wave wait for that load there (FP32-bulk).
  R qz[NZ][4];
  R pre_n2 = 0, pre_p2 = 0, pre_row[NA], pre_col[NA];
  auto fetch_z = [&](int k, int s) {
#pragma unroll
    for (int a = 0; a < NZ; ++a) qz[a][s] = own_ok ? A[zarr[a]][N1N0 * k + own_off] : (R)0;
  };
  // The curl reads A_x (arrays 0, 3) only at y +- 1 and A_y (arrays 1, 4) only at x +- 1: they
  // need no halo rows and no halo columns respectively.
  auto need_row = [](int a) { return a != 0 && a != 3; };
  auto need_col = [](int a) { return a != 1 && a != 4; };
  auto fetch_plane = [&](int k) {  // what plane k stages besides the queued own values
    const long b = N1N0 * k;
    if (own_ok) {
      pre_n2 = A[2][b + own_off];
      pre_p2 = A[5][b + own_off];
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      if (need_row(a) && hrow_ok) pre_row[a] = A[a][b + hrow_off];
      if (need_col(a) && hcol_ok) pre_col[a] = A[a][b + hcol_off];
    }
  };
  fetch_z(kb - 1, 0);
  fetch_z(kb, 1);
  fetch_z(kb + 1, 2);
  fetch_plane(kb);
  const double mdt = q.mdt, dx2 = q.dx2, dy2 = q.dy2, dz2 = q.dz2;
  auto dt_ = [&](double x) { return div_rn(x, mdt, q.rmdt); };
  auto dx_ = [&](double x) { return div_rn(x, dx2, q.rdx2); };
  auto dy_ = [&](double x) { return div_rn(x, dy2, q.rdy2); };
  auto dz_ = [&](double x) { return div_rn(x, dz2, q.rdz2); };
  long m = N1N0 * kb + own_off;
  for (int k = kb; k < ke; ++k, m += N1N0) {
    // stage plane k
    if (own_ok) {
      L[0 * P + own_slot] = (double)qz[0][1];
      L[1 * P + own_slot] = (double)qz[1][1];
      L[2 * P + own_slot] = (double)pre_n2;
      L[3 * P + own_slot] = (double)qz[2][1];
      L[4 * P + own_slot] = (double)qz[3][1];
      L[5 * P + own_slot] = (double)pre_p2;
      if (SC) L[6 * P + own_slot] = (double)qz[NZ - 1][1];
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      if (need_row(a) && hrow_ok) L[a * P + hrow_slot] = (double)pre_row[a];
      if (need_col(a) && hcol_ok) L[a * P + hcol_slot] = (double)pre_col[a];
    }
    __syncthreads();
    if (k + 1 < ke) fetch_plane(k + 1);
    if (k + 2 <= ke) fetch_z(k + 2, 3);
    if (active) {
      const double* n1l = L + 1 * P + own_slot;
      const double* n2l = L + 2 * P + own_slot;
      const double* p1l = L + 4 * P + own_slot;
      const double* p2l = L + 5 * P + own_slot;
      const double* n0l = L + 0 * P + own_slot;
      const double* p0l = L + 3 * P + own_slot;
      double ex = dt_((double)qz[2][1]) - dt_((double)qz[0][1]);
      double ey = dt_((double)qz[3][1]) - dt_((double)qz[1][1]);
      float ez = (float)dt_(p2l[0]);
      ez = (float)((double)ez - dt_(n2l[0]));
      if (SC) {
        const double* fl = L + 6 * P + own_slot;
        ex = ex - dx_(fl[W] - fl[-W]);
        ey = ey - dy_(fl[1] - fl[-1]);
        ez = (float)((double)ez - dz_((double)qz[NZ - 1][2] - (double)qz[NZ - 1][0]));
      }
      const float bx = (float)(0.5 * (dy_(n2l[1] - n2l[-1]) - dz_((double)qz[1][2] - (double)qz[1][0]) +
                                      dy_(p2l[1] - p2l[-1]) - dz_((double)qz[3][2] - (double)qz[3][0])));
      const float by = (float)(0.5 * (dz_((double)qz[0][2] - (double)qz[0][0]) - dx_(n2l[W] - n2l[-W]) +
                                      dz_((double)qz[2][2] - (double)qz[2][0]) - dx_(p2l[W] - p2l[-W])));
      const float bz = (float)(0.5 * (dx_(n1l[W] - n1l[-W]) - dy_(n0l[1] - n0l[-1]) +
                                      dx_(p1l[W] - p1l[-W]) - dy_(p0l[1] - p0l[-1])));
      const f2 v0 = {(float)ex, (float)ey}, v1 = {ez, bx}, v2 = {by, bz};
      auto put = [&](long node) {  // E/B is read by later kernels only: stream past L2
        st_stream(ebg, kEBPairs * node, v0);
        st_stream(ebg, kEBPairs * node + 1, v1);
        st_stream(ebg, kEBPairs * node + 2, v2);
      };
      put(m);
      if (k == 1) put(m - N1N0);
      if (k == N2 - 2) put(m + N1N0);
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < NZ; ++a) {
      qz[a][0] = qz[a][1];
      qz[a][1] = qz[a][2];
      qz[a][2] = qz[a][3];
    }
  }
}

template <typename R, bool SC, int TI, int K>
__global__ __launch_bounds__(kTileJ* TI) void k_eval_lds(FieldSet An, FieldSet Ap, float* __restrict__ eb, int N0,
                                                         int N1, int N2, int tilesJ, int tilesI, int klo, int khi,
                                                         EvalConst q, const int* __restrict__ zr, int pb0, int pb1) {
  eval_lds_body<R, SC, TI, K>(An, Ap, eb, N0, N1, N2, tilesJ, tilesI, klo, khi, q, zr, pb0, pb1,
                              xcd_logical_block(blockIdx.x, gridDim.x));
}

// ---- pipelined step: E/B of step n fused with the J-free part of the next interior update ----
//
// Once A^{n+1} is complete (interior, seed injection and Mur boundaries), the two field passes
// that remain before the next deposit read the same two levels: the E/B evaluation of step n
// reads A^n and A^{n+1}, and the interior update of step n+1 reads A^{n+1} (stencil) and A^n
// (its A^{n-1}).  Only the update's last term, a4 J^{n+1}, waits for the deposit.  The update
// (src/database.cpp:44-134) sums its terms left to right with the source last, so
//   A^{n+2} = X + a4 J,  X = a0 A^{n+1} - A^n + (transverse terms) + a3 (z terms)
// splits exactly: this kernel writes X (into the A^{n-1} buffer, free once the boundaries of
// A^{n+1} are done) and the E/B of step n; the row-tiled deposit then writes X + a4 J in place
// of J.  In FP64 the result is the unsplit update's bit for bit; in FP32 X is rounded to float
// once before the source is added.
//
// A workgroup owns TI x-rows x 64 y-nodes of all three components and marches K planes: A^{n+1}
// with a one-node halo ring in a three-plane LDS ring per component (the stencil's planes k-1,
// k, k+1), A^n of plane k with its ring in one LDS plane per component (the curl's transverse
// neighbours), and the z neighbours of A^n_x, A^n_y in a register queue.  Same expressions, in
// the same order, as k_interior_lds (without the source) and k_eval_lds (without phi).
struct StencilConst {
  double a0, a1, a2, a3, alpha, beta;
};
#ifndef MITHRA_STENCIL_WAVES
#define MITHRA_STENCIL_WAVES 4
#endif
constexpr int kStencilWaves = MITHRA_STENCIL_WAVES;  // waves per SIMD the register budget allows

template <typename R, bool NSFD, int TI, int K, bool SC = false>
__global__ __launch_bounds__(kTileJ* TI, SC ? 3 : kStencilWaves) void k_stencil_eb(
    FieldSet An1, FieldSet An, FieldSet X, float* __restrict__ eb, int N0, int N1, int N2, int tilesJ, int tilesI,
    StencilConst s, EvalConst q, const int* __restrict__ zr, int pb0, int pb1) {
  // Components: A_x, A_y, A_z, and phi under space charge (the same stencil; its E/B terms are
  // the gradient of phi^n, as in eval_lds_body).
  constexpr int NC = SC ? 4 : 3;
  constexpr int W = kTileJ + 2, P = (TI + 2) * W;
  __shared__ double L1[3 * NC * P];  // A^{n+1}: [component][slot][P]
  __shared__ double L0[NC * P];      // A^n, plane k: [component][P]
  int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int tj = lb % tilesJ;
  lb /= tilesJ;
  const int ti = lb % tilesI;
  const int kc = lb / tilesI;
  const int kb = 1 + kc * K;
  const int ke = min(kb + K, N2 - 1);
  if (kb >= ke) return;  // uniform over the workgroup
  const bool ebneed = !zr || lazy_needed(kb, ke, zr, pb0, pb1);
  const gptr<f2> ebg = G(reinterpret_cast<f2*>(eb));
  const int lane = threadIdx.x % kTileJ, w = threadIdx.x / kTileJ;
  const int j0 = tj * kTileJ, i0 = 1 + ti * TI;
  const int j = j0 + lane, i = i0 + w;
  const bool active = i <= N0 - 2 && j >= 1 && j <= N1 - 2;
  const long N1N0 = (long)N1 * N0;
  gptr<const R> p[NC], n[NC];
  gptr<R> x[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    p[c] = G((const R*)component(An1, c));
    n[c] = G((const R*)component(An, c));
    x[c] = G((R*)component(X, c));
  }
  // staged per plane by this thread: its own node, and (as in k_interior_lds) a halo row node
  // (waves 0 and 1) or a halo column node (lanes < 2 TI of wave 0)
  const bool own_ok = i <= N0 - 1 && j <= N1 - 1;
  const long own_off = (long)N1 * i + j;
  const int own_slot = (w + 1) * W + lane + 1;
  int hrow_i = -1, hrow_slot = 0;
  if (w == 0) { hrow_i = i0 - 1; hrow_slot = lane + 1; }
  if (w == 1) { hrow_i = i0 + TI; hrow_slot = (TI + 1) * W + lane + 1; }
  const bool hrow_ok = hrow_i >= 0 && hrow_i <= N0 - 1 && j <= N1 - 1;
  const long hrow_off = (long)N1 * hrow_i + j;
  int hcol_j = -1, hcol_i = 0, hcol_slot = 0;
  if (w == 0 && lane < TI) { hcol_i = i0 + lane; hcol_j = j0 - 1; hcol_slot = (lane + 1) * W; }
  if (w == 0 && lane >= TI && lane < 2 * TI) {
    hcol_i = i0 + lane - TI; hcol_j = j0 + kTileJ; hcol_slot = (lane - TI + 1) * W + kTileJ + 1;
  }
  const bool hcol_ok = hcol_j >= 0 && hcol_j <= N1 - 1 && hcol_i <= N0 - 1;
  const long hcol_off = (long)N1 * hcol_i + hcol_j;
  // A^{n+1} of the plane to stage next.  Prefetched values stay in the storage type until they
  // are used: a conversion right after a load would make the wave wait for that load there,
  // and the prefetch would overlap nothing (FP32-bulk).
  R p_own[NC] = {}, p_row[NC] = {}, p_col[NC] = {};
  auto fetch_p = [&](int k) {
    const long b = N1N0 * k;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (own_ok) p_own[c] = p[c][b + own_off];
      if (hrow_ok) p_row[c] = p[c][b + hrow_off];
      if (hcol_ok) p_col[c] = p[c][b + hcol_off];
    }
  };
  auto stage_p = [&](int slot) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      double* d = L1 + (c * 3 + slot) * P;
      if (own_ok) d[own_slot] = (double)p_own[c];
      if (hrow_ok) d[hrow_slot] = (double)p_row[c];
      if (hcol_ok) d[hcol_slot] = (double)p_col[c];
    }
  };
  // A^n: own A_x, A_y (and phi) at planes k-1 .. k+2 (qx, qy, qf), own A_z at k and k+1, halo
  // of the next plane.  The curl reads A^n_x only at y +- 1 and A^n_y only at x +- 1, so A^n_x
  // needs no halo rows and A^n_y no halo columns; the gradient of phi needs both.
  R qx[4] = {}, qy[4] = {}, qf[4] = {}, qz = 0, qz_next = 0, n_row[NC] = {}, n_col[NC] = {};
  auto fetch_n_halo = [&](int k) {
    const long b = N1N0 * k;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c != 0 && hrow_ok) n_row[c] = n[c][b + hrow_off];
      if (c != 1 && hcol_ok) n_col[c] = n[c][b + hcol_off];
    }
  };
  fetch_p(kb - 1);
  stage_p(0);
  fetch_p(kb);
  stage_p(1);
  fetch_p(kb + 1);
  if (own_ok) {
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      qx[t] = n[0][N1N0 * (kb - 1 + t) + own_off];
      qy[t] = n[1][N1N0 * (kb - 1 + t) + own_off];
      if (SC) qf[t] = n[NC - 1][N1N0 * (kb - 1 + t) + own_off];
    }
    qz = n[2][N1N0 * kb + own_off];
  }
  fetch_n_halo(kb);
  const double mdt = q.mdt, dx2 = q.dx2, dy2 = q.dy2, dz2 = q.dz2;
  auto dt_ = [&](double v) { return div_rn(v, mdt, q.rmdt); };
  auto dx_ = [&](double v) { return div_rn(v, dx2, q.rdx2); };
  auto dy_ = [&](double v) { return div_rn(v, dy2, q.rdy2); };
  auto dz_ = [&](double v) { return div_rn(v, dz2, q.rdz2); };
  long m = N1N0 * kb + own_off;
  for (int k = kb; k < ke; ++k, m += N1N0) {
    const int s0 = (k - kb + 1) % 3, sp = (k - kb + 2) % 3, sm = (k - kb) % 3;
    stage_p(sp);
    {
      const double own[4] = {(double)qx[1], (double)qy[1], (double)qz, (double)qf[1]};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        double* d = L0 + c * P;
        if (own_ok) d[own_slot] = own[c];
        if (c != 0 && hrow_ok) d[hrow_slot] = (double)n_row[c];
        if (c != 1 && hcol_ok) d[hcol_slot] = (double)n_col[c];
      }
    }
    __syncthreads();
    if (k + 2 <= ke) fetch_p(k + 2);
    if (k + 1 < ke) {
      fetch_n_halo(k + 1);
      if (own_ok) {
        qx[3] = n[0][m + 2 * N1N0];
        qy[3] = n[1][m + 2 * N1N0];
        if (SC) qf[3] = n[NC - 1][m + 2 * N1N0];
        qz_next = n[2][m + N1N0];
      }
    }
    if (active) {
      const double v1[4] = {(double)qx[1], (double)qy[1], (double)qz, (double)qf[1]};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const double* c0 = L1 + (c * 3 + s0) * P + own_slot;
        const double* cp = L1 + (c * 3 + sp) * P + own_slot;
        const double* cm = L1 + (c * 3 + sm) * P + own_slot;
        double r;
        if (NSFD) {
          double tx = c0[W] + c0[-W] + s.beta * (cp[W] + cm[W] + cp[-W] + cm[-W]);
          double ty = c0[1] + c0[-1] + s.beta * (cp[1] + cm[1] + cp[-1] + cm[-1]);
          r = s.a0 * c0[0] - v1[c] + s.alpha * (s.a1 * tx + s.a2 * ty) + s.a3 * (cp[0] + cm[0]);
        } else {
          r = s.a0 * c0[0] - v1[c] + s.a1 * (c0[W] + c0[-W]) + s.a2 * (c0[1] + c0[-1]) + s.a3 * (cp[0] + cm[0]);
        }
        st_stream(x[c], m, (R)r);  // X and E/B are not read again here: keep L2 for the halos
      }
      if (ebneed) {
        const double* n0l = L0 + own_slot;
        const double* n1l = L0 + P + own_slot;
        const double* n2l = L0 + 2 * P + own_slot;
        const double* p0l = L1 + (0 * 3 + s0) * P + own_slot;
        const double* p1l = L1 + (1 * 3 + s0) * P + own_slot;
        const double* p2l = L1 + (2 * 3 + s0) * P + own_slot;
        const double p0p = L1[(0 * 3 + sp) * P + own_slot], p0m = L1[(0 * 3 + sm) * P + own_slot];
        const double p1p = L1[(1 * 3 + sp) * P + own_slot], p1m = L1[(1 * 3 + sm) * P + own_slot];
        double ex = dt_(p0l[0]) - dt_((double)qx[1]);
        double ey = dt_(p1l[0]) - dt_((double)qy[1]);
        float ez = (float)dt_(p2l[0]);
        ez = (float)((double)ez - dt_(n2l[0]));
        if (SC) {  // minus the gradient of phi^n (eval_lds_body's expressions)
          const double* fl = L0 + (NC - 1) * P + own_slot;
          ex = ex - dx_(fl[W] - fl[-W]);
          ey = ey - dy_(fl[1] - fl[-1]);
          ez = (float)((double)ez - dz_((double)qf[2] - (double)qf[0]));
        }
        const float bx = (float)(0.5 * (dy_(n2l[1] - n2l[-1]) - dz_((double)qy[2] - (double)qy[0]) +
                                        dy_(p2l[1] - p2l[-1]) - dz_(p1p - p1m)));
        const float by = (float)(0.5 * (dz_((double)qx[2] - (double)qx[0]) - dx_(n2l[W] - n2l[-W]) +
                                        dz_(p0p - p0m) - dx_(p2l[W] - p2l[-W])));
        const float bz = (float)(0.5 * (dx_(n1l[W] - n1l[-W]) - dy_(n0l[1] - n0l[-1]) +
                                        dx_(p1l[W] - p1l[-W]) - dy_(p0l[1] - p0l[-1])));
        const f2 v0 = {(float)ex, (float)ey}, vv1 = {ez, bx}, v2 = {by, bz};
        auto put = [&](long node) {
          st_stream(ebg, kEBPairs * node, v0);
          st_stream(ebg, kEBPairs * node + 1, vv1);
          st_stream(ebg, kEBPairs * node + 2, v2);
        };
        put(m);
        if (k == 1) put(m - N1N0);
        if (k == N2 - 2) put(m + N1N0);
      }
    }
    __syncthreads();
    qx[0] = qx[1]; qx[1] = qx[2]; qx[2] = qx[3];
    qy[0] = qy[1]; qy[1] = qy[2]; qy[2] = qy[3];
    qf[0] = qf[1]; qf[1] = qf[2]; qf[2] = qf[3];
    qz = qz_next;
  }
}

// The flat form of the fused kernel (see interior_flat_body): A^{n+1}'s three planes and their
// neighbours in registers, A^n's transverse neighbours from L1/L2.
template <typename R, bool NSFD, bool SC>
__global__ __launch_bounds__(kFlatThreads) void k_stencil_eb_flat(FieldSet An1, FieldSet An, FieldSet X,
                                                                  float* __restrict__ eb, int N0, int N1, int N2,
                                                                  int tiles, int K, StencilConst s, EvalConst q,
                                                                  const int* __restrict__ zr, int pb0, int pb1) {
  constexpr int NC = SC ? 4 : 3;
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  FlatNode f;
  if (!flat_node(lb % tiles, lb / tiles, K, 1, N2 - 2, N0, N1, f)) return;
  const bool ebneed = !zr || lazy_needed(f.kb, f.ke, zr, pb0, pb1);
  const gptr<f2> ebg = G(reinterpret_cast<f2*>(eb));
  const long N1N0 = (long)N1 * N0;
  gptr<const R> p[NC], n[NC];
  gptr<R> x[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    p[c] = G((const R*)component(An1, c));
    n[c] = G((const R*)component(An, c));
    x[c] = G((R*)component(X, c));
  }
  const double mdt = q.mdt, dx2 = q.dx2, dy2 = q.dy2, dz2 = q.dz2;
  auto dt_ = [&](double v) { return div_rn(v, mdt, q.rmdt); };
  auto dx_ = [&](double v) { return div_rn(v, dx2, q.rdx2); };
  auto dy_ = [&](double v) { return div_rn(v, dy2, q.rdy2); };
  auto dz_ = [&](double v) { return div_rn(v, dz2, q.rdz2); };
  long m = f.m;
  RawPlane<R> rm[NC], r0[NC], rp[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    rm[c] = raw_plane<R>(p[c], m - N1N0, N1);
    r0[c] = raw_plane<R>(p[c], m, N1);
  }
  // A^n_x, A^n_y (and phi^n) at planes k-1, k, k+1
  double qx[3], qy[3], qf[3];
  qx[0] = rd(n[0], m - N1N0); qx[1] = rd(n[0], m);
  qy[0] = rd(n[1], m - N1N0); qy[1] = rd(n[1], m);
  if (SC) { qf[0] = rd(n[NC - 1], m - N1N0); qf[1] = rd(n[NC - 1], m); }
  for (int k = f.kb; k < f.ke; ++k, m += N1N0) {
#pragma unroll
    for (int c = 0; c < NC; ++c) rp[c] = raw_plane<R>(p[c], m + N1N0, N1);
    qx[2] = rd(n[0], m + N1N0);
    qy[2] = rd(n[1], m + N1N0);
    if (SC) qf[2] = rd(n[NC - 1], m + N1N0);
    const double qz = rd(n[2], m);
    const double v1[4] = {qx[1], qy[1], qz, SC ? qf[1] : 0.0};
    Plane5 pm[NC], p0[NC], pp[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      pm[c] = rm[c].wide();
      p0[c] = r0[c].wide();
      pp[c] = rp[c].wide();
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      double r;
      if (NSFD) {
        const double tx = p0[c].xp + p0[c].xm + s.beta * (pp[c].xp + pm[c].xp + pp[c].xm + pm[c].xm);
        const double ty = p0[c].yp + p0[c].ym + s.beta * (pp[c].yp + pm[c].yp + pp[c].ym + pm[c].ym);
        r = s.a0 * p0[c].c - v1[c] + s.alpha * (s.a1 * tx + s.a2 * ty) + s.a3 * (pp[c].c + pm[c].c);
      } else {
        r = s.a0 * p0[c].c - v1[c] + s.a1 * (p0[c].xp + p0[c].xm) + s.a2 * (p0[c].yp + p0[c].ym) +
            s.a3 * (pp[c].c + pm[c].c);
      }
      st_stream(x[c], m, (R)r);
    }
    if (ebneed) {
      double ex = dt_(p0[0].c) - dt_(qx[1]);
      double ey = dt_(p0[1].c) - dt_(qy[1]);
      float ez = (float)dt_(p0[2].c);
      ez = (float)((double)ez - dt_(qz));
      if (SC) {  // minus the gradient of phi^n
        ex = ex - dx_(rd(n[NC - 1], m + N1) - rd(n[NC - 1], m - N1));
        ey = ey - dy_(rd(n[NC - 1], m + 1) - rd(n[NC - 1], m - 1));
        ez = (float)((double)ez - dz_(qf[2] - qf[0]));
      }
      const float bx = (float)(0.5 * (dy_(rd(n[2], m + 1) - rd(n[2], m - 1)) - dz_(qy[2] - qy[0]) +
                                      dy_(p0[2].yp - p0[2].ym) - dz_(pp[1].c - pm[1].c)));
      const float by = (float)(0.5 * (dz_(qx[2] - qx[0]) - dx_(rd(n[2], m + N1) - rd(n[2], m - N1)) +
                                      dz_(pp[0].c - pm[0].c) - dx_(p0[2].xp - p0[2].xm)));
      const float bz = (float)(0.5 * (dx_(rd(n[1], m + N1) - rd(n[1], m - N1)) - dy_(rd(n[0], m + 1) - rd(n[0], m - 1)) +
                                      dx_(p0[1].xp - p0[1].xm) - dy_(p0[0].yp - p0[0].ym)));
      const f2 v0 = {(float)ex, (float)ey}, vv1 = {ez, bx}, v2 = {by, bz};
      auto put = [&](long node) {
        st_stream(ebg, kEBPairs * node, v0);
        st_stream(ebg, kEBPairs * node + 1, vv1);
        st_stream(ebg, kEBPairs * node + 2, v2);
      };
      put(m);
      if (k == 1) put(m - N1N0);
      if (k == N2 - 2) put(m + N1N0);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      rm[c] = r0[c];
      r0[c] = rp[c];
    }
    qx[0] = qx[1]; qx[1] = qx[2];
    qy[0] = qy[1]; qy[1] = qy[2];
    if (SC) { qf[0] = qf[1]; qf[1] = qf[2]; }
  }
}

// ---- batched forms: persistent workgroups walking a table of (instance, local tile) ---------
// Workgroup b takes entries r * G + l(b), r = 0, 1, ..., where l gives every XCD a contiguous
// run of entries, so neighbouring tiles of one instance meet in one L2.
__device__ inline int batch_entry(int r) { return r * (int)gridDim.x + xcd_logical_block(blockIdx.x, gridDim.x); }

template <typename R, bool NSFD, int TI, int K, bool LDS>
__global__ __launch_bounds__(kTileJ* TI) void kb_interior(const BatchView* __restrict__ V, BatchTiles T) {
  for (int r = 0;; ++r) {
    const int t = batch_entry(r);
    if (t >= T.n) break;
    const int2 e = T.t[t];
    const BatchView& v = V[e.x];
    if (v.active) {
      if constexpr (LDS) {
        MurYFace yf;  // a local copy: stores to the potentials cannot alias it
        for (int q = 0; q < 5; ++q) yf.B[q] = v.mur.cB[q];
        yf.mask = v.faces;
        interior_lds_body<R, NSFD, TI, K, true>(v.lvl[v.i_n], v.lvl[v.i_nm1], v.lvl[v.i_np1], v.ncomp, v.N0, v.N1,
                                                v.N2, v.tilesJ, v.tilesI, v.chunks, v.a[0], v.a[1], v.a[2], v.a[3],
                                                v.a[4], v.a[5], v.alpha, v.beta, e.y, yf);
      } else {
        MurYFace yf;
        for (int q = 0; q < 5; ++q) yf.B[q] = v.mur.cB[q];
        yf.mask = v.faces;
        interior_body<R, NSFD, TI, K, true>(v.lvl[v.i_n], v.lvl[v.i_nm1], v.lvl[v.i_np1], v.ncomp, v.N0, v.N1, v.N2,
                                            v.tilesJ, v.tilesI, v.chunks, v.a[0], v.a[1], v.a[2], v.a[3], v.a[4],
                                            v.a[5], v.alpha, v.beta, e.y, yf);
      }
    }
    if constexpr (LDS) __syncthreads();  // the LDS ring is reused by the next tile
  }
}

template <typename R, int TI, int K, bool LDS>
__global__ __launch_bounds__(kTileJ* TI) void kb_eval(const BatchView* __restrict__ V, BatchTiles T) {
  for (int r = 0;; ++r) {
    const int t = batch_entry(r);
    if (t >= T.n) break;
    const int2 e = T.t[t];
    const BatchView& v = V[e.x];
    if (v.active) {
      const EvalConst q = v.ev;  // a local copy: stores to eb cannot alias it
      if constexpr (LDS) {
        if (v.ncomp == 4)  // space charge: E includes -grad phi^n
          eval_lds_body<R, true, TI, K>(v.lvl[v.i_n], v.lvl[v.i_np1], v.eb, v.N0, v.N1, v.N2, v.tilesJ, v.tilesI, 1,
                                        v.N2 - 2, q, nullptr, 0, -1, e.y);
        else
          eval_lds_body<R, false, TI, K>(v.lvl[v.i_n], v.lvl[v.i_np1], v.eb, v.N0, v.N1, v.N2, v.tilesJ, v.tilesI,
                                         1, v.N2 - 2, q, nullptr, 0, -1, e.y);
      } else {
        if (v.ncomp == 4)
          eval_body<R, true, TI, K>(v.lvl[v.i_n], v.lvl[v.i_np1], v.eb, v.N0, v.N1, v.N2, v.tilesJ, v.tilesI, 1,
                                    v.N2 - 2, q, nullptr, 0, -1, e.y);
        else
          eval_body<R, false, TI, K>(v.lvl[v.i_n], v.lvl[v.i_np1], v.eb, v.N0, v.N1, v.N2, v.tilesJ, v.tilesI, 1,
                                     v.N2 - 2, q, nullptr, 0, -1, e.y);
      }
    }
    if constexpr (LDS) __syncthreads();
  }
}

// The flat forms: v.tilesI tiles of a plane, v.planes / v.eplanes planes per entry.
template <typename R, bool NSFD>
__global__ __launch_bounds__(kFlatThreads) void kb_interior_flat(const BatchView* __restrict__ V, BatchTiles T) {
  for (int r = 0;; ++r) {
    const int t = batch_entry(r);
    if (t >= T.n) break;
    const int2 e = T.t[t];
    const BatchView& v = V[e.x];
    if (!v.active) continue;
    MurYFace yf;  // a local copy: stores to the potentials cannot alias it
    for (int q = 0; q < 5; ++q) yf.B[q] = v.mur.cB[q];
    yf.mask = v.faces;
    if (v.faces)
      interior_flat_body<R, NSFD, true>(v.lvl[v.i_n], v.lvl[v.i_nm1], v.lvl[v.i_np1], v.ncomp, v.N0, v.N1, v.N2,
                                        v.tilesI, v.chunks, v.planes, v.a[0], v.a[1], v.a[2], v.a[3], v.a[4], v.a[5],
                                        v.alpha, v.beta, e.y, yf);
    else
      interior_flat_body<R, NSFD, false>(v.lvl[v.i_n], v.lvl[v.i_nm1], v.lvl[v.i_np1], v.ncomp, v.N0, v.N1, v.N2,
                                         v.tilesI, v.chunks, v.planes, v.a[0], v.a[1], v.a[2], v.a[3], v.a[4], v.a[5],
                                         v.alpha, v.beta, e.y, yf);
  }
}

template <typename R>
__global__ __launch_bounds__(kFlatThreads) void kb_eval_flat(const BatchView* __restrict__ V, BatchTiles T) {
  for (int r = 0;; ++r) {
    const int t = batch_entry(r);
    if (t >= T.n) break;
    const int2 e = T.t[t];
    const BatchView& v = V[e.x];
    if (!v.active) continue;
    const EvalConst q = v.ev;  // a local copy: stores to eb cannot alias it
    if (v.ncomp == 4)
      eval_flat_body<R, true>(v.lvl[v.i_n], v.lvl[v.i_np1], v.eb, v.N0, v.N1, v.N2, v.tilesI, v.eplanes, 1, v.N2 - 2,
                              q, nullptr, 0, -1, e.y);
    else
      eval_flat_body<R, false>(v.lvl[v.i_n], v.lvl[v.i_np1], v.eb, v.N0, v.N1, v.N2, v.tilesI, v.eplanes, 1, v.N2 - 2,
                               q, nullptr, 0, -1, e.y);
  }
}

// TF/SF injection of the seeded instances: entry .y = block of 256 nodes of the list.
template <typename R>
__global__ __launch_bounds__(256) void kb_tfsf(const BatchView* __restrict__ V, BatchTiles T) {
  for (int r = 0;; ++r) {
    const int t = batch_entry(r);
    if (t >= T.n) break;
    const int2 e = T.t[t];
    const BatchView& v = V[e.x];
    if (!v.active || !v.seeded) continue;
    tfsf_body<R>(v.lvl[v.i_np1], v.N0, v.N1, v.N2, v.grid, v.seed, v.time, v.a[1], v.a[2], v.a[3],
                 (long)e.y * 256 + threadIdx.x);
  }
}

// Mur faces, or edges and corners: entry .y = comp * blocks_per_comp + block
template <typename R, bool RIMS>
__global__ __launch_bounds__(256) void kb_mur(const BatchView* __restrict__ V, BatchTiles T) {
  for (int r = 0;; ++r) {
    const int t = batch_entry(r);
    if (t >= T.n) break;
    const int2 e = T.t[t];
    const BatchView& v = V[e.x];
    if (!v.active) continue;
    const FieldSet P = v.lvl[v.i_np1], N = v.lvl[v.i_n], M = v.lvl[v.i_nm1];
    if (RIMS) {
      const int nb = (int)mur_rim_blocks(v.N0, v.N1, v.N2);
      mur_rims_body<R>(P, N, M, v.ncomp, v.N0, v.N1, v.N2, v.mur, e.y % nb, nb, e.y / nb);
    } else {
      const int nb = (int)((mur_face_count(v.N0, v.N1, v.N2, v.faces) + 255) / 256);
      mur_faces_body<R>(P, N, M, v.ncomp, v.N0, v.N1, v.N2, v.mur, (long)(e.y % nb) * 256 + threadIdx.x, e.y / nb,
                        v.faces);
    }
  }
}

__global__ void k_fill_zero(uint4* p, size_t n16) {
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n16; t += (size_t)gridDim.x * blockDim.x)
    p[t] = make_uint4(0u, 0u, 0u, 0u);
}

__global__ void k_fill_zero_bytes(unsigned char* p, size_t n) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0;
}

// Planes per workgroup of the flat forms for `tile_planes` workgroup-planes: eight, the fastest
// from 64 x 64 x 512 nodes to 211 x 211 x 1531 (four and sixteen are within 4 %; thirty-two is
// 20-50 % slower at 71 x 71 x 397), fewer while that leaves under 1024 workgroups, four for a CU:
// 32 x 32 x 128 takes 9.9 us with eight planes and 7.7 with two, 45 x 45 x 203 13.4 and 12.1.
int flat_planes_for(long tile_planes) {
  int K = 8;
  while (K > 1 && tile_planes / K < 1024) K /= 2;
  return K;
}

EvalConst eval_const(const mithra_grid& g) {
  EvalConst q;
  q.mdt = -g.dt; q.dx2 = 2.0 * g.dx; q.dy2 = 2.0 * g.dy; q.dz2 = 2.0 * g.dz;
  q.rmdt = 1.0 / q.mdt; q.rdx2 = 1.0 / q.dx2; q.rdy2 = 1.0 / q.dy2; q.rdz2 = 1.0 / q.dz2;
  return q;
}

template <typename R, bool NSFD>
hipError_t interior_flat_launch(Domain* d, int mask) {
  const mithra_grid& g = d->g;
  const int tiles = flat_tiles(g.N0, g.N1), K = flat_planes_for((long)tiles * (g.N2 - 2) * d->ncomp);
  const int chunks = (g.N2 - 2 + K - 1) / K;
  const dim3 grid((unsigned)((long)tiles * chunks * d->ncomp));
  const double* a = d->co.a;
  MurYFace yf;
  for (int q = 0; q < 5; ++q) yf.B[q] = d->co.cB[q];
  yf.mask = mask;
  if (mask)
    hipLaunchKernelGGL((k_interior_flat<R, NSFD, true>), grid, dim3(kFlatThreads), 0, d->stream, d->lvl[d->i_n],
                       d->lvl[d->i_nm1], d->lvl[d->i_np1], d->ncomp, g.N0, g.N1, g.N2, tiles, chunks, K, a[0], a[1],
                       a[2], a[3], a[4], a[5], d->co.alpha, d->co.beta, yf);
  else
    hipLaunchKernelGGL((k_interior_flat<R, NSFD, false>), grid, dim3(kFlatThreads), 0, d->stream, d->lvl[d->i_n],
                       d->lvl[d->i_nm1], d->lvl[d->i_np1], d->ncomp, g.N0, g.N1, g.N2, tiles, chunks, K, a[0], a[1],
                       a[2], a[3], a[4], a[5], d->co.alpha, d->co.beta, yf);
  return hipGetLastError();
}

template <typename R, bool SC>
hipError_t eval_flat_launch(Domain* d, int klo, int khi, const int* zr, int pb0, int pb1) {
  const mithra_grid& g = d->g;
  const int planes = khi - klo + 1, tiles = flat_tiles(g.N0, g.N1), K = flat_planes_for((long)tiles * planes);
  const int chunks = (planes + K - 1) / K;
  hipLaunchKernelGGL((k_eval_flat<R, SC>), dim3((unsigned)((long)tiles * chunks)), dim3(kFlatThreads), 0, d->stream,
                     d->lvl[d->i_n], d->lvl[d->i_np1], d->eb, g.N0, g.N1, g.N2, tiles, K, klo, khi, eval_const(g), zr,
                     pb0, pb1);
  return hipGetLastError();
}

template <typename R, bool NSFD, bool SC>
hipError_t stencil_eb_flat_launch(Domain* d, const int* zr, int pb0, int pb1) {
  const mithra_grid& g = d->g;
  const int tiles = flat_tiles(g.N0, g.N1), K = flat_planes_for((long)tiles * (g.N2 - 2));
  const int chunks = (g.N2 - 2 + K - 1) / K;
  const double* a = d->co.a;
  const StencilConst s = {a[0], a[1], a[2], a[3], d->co.alpha, d->co.beta};
  hipLaunchKernelGGL((k_stencil_eb_flat<R, NSFD, SC>), dim3((unsigned)((long)tiles * chunks)), dim3(kFlatThreads), 0,
                     d->stream, d->lvl[d->i_np1], d->lvl[d->i_n], d->lvl[d->i_nm1], d->eb, g.N0, g.N1, g.N2, tiles, K,
                     s, eval_const(g), zr, pb0, pb1);
  return hipGetLastError();
}

// Tile shapes of the marched field kernels: rows of x per workgroup (one wavefront of 64 y
// nodes per row) and z planes per workgroup.  Shape 0, the default, is the flat form: its four
// wavefronts lie end to end over the plane, and it marches at most eight planes.  Every shape
// computes the same values; the autotuner (capi) picks the fastest per domain.
template <typename R, bool NSFD, int TI, int K, bool LDS = false>
hipError_t interior_launch(Domain* d, int ymask) {
  const mithra_grid& g = d->g;
  const int tilesJ = (g.N1 + kTileJ - 1) / kTileJ;
  const int tilesI = (g.N0 - 2 + TI - 1) / TI;
  const int chunks = (g.N2 - 2 + K - 1) / K;
  const long nblk = (long)tilesJ * tilesI * chunks * d->ncomp;
  const double* a = d->co.a;
  MurYFace yf;
  for (int q = 0; q < 5; ++q) yf.B[q] = d->co.cB[q];
  yf.mask = ymask;
  if constexpr (LDS) {
    if (ymask)
      hipLaunchKernelGGL((k_interior_lds<R, NSFD, TI, K, true>), dim3((unsigned)nblk), dim3(kTileJ * TI), 0,
                         d->stream, d->lvl[d->i_n], d->lvl[d->i_nm1], d->lvl[d->i_np1], d->ncomp, g.N0, g.N1, g.N2,
                         tilesJ, tilesI, chunks, a[0], a[1], a[2], a[3], a[4], a[5], d->co.alpha, d->co.beta, yf);
    else
      hipLaunchKernelGGL((k_interior_lds<R, NSFD, TI, K, false>), dim3((unsigned)nblk), dim3(kTileJ * TI), 0,
                         d->stream, d->lvl[d->i_n], d->lvl[d->i_nm1], d->lvl[d->i_np1], d->ncomp, g.N0, g.N1, g.N2,
                         tilesJ, tilesI, chunks, a[0], a[1], a[2], a[3], a[4], a[5], d->co.alpha, d->co.beta, yf);
  } else if (ymask) {
    hipLaunchKernelGGL((k_interior<R, NSFD, TI, K, true>), dim3((unsigned)nblk), dim3(kTileJ * TI), 0, d->stream,
                       d->lvl[d->i_n], d->lvl[d->i_nm1], d->lvl[d->i_np1], d->ncomp, g.N0, g.N1, g.N2, tilesJ, tilesI,
                       chunks, a[0], a[1], a[2], a[3], a[4], a[5], d->co.alpha, d->co.beta, yf);
  } else {
    hipLaunchKernelGGL((k_interior<R, NSFD, TI, K, false>), dim3((unsigned)nblk), dim3(kTileJ * TI), 0, d->stream,
                       d->lvl[d->i_n], d->lvl[d->i_nm1], d->lvl[d->i_np1], d->ncomp, g.N0, g.N1, g.N2, tilesJ, tilesI,
                       chunks, a[0], a[1], a[2], a[3], a[4], a[5], d->co.alpha, d->co.beta, yf);
  }
  return hipGetLastError();
}

template <typename R, bool SC, int TI, int K, bool LDS = false>
hipError_t eval_launch(Domain* d, int klo, int khi, const int* zr, int pb0, int pb1) {
  const mithra_grid& g = d->g;
  const int tilesJ = (g.N1 + kTileJ - 1) / kTileJ;
  const int tilesI = (g.N0 - 2 + TI - 1) / TI;
  const int chunks = (khi - klo + 1 + K - 1) / K;
  const long nblk = (long)tilesJ * tilesI * chunks;
  const EvalConst q = eval_const(g);
  if constexpr (LDS)
    hipLaunchKernelGGL((k_eval_lds<R, SC, TI, K>), dim3((unsigned)nblk), dim3(kTileJ * TI), 0, d->stream,
                       d->lvl[d->i_n], d->lvl[d->i_np1], d->eb, g.N0, g.N1, g.N2, tilesJ, tilesI, klo, khi, q, zr, pb0, pb1);
  else
    hipLaunchKernelGGL((k_eval_eb<R, SC, TI, K>), dim3((unsigned)nblk), dim3(kTileJ * TI), 0, d->stream,
                       d->lvl[d->i_n], d->lvl[d->i_np1], d->eb, g.N0, g.N1, g.N2, tilesJ, tilesI, klo, khi, q, zr, pb0, pb1);
  return hipGetLastError();
}

template <typename R, bool FLAG>
hipError_t field_variant(Domain* d, int kernel, int v, int klo, int khi, const int* zr = nullptr, int pb0 = 0,
                         int pb1 = -1, int ymask = 0) {
  // kernel 0: interior (FLAG = NSFD), kernel 1: E/B evaluation (FLAG = space charge)
#define MITHRA_VARIANT(idx, TI, K)                                                            \
  case idx:                                                                                    \
    return kernel == 0 ? interior_launch<R, FLAG, TI, K>(d, ymask) : eval_launch<R, FLAG, TI, K>(d, klo, khi, zr, pb0, pb1);
  switch (v) {
    case 0: return kernel == 0 ? interior_flat_launch<R, FLAG>(d, ymask) : eval_flat_launch<R, FLAG>(d, klo, khi, zr, pb0, pb1);
    MITHRA_VARIANT(1, 2, 64)
    MITHRA_VARIANT(2, 4, 32)
    MITHRA_VARIANT(3, 4, 128)
    MITHRA_VARIANT(4, 8, 32)
    MITHRA_VARIANT(5, 8, 64)
    MITHRA_VARIANT(6, 16, 32)
  }
  static_assert(kTileVariants == 10, "variant table and switch disagree");
  // variants 7..9: the LDS-staged (2.5-D blocked) forms of both kernels
  switch (v) {
    case 7: return kernel == 0 ? interior_launch<R, FLAG, 4, 64, true>(d, ymask) : eval_launch<R, FLAG, 4, 64, true>(d, klo, khi, zr, pb0, pb1);
    case 8: return kernel == 0 ? interior_launch<R, FLAG, 8, 64, true>(d, ymask) : eval_launch<R, FLAG, 8, 64, true>(d, klo, khi, zr, pb0, pb1);
    case 9: return kernel == 0 ? interior_launch<R, FLAG, 16, 64, true>(d, ymask) : eval_launch<R, FLAG, 16, 64, true>(d, klo, khi, zr, pb0, pb1);
  }
#undef MITHRA_VARIANT
  return hipErrorInvalidValue;
}

// Below this many nodes the flat forms are the faster ones in FP64 too.  The tiled forms with LDS
// planes read a node's neighbours once from L2 but march serially; they win once the
// levels no longer fit the 256 MB last-level cache and the workgroups suffice.  The line is the interior
// update's, us flat / 4 x 64 tiles: 64 x 64 x 1024 135 / 142, 96 x 96 x 600 169 / 164, 128 x 128 x 330 158 / 157
// (206 / 173 with phi), 128 x 128 x 500 232 / 191; ragged meshes cross later (150 x 150 x 360 218 / 257, 200 x
// 210 x 340 370 / 405).  The fused kernel's own line would lie at some 8 million nodes: 32 x 32 x 128 with phi 12 /
// 163, 71 x 71 x 397 60 / 182, 90 x 90 x 301 77 / 165, 131 x 147 x 260 107 / 183 (192 / 256 with phi),
// 96 x 96 x 600 115 / 185, 150 x 150 x 360 259 / 265, 128 x 128 x 500 247 / 226, 128 x 128 x 850 406 / 354,
// 128 x 128 x 1024 463 / 369; so that it is not the fastest shape on meshes of 5 to 8 million.
constexpr long kFlatNodes = 5000000;

template <typename R, bool NSFD, int TI, int K, bool SC>
hipError_t stencil_eb_launch(Domain* d, const int* zr, int pb0, int pb1) {
  const mithra_grid& g = d->g;
  const int tilesJ = (g.N1 + kTileJ - 1) / kTileJ;
  const int tilesI = (g.N0 - 2 + TI - 1) / TI;
  const int chunks = (g.N2 - 2 + K - 1) / K;
  const long nblk = (long)tilesJ * tilesI * chunks;
  const double* a = d->co.a;
  const StencilConst s = {a[0], a[1], a[2], a[3], d->co.alpha, d->co.beta};
  const EvalConst q = eval_const(g);
  hipLaunchKernelGGL((k_stencil_eb<R, NSFD, TI, K, SC>), dim3((unsigned)nblk), dim3(kTileJ * TI), 0, d->stream,
                     d->lvl[d->i_np1], d->lvl[d->i_n], d->lvl[d->i_nm1], d->eb, g.N0, g.N1, g.N2, tilesJ, tilesI, s,
                     q, zr, pb0, pb1);
  return hipGetLastError();
}

template <typename R, bool NSFD, bool SC = false>
hipError_t stencil_eb_variant(Domain* d, const int* zr, int pb0, int pb1) {
  static_assert(kFusedVariants == 4, "variant table and switch disagree");
  switch (d->tile_fused) {
    // the flat form up to kFlatNodes (see there)
    case 0:
      if (d->nodes < kFlatNodes) return stencil_eb_flat_launch<R, NSFD, SC>(d, zr, pb0, pb1);
      return stencil_eb_launch<R, NSFD, 4, 64, SC>(d, zr, pb0, pb1);
    case 1: return stencil_eb_launch<R, NSFD, 8, 64, SC>(d, zr, pb0, pb1);
    // under space charge 16-row tiles need more than the 128 registers a 1024-thread
    // workgroup allows (they spill): that variant runs the 8-row form
    case 2:
      if constexpr (SC) return stencil_eb_launch<R, NSFD, 8, 64, SC>(d, zr, pb0, pb1);
      else return stencil_eb_launch<R, NSFD, 16, 64, SC>(d, zr, pb0, pb1);
    case 3: return stencil_eb_launch<R, NSFD, 8, 128, SC>(d, zr, pb0, pb1);
  }
  return hipErrorInvalidValue;
}

template <typename R>
hipError_t stencil_eb_impl(Domain* d) {
  const int* zr = nullptr;
  int pb0 = 0, pb1 = -1;
  if (d->lazy_fields && d->zrange_valid) {
    if (const hipError_t e = launch_zrange(d); e != hipSuccess) return e;
    zr = d->zrange;
    lazy_planes(d, &pb0, &pb1);
  }
  if (d->ncomp == 4)
    return d->g.solver == MITHRA_SOLVER_NSFD ? stencil_eb_variant<R, true, true>(d, zr, pb0, pb1)
                                             : stencil_eb_variant<R, false, true>(d, zr, pb0, pb1);
  return d->g.solver == MITHRA_SOLVER_NSFD ? stencil_eb_variant<R, true>(d, zr, pb0, pb1)
                                           : stencil_eb_variant<R, false>(d, zr, pb0, pb1);
}

template <typename R>
hipError_t interior_impl(Domain* d, bool fuse_faces) {
  const int ymask = fuse_faces ? faces_mask(d->tile_interior, d->g.N1) : 0;
  const hipError_t e = d->g.solver == MITHRA_SOLVER_NSFD
                           ? field_variant<R, true>(d, 0, d->tile_interior, 0, 0, nullptr, 0, -1, ymask)
                           : field_variant<R, false>(d, 0, d->tile_interior, 0, 0, nullptr, 0, -1, ymask);
  d->faces_pending = e == hipSuccess ? ymask : 0;
  return e;
}

template <typename R>
hipError_t tfsf_sg_impl(Domain* d, double time, const mithra_seed* seed) {
  const mithra_grid& g = d->g;
  const long ni = g.N0 - 4, nj = g.N1 - 4, nk = g.N2 - 4;
  const long blocks[4] = {4 * nj * nk, 4 * ni * nk, 2 * ni * nj, 2 * ni * nj};
  const long n = blocks[0] + blocks[1] + blocks[2] + blocks[3];
  if (n <= 0) return hipSuccess;
  if (d->sg_cap < n) {
    hipError_t e = hipStreamSynchronize(d->stream);
    if (e != hipSuccess) return e;
    (void)hipFree(d->sg_buf);
    d->sg_buf = nullptr;
    d->sg_cap = 0;
    if ((e = hipMalloc(&d->sg_buf, (size_t)n * (4 * sizeof(double) + sizeof(int)))) != hipSuccess) return e;
    d->sg_cap = n;
  }
  double* term = (double*)d->sg_buf;
  double* run = term + n;
  int* reset = (int*)(run + 3 * n);
  const unsigned grid = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(k_sg_terms, dim3(grid), dim3(256), 0, d->stream, g, *seed, time, n, term, reset);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_sg_running, dim3(1), dim3(64), 0, d->stream, *seed, n, term, reset, run);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const double coef[4] = {d->co.a[1], d->co.a[2], d->co.a[3], d->co.a[3]};
  long first = 0;
  for (int b = 0; b < 4; ++b) {
    if (blocks[b] > 0) {
      hipLaunchKernelGGL((k_sg_apply<R>), dim3((unsigned)((blocks[b] + 255) / 256)), dim3(256), 0, d->stream,
                         d->lvl[d->i_np1], g, first, blocks[b], run, coef[b]);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    first += blocks[b];
  }
  return hipSuccess;
}

template <typename R>
hipError_t tfsf_impl(Domain* d, double time, const mithra_seed* seed) {
  const mithra_grid& g = d->g;
  // the standing types are not handled by Seed::fields: its output stays the zero vector the
  // update starts from (src/classes.cpp:758-851, src/fdtd.cpp:239), so nothing is injected
  if (seed->seed_type >= MITHRA_SEED_STANDING_PLANEWAVE) return hipSuccess;
  if (seed->seed_type == MITHRA_SEED_SUPERGAUSSIANBEAM) return tfsf_sg_impl<R>(d, time, seed);
  hipLaunchKernelGGL((k_tfsf<R>), dim3((unsigned)((tfsf_count(g.N0, g.N1, g.N2) + 255) / 256)), dim3(256), 0,
                     d->stream, d->lvl[d->i_np1], g.N0, g.N1, g.N2, g, *seed, time, d->co.a[1], d->co.a[2],
                     d->co.a[3]);
  return hipGetLastError();
}

template <typename R>
hipError_t boundaries_impl(Domain* d) {
  const mithra_grid& g = d->g;
  const MurCoeffs c = mur_coeffs(d->co);
  FieldSet P = d->lvl[d->i_np1], N = d->lvl[d->i_n], M = d->lvl[d->i_nm1];
  const int mask = d->faces_pending;  // faces the interior launch already updated
  d->faces_pending = 0;
  const long nf = mur_face_count(g.N0, g.N1, g.N2, mask);
  hipLaunchKernelGGL((k_mur_faces<R>), dim3((unsigned)((nf + 255) / 256), d->ncomp), dim3(256), 0, d->stream, P, N, M,
                     d->ncomp, g.N0, g.N1, g.N2, c, mask);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || g.truncation_order != 2) return e;
  hipLaunchKernelGGL((k_mur_rims<R>), dim3((unsigned)mur_rim_blocks(g.N0, g.N1, g.N2), d->ncomp), dim3(256), 0,
                     d->stream, P, N, M, d->ncomp, g.N0, g.N1, g.N2, c);
  return hipGetLastError();
}

template <typename R>
hipError_t eval_impl(Domain* d, int klo, int khi, const int* zr = nullptr, int pb0 = 0, int pb1 = -1) {
  klo = std::max(klo, 1);
  khi = std::min(khi, d->g.N2 - 2);
  if (klo > khi) return hipSuccess;
  return d->g.space_charge ? field_variant<R, true>(d, 1, d->tile_eval, klo, khi, zr, pb0, pb1)
                           : field_variant<R, false>(d, 1, d->tile_eval, klo, khi, zr, pb0, pb1);
}

}  // namespace

extern const int kTileShapes[kTileVariants][2] = {{0, 8}, {2, 64}, {4, 32}, {4, 128}, {8, 32},
                                                  {8, 64}, {16, 32}, {4, 64}, {8, 64}, {16, 64}};

// The shapes a domain starts with.  In FP32 the flat interior update is the fastest at every size
// tried; in FP64 the LDS-staged 4 x 64 tiles from kFlatNodes on (see there).  The E/B evaluation
// reads more neighbours: its LDS forms win from 8M nodes in FP64 (128 x 128 x 512 139 against
// 165 us, 128 x 128 x 1024 263 / 323, 211 x 211 x 1531 1273 / 1357) and in FP32 from 16M nodes when
// the 64-node rows of the tiles waste few lanes (128 x 128 x 1024 186 / 215; but 150 x 150 x 1000
// 318 flat, 323 tiled).  The 8-row tiles fetch fewer halo rows, the 4-row ones suit ragged meshes.
// The fused kernel's 4-row tiles are ahead of the 8-row ones below 12 million nodes (128 x 128 x 500 226 / 255, x 670
// 286 / 324), behind from there where rows fill (x 850 354 / 348, x 970 376 / 368), and ahead on ragged
// meshes (200 x 210 x 340 521 / 617).
int default_tile(const Domain* d, int kernel) {
  const int N1 = d->g.N1;
  const bool f64 = d->precision == MITHRA_PRECISION_FP64, aligned = 10 * ((N1 + 63) / 64 * 64) < 11 * N1;
  if (kernel == 0) return f64 && d->nodes >= kFlatNodes ? 7 : 0;
  if (kernel == 1) return f64 ? (d->nodes < 8000000 ? 0 : aligned ? 8 : 7) : (d->nodes >= 16000000 && aligned ? 8 : 0);
  return d->nodes >= 16000000 && aligned ? 1 : 0;  // the fused kernel
}

int flat_tiles(int N0, int N1) { return (int)(((long)N1 * (N0 - 2) + kFlatThreads - 1) / kFlatThreads); }

int flat_planes(long tile_planes) { return flat_planes_for(tile_planes); }

hipError_t launch_interior(Domain* d, bool fuse_faces) {
  return d->precision == MITHRA_PRECISION_FP64 ? interior_impl<double>(d, fuse_faces)
                                               : interior_impl<float>(d, fuse_faces);
}

extern const int kFusedShapes[kFusedVariants][2] = {{4, 64}, {8, 64}, {16, 64}, {8, 128}};

hipError_t launch_stencil_eb(Domain* d) {
  if ((d->ncomp != 3 && d->ncomp != 4) || d->tile_fused < 0 || d->tile_fused >= kFusedVariants)
    return hipErrorInvalidValue;
  return d->precision == MITHRA_PRECISION_FP64 ? stencil_eb_impl<double>(d) : stencil_eb_impl<float>(d);
}

hipError_t launch_tfsf(Domain* d, double time, const mithra_seed* seed) {
  return d->precision == MITHRA_PRECISION_FP64 ? tfsf_impl<double>(d, time, seed) : tfsf_impl<float>(d, time, seed);
}

hipError_t launch_boundaries(Domain* d) {
  return d->precision == MITHRA_PRECISION_FP64 ? boundaries_impl<double>(d) : boundaries_impl<float>(d);
}

hipError_t launch_eval_eb(Domain* d) { return launch_eval_eb_range(d, 1, d->g.N2 - 2); }

hipError_t launch_eval_eb_step(Domain* d) {
  if (!d->lazy_fields || !d->zrange_valid) return launch_eval_eb(d);
  if (const hipError_t e = launch_zrange(d); e != hipSuccess) return e;
  int pb0, pb1;
  lazy_planes(d, &pb0, &pb1);
  return d->precision == MITHRA_PRECISION_FP64 ? eval_impl<double>(d, 1, d->g.N2 - 2, d->zrange, pb0, pb1)
                                               : eval_impl<float>(d, 1, d->g.N2 - 2, d->zrange, pb0, pb1);
}

hipError_t launch_eval_eb_range(Domain* d, int klo, int khi) {
  return d->precision == MITHRA_PRECISION_FP64 ? eval_impl<double>(d, klo, khi) : eval_impl<float>(d, klo, khi);
}

hipError_t launch_fill_zero(Domain* d, void* ptr, size_t bytes) {
  // A fill kernel rather than hipMemsetAsync, so the step stays safe to capture in a graph.
  const size_t n16 = bytes / 16, tail = bytes % 16;
  if (n16) {
    unsigned blocks = (unsigned)((n16 + 255) / 256);
    if (blocks > 65536u) blocks = 65536u;
    hipLaunchKernelGGL(k_fill_zero, dim3(blocks), dim3(256), 0, d->stream, (uint4*)ptr, n16);
  }
  if (tail)
    hipLaunchKernelGGL(k_fill_zero_bytes, dim3(1), dim3(64), 0, d->stream, (unsigned char*)ptr + n16 * 16, tail);
  return hipGetLastError();
}


// ---- batched launchers --------------------------------------------------------------------
template <typename R, int TI, int K, bool LDS>
hipError_t batch_field(BatchView* V, BatchTiles T, int kernel, int nsfd, hipStream_t s) {
  // workgroups resident per CU, by shape: LDS forms are register- or LDS-bound, the others small
  const int per_cu = LDS ? (TI >= 16 ? 1 : TI >= 8 ? 2 : 4) : (TI >= 16 ? 2 : TI >= 8 ? 4 : 8);
  const int g = batch_grid(T.n, per_cu);
  if (kernel == 0) {
    if (nsfd) hipLaunchKernelGGL((kb_interior<R, true, TI, K, LDS>), dim3(g), dim3(kTileJ * TI), 0, s, V, T);
    else hipLaunchKernelGGL((kb_interior<R, false, TI, K, LDS>), dim3(g), dim3(kTileJ * TI), 0, s, V, T);
  } else {
    hipLaunchKernelGGL((kb_eval<R, TI, K, LDS>), dim3(g), dim3(kTileJ * TI), 0, s, V, T);
  }
  return hipGetLastError();
}

template <typename R>
hipError_t batch_field_variant(BatchView* V, BatchTiles T, int kernel, int variant, int nsfd, hipStream_t s) {
  if (T.n == 0) return hipSuccess;
  switch (variant) {
    case 0: {
      const dim3 g(batch_grid(T.n, 8)), b(kFlatThreads);
      if (kernel == 1) hipLaunchKernelGGL((kb_eval_flat<R>), g, b, 0, s, V, T);
      else if (nsfd) hipLaunchKernelGGL((kb_interior_flat<R, true>), g, b, 0, s, V, T);
      else hipLaunchKernelGGL((kb_interior_flat<R, false>), g, b, 0, s, V, T);
      return hipGetLastError();
    }
    case 1: return batch_field<R, 2, 64, false>(V, T, kernel, nsfd, s);
    case 2: return batch_field<R, 4, 32, false>(V, T, kernel, nsfd, s);
    case 3: return batch_field<R, 4, 128, false>(V, T, kernel, nsfd, s);
    case 4: return batch_field<R, 8, 32, false>(V, T, kernel, nsfd, s);
    case 5: return batch_field<R, 8, 64, false>(V, T, kernel, nsfd, s);
    case 6: return batch_field<R, 16, 32, false>(V, T, kernel, nsfd, s);
    case 7: return batch_field<R, 4, 64, true>(V, T, kernel, nsfd, s);
    case 8: return batch_field<R, 8, 64, true>(V, T, kernel, nsfd, s);
    case 9: return batch_field<R, 16, 64, true>(V, T, kernel, nsfd, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_batch_interior(BatchView* V, BatchTiles T, int variant, int precision, int nsfd, hipStream_t s) {
  return precision == MITHRA_PRECISION_FP64 ? batch_field_variant<double>(V, T, 0, variant, nsfd, s)
                                            : batch_field_variant<float>(V, T, 0, variant, nsfd, s);
}

hipError_t launch_batch_eval(BatchView* V, BatchTiles T, int variant, int precision, hipStream_t s) {
  return precision == MITHRA_PRECISION_FP64 ? batch_field_variant<double>(V, T, 1, variant, 0, s)
                                            : batch_field_variant<float>(V, T, 1, variant, 0, s);
}

hipError_t launch_batch_tfsf(BatchView* V, BatchTiles T, int precision, hipStream_t s) {
  if (!T.n) return hipSuccess;
  if (precision == MITHRA_PRECISION_FP64)
    hipLaunchKernelGGL((kb_tfsf<double>), dim3(batch_grid(T.n, 8)), dim3(256), 0, s, V, T);
  else
    hipLaunchKernelGGL((kb_tfsf<float>), dim3(batch_grid(T.n, 8)), dim3(256), 0, s, V, T);
  return hipGetLastError();
}

long tfsf_nodes(int N0, int N1, int N2) { return tfsf_count(N0, N1, N2); }

template <typename R>
hipError_t batch_mur_impl(BatchView* V, BatchTiles faces, BatchTiles rims, hipStream_t s) {
  if (faces.n) hipLaunchKernelGGL((kb_mur<R, false>), dim3(batch_grid(faces.n, 8)), dim3(256), 0, s, V, faces);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (rims.n) hipLaunchKernelGGL((kb_mur<R, true>), dim3(batch_grid(rims.n, 8)), dim3(256), 0, s, V, rims);
  return hipGetLastError();
}

hipError_t launch_batch_mur(BatchView* V, BatchTiles faces, BatchTiles rims, int precision, hipStream_t s) {
  return precision == MITHRA_PRECISION_FP64 ? batch_mur_impl<double>(V, faces, rims, s)
                                            : batch_mur_impl<float>(V, faces, rims, s);
}

}  // namespace mithra

namespace {

// Runs one of the analytic-seed kernels over n host points: inputs in (n_in arrays of per[i]
// doubles per point), one output of per_out doubles per point.
template <typename Launch>
int eval_points(long n, std::initializer_list<std::pair<const double*, int>> in, int per_out, double* out,
                Launch launch) {
  if (n < 0 || (n > 0 && !out)) return MITHRA_E_ARG;
  for (const auto& a : in)
    if (n > 0 && !a.first) return MITHRA_E_ARG;
  if (n == 0) return MITHRA_OK;
  std::vector<double*> dev;
  hipError_t e = hipSuccess;
  auto cleanup = [&]() {
    for (double* p : dev) (void)hipFree(p);
  };
  for (const auto& a : in) {
    double* p = nullptr;
    if ((e = hipMalloc(&p, sizeof(double) * a.second * n)) != hipSuccess) break;
    dev.push_back(p);
    if ((e = hipMemcpy(p, a.first, sizeof(double) * a.second * n, hipMemcpyHostToDevice)) != hipSuccess) break;
  }
  double* o = nullptr;
  if (e == hipSuccess && (e = hipMalloc(&o, sizeof(double) * per_out * n)) == hipSuccess) dev.push_back(o);
  if (e == hipSuccess) {
    launch(dev.data(), o, (unsigned)((n + 255) / 256));
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(out, o, sizeof(double) * per_out * n, hipMemcpyDeviceToHost);
  cleanup();
  if (e == hipErrorOutOfMemory) return MITHRA_E_NOMEM;
  return e == hipSuccess ? MITHRA_OK : MITHRA_E_HIP - (int)e;
}

bool signal_valid(const mithra_seed* s) { return s->signal_type >= MITHRA_SIGNAL_NEUMANN && s->signal_type <= MITHRA_SIGNAL_INVGAUSSIAN; }

}  // namespace

extern "C" {

int mithra_signal_evaluate(const mithra_seed* seed, const double* t, const double* phase, long n, double* out) {
  if (!seed || !signal_valid(seed)) return MITHRA_E_ARG;
  const mithra_seed s = *seed;
  return eval_points(n, {{t, 1}, {phase, 1}}, 1, out, [&](double** in, double* o, unsigned blocks) {
    hipLaunchKernelGGL(mithra::k_signal_eval, dim3(blocks), dim3(256), 0, 0, s, in[0], in[1], n, o);
  });
}

int mithra_seed_evaluate(const mithra_seed* seed, const double* r, const double* time, long n, double* a) {
  if (!seed || !signal_valid(seed)) return MITHRA_E_ARG;
  if (seed->seed_type < MITHRA_SEED_PLANEWAVE || seed->seed_type > MITHRA_SEED_STANDING_SUPERGAUSSIANBEAM)
    return MITHRA_E_ARG;
  if (n < 0 || (n > 0 && (!r || !time || !a))) return MITHRA_E_ARG;
  if (seed->seed_type >= MITHRA_SEED_STANDING_PLANEWAVE) {  // Seed::fields leaves the zero vector as it is
    for (long q = 0; q < 3 * n; ++q) a[q] = 0.0;
    return MITHRA_OK;
  }
  const mithra_seed s = *seed;
  if (s.seed_type == MITHRA_SEED_SUPERGAUSSIANBEAM) {
    // one output vector, zeroed once and passed to every point in turn, as the injection loop
    // passes it (src/fdtd.cpp:239, :307-373)
    if (n == 0) return MITHRA_OK;
    double* term = nullptr;
    int* reset = nullptr;
    if (hipMalloc(&term, sizeof(double) * n) != hipSuccess || hipMalloc(&reset, sizeof(int) * n) != hipSuccess) {
      (void)hipFree(term);
      return MITHRA_E_NOMEM;
    }
    const int rc = eval_points(n, {{r, 3}, {time, 1}}, 3, a, [&](double** in, double* o, unsigned blocks) {
      hipLaunchKernelGGL(mithra::k_sg_point_terms, dim3(blocks), dim3(256), 0, 0, s, in[0], in[1], n, term, reset);
      hipLaunchKernelGGL(mithra::k_sg_running, dim3(1), dim3(64), 0, 0, s, n, term, reset, o);
    });
    (void)hipFree(term);
    (void)hipFree(reset);
    return rc;
  }
  return eval_points(n, {{r, 3}, {time, 1}}, 3, a, [&](double** in, double* o, unsigned blocks) {
    hipLaunchKernelGGL(mithra::k_seed_eval, dim3(blocks), dim3(256), 0, 0, s, in[0], in[1], n, o);
  });
}

}  // extern "C"
