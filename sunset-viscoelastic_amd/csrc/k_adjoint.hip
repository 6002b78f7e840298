// k_adjoint.hip -- hand-written reverse mode of the direct-form (DI) RK3 step
// at a fixed time step: the vector-Jacobian product of calc_all_rhs
// (rhs_di.F90:47-476 with the full-gradient reading of calc_rhs_c), of the
// four RK stages and registers (step.F90:281-409), of the hyperviscous filter
// (calc_filtered_var, derivatives.F90:360-414) and of the mass correction
// (rhs_di.F90:667-720), and checkpointed rollouts of a trace loss.
//
// Stencil transposes without atomics: every forward link (i -> j, weights w)
// is stored once more in a transposed SELL-64 layout keyed by j, so the
// adjoint of "D_i = sum_k w_ik G_j - G_i sum_k w_ik" is a gather
//   Gbar_j += sum_{(i,k): j_k = i's link} w_ik Dbar_i
// over the transposed list of j in a fixed order (ascending i): deterministic.
//
// Each RK stage's adjoint has two parts:
//   pointwise    Rbar_i and the stage tape (own gather record G_i and
//                derivative values D_i written by the forward stage) -> the
//                adjoints of the 14 derivative values Dbar_i (+3 Laplacians of
//                c with Mdiff) and the own-node adjoint of G_i
//   transposed   gather of Dbar, G -> U (u = rou/ro), and the RK register
//                recurrences that give the previous stage's Rbar
// The pointwise part of stage k-1 needs only node i's own Rbar, so it runs
// inside the transposed gather of stage k (two buffer sets, ping-pong), and
// the pointwise part of stage 4 inside the fused mass-correction + filter
// adjoint: one step's adjoint is six launches (a per-segment sum, the filter,
// four transposed gathers; five of a small node set, whose filter makes the sum).
// Rollouts keep the state every `checkpoint` steps; the adjoint recomputes one
// checkpoint interval with the tape on and walks it backwards; the last
// interval's tape is written by the rollout itself where it is wanted (want_tape).
#include <string.h>

#include <algorithm>
#include <memory>

#include "sv_internal.h"
#include "sweep.h"

namespace {

constexpr int BS = SV_BLOCK;

#ifndef SV_ADJ_BATCH
#define SV_ADJ_BATCH 4     // transposed links per batch of requests
#endif
// The reverse sweeps run blocks of AB threads, BS/AB of them per 256-node
// block of the node layout, so that small node sets (a 128x128 lattice is 64
// such blocks) still occupy every CU.
#ifndef SV_ADJ_THREADS
#define SV_ADJ_THREADS 64
#endif
constexpr int AB = SV_ADJ_THREADS;
constexpr int SUBS = BS / AB;
static_assert(BS % AB == 0 && AB % 64 == 0, "adjoint blocks are whole waves dividing SV_BLOCK");

__device__ __forceinline__ void ld6(const double *p, double f[6]) {
  const double2 *q = reinterpret_cast<const double2 *>(p);
  const double2 a = q[0], b = q[1], c = q[2];
  f[0] = a.x; f[1] = a.y; f[2] = b.x; f[3] = b.y; f[4] = c.x; f[5] = c.y;
}

__device__ __forceinline__ void st6(double *p, const double f[6]) {
  double2 *q = reinterpret_cast<double2 *>(p);
  q[0] = double2{f[0], f[1]};
  q[1] = double2{f[2], f[3]};
  q[2] = double2{f[4], f[5]};
}

struct NodeRef {
  int sg, i, ii;
  bool act;
};

// node of this thread in sub-block sb (AB threads) of the node layout
__device__ __forceinline__ NodeRef node_ref_sub(const int *blk_seg, const sv_segk *seg, int sb) {
  NodeRef r;
  const int bid = sb / SUBS;
  r.sg = blk_seg[bid];
  const sv_segk &S = seg[r.sg];
  const int li = (bid - S.blk0) * BS + (sb % SUBS) * AB + (int)threadIdx.x;
  r.act = li < S.npfb;
  r.i = S.base + li;
  r.ii = r.act ? r.i : S.base;
  return r;
}

// node of this thread when LPN lanes share a node (LPN = 1 or 4): a block of
// AB threads covers AB / LPN consecutive nodes, BS * LPN / AB blocks per
// 256-node block of the node layout
template <int LPN>
__device__ __forceinline__ NodeRef node_ref_lanes(const int *blk_seg, const sv_segk *seg,
                                                  int sb) {
  if (LPN == 1) return node_ref_sub(blk_seg, seg, sb);
  constexpr int NPB = AB / LPN, SUBL = BS / NPB;
  NodeRef r;
  const int bid = sb / SUBL;
  r.sg = blk_seg[bid];
  const sv_segk &S = seg[r.sg];
  const int li = (bid - S.blk0) * BS + (sb % SUBL) * NPB + (int)threadIdx.x / LPN;
  r.act = li < S.npfb;
  r.i = S.base + li;
  r.ii = r.act ? r.i : S.base;
  return r;
}

// sum of v over the 4 lanes of a quad (DPP quad_perm [1,0,3,2] then
// [2,3,0,1]); every lane of the quad ends with the same value
__device__ __forceinline__ double quad_sum(double v) {
  int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, false);
  int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, false);
  v = v + __hiloint2double(hi, lo);
  lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x4E, 0xF, 0xF, false);
  hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x4E, 0xF, 0xF, false);
  return v + __hiloint2double(hi, lo);
}

__device__ __forceinline__ NodeRef node_ref(const int *blk_seg, const sv_segk *seg, int bid) {
  NodeRef r;
  r.sg = blk_seg[bid];
  const sv_segk &S = seg[r.sg];
  const int li = (bid - S.blk0) * BS + (int)threadIdx.x;
  r.act = li < S.npfb;
  r.i = S.base + li;
  r.ii = r.act ? r.i : S.base;
  return r;
}

// ---- pointwise adjoint of the DI right-hand side ------------------------
// Dbar record [ntot][16]: rx ry | ux uy lu | vx vy lv | cxx_x cxx_y | cxy_x
// cxy_y | cyy_x cyy_y | 0 0; with Mdiff a second record [ntot][4]: the
// Laplacian adjoints of cxx, cxy, cyy.
struct PointArgs {
  const int *blk_seg;
  const sv_segk *seg;
  const double *tG, *tD;     // stage tape
  const double *Rbar;        // [ntot][SV_US]
  const double *gsx, *gsy, *lsum;
  double *dbar, *dbarm, *own;
  double *pacc;              // [ntot][4] parameter-gradient accumulators (or null):
                             // d/d(visc_solvent), d/d(cp), d/d(lambda), d/d(eps)
};

// what the pointwise adjoint reads of a node: its tape, the sums of its weights
// and its parameter accumulators
struct PointOwn {
  double g[6], sx, sy, sl;
  double2 D[7], p0, p1;
};

__device__ __forceinline__ PointOwn load_point(const PointArgs &a, int i) {
  PointOwn o;
  ld6(a.tG + (size_t)i * SV_US, o.g);
  const double2 *d = reinterpret_cast<const double2 *>(a.tD + (size_t)i * SV_TAPE_D);
#pragma unroll
  for (int q = 0; q < 7; q++) o.D[q] = d[q];
  o.sx = a.gsx[i]; o.sy = a.gsy[i]; o.sl = a.lsum[i];
  if (a.pacc) {
    const double2 *p = reinterpret_cast<const double2 *>(a.pacc + (size_t)i * 4);
    o.p0 = p[0];
    o.p1 = p[1];
  }
  return o;
}

// the pointwise adjoint of one (active) node, Rbar given in registers
template <bool MDIFF>
__device__ __forceinline__ void adj_point_node(const PointArgs &a, const NodeRef &nr,
                                               const double rb[6], const PointOwn &own) {
  const int i = nr.i;
  const sv_physk &P = a.seg[nr.sg].pk;
  const double *g = own.g;
  const double ro = g[0], u = g[1], v = g[2], cxx = g[3], cxy = g[4], cyy = g[5];
  const double rx = own.D[0].x, ry = own.D[0].y, ux = own.D[1].x, uy = own.D[1].y;
  const double lu = own.D[2].x, vx = own.D[2].y, vy = own.D[3].x, lv = own.D[3].y;
  const double gxx_x = own.D[4].x, gxx_y = own.D[4].y, gxy_x = own.D[5].x, gxy_y = own.D[5].y;
  const double gyy_x = own.D[6].x, gyy_y = own.D[6].y;
  const double Ab = rb[0], Bu = rb[1], Bv = rb[2], Xb = rb[3], Yb = rb[4], Zb = rb[5];
  // forward intermediates the adjoint needs
  const double r_ro = -ro * (ux + vy) - (u * rx + v * ry);
  const double fr = -(1.0 - P.eps * 2.0 + P.eps * (cxx + cyy + 1.0)) / P.lambda;
  double bro = 0, bu = 0, bv = 0, bcxx = 0, bcxy = 0, bcyy = 0;
  double brx = 0, bry = 0, bux = 0, buy = 0, blu = 0, bvx = 0, bvy = 0, blv = 0;
  double bgxx_x = 0, bgxx_y = 0, bgxy_x = 0, bgxy_y = 0, bgyy_x = 0, bgyy_y = 0;
  // r_rou = -tsu - csq*rx + ro*bfx + fx + cs*lu + cp*(cxx_x + cxy_y)
  const double btsu = -Bu, btsv = -Bv;
  brx += -P.csq * Bu;
  bry += -P.csq * Bv;
  bro += P.bfx * Bu + P.bfy * Bv;
  blu += P.coef_solvent * Bu;
  blv += P.coef_solvent * Bv;
  bgxx_x += P.coef_polymeric * Bu;
  bgxy_y += P.coef_polymeric * Bu;
  bgxy_x += P.coef_polymeric * Bv;
  bgyy_y += P.coef_polymeric * Bv;
  // tsu = ro*(u*ux + v*uy) - u*r_ro ; tsv = ro*(u*vx + v*vy) - v*r_ro
  bro += (u * ux + v * uy) * btsu + (u * vx + v * vy) * btsv;
  bu += ro * ux * btsu - r_ro * btsu + ro * vx * btsv;
  bv += ro * uy * btsu + ro * vy * btsv - r_ro * btsv;
  bux += ro * u * btsu;
  buy += ro * v * btsu;
  bvx += ro * u * btsv;
  bvy += ro * v * btsv;
  const double Ar = Ab - u * btsu - v * btsv;
  // r_ro = -ro*(ux + vy) - (u*rx + v*ry)
  bro += -(ux + vy) * Ar;
  bux += -ro * Ar;
  bvy += -ro * Ar;
  bu += -rx * Ar;
  brx += -u * Ar;
  bv += -ry * Ar;
  bry += -v * Ar;
  // advection of c
  bu += -(gxx_x * Xb + gxy_x * Yb + gyy_x * Zb);
  bv += -(gxx_y * Xb + gxy_y * Yb + gyy_y * Zb);
  bgxx_x += -u * Xb; bgxx_y += -v * Xb;
  bgxy_x += -u * Yb; bgxy_y += -v * Yb;
  bgyy_x += -u * Zb; bgyy_y += -v * Zb;
  // upper-convected terms
  bux += 2.0 * cxx * Xb + cxy * Yb;
  buy += 2.0 * cxy * Xb + cyy * Yb;
  bvx += cxx * Yb + 2.0 * cxy * Zb;
  bvy += cxy * Yb + 2.0 * cyy * Zb;
  bcxx += 2.0 * ux * Xb + vx * Yb;
  bcxy += 2.0 * uy * Xb + (ux + vy) * Yb + 2.0 * vx * Zb;
  bcyy += uy * Yb + 2.0 * vy * Zb;
  // relaxation fr*(c - I), fr = -(1 - 2 eps + eps*(cxx + cyy + 1))/lambda
  bcxx += fr * Xb;
  bcxy += fr * Yb;
  bcyy += fr * Zb;
  const double bfr = (cxx - 1.0) * Xb + cxy * Yb + (cyy - 1.0) * Zb;
  const double dfr = -P.eps / P.lambda * bfr;
  bcxx += dfr;
  bcyy += dfr;
  double blxx = 0, blxy = 0, blyy = 0;
  if (MDIFF) { blxx = P.Mdiff * Xb; blxy = P.Mdiff * Yb; blyy = P.Mdiff * Zb; }
  // D_i = sum_k w G_j - G_i * sum: own-node share
  const double sx = own.sx, sy = own.sy, sl = own.sl;
  double o[6];
  o[0] = bro - (sx * brx + sy * bry);
  o[1] = bu - (sx * bux + sy * buy + sl * blu);
  o[2] = bv - (sx * bvx + sy * bvy + sl * blv);
  o[3] = bcxx - (sx * bgxx_x + sy * bgxx_y + sl * blxx);
  o[4] = bcxy - (sx * bgxy_x + sy * bgxy_y + sl * blxy);
  o[5] = bcyy - (sx * bgyy_x + sy * bgyy_y + sl * blyy);
  st6(a.own + (size_t)i * SV_US, o);
  double2 *T = reinterpret_cast<double2 *>(a.dbar + (size_t)i * SV_TAPE_D);
  T[0] = double2{brx, bry}; T[1] = double2{bux, buy}; T[2] = double2{blu, bvx};
  T[3] = double2{bvy, blv}; T[4] = double2{bgxx_x, bgxx_y}; T[5] = double2{bgxy_x, bgxy_y};
  T[6] = double2{bgyy_x, bgyy_y}; T[7] = double2{0.0, 0.0};
  if (MDIFF) {
    double2 *M = reinterpret_cast<double2 *>(a.dbarm + (size_t)i * 4);
    M[0] = double2{blxx, blxy};
    M[1] = double2{blyy, 0.0};
  }
  if (a.pacc) {
    // r_rou, r_rov hold visc_solvent*(lu, lv) and cp*(div c); the conformation
    // source fr*(c - I) holds lambda and eps through fr
    double2 *Pq = reinterpret_cast<double2 *>(a.pacc + (size_t)i * 4);
    double2 p0 = own.p0, p1 = own.p1;
    p0.x += Bu * lu + Bv * lv;
    p0.y += Bu * (gxx_x + gxy_y) + Bv * (gxy_x + gyy_y);
    p1.x += bfr * (-fr / P.lambda);
    p1.y += bfr * (-(cxx + cyy - 1.0) / P.lambda);
    Pq[0] = p0;
    Pq[1] = p1;
  }
}

template <bool MDIFF>
__global__ __launch_bounds__(AB) void k_adj_point(PointArgs a) {
  const NodeRef nr = node_ref_sub(a.blk_seg, a.seg, sv_xcd_block());
  if (!nr.act) return;
  double rb[6];
  ld6(a.Rbar + (size_t)nr.i * SV_US, rb);
  adj_point_node<MDIFF>(a, nr, rb, load_point(a, nr.i));
}

// ---- transposed gather + G->U + RK register recurrences ------------------
struct TransArgs {
  const int *blk_seg;
  const sv_segk *seg;
  const int64_t *toff;       // transposed SELL
  const int *tcnt, *tcol;
  const double *tw3;
  const double *dbar, *dbarm, *own;
  const double *tG;          // stage tape (ro, u, v of node j)
  const sv_ctrl *ctrl;       // RK coefficients (dt included)
  double *Ubar;              // STAGE 1 / 0: output
  double *Rbar;              // STAGE 2..4: next (earlier) stage's Rbar
  double *regbar;            // STAGE 2..4: in/out
  double seed;               // STAGE 1: loss seed added to cxx and cyy
  double *psum;              // STAGE 1: per-sub-block sum of Ubar_ro (mass correction)
  PointArgs nxt;             // STAGE 2..4: the pointwise adjoint of stage STAGE-1,
                             // fused (its Rbar stays in registers)
  const int4 *krange;        // halos of the transposed lists (k_adj_trans_h)
  const int64_t *hoff;
  const int *hidx;
  const uint16_t *lcol;
};

// a node's own values in a transposed gather
struct TransOwn {
  double o[6], g[6], rg[6];
  PointOwn p;
};

template <int STAGE>
__device__ __forceinline__ TransOwn load_own(const TransArgs &a, int j) {
  TransOwn w;
  ld6(a.own + (size_t)j * SV_US, w.o);
  ld6(a.tG + (size_t)j * SV_US, w.g);
  if (STAGE >= 1) ld6(a.regbar + (size_t)j * SV_US, w.rg);
  if (STAGE >= 2) w.p = load_point(a.nxt, j);
  return w;
}

// Own-node part of a transposed gather: G -> U and the RK register recurrences.
// Returns Ubar_ro (STAGE 1).
template <int STAGE, bool MDIFF>
__device__ __forceinline__ double trans_point(const TransArgs &a, const NodeRef &nr,
                                              const double acc[6], const TransOwn &w) {
  const int j = nr.i;
  double G[6];
#pragma unroll
  for (int f = 0; f < 6; f++) G[f] = w.o[f] + acc[f];
  // G = (ro, rou/ro, rov/ro, c) -> U
  const double ooro = 1.0 / w.g[0];
  double Ub[6];
  Ub[0] = G[0] - (G[1] * w.g[1] + G[2] * w.g[2]) * ooro;
  Ub[1] = G[1] * ooro;
  Ub[2] = G[2] * ooro;
  Ub[3] = G[3]; Ub[4] = G[4]; Ub[5] = G[5];
  if constexpr (STAGE == 0) {
    st6(a.Ubar + (size_t)j * SV_US, Ub);
  } else if constexpr (STAGE == 1) {
#pragma unroll
    for (int f = 0; f < 6; f++) Ub[f] += w.rg[f];
    Ub[3] += a.seed;
    Ub[5] += a.seed;
    st6(a.Ubar + (size_t)j * SV_US, Ub);
    return Ub[0];
  } else {
    // U_k = reg_{k-2} + a_{k-1} R_{k-1};  reg_{k-1} = reg_{k-2} + b_{k-1} R_{k-1}
    const sv_ctrl *C = a.ctrl + nr.sg;
    const double ra = C->RKa[STAGE - 2], rbk = C->RKb[STAGE - 2];
    double rg[6], Rn[6];
#pragma unroll
    for (int f = 0; f < 6; f++) {
      Rn[f] = ra * Ub[f] + rbk * w.rg[f];
      rg[f] = Ub[f] + w.rg[f];
    }
    st6(a.regbar + (size_t)j * SV_US, rg);
    adj_point_node<MDIFF>(a.nxt, nr, Rn, w.p);
  }
  return 0.0;
}

// stencil-adjoint record of a node: d0..d6, and with Mdiff m0, m1.  (Named
// members: arrays of them end up in scratch memory.)
struct DRec {
  double2 d0, d1, d2, d3, d4, d5, d6, m0, m1;
};
template <bool MDIFF>
__device__ __forceinline__ DRec load_rec(const double *d, const double *m) {
  const double2 *q = reinterpret_cast<const double2 *>(d);
  const double2 *p = reinterpret_cast<const double2 *>(m);
  DRec r;
  r.d0 = q[0]; r.d1 = q[1]; r.d2 = q[2]; r.d3 = q[3]; r.d4 = q[4]; r.d5 = q[5]; r.d6 = q[6];
  if (MDIFF) { r.m0 = p[0]; r.m1 = p[1]; }
  return r;
}

// one transposed link: the record of node i weighted by the link's gradient and
// Laplacian weights
template <bool MDIFF>
__device__ __forceinline__ void trans_link(double acc[6], double wx, double wy, double wl,
                                           const DRec &r) {
  acc[0] += wx * r.d0.x + wy * r.d0.y;
  acc[1] += wx * r.d1.x + wy * r.d1.y + wl * r.d2.x;
  acc[2] += wx * r.d2.y + wy * r.d3.x + wl * r.d3.y;
  acc[3] += wx * r.d4.x + wy * r.d4.y;
  acc[4] += wx * r.d5.x + wy * r.d5.y;
  acc[5] += wx * r.d6.x + wy * r.d6.y;
  if (MDIFF) {
    acc[3] += wl * r.m0.x;
    acc[4] += wl * r.m0.y;
    acc[5] += wl * r.m1.x;
  }
}

// STAGE 0: plain vector-Jacobian product of calc_all_rhs (Ubar = J^T Rbar).
// LPN lanes per node: lane r of a node sums its links r, r + LPN, ... and the
// quad's partial sums are added in a fixed order (small node sets, where one
// lane per node leaves most of the chip idle and each lane walks ~70 links).
template <int STAGE, bool MDIFF, int LPN>
__global__ __launch_bounds__(AB) void k_adj_trans(TransArgs a) {
  __shared__ double red[AB];
  const int bid = sv_xcd_block();
  const NodeRef nr = node_ref_lanes<LPN>(a.blk_seg, a.seg, bid);
  const int j = nr.i, jj = nr.ii;
  const int lr = (int)threadIdx.x % LPN;
  const int64_t b = a.toff[jj >> 6] + (jj & 63);
  const int K = nr.act ? a.tcnt[jj] : 0;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  // links in batches of SV_ADJ_BATCH: every index and weight of a batch, then
  // every gathered record, are requested before the first sum, so the
  // dependent index -> record loads cost one memory round trip per batch
  // rather than per link (the sums keep the link order)
  int k = lr;
  for (; k + (SV_ADJ_BATCH - 1) * LPN < K; k += SV_ADJ_BATCH * LPN) {
    int ix[SV_ADJ_BATCH];
    double wx[SV_ADJ_BATCH], wy[SV_ADJ_BATCH], wl[SV_ADJ_BATCH];
#pragma unroll
    for (int u = 0; u < SV_ADJ_BATCH; u++) {
      const int64_t e = b + (int64_t)(k + u * LPN) * SV_WAVE;
      ix[u] = a.tcol[e];
      wx[u] = a.tw3[sv_w3(e, 0)];
      wy[u] = a.tw3[sv_w3(e, 1)];
      wl[u] = a.tw3[sv_w3(e, 2)];
    }
    DRec d[SV_ADJ_BATCH];
#pragma unroll
    for (int u = 0; u < SV_ADJ_BATCH; u++)
      d[u] = load_rec<MDIFF>(a.dbar + (size_t)ix[u] * SV_TAPE_D, a.dbarm + (size_t)ix[u] * 4);
#pragma unroll
    for (int u = 0; u < SV_ADJ_BATCH; u++) trans_link<MDIFF>(acc, wx[u], wy[u], wl[u], d[u]);
  }
  for (; k < K; k += LPN) {
    const int64_t e = b + (int64_t)k * SV_WAVE;
    const int i = a.tcol[e];
    trans_link<MDIFF>(acc, a.tw3[sv_w3(e, 0)], a.tw3[sv_w3(e, 1)], a.tw3[sv_w3(e, 2)],
                      load_rec<MDIFF>(a.dbar + (size_t)i * SV_TAPE_D, a.dbarm + (size_t)i * 4));
  }
  if (LPN == 4) {
#pragma unroll
    for (int f = 0; f < 6; f++) acc[f] = quad_sum(acc[f]);
  }
  double part = 0.0;
  if (nr.act && lr == 0) part = trans_point<STAGE, MDIFF>(a, nr, acc, load_own<STAGE>(a, j));
  if (STAGE == 1) {
    red[threadIdx.x] = part;
    __syncthreads();
    for (int s = AB / 2; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) a.psum[bid] = red[0];
  }
}

// ---- halo-staged forms ----------------------------------------------------
// A workgroup per 64 slots stages the records of its transposed halo (~4 per
// node on a lattice) in LDS, as the forward sweeps do, and four wavefronts walk
// a quarter of each list, their partial sums added in order.  The gathers
// from memory they replace (14 doubles a link in 16-byte pieces of 64 records)
// are bound by the CU's address rate.  A stage of 16k nodes, order 6: 30 -> 12 us;
// filter and sum: 16.2 -> 10.1.  Records of 14 doubles (18 with polymer diffusion) and 6: odd
// multiples of 16 bytes, which spread over the LDS banks.
constexpr int AW = 4;
template <bool MDIFF>
constexpr int trans_rec() { return MDIFF ? 18 : 14; }

// the six sums of the other wavefronts, added to wave 0's in their order
__device__ __forceinline__ void add_sums(double *lds, int w, double acc[6]) {
  const int lane = (int)threadIdx.x & (SV_WAVE - 1);
  __syncthreads();   // the halo has been read
  if (w > 0)
#pragma unroll
    for (int q = 0; q < 6; q++) lds[((w - 1) * 6 + q) * SV_WAVE + lane] = acc[q];
  __syncthreads();
  if (w > 0) return;
#pragma unroll
  for (int v = 0; v < AW - 1; v++)
#pragma unroll
    for (int q = 0; q < 6; q++) acc[q] += lds[(v * 6 + q) * SV_WAVE + lane];
}
constexpr size_t SUMS_LDS = sizeof(double) * (AW - 1) * 6 * SV_WAVE;

__device__ __forceinline__ NodeRef node_ref_slice(const int *blk_seg, const sv_segk *seg, int s) {
  NodeRef r;
  r.sg = blk_seg[s / (BS / SV_WAVE)];
  const sv_segk &S = seg[r.sg];
  r.i = s * SV_WAVE + ((int)threadIdx.x & (SV_WAVE - 1));
  r.act = r.i - S.base < S.npfb;
  r.ii = r.act ? r.i : S.base;
  return r;
}

template <int STAGE, bool MDIFF>
__global__ __launch_bounds__(AW * SV_WAVE) void k_adj_trans_h(TransArgs a) {
  extern __shared__ double hl[];
  constexpr int RS = trans_rec<MDIFF>(), U = 3, NT = AW * SV_WAVE;
  const int s = sv_xcd_block();
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / SV_WAVE);
  const NodeRef nr = node_ref_slice(a.blk_seg, a.seg, s);
  const Share<AW> sh(w, a.tcnt[nr.i], a.krange[s].x, a.krange[s].y);
  const int64_t o = a.toff[s] + (int64_t)sh.k0 * SV_WAVE;
  const int64_t h0 = a.hoff[s];
  const int nh = (int)(a.hoff[s + 1] - h0);
  const Stream<uint32_t, 1, false> sc(a.lcol + o, sh.KM);
  const Stream<dbl2, 3, false> sw(a.tw3 + 3 * o, sh.KM);
  uint32_t jc[2][U];
  dbl2 wg[2][2 * U], wl[2][U];
  auto load = [&](int b, int u, int p) {
    jc[b][u] = sc.at(p, u, 0);
    wg[b][2 * u] = sw.at(p, u, 0); wg[b][2 * u + 1] = sw.at(p, u, 1); wl[b][u] = sw.at(p, u, 2);
  };
  const int *hx = a.hidx + h0;
  HaloKeys<SV_WAVE, NT> keys;
  if (nh > 0) keys.get(hx, threadIdx.x, nh);
  __builtin_amdgcn_sched_barrier(0);
  const int p0 = entry_at(0);
#pragma unroll
  for (int u = 0; u < U; u++) load(0, u, 2 * u < sh.K ? p0 : OUT_OF_RANGE);
  TransOwn own;
  if (w == 0) own = load_own<STAGE>(a, nr.ii);
  halo_stage<SV_WAVE, NT>(
      hx, nh, keys,
      [&](int j) {
        return load_rec<MDIFF>(a.dbar + (size_t)j * SV_TAPE_D, a.dbarm + (size_t)j * 4);
      },
      [&](int h, int, const DRec &r) {
        double2 *q = reinterpret_cast<double2 *>(hl + (size_t)h * RS);
        q[0] = r.d0; q[1] = r.d1; q[2] = r.d2; q[3] = r.d3; q[4] = r.d4; q[5] = r.d5; q[6] = r.d6;
        if (MDIFF) { q[7] = r.m0; q[8] = r.m1; }
      });
  __syncthreads();
  double acc[6] = {0, 0, 0, 0, 0, 0};
  walk_links<U, DRec>(
      sh.K, sh.KF, sh.KM, load,
      [&](int b, int l) {
        const double *q = hl + (size_t)RS * (l & 1 ? jc[b][l / 2] >> 16 : jc[b][l / 2] & 0xffff);
        return load_rec<MDIFF>(q, q + 14);
      },
      [&](const DRec &r, int b, int l) {
        trans_link<MDIFF>(acc, wg[b][l].x, wg[b][l].y, l & 1 ? wl[b][l / 2].y : wl[b][l / 2].x, r);
      });
  add_sums(hl, w, acc);
  if (w > 0) return;
  double part = 0.0;
  if (nr.act) part = trans_point<STAGE, MDIFF>(a, nr, acc, own);
  if (STAGE == 1) {
    part = wave_sum(part);
    if (threadIdx.x == 0) a.psum[s] = part;
  }
}

// per-block sums of Ubar_ro (the start of a backward sweep), in the block
// layout of the LPN sweeps that write psum afterwards
template <int LPN>
__global__ __launch_bounds__(AB) void k_adj_sum(const int *blk_seg, const sv_segk *seg,
                                                const double *Ubar, double *psum) {
  __shared__ double red[AB];
  const int bid = sv_xcd_block();
  const NodeRef nr = node_ref_lanes<LPN>(blk_seg, seg, bid);
  red[threadIdx.x] = (nr.act && (int)threadIdx.x % LPN == 0) ? Ubar[(size_t)nr.i * SV_US] : 0.0;
  __syncthreads();
  for (int s = AB / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) psum[bid] = red[0];
}

// mass-correction adjoint: sbar[seg] = sum_j Ubar_ro,j / sum_j vol_j (one block
// per segment, over the segment's sub-block sums), then Ubar_ro,i -= vol_i * sbar
__global__ __launch_bounds__(1024) void k_adj_sum_reduce(const sv_segk *seg, const double *psum,
                                                         int subl, double *sbar) {
  __shared__ double s1[1024];
  const sv_segk &S = seg[blockIdx.x];
  double a = 0.0;
  for (int k = threadIdx.x; k < S.nblk * subl; k += 1024) a += psum[S.blk0 * subl + k];
  s1[threadIdx.x] = a;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) s1[threadIdx.x] += s1[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) sbar[blockIdx.x] = s1[0] / S.volsum;
}

// mass-correction + filter adjoint, fused with the pointwise adjoint of
// stage 4: Uf_i = Ubar_i - [ro] vol_i sbar (evaluated for every gathered i),
// Ustar_j = Uf_j - hsum_j Uf_j + sum_t wh_t Uf_{i_t}; regbar_3 = Ustar,
// Rbar_4 = b_4 Ustar (registers) -> stage-4 pointwise adjoint
struct FiltArgs {
  const int *blk_seg;
  const sv_segk *seg;
  const int64_t *toff;
  const int *tcnt, *tcol;
  const double *twh, *hsum, *vol, *sbar;
  const double *Ubar;
  const sv_ctrl *ctrl;
  double *regbar;
  PointArgs p4;
  const int4 *krange;        // halos of the transposed lists (k_adj_filter_h)
  const int64_t *hoff;
  const int *hidx;
  const uint16_t *lcol;
  const double *psum;        // k_adj_filter_h: the npsum sums whose total it makes
  int npsum;                 // itself instead of reading sbar (0: reads it)
};

// a node's own values in the filter's adjoint
struct FiltOwn {
  double f[6], vol, hs;
  PointOwn p;
};

__device__ __forceinline__ FiltOwn load_own(const FiltArgs &a, int j) {
  FiltOwn w;
  ld6(a.Ubar + (size_t)j * SV_US, w.f);
  w.vol = a.vol[j];
  w.hs = a.hsum[j];
  w.p = load_point(a.p4, j);
  return w;
}

// own-node part: the filter's adjoint, then the pointwise adjoint of stage 4
template <bool MDIFF>
__device__ __forceinline__ void filt_point(const FiltArgs &a, const NodeRef &nr, double sv,
                                           const double acc[6], FiltOwn &w) {
  double out[6], rb[6];
  w.f[0] -= w.vol * sv;
  const double b4 = a.ctrl[nr.sg].RKb[3];
#pragma unroll
  for (int q = 0; q < 6; q++) {
    out[q] = w.f[q] - w.hs * w.f[q] + acc[q];
    rb[q] = b4 * out[q];
  }
  st6(a.regbar + (size_t)nr.i * SV_US, out);
  adj_point_node<MDIFF>(a.p4, nr, rb, w.p);
}

template <bool MDIFF, int LPN>
__global__ __launch_bounds__(AB) void k_adj_filter(FiltArgs a) {
  const NodeRef nr = node_ref_lanes<LPN>(a.blk_seg, a.seg, sv_xcd_block());
  const int j = nr.i, jj = nr.ii;
  const int lr = (int)threadIdx.x % LPN;
  const int64_t b = a.toff[jj >> 6] + (jj & 63);
  const int K = nr.act ? a.tcnt[jj] : 0;
  const double sv = a.sbar[nr.sg];
  double acc[6] = {0, 0, 0, 0, 0, 0};
  int k = lr;
  // batched as in k_adj_trans, lane lr of a node taking links lr, lr + LPN, ...
  for (; k + (SV_ADJ_BATCH - 1) * LPN < K; k += SV_ADJ_BATCH * LPN) {
    int ix[SV_ADJ_BATCH];
    double w[SV_ADJ_BATCH], f[SV_ADJ_BATCH][6], vo[SV_ADJ_BATCH];
#pragma unroll
    for (int u = 0; u < SV_ADJ_BATCH; u++) {
      const int64_t e = b + (int64_t)(k + u * LPN) * SV_WAVE;
      ix[u] = a.tcol[e];
      w[u] = a.twh[sv_pair(e)];
    }
#pragma unroll
    for (int u = 0; u < SV_ADJ_BATCH; u++) {
      ld6(a.Ubar + (size_t)ix[u] * SV_US, f[u]);
      vo[u] = a.vol[ix[u]];
    }
#pragma unroll
    for (int u = 0; u < SV_ADJ_BATCH; u++) {
      f[u][0] -= vo[u] * sv;
#pragma unroll
      for (int q = 0; q < 6; q++) acc[q] += w[u] * f[u][q];
    }
  }
  for (; k < K; k += LPN) {
    const int64_t e = b + (int64_t)k * SV_WAVE;
    const int i = a.tcol[e];
    const double w = a.twh[sv_pair(e)];
    double f[6];
    ld6(a.Ubar + (size_t)i * SV_US, f);
    f[0] -= a.vol[i] * sv;
#pragma unroll
    for (int q = 0; q < 6; q++) acc[q] += w * f[q];
  }
  if (LPN == 4) {
#pragma unroll
    for (int q = 0; q < 6; q++) acc[q] = quad_sum(acc[q]);
  }
  if (!nr.act || lr != 0) return;
  FiltOwn own = load_own(a, j);
  filt_point<MDIFF>(a, nr, sv, acc, own);
}

// the filter's adjoint with halos (see k_adj_trans_h).  Of a small node set every
// wavefront makes the mass correction's sum itself: a launch less.
constexpr int SMALL_SUMS = 512;
template <bool MDIFF>
__global__ __launch_bounds__(AW * SV_WAVE) void k_adj_filter_h(FiltArgs a) {
  extern __shared__ double hl[];
  constexpr int U = 4, NT = AW * SV_WAVE;
  const int s = sv_xcd_block();
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / SV_WAVE);
  const NodeRef nr = node_ref_slice(a.blk_seg, a.seg, s);
  const Share<AW> sh(w, a.tcnt[nr.i], a.krange[s].z, a.krange[s].w);
  const int64_t o = a.toff[s] + (int64_t)sh.k0 * SV_WAVE;
  const int64_t h0 = a.hoff[s];
  const int nh = (int)(a.hoff[s + 1] - h0);
  const Stream<uint32_t, 1, false> sc(a.lcol + o, sh.KM);
  const Stream<dbl2, 1, false> sw(a.twh + o, sh.KM);
  uint32_t jc[2][U];
  dbl2 wf[2][U];
  auto load = [&](int b, int u, int p) {
    jc[b][u] = sc.at(p, u, 0);
    wf[b][u] = sw.at(p, u, 0);
  };
  const int *hx = a.hidx + h0;
  HaloKeys<SV_WAVE, NT> keys;
  if (nh > 0) keys.get(hx, threadIdx.x, nh);
  double sv;
  if (a.npsum > 0) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < SMALL_SUMS / SV_WAVE; k++) {
      const int q = k * SV_WAVE + ((int)threadIdx.x & (SV_WAVE - 1));
      v += q < a.npsum ? a.psum[q] : 0.0;
    }
    sv = wave_sum(v) / a.seg[nr.sg].volsum;
  } else {
    sv = a.sbar[nr.sg];
  }
  __builtin_amdgcn_sched_barrier(0);
  const int p0 = entry_at(0);
#pragma unroll
  for (int u = 0; u < U; u++) load(0, u, 2 * u < sh.K ? p0 : OUT_OF_RANGE);
  FiltOwn own;
  if (w == 0) own = load_own(a, nr.ii);
  struct Rec {
    double2 d[3];
    double vol;
  };
  halo_stage<SV_WAVE, NT>(
      hx, nh, keys,
      [&](int j) {
        const double2 *q = reinterpret_cast<const double2 *>(a.Ubar + (size_t)j * SV_US);
        return Rec{{q[0], q[1], q[2]}, a.vol[j]};
      },
      [&](int h, int, const Rec &r) {
        double2 *q = reinterpret_cast<double2 *>(hl + (size_t)h * SV_US);
        q[0] = double2{r.d[0].x - r.vol * sv, r.d[0].y};
        q[1] = r.d[1];
        q[2] = r.d[2];
      });
  __syncthreads();
  double acc[6] = {0, 0, 0, 0, 0, 0};
  struct Rec6 {
    double2 d[3];
  };
  walk_links<U, Rec6>(
      sh.K, sh.KF, sh.KM, load,
      [&](int b, int l) {
        const double2 *q = reinterpret_cast<const double2 *>(
            hl + (size_t)SV_US * (l & 1 ? jc[b][l / 2] >> 16 : jc[b][l / 2] & 0xffff));
        return Rec6{{q[0], q[1], q[2]}};
      },
      [&](const Rec6 &r, int b, int l) {
        const double wt = l & 1 ? wf[b][l / 2].y : wf[b][l / 2].x;
#pragma unroll
        for (int q = 0; q < 3; q++) {
          acc[2 * q] += wt * r.d[q].x;
          acc[2 * q + 1] += wt * r.d[q].y;
        }
      });
  add_sums(hl, w, acc);
  if (w == 0 && nr.act) filt_point<MDIFF>(a, nr, sv, acc, own);
}

// trace loss of the state: per-block sums of (cxx + cyy - 2) after each step,
// then one block per step and one thread that adds the steps' means to lacc in
// their order
__global__ __launch_bounds__(BS) void k_loss_part(const int *blk_seg, const sv_segk *seg,
                                                  const double *U, double *part) {
  __shared__ double red[BS];
  const int bid = sv_xcd_block();
  const NodeRef nr = node_ref(blk_seg, seg, bid);
  double v = 0.0;
  if (nr.act) {
    const double *r = U + (size_t)nr.i * SV_US;
    v = r[3] + r[5] - 2.0;
  }
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = BS / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[bid] = red[0];
}

__global__ __launch_bounds__(1024) void k_loss_steps(const sv_segk *seg, const double *part,
                                                     double *mean) {
  __shared__ double s1[1024];
  const sv_segk &S = seg[0];
  const double *p = part + (size_t)blockIdx.x * S.nblk;
  double a = 0.0;
  for (int k = threadIdx.x; k < S.nblk; k += 1024) a += p[k];
  s1[threadIdx.x] = a;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) s1[threadIdx.x] += s1[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) mean[blockIdx.x] = s1[0] / S.npfb;
}

__global__ void k_loss_add(int steps, const double *mean, double *lacc) {
  double a = *lacc;
  for (int s = 0; s < steps; s++) a += mean[s];
  *lacc = a;
}

// sums of the parameter-gradient accumulators over the real nodes (one block,
// fixed order: deterministic)
__global__ __launch_bounds__(1024) void k_param_reduce(const double *pacc, int n, double *out) {
  __shared__ double s1[4][1024];
  double a[4] = {0, 0, 0, 0};
  for (int k = threadIdx.x; k < n; k += 1024)
    for (int q = 0; q < 4; q++) a[q] += pacc[(size_t)k * 4 + q];
  for (int q = 0; q < 4; q++) s1[q][threadIdx.x] = a[q];
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
      for (int q = 0; q < 4; q++) s1[q][threadIdx.x] += s1[q][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x < 4) out[threadIdx.x] = s1[threadIdx.x][0];
}

__global__ void k_zero(double *p, int64_t n) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = 0.0;
}

}  // namespace

// ---- host side ------------------------------------------------------------
constexpr int LOSS_STEPS = 32;

struct sv_adj {
  int every = 20;            // checkpoint interval (steps)
  sv_loopl TL;               // transposed stencil (SELL-64 over j)
  bool halo = false;         // its halos fit: the halo-staged sweeps
  // adjoint records [ntot][SV_US] and stencil-adjoint records
  double *Ubar = nullptr, *Rbar = nullptr, *regbar = nullptr;
  // stencil-adjoint records of two consecutive stages (ping-pong: a fused
  // kernel reads stage k's while writing stage k-1's)
  double *own[2] = {nullptr, nullptr}, *dbar[2] = {nullptr, nullptr};
  double *dbarm[2] = {nullptr, nullptr};
  double *psum = nullptr, *sbar = nullptr;
  double *lpart = nullptr, *lmean = nullptr, *lacc = nullptr;   // loss sums of lsteps steps
  int lsteps = 0;
  double *pacc = nullptr, *pred = nullptr;   // parameter-gradient accumulators, sums
  double pgrad[3] = {0, 0, 0};               // d/d(Wi, beta, epsPTT) of the last VJP
  // rollout: checkpoints of U records, the end state, the tape of one interval
  int T = 0;                 // steps of the last forward rollout
  std::vector<double *> ckpt;
  std::vector<sv_ctrl> ckpt_ctrl;
  double *Uend = nullptr;
  sv_ctrl ctrl_end{};
  std::vector<double *> tape;    // [every][8]
  // the tape holds the last interval of the last rollout; tape_used: a reverse
  // sweep has followed the last rollout that wrote one
  bool taped = false, tape_used = true;
  double t_fwd = 0, t_bwd = 0;   // ms of the last rollout / vjp
  int recomputed = 0;            // steps that the last vjp computed again
  int lpn = 1;                   // lanes per node of the transposed gathers (1 or 4)
};

// sub-blocks per 256-node block of the reverse sweeps with lpn lanes per node
static int subl_of(int lpn) { return SUBS * lpn; }

void sv_adj_free(sv_ctx *c) {
  delete c->adj;
  c->adj = nullptr;
}

static int adj_alloc(sv_ctx *c, double **p, size_t n) {
  return sv_alloc(c, (void **)p, sizeof(double) * (n ? n : 1));
}

static int zero_dev(sv_ctx *c, double *p, int64_t n) {
  if (n <= 0) return 0;
  k_zero<<<(unsigned)((n + 255) / 256), 256, 0, c->stream>>>(p, n);
  SV_HIP(c, hipGetLastError());
  return 0;
}

// tape of `steps` steps; what is missing in one allocation
static int ensure_tape(sv_ctx *c, sv_adj *A, int steps) {
  const size_t N = (size_t)c->ntot;
  const int more = steps - (int)A->tape.size() / 8;
  if (more <= 0) return 0;
  double *p = nullptr;
  if (adj_alloc(c, &p, (size_t)more * 4 * (SV_US + SV_TAPE_D) * N)) return SV_E_NOMEM;
  for (int k = 0; k < 8 * more; k++) {
    A->tape.push_back(p);
    p += ((k & 1) ? SV_TAPE_D : SV_US) * N;
  }
  return 0;
}

// Whether a rollout writes the tape of its last interval (of `steps` steps), so
// that the reverse sweep need not compute the interval again (75 us a step of
// 16k nodes; writing costs 176 bytes a node and stage beside the ~2 kB read).
// Asked for ("rollout_tape" 1): where the tape takes at most a quarter of the
// free memory.  Left to the library (-1): into the memory of an earlier reverse
// sweep only, since whether this rollout will have one is not known (20 steps of
// 1M nodes take 14 GB), and not after a rollout whose tape nothing read.
static bool want_tape(sv_ctx *c, sv_adj *A, int steps) {
  const int more = std::max(0, steps - (int)A->tape.size() / 8);
  if (c->rollout_tape <= 0) return c->rollout_tape < 0 && A->tape_used && more == 0;
  if (more > 0) {
    size_t free_b = 0, total = 0;
    if (hipMemGetInfo(&free_b, &total) != hipSuccess) return false;
    const size_t per = sizeof(double) * 4 * (SV_US + SV_TAPE_D) * (size_t)c->ntot;
    if (per * more > free_b / 4) return false;
  }
  return ensure_tape(c, A, steps) == 0;
}

bool sv_adj_stat(sv_ctx *c, const char *what, double *v) {
  const sv_adj *A = c->adj;
  if (!strcmp(what, "tape_steps")) *v = A ? (double)(A->tape.size() / 8) : 0.0;
  else if (!strcmp(what, "tape_written")) *v = A && A->taped;
  else if (!strcmp(what, "vjp_recomputed")) *v = A ? A->recomputed : 0;
  else return false;
  return true;
}

void sv_adj_drop_tape(sv_ctx *c) {
  if (c->adj) c->adj->taped = false;
}

// pointwise-adjoint arguments for stage k (1..4) of a tape slot, buffer set q
static PointArgs point_args(sv_ctx *c, sv_adj *A, double *const *tape, int k, int q) {
  return PointArgs{c->blk_seg, c->segk, tape[2 * (k - 1)], tape[2 * (k - 1) + 1], A->Rbar,
                   c->L.gsx, c->L.gsy, c->L.lsum, A->dbar[q], A->dbarm[q], A->own[q],
                   A->pacc};
}

// Sum the accumulators and map d/d(visc_solvent, cp, lambda, eps) to the
// parameters through the derived constants (load_data.F90:132-148):
// visc_solvent = beta*vt, lambda = Wi*L/U, cp = (1 - beta)*vt/lambda.
static int param_grad_finish(sv_ctx *c, sv_adj *A) {
  k_param_reduce<<<1, 1024, 0, c->stream>>>(A->pacc, c->npfb, A->pred);
  SV_HIP(c, hipGetLastError());
  double g[4];
  SV_HIP(c, hipMemcpyAsync(g, A->pred, sizeof(g), hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  const sv_physk &P = c->pk;
  const double vt = P.visc_total, lam = P.lambda, cp = P.coef_polymeric;
  const double dlam_dWi = P.L_char / P.U_char;
  A->pgrad[0] = g[2] * dlam_dWi - g[1] * cp / lam * dlam_dWi;
  A->pgrad[1] = g[0] * vt - g[1] * vt / lam;
  A->pgrad[2] = g[3];
  return 0;
}

// LDS of the transposed gathers' largest halo
static size_t trans_lds(sv_ctx *c, sv_adj *A) {
  return sizeof(double) * (c->any_mdiff ? trans_rec<true>() : trans_rec<false>()) *
         (size_t)A->TL.hmax;
}

// transposed gather of stage STAGE (its records in buffer set q); for STAGE
// 2..4 fused with the pointwise adjoint of STAGE-1 into buffer set 1-q
template <int STAGE>
static int adj_trans(sv_ctx *c, sv_adj *A, double *const *tape, int q, double seed) {
  const int k = STAGE == 0 ? 1 : STAGE;
  const sv_loopl &L = A->TL;
  TransArgs t{c->blk_seg, c->segk, L.off, L.cnt, L.col, L.w3,
              A->dbar[q], A->dbarm[q], A->own[q], tape[2 * (k - 1)], c->ctrl, A->Ubar, A->Rbar,
              A->regbar, seed, A->psum, PointArgs{}, L.krange, L.hoff, L.hidx, L.lcol};
  if (STAGE >= 2) t.nxt = point_args(c, A, tape, STAGE - 1, 1 - q);
  if (A->halo) {
    const int grid = c->nblk * (BS / SV_WAVE), nt = AW * SV_WAVE;
    const size_t shm = std::max(SUMS_LDS, trans_lds(c, A));
    if (c->any_mdiff) k_adj_trans_h<STAGE, true><<<grid, nt, shm, c->stream>>>(t);
    else k_adj_trans_h<STAGE, false><<<grid, nt, shm, c->stream>>>(t);
    SV_HIP(c, hipGetLastError());
    return 0;
  }
  const int grid = c->nblk * subl_of(A->lpn);
  if (A->lpn == 4) {
    if (c->any_mdiff) k_adj_trans<STAGE, true, 4><<<grid, AB, 0, c->stream>>>(t);
    else k_adj_trans<STAGE, false, 4><<<grid, AB, 0, c->stream>>>(t);
  } else {
    if (c->any_mdiff) k_adj_trans<STAGE, true, 1><<<grid, AB, 0, c->stream>>>(t);
    else k_adj_trans<STAGE, false, 1><<<grid, AB, 0, c->stream>>>(t);
  }
  SV_HIP(c, hipGetLastError());
  return 0;
}

// calc_all_rhs vector-Jacobian product at tape slot 0 (Rbar in A->Rbar)
static int adj_rhs(sv_ctx *c, sv_adj *A, double *const *tape) {
  const PointArgs p = point_args(c, A, tape, 1, 0);
  if (c->any_mdiff) k_adj_point<true><<<c->nblk * SUBS, AB, 0, c->stream>>>(p);
  else k_adj_point<false><<<c->nblk * SUBS, AB, 0, c->stream>>>(p);
  SV_HIP(c, hipGetLastError());
  return adj_trans<0>(c, A, tape, 0, 0.0);
}

// adjoint of one step (tape slot): Ubar (after the step, with its mass sums
// in psum) -> Ubar (before the step) + seed on cxx, cyy.  Six launches.
static int adj_step(sv_ctx *c, sv_adj *A, double *const *tape, double seed) {
  const sv_loopl &L = A->TL;
  const int subl = subl_of(A->lpn), grid = c->nblk * subl;
  const bool small = A->halo && grid <= SMALL_SUMS;
  if (!small) k_adj_sum_reduce<<<c->nseg, 1024, 0, c->stream>>>(c->segk, A->psum, subl, A->sbar);
  FiltArgs f{c->blk_seg, c->segk, L.off, L.cnt, L.col, L.wh, c->L.hsum, c->L.vol,
             A->sbar, A->Ubar, c->ctrl, A->regbar, point_args(c, A, tape, 4, 0), L.krange, L.hoff,
             L.hidx, L.lcol, A->psum, small ? grid : 0};
  if (A->halo) {
    const size_t shm = std::max(SUMS_LDS, sizeof(double) * SV_US * (size_t)L.hmax);
    if (c->any_mdiff) k_adj_filter_h<true><<<grid, AW * SV_WAVE, shm, c->stream>>>(f);
    else k_adj_filter_h<false><<<grid, AW * SV_WAVE, shm, c->stream>>>(f);
  } else if (A->lpn == 4) {
    if (c->any_mdiff) k_adj_filter<true, 4><<<grid, AB, 0, c->stream>>>(f);
    else k_adj_filter<false, 4><<<grid, AB, 0, c->stream>>>(f);
  } else {
    if (c->any_mdiff) k_adj_filter<true, 1><<<grid, AB, 0, c->stream>>>(f);
    else k_adj_filter<false, 1><<<grid, AB, 0, c->stream>>>(f);
  }
  SV_HIP(c, hipGetLastError());
  if (int rc = adj_trans<4>(c, A, tape, 0, 0.0)) return rc;   // + point 3 -> set 1
  if (int rc = adj_trans<3>(c, A, tape, 1, 0.0)) return rc;   // + point 2 -> set 0
  if (int rc = adj_trans<2>(c, A, tape, 0, 0.0)) return rc;   // + point 1 -> set 1
  return adj_trans<1>(c, A, tape, 1, seed);
}

// the loss of the state after a step; the steps' sums are added up LOSS_STEPS at
// a time, and when last
static int loss_accumulate(sv_ctx *c, sv_adj *A, bool last) {
  k_loss_part<<<c->nblk, BS, 0, c->stream>>>(c->blk_seg, c->segk, c->U,
                                             A->lpart + (size_t)A->lsteps * c->nblk);
  if (++A->lsteps == LOSS_STEPS || last) {
    k_loss_steps<<<A->lsteps, 1024, 0, c->stream>>>(c->segk, A->lpart, A->lmean);
    k_loss_add<<<1, 1, 0, c->stream>>>(A->lsteps, A->lmean, A->lacc);
    A->lsteps = 0;
  }
  SV_HIP(c, hipGetLastError());
  return 0;
}

// caller-order arrays <-> loop-order records
static int upload_records(sv_ctx *c, double *dst, const double *const f[6]) {
  const int n = c->npfb;
  const std::vector<int> &P = c->L.hperm;
  std::vector<double> rec((size_t)SV_US * c->ntot, 0.0);
  for (int q = 0; q < 6; q++)
    if (f && f[q])
      for (int k = 0; k < n; k++) rec[(size_t)SV_US * k + q] = f[q][P[k]];
  SV_HIP(c, hipMemcpy(dst, rec.data(), sizeof(double) * rec.size(), hipMemcpyHostToDevice));
  return 0;
}

static int download_records(sv_ctx *c, const double *src, double *const f[6]) {
  const int n = c->npfb;
  const std::vector<int> &P = c->L.hperm;
  std::vector<double> rec((size_t)SV_US * n);
  SV_HIP(c, hipMemcpy(rec.data(), src, sizeof(double) * rec.size(), hipMemcpyDeviceToHost));
  for (int q = 0; q < 6; q++)
    if (f[q])
      for (int k = 0; k < n; k++) f[q][P[k]] = rec[(size_t)SV_US * k + q];
  return 0;
}

// caller-order device arrays <-> loop-order records, on the device
struct Fields6 {
  const double *f[6];
};
struct OutFields6 {
  double *f[6];
};

__global__ void k_gather_records(int n, const int *perm, Fields6 in, double *rec) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = perm[k];
#pragma unroll
  for (int q = 0; q < 6; q++) rec[(size_t)SV_US * k + q] = in.f[q] ? in.f[q][i] : 0.0;
}

__global__ void k_scatter_records(int n, const int *perm, const double *rec, OutFields6 out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = perm[k];
#pragma unroll
  for (int q = 0; q < 6; q++)
    if (out.f[q]) out.f[q][i] = rec[(size_t)SV_US * k + q];
}

// The eleven output fields of sv_get_state in the caller's node order, field
// after field (out[q * n + i]): ro, rou, rov from the registers, u, v from the
// gather records, psi (LC; left untouched in DI) from the registers, c from
// the gather records.
__global__ void k_get_fields(int n, const int *perm, const double *U, const double *G, int gs,
                             int lc, double *out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = perm[k];
  const double *u = U + (size_t)SV_US * k;
  const double *g = G + (size_t)gs * k;
  out[0 * (size_t)n + i] = u[0];
  out[1 * (size_t)n + i] = u[1];
  out[2 * (size_t)n + i] = u[2];
  out[3 * (size_t)n + i] = g[SV_G_U];
  out[4 * (size_t)n + i] = g[SV_G_V];
  if (lc) {
    out[5 * (size_t)n + i] = u[3];
    out[6 * (size_t)n + i] = u[4];
    out[7 * (size_t)n + i] = u[5];
  }
  out[8 * (size_t)n + i] = g[SV_G_CXX];
  out[9 * (size_t)n + i] = g[SV_G_CXY];
  out[10 * (size_t)n + i] = g[SV_G_CYY];
}

// nf fields of n values from loop order (in[f * n + k]) to the caller's
// order (out[f * n + perm[k]])
__global__ void k_to_caller_order(int n, int nf, const int *perm, const double *in,
                                  double *out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int i = perm[k];
  for (int f = 0; f < nf; f++) out[(size_t)f * n + i] = in[(size_t)f * n + k];
}

int sv_dev_to_caller_order(sv_ctx *c, int nf, const double *in, double *out) {
  const int n = c->npfb;
  k_to_caller_order<<<(n + 255) / 256, 256, 0, c->stream>>>(n, nf, c->L.perm, in, out);
  SV_HIP(c, hipGetLastError());
  return 0;
}

int sv_dev_get_fields(sv_ctx *c, int base, int n, double *out) {
  k_get_fields<<<(n + 255) / 256, 256, 0, c->stream>>>(
      n, c->L.perm + base, c->U + (size_t)base * SV_US, c->GA + (size_t)base * c->gs, c->gs,
      c->cfg.form == SV_FORM_LC, out);
  SV_HIP(c, hipGetLastError());
  return 0;
}

int sv_dev_gather_records(sv_ctx *c, double *dst, const double *const f[6]) {
  Fields6 in{};
  for (int q = 0; q < 6; q++) in.f[q] = f ? f[q] : nullptr;
  const int n = c->npfb;
  k_gather_records<<<(n + 255) / 256, 256, 0, c->stream>>>(n, c->L.perm, in, dst);
  SV_HIP(c, hipGetLastError());
  return 0;
}

int sv_dev_scatter_records(sv_ctx *c, const double *src, double *const f[6]) {
  OutFields6 out{};
  for (int q = 0; q < 6; q++) out.f[q] = f[q];
  const int n = c->npfb;
  k_scatter_records<<<(n + 255) / 256, 256, 0, c->stream>>>(n, c->L.perm, src, out);
  SV_HIP(c, hipGetLastError());
  return 0;
}

#define SV_ADJ_CHECK(c, cond, ...)                            \
  do {                                                        \
    if (!(cond)) return sv_fail((c), SV_E_ARG, __VA_ARGS__);  \
  } while (0)

// the control block after the work queued on the context's stream
static int read_ctrl(sv_ctx *c, sv_ctrl *h) {
  SV_HIP(c, hipMemcpyAsync(h, c->ctrl, sizeof(*h), hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}

// how the reverse sweeps gather
static int choose_gathers(sv_ctx *c) {
  sv_adj *A = c->adj;
  // lanes per node of the transposed gathers: 4 when one lane per node would
  // give fewer than 8 waves per CU (e.g. a 128x128 lattice: 256 waves)
  int ncu = 0;
  SV_HIP(c, hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
  const int64_t waves = (int64_t)c->nblk * SUBS;
  A->lpn = c->adj_lanes == 1 || c->adj_lanes == 4 ? c->adj_lanes
           : (waves < 8 * (int64_t)ncu ? 4 : 1);
  // staged halos where they fit (for either records), one slice a workgroup
  // (adj_lanes asks for the gathers from memory)
  A->halo = c->adj_lanes == 0 && A->TL.halo &&
            sizeof(double) * trans_rec<true>() * A->TL.hmax <= (size_t)SV_HALO_LDS_MAX;
  if (A->halo) A->lpn = 1;
  return 0;
}

// Where the lists cannot be made the adjoint goes (its buffers with the node
// set), so that no reverse sweep runs on lists of the old layout.
int sv_adj_new_layout(sv_ctx *c) {
  sv_adj *A = c->adj;
  if (!A) return 0;
  A->taped = false;
  sv_free_layout(c, A->TL);
  int rc = sv_dev_build_transpose(c, A->TL);
  if (!rc) rc = choose_gathers(c);
  if (rc) {
    sv_free_layout(c, A->TL);
    sv_adj_free(c);
  }
  return rc;
}

extern "C" {

int sv_adj_setup(sv_ctx *c, int32_t checkpoint_every) {
  SV_ADJ_CHECK(c, c && c->have_state, "sv_set_initial must come first");
  SV_ADJ_CHECK(c, !c->is_ensemble, "not available on an ensemble context");
  SV_ADJ_CHECK(c, c->cfg.form == SV_FORM_DI, "the adjoint is implemented for the DI form");
  SV_ADJ_CHECK(c, c->nb == 0, "the adjoint is implemented for node sets without boundary nodes");
  SV_ADJ_CHECK(c, !c->has_mirror, "the adjoint is implemented for periodic node sets (no "
               "symmetric/no-slip mirror ghosts)");
  SV_ADJ_CHECK(c, checkpoint_every >= 1 && checkpoint_every <= 1000,
               "checkpoint interval must be in [1, 1000]");
  SV_HIP(c, hipSetDevice(c->device));
  sv_ctrl h{};
  if (int rc = read_ctrl(c, &h)) return rc;
  SV_ADJ_CHECK(c, h.dt_mode == SV_DT_FIXED,
               "the adjoint needs a fixed time step (sv_set_control with SV_DT_FIXED)");
  if (!c->adj) {   // whole or not at all
    std::unique_ptr<sv_adj> A(new sv_adj());
    const size_t R = (size_t)SV_US * c->ntot, N = c->ntot;
    int rc = sv_dev_build_transpose(c, A->TL);
    if (!rc)
      rc = sv_alloc_all(
          c, {sv_want(&A->Ubar, R), sv_want(&A->Rbar, R), sv_want(&A->regbar, R),
              sv_want(&A->own[0], R), sv_want(&A->own[1], R), sv_want(&A->dbar[0], SV_TAPE_D * N),
              sv_want(&A->dbar[1], SV_TAPE_D * N), sv_want(&A->dbarm[0], 4 * N),
              sv_want(&A->dbarm[1], 4 * N), sv_want(&A->psum, (size_t)c->nblk * subl_of(4)),
              sv_want(&A->sbar, c->nseg), sv_want(&A->lpart, (size_t)LOSS_STEPS * c->nblk),
              sv_want(&A->lmean, LOSS_STEPS), sv_want(&A->lacc, c->nseg), sv_want(&A->Uend, R),
              sv_want(&A->pacc, 4 * N), sv_want(&A->pred, 4)});
    if (rc) {
      sv_free_layout(c, A->TL);
      return rc;
    }
    c->adj = A.release();
  }
  if (c->adj->every != checkpoint_every) c->adj->taped = false;
  c->adj->every = checkpoint_every;
  return choose_gathers(c);
}

// calc_all_rhs vector-Jacobian product at the current state: ubar = J^T rbar
int sv_rhs_vjp(sv_ctx *c, const double *const rbar[6], double *const ubar[6]) {
  SV_ADJ_CHECK(c, c && c->adj, "sv_adj_setup must come first");
  SV_ADJ_CHECK(c, rbar && ubar, "null argument");
  sv_adj *A = c->adj;
  SV_HIP(c, hipSetDevice(c->device));
  if (int rc = ensure_tape(c, A, 1)) return rc;
  A->taped = false;
  {
    DevTmp<double> scratch;
    SV_HIP(c, scratch.alloc(c, 6 * (size_t)c->npfb));
    if (int rc = sv_dev_rhs(c, 1, scratch, A->tape[0], A->tape[1])) return rc;
  }
  if (int r2 = upload_records(c, A->Rbar, rbar)) return r2;
  if (int r2 = zero_dev(c, A->pacc, (int64_t)4 * c->ntot)) return r2;
  if (int r2 = adj_rhs(c, A, A->tape.data())) return r2;
  if (int r2 = param_grad_finish(c, A)) return r2;
  return download_records(c, A->Ubar, ubar);
}

// nsteps of the fixed-dt loop from the current state, storing checkpoints;
// *loss = (1/nsteps) sum_t mean_i (cxx + cyy - 2) after each step
int sv_rollout_forward(sv_ctx *c, int32_t nsteps, double *loss) {
  SV_ADJ_CHECK(c, c && c->adj, "sv_adj_setup must come first");
  SV_ADJ_CHECK(c, nsteps >= 1, "nsteps must be >= 1");
  sv_adj *A = c->adj;
  SV_HIP(c, hipSetDevice(c->device));
  {
    sv_ctrl h{};
    if (int rc = read_ctrl(c, &h)) return rc;
    SV_ADJ_CHECK(c, h.dt_mode == SV_DT_FIXED, "the adjoint needs a fixed time step");
  }
  const int nck = (nsteps + A->every - 1) / A->every;
  const size_t R = (size_t)SV_US * c->ntot;
  while ((int)A->ckpt.size() < nck) {
    double *p = nullptr;
    if (adj_alloc(c, &p, R)) return SV_E_NOMEM;
    A->ckpt.push_back(p);
  }
  A->ckpt_ctrl.assign(nck, sv_ctrl{});
  const bool tape = want_tape(c, A, nsteps - (nck - 1) * A->every);
  A->taped = false;
  A->lsteps = 0;
  if (int rc = zero_dev(c, A->lacc, c->nseg)) return rc;
  EventTmp e0, e1;
  SV_HIP(c, e0.create());
  SV_HIP(c, e1.create());
  SV_HIP(c, hipEventRecord(e0, c->stream));
  for (int s = 0; s < nsteps; s++) {
    if (s % A->every == 0) {
      const int k = s / A->every;
      SV_HIP(c, hipMemcpyAsync(A->ckpt[k], c->U, sizeof(double) * R, hipMemcpyDeviceToDevice,
                               c->stream));
      SV_HIP(c, hipMemcpyAsync(&A->ckpt_ctrl[k], c->ctrl, sizeof(sv_ctrl),
                               hipMemcpyDeviceToHost, c->stream));
    }
    const int t = s - (nck - 1) * A->every;   // step of the last interval
    if (tape && t >= 0) {
      if (int rc = sv_dev_step_tape(c, A->tape.data() + 8 * t)) return rc;
    } else if (int rc = sv_dev_step(c, nullptr)) {
      return rc;
    }
    if (int rc = loss_accumulate(c, A, s + 1 == nsteps)) return rc;
  }
  SV_HIP(c, hipEventRecord(e1, c->stream));
  SV_HIP(c, hipMemcpyAsync(A->Uend, c->U, sizeof(double) * R, hipMemcpyDeviceToDevice,
                           c->stream));
  SV_HIP(c, hipMemcpyAsync(&A->ctrl_end, c->ctrl, sizeof(sv_ctrl), hipMemcpyDeviceToHost,
                           c->stream));
  double acc = 0.0;
  SV_HIP(c, hipMemcpyAsync(&acc, A->lacc, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  float ms = 0;
  SV_HIP(c, hipEventElapsedTime(&ms, e0, e1));
  A->t_fwd = ms;
  A->T = nsteps;
  A->taped = tape;
  if (tape) A->tape_used = false;
  if (loss) *loss = acc / nsteps;
  return 0;
}

// Gradient of  loss_bar * L + <ubar_final, U_T>  with respect to the state
// (ro, rou, rov, cxx, cxy, cyy) at the start of the last sv_rollout_forward.
// ubar_final may be NULL (or hold NULL fields).  The context's state is left
// at the end of the rollout.
// the loss term's seed on cxx and cyy of every real node's record
__global__ void k_seed_loss(int n, double seed, double *rec) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  rec[(size_t)SV_US * k + 3] += seed;
  rec[(size_t)SV_US * k + 5] += seed;
}

static int rollout_vjp(sv_ctx *c, double loss_bar, const double *const ubar_final[6],
                       double *const grad0[6], bool device_io) {
  SV_ADJ_CHECK(c, c && c->adj && c->adj->T > 0, "sv_rollout_forward must come first");
  SV_ADJ_CHECK(c, grad0, "null output");
  sv_adj *A = c->adj;
  SV_HIP(c, hipSetDevice(c->device));
  const int T = A->T, E = A->every;
  const bool taped = A->taped;
  if (int rc = ensure_tape(c, A, std::min(T, E))) return rc;
  A->taped = false;
  A->tape_used = true;
  const double seed = loss_bar / ((double)T * c->npfb);
  const size_t R = (size_t)SV_US * c->ntot;
  if (device_io) {
    if (int rc = zero_dev(c, A->Ubar, (int64_t)R)) return rc;
    if (int rc = sv_dev_gather_records(c, A->Ubar, ubar_final)) return rc;
  } else if (int rc = upload_records(c, A->Ubar, ubar_final)) {
    return rc;
  }
  k_seed_loss<<<(c->npfb + 255) / 256, 256, 0, c->stream>>>(c->npfb, seed, A->Ubar);
  SV_HIP(c, hipGetLastError());
  EventTmp e0, e1;
  SV_HIP(c, e0.create());
  SV_HIP(c, e1.create());
  SV_HIP(c, hipEventRecord(e0, c->stream));
  if (int rc = zero_dev(c, A->pacc, (int64_t)4 * c->ntot)) return rc;
  if (A->lpn == 4)
    k_adj_sum<4><<<c->nblk * subl_of(4), AB, 0, c->stream>>>(c->blk_seg, c->segk, A->Ubar,
                                                             A->psum);
  else
    k_adj_sum<1><<<c->nblk * SUBS, AB, 0, c->stream>>>(c->blk_seg, c->segk, A->Ubar, A->psum);
  SV_HIP(c, hipGetLastError());
  const int nck = (T + E - 1) / E;
  A->recomputed = 0;
  for (int k = nck - 1; k >= 0; k--) {
    const int s0 = k * E, s1 = std::min(T, s0 + E);
    if (taped && k == nck - 1) {   // the rollout wrote its tape
      SV_HIP(c, hipMemcpyAsync(c->ctrl, &A->ctrl_end, sizeof(sv_ctrl), hipMemcpyHostToDevice,
                               c->stream));
    } else {
      // recompute the interval from its checkpoint with the tape on
      SV_HIP(c, hipMemcpyAsync(c->U, A->ckpt[k], sizeof(double) * R, hipMemcpyDeviceToDevice,
                               c->stream));
      SV_HIP(c, hipMemcpyAsync(c->ctrl, &A->ckpt_ctrl[k], sizeof(sv_ctrl),
                               hipMemcpyHostToDevice, c->stream));
      if (int rc = sv_dev_init_state(c)) return rc;
      A->recomputed += s1 - s0;
      for (int s = s0; s < s1; s++)
        if (int rc = sv_dev_step_tape(c, A->tape.data() + 8 * (s - s0))) return rc;
    }
    for (int s = s1 - 1; s >= s0; s--)
      if (int rc = adj_step(c, A, A->tape.data() + 8 * (s - s0), s >= 1 ? seed : 0.0))
        return rc;
  }
  SV_HIP(c, hipEventRecord(e1, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  float ms = 0;
  SV_HIP(c, hipEventElapsedTime(&ms, e0, e1));
  A->t_bwd = ms;
  if (int rc = param_grad_finish(c, A)) return rc;
  if (device_io) {
    if (int rc = sv_dev_scatter_records(c, A->Ubar, grad0)) return rc;
    SV_HIP(c, hipStreamSynchronize(c->stream));
  } else if (int rc = download_records(c, A->Ubar, grad0)) {
    return rc;
  }
  // leave the state at the end of the rollout
  SV_HIP(c, hipMemcpy(c->U, A->Uend, sizeof(double) * R, hipMemcpyDeviceToDevice));
  SV_HIP(c, hipMemcpy(c->ctrl, &A->ctrl_end, sizeof(sv_ctrl), hipMemcpyHostToDevice));
  return sv_dev_init_state(c);
}

int sv_rollout_vjp(sv_ctx *c, double loss_bar, const double *const ubar_final[6],
                   double *const grad0[6]) {
  return rollout_vjp(c, loss_bar, ubar_final, grad0, false);
}

int sv_rollout_vjp_device(sv_ctx *c, double loss_bar, const double *const ubar_final[6],
                          double *const grad0[6], void *stream) {
  SV_ADJ_CHECK(c, c && grad0, "null argument");
  for (int q = 0; q < 6; q++) {
    if (int rc = sv_check_device_ptr(c, grad0[q], "grad0")) return rc;
    if (ubar_final && ubar_final[q])
      if (int rc = sv_check_device_ptr(c, ubar_final[q], "ubar_final")) return rc;
  }
  // the caller's stream, the null stream included (a framework's default
  // stream): its pending work on the arrays completes first
  SV_HIP(c, hipStreamSynchronize((hipStream_t)stream));
  return rollout_vjp(c, loss_bar, ubar_final, grad0, true);
}

int sv_adj_param_grad(sv_ctx *c, double grad[3]) {
  SV_ADJ_CHECK(c, c && c->adj && grad, "sv_adj_setup must come first");
  for (int k = 0; k < 3; k++) grad[k] = c->adj->pgrad[k];
  return 0;
}

int sv_adj_timing(sv_ctx *c, double *fwd_ms, double *vjp_ms) {
  SV_ADJ_CHECK(c, c && c->adj, "sv_adj_setup must come first");
  if (fwd_ms) *fwd_ms = c->adj->t_fwd;
  if (vjp_ms) *vjp_ms = c->adj->t_bwd;
  return 0;
}

}  // extern "C"
