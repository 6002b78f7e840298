// k_step.hip -- device-resident RK3(2)4[2R+]C step (step_rk3_4S_2R_EE,
// step.F90:218-512) with the right-hand sides of rhs_lc.F90 / rhs_di.F90 and
// filter_variables, set_tstep and set_tstep_PID.
//
// One step is 8 launches, all reading their scalars from the device control
// block so the step can be captured once and replayed as a hipGraph.  Up to
// 32768 nodes it is 6: a launch of a single block costs 4.4 us there, a tenth of
// the step, and the few partial results are reduced by every workgroup of the
// kernel that needs them (k_dt's work at the head of stage 1, k_reduce's in
// k_apply_state), in the same order:
//   k_dt          (1 block)  set_tstep + set_tstep_PID, emax history shift,
//                            dt-scaled RK coefficients
//   k_stage<1..4>            ONE gather sweep per stage: every gradient and
//                            Laplacian the RHS needs (the reference makes 11
//                            separate sweeps, rhs_lc.F90:64-402), then the
//                            pointwise RHS and the low-storage RK update
//   k_filter                 hyperviscous filter of the evolved fields
//                            (calc_filtered_var, derivatives.F90:360-414) and
//                            the conformation tensor of the filtered psi
//   k_reduce      (1 block)  mass correction (rhs_lc.F90:871-890), emax,
//                            itime += 1
//   k_apply_state            rho -= drho, u = rou/rho, dt partial minima
// Ghost nodes do not exist at run time: periodic links point at the parent
// (mirror copies are exact copies, mirror_boundaries.F90:263-352).
// Reductions are a fixed-order two-level tree, so results are bitwise
// reproducible run to run.
//
// Memory layout of the state (records, see sv_internal.h): what a neighbour
// gather needs of node j sits in one packed 80-byte record (LC) or 48-byte
// record (DI), so a link costs at most two cache lines instead of one line
// per field, and records of adjacent nodes share lines.
#include <algorithm>

#include "sv_internal.h"
#include "sweep.h"

namespace {

constexpr int BS = SV_BLOCK;   // threads per block of the node kernels
constexpr int SPB = BS / SV_WAVE;   // slices (and partial results) per block

// Pairs of links per batch in the halo-staged sweeps (the global streams are
// prefetched one batch ahead), by threads per workgroup: a small node set has
// one wave per SIMD at most and needs many requests per wave (128^2 order 6,
// stage: 1 pair 24 us, 2 15.6, 3 14.2); a large one has twelve waves per CU and
// is slower with more (1024^2: 1 pair 421 us, 2 436).
template <int NB>
struct HaloU {
  static constexpr int U = NB == 64 ? 3 : NB == 128 ? 2 : 1;   // stage sweeps
  static constexpr int UF = NB == 64 ? 4 : 2;                  // the filter
};
// the stencil arrays of the sweeps that gather from memory: read once per sweep,
// loaded non-temporally so that they do not displace the gathered records
template <typename T>
__device__ __forceinline__ T ld_stream(const T *p) {
  return __builtin_nontemporal_load(p);
}

// The node handled by this thread: segment of the block, concatenated index i,
// a safe index ii (= i, or the segment's first node for an idle lane).
struct NodeRef {
  int sg, i, ii;
  bool act;
};

// bid: workgroup of NB consecutive slots (NB divides SV_BLOCK); waves past
// them (a list shared by several) repeat its slots
template <int NB = BS>
__device__ __forceinline__ NodeRef node_ref(const int *blk_seg, const sv_segk *seg, int bid) {
  NodeRef r;
  r.sg = blk_seg[bid / (BS / NB)];
  const sv_segk &S = seg[r.sg];
  r.i = bid * NB + (int)threadIdx.x % NB;
  r.act = r.i - S.base < S.npfb;
  r.ii = r.act ? r.i : S.base;
  return r;
}

// Logical workgroup of NB slots: the XCD-aware index, through a launch group's
// block list (256-slot blocks) when the launch covers a subset
template <int NB>
__device__ __forceinline__ int logical_wg(const int *blist) {
  constexpr int SUB = BS / NB;
  const int b = sv_xcd_block();
  return blist ? blist[b / SUB] * SUB + b % SUB : b;
}

// ---- conformation algebra (conf_transforms.F90) -------------------------
// 2D eigens (:399-444); R column-major R[0]=R11 R[1]=R21 R[2]=R12 R[3]=R22
__device__ __forceinline__ void eigens2(double a, double b, double d, double &l1, double &l2,
                                        double R[4]) {
  if (fabs(b) <= 1.0e-16) {
    l1 = a; l2 = d;
    R[0] = 1.0; R[1] = 0.0; R[2] = 0.0; R[3] = 1.0;
    return;
  }
  const double tr = a + d;
  const double det = a * d - b * b;
  double t = 0.25 * tr * tr - det;
  if (t <= 1.0e-16) t = 0.0;
  t = sqrt(t);
  l1 = 0.5 * tr + t;
  l2 = 0.5 * tr - t;
  double r11 = l1 - d, r21 = b;
  const double nrm = sqrt(r11 * r11 + r21 * r21);
  r11 = r11 / nrm;
  r21 = r21 / nrm;
  R[0] = r11; R[1] = r21; R[2] = -r21; R[3] = r11;
}

// log_conf_c_from_psi (:133-169): C = R diag(exp L) R^T
__device__ __forceinline__ void c_from_psi(double pxx, double pxy, double pyy, double &cxx,
                                           double &cxy, double &cyy) {
  double l1, l2, R[4];
  eigens2(pxx, pxy, pyy, l1, l2, R);
  const double e1 = exp(l1), e2 = exp(l2);
  const double i11 = e1 * R[0], i12 = e1 * R[1], i21 = e2 * R[2], i22 = e2 * R[3];
  cxx = R[0] * i11 + R[2] * i21;
  cxy = R[1] * i11 + R[3] * i21;
  cyy = R[1] * i12 + R[3] * i22;
}

// calc_rhs_logconf pointwise part (rhs_lc.F90:416-557)
__device__ __forceinline__ void rhs_logconf(double u, double v, double ux, double uy, double vx,
                                            double vy, double pxx, double pxy, double pyy,
                                            double gpxx_x, double gpxx_y, double gpxy_x,
                                            double gpxy_y, double gpyy_x, double gpyy_y,
                                            bool first, double eps, double lam, double &rxx,
                                            double &rxy, double &ryy) {
  const double adxx = -(u * gpxx_x + v * gpxx_y + 0.0);
  const double adxy = -(u * gpxy_x + v * gpxy_y + 0.0);
  const double adyy = -(u * gpyy_x + v * gpyy_y + 0.0);
  double L1, L2, R[4];
  eigens2(pxx, pxy, pyy, L1, L2, R);
  L1 = exp(L1);
  L2 = exp(L2);
  const double tr_c = L1 + L2;
  const double G11 = ux, G12 = uy, G21 = vx, G22 = vy;
  const double GR11 = G11 * R[0] + G12 * R[1], GR12 = G11 * R[2] + G12 * R[3];
  const double GR21 = G21 * R[0] + G22 * R[1], GR22 = G21 * R[2] + G22 * R[3];
  const double M11 = R[0] * GR11 + R[1] * GR21, M12 = R[0] * GR12 + R[1] * GR22;
  const double M21 = R[2] * GR11 + R[3] * GR21, M22 = R[2] * GR12 + R[3] * GR22;
  double om = L2 * M12 + L1 * M21;
  if (fabs(L2 - L1) <= 1.0e-30) om = 0.0;
  else om = om / (L2 - L1);
  double B11, B12, B22, O11, O12, O21, O22;
  {
    const double i11 = M11 * R[0], i12 = M11 * R[1], i21 = M22 * R[2], i22 = M22 * R[3];
    B11 = R[0] * i11 + R[2] * i21;
    B12 = R[0] * i12 + R[2] * i22;
    B22 = R[1] * i12 + R[3] * i22;
  }
  {
    const double i11 = om * R[2], i12 = om * R[3], i21 = -om * R[0], i22 = -om * R[1];
    O11 = R[0] * i11 + R[2] * i21;
    O12 = R[0] * i12 + R[2] * i22;
    O21 = R[1] * i11 + R[3] * i21;
    O22 = R[1] * i12 + R[3] * i22;
  }
  if (first) {   // rhs_lc.F90:503-506
    O11 = O12 = O21 = O22 = 0.0;
    B11 = 0.5 * (G11 + G11);
    B12 = 0.5 * (G12 + G21);
    B22 = 0.5 * (G22 + G22);
  }
  const double UC11 = (O11 * pxx + O12 * pxy) - (pxx * O11 + pxy * O21) + 2.0 * B11;
  const double UC12 = (O11 * pxy + O12 * pyy) - (pxx * O12 + pxy * O22) + 2.0 * B12;
  const double UC22 = (O21 * pxy + O22 * pyy) - (pxy * O12 + pyy * O22) + 2.0 * B22;
  const double fR = 1.0 - 2.0 * eps + eps * tr_c;
  const double C1 = fR / L1 - fR, C2 = fR / L2 - fR;
  const double i11 = C1 * R[0], i12 = C1 * R[1], i21 = C2 * R[2], i22 = C2 * R[3];
  rxx = adxx + UC11 + (R[0] * i11 + R[2] * i21) / lam;
  rxy = adxy + UC12 + (R[0] * i12 + R[2] * i22) / lam;
  ryy = adyy + UC22 + (R[1] * i12 + R[3] * i22) / lam;
}

// ---- record access ----------------------------------------------------
struct Rec9 {   // gathered fields of one node
  double ro, u, v, cxx, cxy, cyy, pxx, pxy, pyy;
};

template <int FORM>
__device__ __forceinline__ Rec9 load_g(const double *G, int j) {
  constexpr int S = (FORM == SV_FORM_LC) ? SV_GS_LC : SV_GS_DI;
  const double2 *p = reinterpret_cast<const double2 *>(G + (size_t)j * S);
  Rec9 r;
  const double2 a = p[0], b = p[1], c = p[2];
  r.ro = a.x; r.u = a.y; r.v = b.x; r.cxx = b.y; r.cxy = c.x; r.cyy = c.y;
  if (FORM == SV_FORM_LC) {
    const double2 d = p[3];
    r.pxx = d.x; r.pxy = d.y;
    r.pyy = G[(size_t)j * S + SV_G_PYY];
  } else {
    r.pxx = r.pxy = r.pyy = 0.0;
  }
  return r;
}

template <int FORM>
__device__ __forceinline__ void store_g(double *G, int i, const Rec9 &r) {
  constexpr int S = (FORM == SV_FORM_LC) ? SV_GS_LC : SV_GS_DI;
  double2 *p = reinterpret_cast<double2 *>(G + (size_t)i * S);
  p[0] = double2{r.ro, r.u};
  p[1] = double2{r.v, r.cxx};
  p[2] = double2{r.cxy, r.cyy};
  if (FORM == SV_FORM_LC) {
    p[3] = double2{r.pxx, r.pxy};
    p[4] = double2{r.pyy, 0.0};   // the pad too: whole lines reach memory
  }
}

__device__ __forceinline__ void load_u(const double *U, int i, double f[6]) {
  const double2 *p = reinterpret_cast<const double2 *>(U + (size_t)i * SV_US);
  const double2 a = p[0], b = p[1], c = p[2];
  f[0] = a.x; f[1] = a.y; f[2] = b.x; f[3] = b.y; f[4] = c.x; f[5] = c.y;
}

__device__ __forceinline__ void store_u(double *U, int i, const double f[6]) {
  double2 *p = reinterpret_cast<double2 *>(U + (size_t)i * SV_US);
  p[0] = double2{f[0], f[1]};
  p[1] = double2{f[2], f[3]};
  p[2] = double2{f[4], f[5]};
}

struct StageArgs {
  int rhs_stride;       // STAGE 0: length of each rhs_out array
  const int *blk_seg;
  const sv_segk *seg;
  const int64_t *off;
  const int *kcnt;
  const int *col;
  const double *w3;
  const double *gsx, *gsy, *lsum;
  const double *G;      // gathered records (stage input)
  const double *reg_in; // register 1 input (stage 1: the state)
  double *reg_out;      // register 1 output
  double *e;            // error accumulators
  double *Uout;         // stage 4 result
  double *Gout;         // stages 1-3: next gather records
  double *rhs_out;      // STAGE 0: six arrays of npfb
  const double *fx;
  const sv_ctrl *ctrl;  // [nseg]
  double *partial;      // stage 4: max error per slice
  // stage 1 of small node sets: the limits' partial minima, and the control
  // values made from them and ctrl (another array: other workgroups still read)
  const double *pcfl, *pvisc;
  sv_ctrl *ctrl_out;
  int rk1;              // STAGE 0: reference stage counter is 1
  // DI only, nullable: the stage's own gather record [ntot][SV_US] and its
  // derivative values [ntot][16] (rx ry ux uy lu vx vy lv, cxx_x cxx_y, cxy_x
  // cxy_y, cyy_x cyy_y, 0 0), the tape the adjoint sweep reads
  double *tapeG, *tapeD;
  const int4 *krange;   // links per slice (sv_loopl)
  // per-block halos (k_stage_h)
  const int64_t *hoff;
  const int *hidx;
  const uint16_t *lcol;
  // boundary nodes (nullable): per loop slot the record index or -1, records
  const int *bidx;
  const double *brec;
  const int *blist;     // launch group's logical blocks (nullable: all blocks)
};

// u_inflow_local of an inflow node as the last apply_time_dependent_bounds
// before stage s of the current step left it (update_u_inflow,
// characteristic_boundaries.F90:256-289): while time <= ramp_time every apply
// sets the ramp value; the applies of this step ran at time0 + RKc[q-1],
// q < s.  s = 1: the value at the start of the step.
__device__ __forceinline__ double uin_now(const sv_physk &P, const sv_ctrl *C, double uin0,
                                          int s) {
  if (P.u_control != 1) return uin0;
  bool set = C->uin_set != 0;
  double v = C->uin_ramp;
#pragma unroll
  for (int q = 1; q < s; q++) {
    const double t = C->time0 + C->RKc[q - 1];
    if (t <= P.ramp_time) {
      set = true;
      v = P.u_start + (P.u_end - P.u_start) * t / P.ramp_time;
    }
  }
  return set ? v : uin0;
}

// apply_time_dependent_bounds on one state record (characteristic_boundaries.F90:
// 176-254): walls hold zero velocity, hard inflows the inflow velocity
__device__ __forceinline__ void bound_apply(const sv_physk &P, int kind, double uin, double f[6]) {
  if (kind == 0) {
    f[1] = 0.0;
    f[2] = 0.0;
  } else if (kind == 1 && P.inflow_type == 1) {
    f[1] = uin * f[0];
    f[2] = 0.0;
  }
}

// Right-hand side of a boundary node: the boundary branches of calc_rhs_ro
// (rhs_lc.F90:144-160), calc_rhs_rovel (:279-367) and, for the conformation,
// calc_rhs_logconf (:564-745) or calc_rhs_c (rhs_di.F90:477-594: on walls the
// upper-convected and relaxation terms with the rotated velocity gradient, the
// polymer diffusion added by the caller; on inflows/outflows zero), then the
// characteristic waves
// (characteristic_boundaries.F90:27-175) applied as calc_rhs_nscbc
// (rhs_lc.F90:752-813).  Wall derivatives are in the normal-tangent frame
// (x component = d/dn, y = d/dt), inflow/outflow ones in x-y.  In the
// log-conformation form the interior conformation right-hand side (r_xx..r_yy
// on entry) is kept on inflow and outflow nodes.  f1..f3: psi (LC) or c (DI).
template <int FORM>
__device__ __forceinline__ void bound_rhs(const sv_physk &P, int kind, double nx, double ny,
                                          double uin, bool first, double ro, double u, double v,
                                          double rx, double ry, double ux, double uy, double vx,
                                          double vy, double lu, double lv, double dcxx_x,
                                          double dcxy_y, double dcxy_x, double dcyy_y,
                                          double f1, double f2, double f3, double &r_ro,
                                          double &r_rou, double &r_rov, double &r_xx,
                                          double &r_xy, double &r_yy) {
  const double csq = P.csq, c = P.cs;
  const double nscbc = 2.87e-1;                   // common_parameter.F90:71
  const double pr = csq * ro, dpdn = csq * rx;
  double L1, L2, L3, L5;
  if (kind == 0) {
    const double dutdt = -ny * uy + nx * vy;
    r_ro = -ro * dutdt - ro * 0.0;
    const double un = u * nx + v * ny;
    const double dundn = nx * ux + ny * vx;
    const double dutdn = -ny * ux + nx * vx;
    L1 = 0.5 * (un - c) * (dpdn - ro * c * dundn);
    L2 = un * (rx - csq * rx / c / c);
    L3 = un * dutdn;
    L5 = 0.5 * (un + c) * (dpdn + ro * c * dundn);
    r_rou = 0.0;
    r_rov = 0.0;
    // velocity gradient rotated to x-y; no advection on a wall
    const double G11 = nx * ux - ny * uy, G12 = ny * ux + nx * uy;
    const double G21 = nx * vx - ny * vy, G22 = ny * vx + nx * vy;
    if (FORM == SV_FORM_LC) {
      rhs_logconf(0.0, 0.0, G11, G12, G21, G22, f1, f2, f3, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0,
                  first, P.eps, P.lambda, r_xx, r_xy, r_yy);
    } else {
      const double cxx = f1, cxy = f2, cyy = f3;
      const double ucxx = 2.0 * G11 * cxx + 2.0 * G12 * cxy + 0.0;
      const double ucxy = G11 * cxy + G12 * cyy + 0.0 + G21 * cxx + G22 * cxy + 0.0;
      const double ucyy = 2.0 * G21 * cxy + 2.0 * G22 * cyy + 0.0;
      const double fr = -(1.0 - P.eps * 2.0 + P.eps * (cxx + cyy + 1.0)) / P.lambda;
      r_xx = ucxx + fr * (cxx - 1.0) + 0.0;
      r_xy = ucxy + fr * cxy + 0.0;
      r_yy = ucyy + fr * (cyy - 1.0) + 0.0;
    }
    L5 = L1;                                      // isothermal wall
  } else {
    r_ro = -v * ry - ro * vy - 0.0 * 0.0 - ro * 0.0;
    L1 = 0.5 * (u - c) * (dpdn - ro * c * ux);
    L2 = u * (rx - csq * rx / c / c);
    L3 = u * vx;
    L5 = 0.5 * (u + c) * (dpdn + ro * c * ux);
    double fvu = P.coef_solvent * lu;
    double fvv = P.coef_solvent * lv;
    fvu = fvu + P.coef_polymeric * (dcxx_x + dcxy_y + 0.0);
    fvv = fvv + P.coef_polymeric * (dcxy_x + dcyy_y + 0.0);
    r_rou = -v * uy - 0.0 * 0.0 + fvu + ro * P.bfx;
    r_rov = -v * vy - 0.0 * 0.0 - csq * ry + fvv + ro * P.bfy;
    if (FORM == SV_FORM_DI) { r_xx = 0.0; r_xy = 0.0; r_yy = 0.0; }   // rhs_di.F90:579-590
    const double Lx = P.Lx;
    if (kind == 1) {
      if (P.inflow_type == 1) {                   // hard inflow
        L2 = 0.0; L3 = 0.0; L5 = L1;
      } else if (P.inflow_type == 2) {            // inflow-outflow
        if (u > 0.0) {
          L2 = 0.0;
          L3 = v * nscbc * c / Lx;
          L5 = (u - uin) * nscbc * (1.0 - u / c) * c * c * 1.0 / Lx;
        } else {
          L2 = 0.0;
          L5 = (pr - P.p_ref) * nscbc * c * 1.0 / 2.0 / Lx;
        }
      } else {                                    // soft inflow
        const double gp2 = csq * ry;
        L2 = 0.0;
        L3 = v * nscbc * c / Lx - v * vy - 0.0 * 0.0 - gp2 / ro;
        L5 = (u - uin) * nscbc * (1.0 - u / c) * c * c * 1.0 / Lx -
             0.5 * (v * gp2 + pr * vy + ro * c * v * uy) -
             0.5 * (0.0 * 0.0 + pr * 0.0 + ro * c * 0.0 * 0.0);
      }
    } else {                                      // outflow
      if (u < c) L1 = (pr - P.p_ref) * nscbc * c * 1.0 / 2.0 / Lx;
      L2 = 0.0;
      if (u <= 0.0) { L2 = 0.0; L3 = 0.0; }
    }
  }
  const double ts = (c * c * L2 + L5 + L1) / c / c;
  r_ro = r_ro - ts;
  r_rou = r_rou - u * ts - (L5 - L1) / c;
  r_rov = r_rov - v * ts - ro * L3;
}

// A control block field by field (a copy of the whole goes through scratch
// memory where the copy lives in registers).
__device__ __forceinline__ void copy_ctrl(const sv_ctrl &a, sv_ctrl &b) {
  b.dt = a.dt; b.time = a.time; b.time0 = a.time0; b.dt_cfl = a.dt_cfl; b.dt_par = a.dt_par;
  b.emax_np1 = a.emax_np1; b.emax_n = a.emax_n; b.emax_nm1 = a.emax_nm1;
#pragma unroll
  for (int k = 0; k < 3; k++) b.RKa[k] = a.RKa[k];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    b.RKb[k] = a.RKb[k]; b.RKbmbh[k] = a.RKbmbh[k]; b.RKc[k] = a.RKc[k];
  }
  b.dro = a.dro;
  b.itime = a.itime; b.dt_mode = a.dt_mode; b.flags = a.flags;
  b.uin_ramp = a.uin_ramp; b.uin_set = a.uin_set;
}

// set_tstep (step.F90:569-622), set_tstep_PID (:624-682) and the start of
// step_rk3_4S_2R_EE (:239-246) from the minima of the advective and viscous
// limits over the nodes
__device__ __forceinline__ void next_dt(const sv_physk &P, double mc, double mv, sv_ctrl &c) {
  c.dt_cfl = 1.0 * mc * P.L_char;
  c.dt_par = (2.0 / 3.0) * mv * P.L_char * P.L_char;
  if (c.dt_mode == SV_DT_PID) {
    const double fA = SV_PID_A * log(SV_PID_TOL / c.emax_np1);
    const double fB = SV_PID_B * log(c.emax_n / SV_PID_TOL);
    const double fC = SV_PID_C * log(SV_PID_TOL / c.emax_nm1);
    double f = SV_PID_K * exp(fA + fB + fC);
    f = fmax(0.5, f);
    f = fmin(1.02, f);
    double dt = c.dt * f;
    const double dmax = fmin(c.dt_cfl, c.dt_par);
    if (dt > dmax) dt = dmax;
    c.dt = dt;
  } else if (c.dt_mode == SV_DT_CFL) {
    c.dt = fmin(c.dt_par, c.dt_cfl);
  }
  c.emax_nm1 = c.emax_n;
  c.emax_n = c.emax_np1;
  const double dt = c.dt;
  c.RKa[0] = dt * SV_RKA1; c.RKa[1] = dt * SV_RKA2; c.RKa[2] = dt * SV_RKA3;
  const double b[4] = {SV_RKB1, SV_RKB2, SV_RKB3, SV_RKB4};
  const double bh[4] = {SV_RKBH1, SV_RKBH2, SV_RKBH3, SV_RKBH4};
  const double cc[4] = {0.0, SV_RKA1, SV_RKA2 + SV_RKB1, 1.0};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    c.RKb[k] = dt * b[k];
    c.RKbmbh[k] = dt * (b[k] - bh[k]);
    c.RKc[k] = dt * cc[k];
  }
  c.time0 = c.time;
}

// The end of a step: mass correction value (rhs_lc.F90:871-890), emax and the
// counters, from the nodes' mass and largest error
__device__ __forceinline__ void end_step(const sv_segk &S, double mass, double err, sv_ctrl &c) {
  c.dro = mass / S.volsum;
  c.emax_np1 = fmax(err, 1.0e-16);       // step.F90:480-485
  if (!(err == err) || !(mass == mass)) c.flags |= 1;
  // the step's four applies of the boundary conditions ran at
  // time0 + RKc[0..3]; the ramped inflow velocity follows the last one at
  // time <= ramp_time (characteristic_boundaries.F90:268-283)
  if (S.pk.u_control == 1)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double t = c.time0 + c.RKc[q];
      if (t <= S.pk.ramp_time) {
        c.uin_set = 1;
        c.uin_ramp = S.pk.u_start + (S.pk.u_end - S.pk.u_start) * t / S.pk.ramp_time;
      }
    }
  c.time = c.time0 + c.RKc[3];
  c.itime = c.itime + 1;               // sunset.F90:99
}

// One wavefront's reductions over the partial results of a segment of at most
// 128 blocks, in the order of k_reduce and k_dt (whose trees halve 1024 entries,
// one per block): two blocks per lane, then the lanes.
constexpr int SMALL_BLOCKS = 128;
struct Partials {
  dbl2 a[2][2], b[2][2];   // two blocks of the two kinds, four slices each
  __device__ __forceinline__ void load(const sv_segk &S, const double *pa, const double *pb,
                                       double none_a, double none_b) {
    const int lane = (int)threadIdx.x & (SV_WAVE - 1);
    const dbl2 *qa = reinterpret_cast<const dbl2 *>(pa) + 2 * (size_t)S.blk0;
    const dbl2 *qb = reinterpret_cast<const dbl2 *>(pb) + 2 * (size_t)S.blk0;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int b0 = lane + k * SV_WAVE;
      const bool in = b0 < S.nblk;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        a[k][h] = in ? qa[2 * b0 + h] : dbl2{none_a, none_a};
        b[k][h] = in ? qb[2 * b0 + h] : dbl2{none_b, none_b};
      }
    }
  }
};
__device__ __forceinline__ double sum_partials(const dbl2 p[2][2]) {
  return wave_sum(((p[0][0].x + p[0][0].y) + (p[0][1].x + p[0][1].y)) +
                  ((p[1][0].x + p[1][0].y) + (p[1][1].x + p[1][1].y)));
}
__device__ __forceinline__ double max_partials(const dbl2 p[2][2]) {
  return wave_max(fmax(fmax(fmax(p[0][0].x, p[0][0].y), fmax(p[0][1].x, p[0][1].y)),
                       fmax(fmax(p[1][0].x, p[1][0].y), fmax(p[1][1].x, p[1][1].y))));
}
__device__ __forceinline__ double min_partials(const dbl2 p[2][2]) {
  return wave_min(fmin(fmin(fmin(p[0][0].x, p[0][0].y), fmin(p[0][1].x, p[0][1].y)),
                       fmin(fmin(p[1][0].x, p[1][0].y), fmin(p[1][1].x, p[1][1].y))));
}

// The neighbour sums of one node in a stage: gradients and Laplacians before
// the own-node term (sum_k w_k f_j), as named in the right-hand side.
struct Sums {
  double rx, ry, ux, uy, vx, vy, lu, lv, axx, ayx, axy, ayy, bxy, byy, cxx_l, cxy_l, cyy_l, q1x, q1y, q2x, q2y, q3x, q3y;
};

// A node's own values in a stage: its gather record, the sums of its weights,
// the RK register and the error accumulators.
struct Own {
  Rec9 s;
  double sx, sy, sl, r1[6], eo[6];
};

template <int FORM, int STAGE>
__device__ __forceinline__ Own load_own(const StageArgs &a, int i) {
  Own o;
  o.s = load_g<FORM>(a.G, i);
  o.sx = a.gsx[i]; o.sy = a.gsy[i]; o.sl = a.lsum[i];
  if (STAGE > 0) load_u(a.reg_in, i, o.r1);
  if (STAGE > 1) load_u(a.e, i, o.eo);
  return o;
}

// Pointwise part of a stage for one node: the right-hand side from the
// gathered sums and the own record, then the RK update.  Returns the node's
// error norm contribution (stage 4).
template <int FORM, int STAGE, bool MDIFF, bool BND>
__device__ __forceinline__ double stage_point(const StageArgs &a, const NodeRef &nr, const Sums &S,
                                              const Own &own, const sv_ctrl *C) {
  const int i = nr.i;
  double rx = S.rx, ry = S.ry, ux = S.ux, uy = S.uy, vx = S.vx, vy = S.vy, lu = S.lu, lv = S.lv;
  double axx = S.axx, ayx = S.ayx, axy = S.axy, ayy = S.ayy, bxy = S.bxy, byy = S.byy, cxx_l = S.cxx_l, cxy_l = S.cxy_l;
  double cyy_l = S.cyy_l, q1x = S.q1x, q1y = S.q1y, q2x = S.q2x, q2y = S.q2y, q3x = S.q3x, q3y = S.q3y;
  (void)ayx; (void)bxy; (void)cxx_l; (void)cxy_l; (void)cyy_l;
  (void)q1x; (void)q1y; (void)q2x; (void)q2y; (void)q3x; (void)q3y;
  double emax_loc = 0.0;
  {
    const double sx = own.sx, sy = own.sy, sl = own.sl;
    const Rec9 s = own.s;
    const double ro = s.ro, u = s.u, v = s.v, cxx = s.cxx, cxy = s.cxy, cyy = s.cyy;
    rx = rx - ro * sx; ry = ry - ro * sy;
    ux = ux - u * sx; uy = uy - u * sy; lu = lu - u * sl;
    vx = vx - v * sx; vy = vy - v * sy; lv = lv - v * sl;
    const sv_physk &P = a.seg[nr.sg].pk;
    // calc_rhs_ro (rhs_lc.F90:127-141)
    const double r_ro = -ro * (ux + vy + 0.0) - (u * rx + v * ry + 0.0 * 0.0);
    int bkind = -1;        // boundary node kind (BND), -1 interior
    double buin0 = 0.0;
    // calc_rhs_rovel (rhs_lc.F90:217-272)
    const double tsu = ro * (u * ux + v * uy + 0.0 * 0.0) - u * r_ro;
    const double tsv = ro * (u * vx + v * vy + 0.0 * 0.0) - v * r_ro;
    const double dcxx_x = axx - cxx * sx;
    const double dcxy_x = axy - cxy * sx;
    const double dcxy_y = ayy - cxy * sy;
    const double dcyy_y = byy - cyy * sy;
    double fvu = P.coef_solvent * lu;
    double fvv = P.coef_solvent * lv;
    fvu = fvu + P.coef_polymeric * (dcxx_x + dcxy_y + 0.0);
    fvv = fvv + P.coef_polymeric * (dcxy_x + dcyy_y + 0.0);
    double bfu = ro * P.bfx;
    const double bfv = ro * P.bfy;
    if (a.fx) bfu = bfu + a.fx[i];
    double r_ro_ = r_ro;
    double r_rou = -tsu - P.csq * rx + bfu + fvu;
    double r_rov = -tsv - P.csq * ry + bfv + fvv;
    double r_xx, r_xy, r_yy;
    if (FORM == SV_FORM_LC) {
      const bool first = (STAGE == 1 || (STAGE == 0 && a.rk1)) && (C->itime == 1);
      rhs_logconf(u, v, ux, uy, vx, vy, s.pxx, s.pxy, s.pyy, q1x - s.pxx * sx,
                  q1y - s.pxx * sy, q2x - s.pxy * sx, q2y - s.pxy * sy, q3x - s.pyy * sx,
                  q3y - s.pyy * sy, first, P.eps, P.lambda, r_xx, r_xy, r_yy);
    } else {
      // calc_rhs_c (rhs_di.F90:417-475) with full gradients of cxx, cyy
      const double gcxx_y = ayx - cxx * sy, gcyy_x = bxy - cyy * sx;
      const double adxx = -(u * dcxx_x + v * gcxx_y + 0.0);
      const double adxy = -(u * dcxy_x + v * dcxy_y + 0.0);
      const double adyy = -(u * gcyy_x + v * dcyy_y + 0.0);
      const double ucxx = 2.0 * ux * cxx + 2.0 * uy * cxy + 0.0;
      const double ucxy = ux * cxy + uy * cyy + 0.0 + vx * cxx + vy * cxy + 0.0;
      const double ucyy = 2.0 * vx * cxy + 2.0 * vy * cyy + 0.0;
      const double fr = -(1.0 - P.eps * 2.0 + P.eps * (cxx + cyy + 1.0)) / P.lambda;
      double mxx = 0.0, mxy = 0.0, myy = 0.0;
      if (MDIFF) {
        mxx = P.Mdiff * (cxx_l - cxx * sl);
        mxy = P.Mdiff * (cxy_l - cxy * sl);
        myy = P.Mdiff * (cyy_l - cyy * sl);
      }
      r_xx = adxx + ucxx + fr * (cxx - 1.0) + mxx;
      r_xy = adxy + ucxy + fr * cxy + mxy;
      r_yy = adyy + ucyy + fr * (cyy - 1.0) + myy;
      if (a.tapeD) {
        double2 *T = reinterpret_cast<double2 *>(a.tapeD + (size_t)i * SV_TAPE_D);
        T[0] = double2{rx, ry}; T[1] = double2{ux, uy}; T[2] = double2{lu, vx};
        T[3] = double2{vy, lv}; T[4] = double2{dcxx_x, gcxx_y}; T[5] = double2{dcxy_x, dcxy_y};
        T[6] = double2{gcyy_x, dcyy_y}; T[7] = double2{0.0, 0.0};
        double2 *Q = reinterpret_cast<double2 *>(a.tapeG + (size_t)i * SV_US);
        Q[0] = double2{ro, u}; Q[1] = double2{v, cxx}; Q[2] = double2{cxy, cyy};
      }
    }
    if (BND) {
      const int jb = a.bidx[i];
      if (jb >= 0) {
        const double *br = a.brec + (size_t)SV_BREC * jb;
        bkind = (int)br[0];
        buin0 = br[3];
        const int s_rhs = STAGE == 0 ? 1 : STAGE;
        const bool first = (STAGE == 1 || (STAGE == 0 && a.rk1)) && (C->itime == 1);
        const double f1 = FORM == SV_FORM_LC ? s.pxx : cxx;
        const double f2 = FORM == SV_FORM_LC ? s.pxy : cxy;
        const double f3 = FORM == SV_FORM_LC ? s.pyy : cyy;
        bound_rhs<FORM>(P, bkind, br[1], br[2], uin_now(P, C, buin0, s_rhs), first, ro, u, v,
                        rx, ry, ux, uy, vx, vy, lu, lv, dcxx_x, dcxy_y, dcxy_x, dcyy_y, f1, f2,
                        f3, r_ro_, r_rou, r_rov, r_xx, r_xy, r_yy);
        if (FORM == SV_FORM_DI && MDIFF && bkind == 0) {
          // polymer diffusion on a wall (rhs_di.F90:396-413, :528-556): the
          // tangential second derivative of c only
          // (calc_laplacian_transverse_only_on_bound, derivatives.F90:329-339),
          // i.e. the wall Laplacian less its normal part ij_wb_grad2(1,:)
          // (labf.F90:594-598 plus the curvature term of :1011), plus the
          // one-sided term that removes the diffusive flux through the wall;
          // both over the four FD rows along the normal
          double fr[4][3];
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const Rec9 q = load_g<FORM>(a.G, (int)br[4 + k]);
            fr[k][0] = q.cxx; fr[k][1] = q.cxy; fr[k][2] = q.cyy;
          }
          const double dx = br[8], ooR = br[9], Lc = br[10];
          const double dx2 = dx * dx;
          const double wn[4] = {(-104.0 / 12.0 / dx2 + 4.0 / dx * ooR) / Lc / Lc,
                                (114.0 / 12.0 / dx2 + -3.0 / dx * ooR) / Lc / Lc,
                                (-56.0 / 12.0 / dx2 + (4.0 / 3.0) / dx * ooR) / Lc / Lc,
                                (11.0 / 12.0 / dx2 + -0.25 / dx * ooR) / Lc / Lc};
          const double wsum = wn[0] + wn[1] + wn[2] + wn[3];
          const double den = 72.0 * dx * dx * Lc * Lc;
          const double c0[3] = {cxx, cxy, cyy};
          const double lap[3] = {cxx_l - cxx * sl, cxy_l - cxy * sl, cyy_l - cyy * sl};
          double m[3];
#pragma unroll
          for (int q = 0; q < 3; q++) {
            const double n2 = wn[0] * fr[0][q] + wn[1] * fr[1][q] + wn[2] * fr[2][q] +
                              wn[3] * fr[3][q] - c0[q] * wsum;
            m[q] = (lap[q] - n2) + (-415.0 * c0[q] + 576.0 * fr[0][q] - 216.0 * fr[1][q] +
                                    64.0 * fr[2][q] - 9.0 * fr[3][q]) / den;
          }
          r_xx = r_xx + P.Mdiff * m[0];
          r_xy = r_xy + P.Mdiff * m[1];
          r_yy = r_yy + P.Mdiff * m[2];
        }
      }
    }
    // ---- RK update (step.F90:291-343, :375-409) ----
    const double rhs[6] = {r_ro_, r_rou, r_rov, r_xx, r_xy, r_yy};
    if (STAGE == 0) {
#pragma unroll
      for (int f = 0; f < 6; f++) a.rhs_out[(size_t)f * a.rhs_stride + i] = rhs[f];
    } else if (STAGE <= 3) {
      const double ra = C->RKa[STAGE - 1], rb = C->RKb[STAGE - 1], rm = C->RKbmbh[STAGE - 1];
      double eo[6], Un[6], ro_[6];
#pragma unroll
      for (int f = 0; f < 6; f++) {
        Un[f] = own.r1[f] + ra * rhs[f];
        ro_[f] = own.r1[f] + rb * rhs[f];
        eo[f] = (STAGE == 1 ? 0.0 : own.eo[f]) + rm * rhs[f];
      }
      store_u(a.reg_out, i, ro_);
      store_u(a.e, i, eo);
      if (BND && bkind >= 0) bound_apply(P, bkind, uin_now(P, C, buin0, STAGE + 1), Un);
      // derived fields for the next stage (step.F90:350-356)
      Rec9 g;
      const double ooro = 1.0 / Un[0];
      g.ro = Un[0];
      g.u = Un[1] * ooro;
      g.v = Un[2] * ooro;
      if (FORM == SV_FORM_LC) {
        g.pxx = Un[3]; g.pxy = Un[4]; g.pyy = Un[5];
        c_from_psi(Un[3], Un[4], Un[5], g.cxx, g.cxy, g.cyy);
      } else {
        g.cxx = Un[3]; g.cxy = Un[4]; g.cyy = Un[5];
        g.pxx = g.pxy = g.pyy = 0.0;
      }
      store_g<FORM>(a.Gout, i, g);
    } else {
      const double rb = C->RKb[3], rm = C->RKbmbh[3];
      double uo[6];
      const double nrm[6] = {1.0, P.err_norm_rou, P.err_norm_rou, 1.0, 1.0, 1.0};
#pragma unroll
      for (int f = 0; f < 6; f++) {
        uo[f] = own.r1[f] + rb * rhs[f];
        const double ef = own.eo[f] + rm * rhs[f];
        emax_loc = fmax(emax_loc, fabs(ef) * nrm[f]);
      }
      if (BND && bkind >= 0) bound_apply(P, bkind, uin_now(P, C, buin0, 5), uo);
      store_u(a.Uout, i, uo);
    }
  }
  return emax_loc;
}

// STAGE 1..4: RK stages; STAGE 0: write the right-hand side into rhs_out.
template <int FORM, int STAGE, bool MDIFF, bool BND>
__global__ __launch_bounds__(BS) void k_stage(StageArgs a) {
  const int bid = sv_logical_block(a.blist);
  const NodeRef nr = node_ref(a.blk_seg, a.seg, bid);
  const int ii = nr.ii;
  const bool act = nr.act;
  const int64_t b = a.off[ii >> 6] + (ii & 63);
  const int K = act ? a.kcnt[ii] : 0;
  double rx = 0, ry = 0, ux = 0, uy = 0, vx = 0, vy = 0, lu = 0, lv = 0;
  double axx = 0, ayx = 0, axy = 0, ayy = 0, bxy = 0, byy = 0;
  double cxx_l = 0, cxy_l = 0, cyy_l = 0;
  double q1x = 0, q1y = 0, q2x = 0, q2y = 0, q3x = 0, q3y = 0;
  auto accum = [&](const Rec9 &r, double wxk, double wyk, double wlk) {
    rx += r.ro * wxk; ry += r.ro * wyk;
    ux += r.u * wxk; uy += r.u * wyk; lu += r.u * wlk;
    vx += r.v * wxk; vy += r.v * wyk; lv += r.v * wlk;
    if (FORM == SV_FORM_LC) {
      axx += r.cxx * wxk;                         // calc_gradient_only(1,cxx)
      axy += r.cxy * wxk; ayy += r.cxy * wyk;     // calc_gradient(cxy)
      byy += r.cyy * wyk;                         // calc_gradient_only(2,cyy)
      q1x += r.pxx * wxk; q1y += r.pxx * wyk;
      q2x += r.pxy * wxk; q2y += r.pxy * wyk;
      q3x += r.pyy * wxk; q3y += r.pyy * wyk;
    } else {
      axx += r.cxx * wxk; ayx += r.cxx * wyk;
      axy += r.cxy * wxk; ayy += r.cxy * wyk;
      bxy += r.cyy * wxk; byy += r.cyy * wyk;
      if (MDIFF) { cxx_l += r.cxx * wlk; cxy_l += r.cxy * wlk; cyy_l += r.cyy * wlk; }
    }
  };
  // Links in pairs, as their weights lie (sv_w3): three 16-byte loads a pair (six
  // of 8 bytes at 16-byte strides: 863 us a step of 400x400 order 6 LC, 670 so),
  // the column indices of the next pair loaded before the current pair is
  // consumed, so each lane keeps two record gathers and the next index loads in
  // flight.  The pair at an odd list's end reads padding.  Summation stays
  // sequential in k.
  constexpr int U = 2;
  int jn[U];
#pragma unroll
  for (int u = 0; u < U; u++) jn[u] = (u < K) ? ld_stream(a.col + b + (int64_t)u * SV_WAVE) : ii;
  for (int k = 0; k < K; k += U) {
    Rec9 r[U];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k + u < K) r[u] = load_g<FORM>(a.G, jn[u]);
    const dbl2 *w = reinterpret_cast<const dbl2 *>(a.w3 + sv_w3(b + (int64_t)k * SV_WAVE, 0));
    const dbl2 wg[U] = {ld_stream(w), ld_stream(w + SV_WAVE)};
    const dbl2 wl = ld_stream(w + 2 * SV_WAVE);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kn = k + U + u;
      jn[u] = (kn < K) ? ld_stream(a.col + b + (int64_t)kn * SV_WAVE) : ii;
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k + u < K) accum(r[u], wg[u].x, wg[u].y, u ? wl.y : wl.x);
  }
  double emax_loc = 0.0;
  if (act) {
    const Sums S{rx, ry, ux, uy, vx, vy, lu, lv, axx, ayx, axy, ayy, bxy, byy, cxx_l, cxy_l, cyy_l, q1x, q1y, q2x, q2y, q3x, q3y};
    emax_loc = stage_point<FORM, STAGE, MDIFF, BND>(a, nr, S, load_own<FORM, STAGE>(a, nr.i),
                                                   a.ctrl + nr.sg);
  }
  if (STAGE == 4) {
    emax_loc = wave_max(emax_loc);
    if ((threadIdx.x & 63) == 0) a.partial[nr.i >> 6] = emax_loc;
  }
}

// ---- halo-staged sweeps ---------------------------------------------------
// A workgroup of NB threads (one per slot of its halo block) first copies the
// gather records of its halo (the distinct neighbours of its nodes: 2.3 per
// node at 256 slots, 3.0 at 128, 4.0 at 64 on an order-6 lattice) into LDS,
// then every link reads its record from LDS by a 16-bit block-local index.
// What bounds it, by size (LC order 6, one RK stage with its launch):
//   1M nodes    HBM: 2.47 GB in 421-439 us, 5.7 TB/s (a plain read of that
//               size reaches 6.95 TB/s non-temporally, a copy 6.2)
//   68k nodes   31 us (40 with 256-slot workgroups and one request pair in
//               flight): one or two waves per SIMD, memory latency and the
//               random LDS reads (50 clocks a link of a wave for 72 bytes a
//               lane, 36 without bank conflicts)
//   16k nodes   11.5 us (34; 14 with one wave per slice): the chain launch ->
//               layout -> keys -> records -> LDS -> links -> pointwise part
// Up to 32768 nodes NW wavefronts walk the links of a slice, each for its own
// fields (flow; conformation; psi), so that every sum keeps the links' order
// and the values do not depend on the split; more threads stage the halo, and
// wave 0 requests the node's own values before it, for the pointwise part that
// it does alone.
// LDS records are the gather records as they are: 10 doubles (80 B, the last
// one a pad) for LC, 6 for DI (48 B), read 16 bytes at a time.  Both strides
// are odd multiples of 16 bytes, so the records' starts spread over all LDS
// banks (64-byte records all start on one of four bank groups).
template <int FORM>
struct HaloL {
  static constexpr int RS = FORM == SV_FORM_LC ? SV_GS_LC : SV_GS_DI;
  static constexpr int BYTES = 8 * RS;
};
// sums handed to wave 0 where the fields of a slice are shared by several waves
constexpr int PARTS_CONF = 9, PARTS_PSI = 6;
template <int FORM>
constexpr int stage_waves() { return FORM == SV_FORM_LC ? 3 : 2; }
static_assert(HaloL<SV_FORM_LC>::BYTES == SV_HALO_REC, "the halo budget counts LC records");


template <int FORM, int STAGE, bool MDIFF, bool BND, int NB, bool NT, int NW>
__global__ __launch_bounds__(NB * NW) void k_stage_h(StageArgs a) {
  extern __shared__ double hl[];
  const int bid = logical_wg<NB>(a.blist);
  // the layout's arrays cover whole blocks (no links past the last node), so
  // nothing of the streams waits for the segment
  const int slot = bid * NB + (int)threadIdx.x % NB;
  const int slice = __builtin_amdgcn_readfirstlane(slot >> 6);
  const int w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NB);
  const int K = a.kcnt[slot];
  const int KF = a.krange[slice].x, KM = a.krange[slice].y;
  const int64_t o = a.off[slice];
  const int64_t h0 = a.hoff[bid];
  const int nh = (int)(a.hoff[bid + 1] - h0);
  const NodeRef nr = node_ref<NB>(a.blk_seg, a.seg, bid);
  const bool act = nr.act;
  double rx = 0, ry = 0, ux = 0, uy = 0, vx = 0, vy = 0, lu = 0, lv = 0;
  double axx = 0, ayx = 0, axy = 0, ayy = 0, bxy = 0, byy = 0;
  double cxx_l = 0, cxy_l = 0, cyy_l = 0;
  double q1x = 0, q1y = 0, q2x = 0, q2y = 0, q3x = 0, q3y = 0;
  constexpr int U = HaloU<NB>::U;
  const Stream<uint32_t, 1, NT> sc(a.lcol + o, KM);
  const Stream<dbl2, 3, NT> sw(a.w3 + 3 * o, KM);
  uint32_t jc[2][U];
  dbl2 wg[2][2 * U], wl[2][U];   // d/dx and d/dy of a link; Laplacian of a pair
  const bool laps = w == 0 || MDIFF;   // this wave's sums hold Laplacians
  auto load = [&](int s, int u, int p) {
    jc[s][u] = sc.at(p, u, 0);
    wg[s][2 * u] = sw.at(p, u, 0); wg[s][2 * u + 1] = sw.at(p, u, 1);
    wl[s][u] = sw.at(NW == 1 || laps ? p : OUT_OF_RANGE, u, 2);
  };
  auto rec = [&](int s, int l) {
    return hl + (size_t)HaloL<FORM>::RS * (l & 1 ? jc[s][l / 2] >> 16 : jc[s][l / 2] & 0xffff);
  };
  // the sums of the momentum and mass balances, of the conformation and of psi
  auto link_flow = [&](double ro, double u, double v, int s, int l) {
    const double wx_ = wg[s][l].x, wy_ = wg[s][l].y;
    const double wl_ = l & 1 ? wl[s][l / 2].y : wl[s][l / 2].x;
    rx += ro * wx_; ry += ro * wy_;
    ux += u * wx_; uy += u * wy_; lu += u * wl_;
    vx += v * wx_; vy += v * wy_; lv += v * wl_;
  };
  auto link_conf = [&](double cxx, double cxy, double cyy, int s, int l) {
    const double wx_ = wg[s][l].x, wy_ = wg[s][l].y;
    axx += cxx * wx_;
    axy += cxy * wx_; ayy += cxy * wy_;
    byy += cyy * wy_;
    if (FORM == SV_FORM_DI) {
      ayx += cxx * wy_;
      bxy += cyy * wx_;
      if (MDIFF) {
        const double wl_ = l & 1 ? wl[s][l / 2].y : wl[s][l / 2].x;
        cxx_l += cxx * wl_; cxy_l += cxy * wl_; cyy_l += cyy * wl_;
      }
    }
  };
  auto link_psi = [&](double pxx, double pxy, double pyy, int s, int l) {
    const double wx_ = wg[s][l].x, wy_ = wg[s][l].y;
    q1x += pxx * wx_; q1y += pxx * wy_;
    q2x += pxy * wx_; q2y += pxy * wy_;
    q3x += pyy * wx_; q3y += pyy * wy_;
  };
  // the halo's keys first, then the first batch of links, in flight while the
  // halo is staged
  const int *hx = a.hidx + h0;
  HaloKeys<NB, NB * NW> keys;
  if (nh > 0) keys.get(hx, threadIdx.x, nh);
  __builtin_amdgcn_sched_barrier(0);
  const int p0 = entry_at(0);
#pragma unroll
  for (int u = 0; u < U; u++) load(0, u, 2 * u < K ? p0 : OUT_OF_RANGE);
  Own own;
  if (NW > 1 && w == 0) own = load_own<FORM, STAGE>(a, nr.ii);
  // the step's control values, made here by every workgroup (small node sets)
  constexpr bool DT = NW > 1 && STAGE == 1;
  Partials lim;
  if (DT && w == 0) lim.load(a.seg[nr.sg], a.pcfl, a.pvisc, 1.0e10, 1.0e10);
  halo_stage<NB, NB * NW>(
      hx, nh, keys, [&](int j) { return load_g<FORM>(a.G, j); },
      [&](int h, int fl, Rec9 r) {
        if (fl) {   // mirror ghost (reapply_mirror_bcs, mirror_boundaries.F90:285-340)
          if (fl != 2) r.u = -r.u;
          if (fl != 1) r.v = -r.v;
          if (fl != 3) { r.cxy = -r.cxy; r.pxy = -r.pxy; }
        }
        store_g<FORM>(hl, h, r);
      });
  __syncthreads();
  if (NW == 1) {
    walk_links<U, Rec9>(
        K, KF, KM, load, [&](int s, int l) { return load_g<FORM>(rec(s, l), 0); },
        [&](const Rec9 &q, int s, int l) {
          link_flow(q.ro, q.u, q.v, s, l);
          link_conf(q.cxx, q.cxy, q.cyy, s, l);
          if (FORM == SV_FORM_LC) link_psi(q.pxx, q.pxy, q.pyy, s, l);
        });
    own = load_own<FORM, STAGE>(a, nr.ii);
  } else {
    // each wave its own fields of every link: the sums keep the links' order
    struct Rec3 {
      double2 a;
      double b;
    };
    auto pair_first = [&](int s, int l, int q) {   // two values, aligned, then one
      const double *r = rec(s, l) + q;
      return Rec3{*reinterpret_cast<const double2 *>(r), r[2]};
    };
    auto pair_last = [&](int s, int l) {           // cxx, then cxy and cyy
      const double *r = rec(s, l) + SV_G_CXX;
      return Rec3{*reinterpret_cast<const double2 *>(r + 1), r[0]};
    };
    auto conf = [&](auto &&f) {
      f(axx); f(axy); f(ayy); f(byy);
      if (FORM == SV_FORM_DI) { f(ayx); f(bxy); }
      if (MDIFF) { f(cxx_l); f(cxy_l); f(cyy_l); }
    };
    auto psi = [&](auto &&f) { f(q1x); f(q1y); f(q2x); f(q2y); f(q3x); f(q3y); };
    if (w == 0)
      walk_links<U, Rec3>(
          K, KF, KM, load, [&](int s, int l) { return pair_first(s, l, 0); },
          [&](const Rec3 &q, int s, int l) { link_flow(q.a.x, q.a.y, q.b, s, l); });
    else if (w == 1)
      walk_links<U, Rec3>(
          K, KF, KM, load, pair_last,
          [&](const Rec3 &q, int s, int l) { link_conf(q.b, q.a.x, q.a.y, s, l); });
    else if (FORM == SV_FORM_LC)
      walk_links<U, Rec3>(
          K, KF, KM, load, [&](int s, int l) { return pair_first(s, l, SV_G_PXX); },
          [&](const Rec3 &q, int s, int l) { link_psi(q.a.x, q.a.y, q.b, s, l); });
    double *psums = hl + part_doubles(PARTS_CONF);
    __syncthreads();   // the halo has been read
    if (w == 1) give_sums(hl, conf);
    if (FORM == SV_FORM_LC && w == 2) give_sums(psums, psi);
    __syncthreads();
    if (w > 0) return;
    take_sums(hl, conf);
    if (FORM == SV_FORM_LC) take_sums(psums, psi);
  }
  const sv_ctrl *C = a.ctrl + nr.sg;
  sv_ctrl cn;
  if (DT) {
    const sv_segk &S = a.seg[nr.sg];
    copy_ctrl(*C, cn);
    next_dt(S.pk, min_partials(lim.a), min_partials(lim.b), cn);
    if (nr.i == S.base) copy_ctrl(cn, a.ctrl_out[nr.sg]);
    C = &cn;
  }
  double emax_loc = 0.0;
  if (act) {
    const Sums S{rx, ry, ux, uy, vx, vy, lu, lv, axx, ayx, axy, ayy, bxy, byy, cxx_l, cxy_l,
                 cyy_l, q1x, q1y, q2x, q2y, q3x, q3y};
    emax_loc = stage_point<FORM, STAGE, MDIFF, BND>(a, nr, S, own, C);
  }
  if (STAGE == 4) {
    emax_loc = wave_max(emax_loc);
    if ((threadIdx.x & 63) == 0) a.partial[nr.i >> 6] = emax_loc;
  }
}

struct FilterArgs {
  const int *blk_seg;
  const sv_segk *seg;
  const int64_t *off;
  const int *kcnt;
  const int *col;
  const double *wh, *hsum, *vol;
  const double *U;   // gathered state records
  double *Uf;        // filtered state records
  double *partial;       // sum of (ro_f - rho_char)*vol per slice
  const int4 *krange;    // links per slice (sv_loopl)
  const int64_t *hoff;   // per-block halos (k_filter_h)
  const int *hidx;
  const uint16_t *lcol;
  const int *blist;       // launch group's logical blocks (nullable: all blocks)
};

// A node's own values in the filter
struct OwnF {
  double f[6], hs, vol;
};

__device__ __forceinline__ OwnF load_own(const FilterArgs &a, int i) {
  OwnF o;
  load_u(a.U, i, o.f);
  o.hs = a.hsum[i];
  o.vol = a.vol[i];
  return o;
}

// Pointwise part of the filter for one node: the filtered record and its
// mass-correction term.
__device__ __forceinline__ double filter_point(const FilterArgs &a, const NodeRef &nr,
                                               const double t[6], const OwnF &o) {
  double g[6];
#pragma unroll
  for (int q = 0; q < 6; q++) g[q] = o.f[q] + (t[q] - o.f[q] * o.hs);
  store_u(a.Uf, nr.i, g);
  return (g[0] - a.seg[nr.sg].pk.rho_char) * o.vol;
}

__global__ __launch_bounds__(BS) void k_filter(FilterArgs a) {
  const int bid = sv_logical_block(a.blist);
  const NodeRef nr = node_ref(a.blk_seg, a.seg, bid);
  const int ii = nr.ii;
  const bool act = nr.act;
  const int64_t b = a.off[ii >> 6] + (ii & 63);
  const int K = act ? a.kcnt[ii] : 0;
  double t[6] = {0, 0, 0, 0, 0, 0};
  // pairs of links with the next pair's column indices prefetched, as k_stage
  constexpr int U = 2;
  int jn[U];
#pragma unroll
  for (int u = 0; u < U; u++) jn[u] = (u < K) ? ld_stream(a.col + b + (int64_t)u * SV_WAVE) : ii;
  for (int k = 0; k < K; k += U) {
    double f[U][6];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k + u < K) load_u(a.U, jn[u], f[u]);
    const dbl2 w = ld_stream(
        reinterpret_cast<const dbl2 *>(a.wh + sv_pair(b + (int64_t)k * SV_WAVE)));
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int kn = k + U + u;
      jn[u] = (kn < K) ? ld_stream(a.col + b + (int64_t)kn * SV_WAVE) : ii;
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k + u < K) {
#pragma unroll
        for (int q = 0; q < 6; q++) t[q] += f[u][q] * (u ? w.y : w.x);
      }
  }
  const double m = wave_sum(act ? filter_point(a, nr, t, load_own(a, nr.i)) : 0.0);
  if ((threadIdx.x & 63) == 0) a.partial[nr.i >> 6] = m;
}

// Halo-staged form of k_filter (see k_stage_h): the block's neighbour state
// records (6 doubles) go to LDS once, links read them by block-local index.
template <int NB, bool NT>
__global__ __launch_bounds__(NB) void k_filter_h(FilterArgs a) {
  extern __shared__ double hl[];
  const int bid = logical_wg<NB>(a.blist);
  const int slot = bid * NB + (int)threadIdx.x;   // as k_stage_h
  const int slice = __builtin_amdgcn_readfirstlane(slot >> 6);
  const int K = a.kcnt[slot];
  const int KF = a.krange[slice].z, KM = a.krange[slice].w;
  const int64_t o = a.off[slice];
  const int64_t h0 = a.hoff[bid];
  const int nh = (int)(a.hoff[bid + 1] - h0);
  const NodeRef nr = node_ref<NB>(a.blk_seg, a.seg, bid);
  const bool act = nr.act;
  double t[6] = {0, 0, 0, 0, 0, 0};
  constexpr int U = HaloU<NB>::UF;
  const Stream<uint32_t, 1, NT> sc(a.lcol + o, KM);
  const Stream<dbl2, 1, NT> sw(a.wh + o, KM);
  uint32_t jc[2][U];
  dbl2 wf[2][U];
  auto load = [&](int s, int u, int p) {
    jc[s][u] = sc.at(p, u, 0);
    wf[s][u] = sw.at(p, u, 0);
  };
  struct Rec6 {
    double2 d0, d1, d2;
  };
  const int *hx = a.hidx + h0;   // keys, first links, halo: as k_stage_h
  HaloKeys<NB, NB> keys;
  if (nh > 0) keys.get(hx, threadIdx.x, nh);
  __builtin_amdgcn_sched_barrier(0);
  const int p0 = entry_at(0);
#pragma unroll
  for (int u = 0; u < U; u++) load(0, u, 2 * u < K ? p0 : OUT_OF_RANGE);
  halo_stage<NB, NB>(
      hx, nh, keys,
      [&](int j) {
        const double2 *q = reinterpret_cast<const double2 *>(a.U + (size_t)j * SV_US);
        return Rec6{q[0], q[1], q[2]};
      },
      [&](int h, int fl, Rec6 r) {
        if (fl) {   // mirror ghost: rho u, rho v and the xy component
          if (fl != 2) r.d0.y = -r.d0.y;
          if (fl != 1) r.d1.x = -r.d1.x;
          if (fl != 3) r.d2.x = -r.d2.x;
        }
        double2 *d = reinterpret_cast<double2 *>(hl + h * 6);
        d[0] = r.d0; d[1] = r.d1; d[2] = r.d2;
      });
  __syncthreads();
  walk_links<U, Rec6>(
      K, KF, KM, load,
      [&](int s, int l) {
        const int j = (int)(l & 1 ? jc[s][l / 2] >> 16 : jc[s][l / 2] & 0xffff);
        const double2 *d = reinterpret_cast<const double2 *>(hl + j * 6);
        return Rec6{d[0], d[1], d[2]};
      },
      [&](const Rec6 &q, int s, int l) {
        const double w = l & 1 ? wf[s][l / 2].y : wf[s][l / 2].x;
        t[0] += q.d0.x * w; t[1] += q.d0.y * w; t[2] += q.d1.x * w;
        t[3] += q.d1.y * w; t[4] += q.d2.x * w; t[5] += q.d2.y * w;
      });
  const double m = wave_sum(act ? filter_point(a, nr, t, load_own(a, nr.ii)) : 0.0);
  if ((threadIdx.x & 63) == 0) a.partial[nr.i >> 6] = m;
}

// mass correction value, emax and the end-of-step counters; one block per
// segment over that segment's per-slice partials
__global__ __launch_bounds__(1024) void k_reduce(const sv_segk *seg, const double *pmass,
                                                 const double *perr, sv_ctrl *ctrl_all) {
  __shared__ double s1[1024], s2[1024];
  const sv_segk &S = seg[blockIdx.x];
  sv_ctrl *ctrl = ctrl_all + blockIdx.x;
  double a = 0.0, m = 0.0;
  // a thread takes the four slices of a block at a time
  static_assert(SPB == 4, "two double2 per block");
  const double2 *pm = reinterpret_cast<const double2 *>(pmass) + 2 * (size_t)S.blk0;
  const double2 *pe = reinterpret_cast<const double2 *>(perr) + 2 * (size_t)S.blk0;
#pragma unroll 4
  for (int k = threadIdx.x; k < S.nblk; k += 1024) {
    const double2 m0 = pm[2 * k], m1 = pm[2 * k + 1], e0 = pe[2 * k], e1 = pe[2 * k + 1];
    a += (m0.x + m0.y) + (m1.x + m1.y);
    m = fmax(fmax(fmax(m, e0.x), fmax(e0.y, e1.x)), e1.y);
  }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = m;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      s1[threadIdx.x] += s1[threadIdx.x + s];
      s2[threadIdx.x] = fmax(s2[threadIdx.x], s2[threadIdx.x + s]);
    }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  end_step(S, s1[0], s2[0], *ctrl);
}

struct ApplyArgs {
  const int *blk_seg;
  const sv_segk *seg;
  const double *Uf;
  double *U;
  double *G;
  const double *s;
  const sv_ctrl *ctrl;   // ctrl[sg].dro is subtracted; nullptr for no correction
  double *pcfl, *pvisc;  // minima for set_tstep per slice
  const int *bidx;       // boundary nodes (nullable), as StageArgs
  const double *brec;
  const double *pmass, *perr;   // REDUCE: partial results, control values (StageArgs)
  sv_ctrl *ctrl_out;
};

// rho -= drho (rhs_lc.F90:887-889); the gather record: u = rou/rho
// (step.F90:514-529), psi and c = exp(psi) (LC); set_tstep partial minima
// (step.F90:579-602).  The record is written here as a whole (the filter
// writing psi and c and this kernel ro, u, v made two partial writes of
// every line).
// REDUCE: the end of the step as well (k_reduce's work), by every wavefront of
// a small node set.
template <int FORM, bool REDUCE>
__global__ __launch_bounds__(BS) void k_apply_state(ApplyArgs a) {
  const NodeRef nr = node_ref(a.blk_seg, a.seg, sv_xcd_block());
  const int i = nr.i;
  const sv_ctrl *C = a.ctrl ? a.ctrl + nr.sg : nullptr;
  double dro = 0.0;
  if (REDUCE) {
    const sv_segk &S = a.seg[nr.sg];
    Partials p;
    p.load(S, a.pmass, a.perr, 0.0, 0.0);
    const double mass = sum_partials(p.a);
    dro = mass / S.volsum;
    if (i - (int)threadIdx.x == S.base) {   // the segment's first block
      const double err = max_partials(p.b);
      if (threadIdx.x == 0) {
        sv_ctrl n;
        copy_ctrl(*C, n);
        end_step(S, mass, err, n);
        copy_ctrl(n, a.ctrl_out[nr.sg]);
      }
    }
  } else if (C) {
    dro = C->dro;
  }
  double mc = 1.0e10, mv = 1.0e10;
  if (nr.act) {
    const sv_physk &P = a.seg[nr.sg].pk;
    double f[6];
    load_u(a.Uf, i, f);
    f[0] = f[0] - dro;
    int bk = -1;
    if (a.bidx) {
      const int jb = a.bidx[i];
      if (jb >= 0) {
        const double *br = a.brec + (size_t)SV_BREC * jb;
        bk = (int)br[0];
        // the apply after filter_variables (step.F90:498)
        // (the values of the step that has just ended)
        if (C) bound_apply(P, bk, uin_now(P, C, br[3], REDUCE ? 5 : 1), f);
      }
    }
    store_u(a.U, i, f);
    const double ooro = 1.0 / f[0];
    const double u = f[1] * ooro, v = f[2] * ooro;
    Rec9 g;
    g.ro = f[0]; g.u = u; g.v = v;
    if (FORM == SV_FORM_LC) {
      g.pxx = f[3]; g.pxy = f[4]; g.pyy = f[5];
      c_from_psi(f[3], f[4], f[5], g.cxx, g.cxy, g.cyy);
    } else {
      g.cxx = f[3]; g.cxy = f[4]; g.cyy = f[5];
    }
    store_g<FORM>(a.G, i, g);
    const double um = sqrt(u * u + v * v + 0.0);
    const double si = a.s[i];
    // slightly smaller on outflows (step.F90:591-595)
    mc = bk == 2 ? 0.8 * si / (um + P.cs) : si / (um + P.cs);
    mv = si * si * f[0] / P.visc_total;
  }
  mc = wave_min(mc);
  mv = wave_min(mv);
  if ((threadIdx.x & 63) == 0) { a.pcfl[i >> 6] = mc; a.pvisc[i >> 6] = mv; }
}

// the next step's control values; one block per segment
__global__ __launch_bounds__(1024) void k_dt(const sv_segk *seg, const double *pcfl,
                                             const double *pvisc, sv_ctrl *ctrl_all) {
  __shared__ double s1[1024], s2[1024];
  const sv_segk &S = seg[blockIdx.x];
  sv_ctrl *c = ctrl_all + blockIdx.x;
  double a = 1.0e10, m = 1.0e10;
  const double2 *p = reinterpret_cast<const double2 *>(pcfl) + 2 * (size_t)S.blk0;
  const double2 *q = reinterpret_cast<const double2 *>(pvisc) + 2 * (size_t)S.blk0;
#pragma unroll 4
  for (int k = threadIdx.x; k < S.nblk; k += 1024) {
    const double2 p0 = p[2 * k], p1 = p[2 * k + 1], q0 = q[2 * k], q1 = q[2 * k + 1];
    a = fmin(fmin(fmin(a, p0.x), fmin(p0.y, p1.x)), p1.y);
    m = fmin(fmin(fmin(m, q0.x), fmin(q0.y, q1.x)), q1.y);
  }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = m;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      s1[threadIdx.x] = fmin(s1[threadIdx.x], s1[threadIdx.x + s]);
      s2[threadIdx.x] = fmin(s2[threadIdx.x], s2[threadIdx.x + s]);
    }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  next_dt(S.pk, s1[0], s2[0], *c);
}

StageArgs stage_args(sv_ctx *c, int stage, const double *Gin, double *Gout) {
  StageArgs a{};
  a.rhs_stride = c->npfb;
  a.blk_seg = c->blk_seg;
  a.seg = c->segk;
  a.off = c->L.off;
  a.kcnt = c->L.cnt_small;
  a.col = c->L.col;
  a.w3 = c->L.w3;
  a.gsx = c->L.gsx; a.gsy = c->L.gsy; a.lsum = c->L.lsum;
  a.G = Gin;
  a.reg_in = (stage == 1) ? c->U : c->reg;
  a.reg_out = c->reg;
  a.e = c->eacc;
  a.Uout = c->U;
  a.Gout = Gout;
  a.fx = c->any_forcing ? c->fx : nullptr;
  a.ctrl = c->ctrl;
  a.krange = c->L.krange;
  a.hoff = c->L.hoff;
  a.hidx = c->L.hidx;
  a.lcol = c->L.lcol;
  a.partial = c->partial;
  a.bidx = c->L.bidx;
  a.brec = c->L.brec;
  return a;
}

// nb: 256-slot blocks of the launch
template <int FORM, int STAGE, bool MDIFF, bool BND>
void launch_sweep(sv_ctx *c, const StageArgs &a, int nb, int hmax) {
  if (!c->L.halo) {
    k_stage<FORM, STAGE, MDIFF, BND><<<nb, BS, 0, c->stream>>>(a);
    return;
  }
  size_t shm = (size_t)hmax * HaloL<FORM>::BYTES;
  const int hb = c->L.hb, grid = nb * (BS / hb);
  if (hb == 64 && c->L.split) {
    constexpr int NW = stage_waves<FORM>();
    shm = std::max(shm, sizeof(double) * part_doubles(PARTS_CONF + PARTS_PSI));
    k_stage_h<FORM, STAGE, MDIFF, BND, 64, false, NW><<<grid, 64 * NW, shm, c->stream>>>(a);
  } else if (hb == 64)
    k_stage_h<FORM, STAGE, MDIFF, BND, 64, false, 1><<<grid, 64, shm, c->stream>>>(a);
  else if (hb == 128 && !c->L.nt)
    k_stage_h<FORM, STAGE, MDIFF, BND, 128, false, 1><<<grid, 128, shm, c->stream>>>(a);
  else if (hb == 128)
    k_stage_h<FORM, STAGE, MDIFF, BND, 128, true, 1><<<grid, 128, shm, c->stream>>>(a);
  else
    k_stage_h<FORM, STAGE, MDIFF, BND, 256, true, 1><<<grid, 256, shm, c->stream>>>(a);
}

template <int FORM, int STAGE>
void launch_stage_grid(sv_ctx *c, const StageArgs &a, int nb, int hmax) {
  const bool bnd = a.bidx != nullptr;
  if (FORM == SV_FORM_DI && c->any_mdiff) {
    if (bnd) launch_sweep<FORM, STAGE, FORM == SV_FORM_DI, true>(c, a, nb, hmax);
    else launch_sweep<FORM, STAGE, FORM == SV_FORM_DI, false>(c, a, nb, hmax);
  } else {
    if (bnd) launch_sweep<FORM, STAGE, false, true>(c, a, nb, hmax);
    else launch_sweep<FORM, STAGE, false, false>(c, a, nb, hmax);
  }
}

// One stage over every block: one launch, or one launch per ensemble launch
// group, each with its own halo budget (its blocks' largest halo).
template <int FORM, int STAGE>
void launch_stage(sv_ctx *c, const StageArgs &a, int nb) {
  if (c->lgroup_mode == 1 && !c->lgroups.empty()) {
    for (const sv_ctx::lgroup &g : c->lgroups) {
      StageArgs b = a;
      b.blist = g.blist;
      launch_stage_grid<FORM, STAGE>(c, b, g.nblk, g.hmax);
    }
    return;
  }
  launch_stage_grid<FORM, STAGE>(c, a, nb, c->L.hmax);
}

void launch_filter_grid(sv_ctx *c, const FilterArgs &f, int nb, int hmax) {
  const size_t shm = sizeof(double) * 6 * (size_t)hmax;
  const int hb = c->L.hb, grid = nb * (BS / hb);
  if (hb == 64) k_filter_h<64, false><<<grid, 64, shm, c->stream>>>(f);
  else if (hb == 128 && !c->L.nt) k_filter_h<128, false><<<grid, 128, shm, c->stream>>>(f);
  else if (hb == 128) k_filter_h<128, true><<<grid, 128, shm, c->stream>>>(f);
  else k_filter_h<256, true><<<grid, 256, shm, c->stream>>>(f);
}

void launch_filter(sv_ctx *c, const FilterArgs &f, int nb) {
  if (!c->L.halo) {
    k_filter<<<nb, BS, 0, c->stream>>>(f);
    return;
  }
  if (c->lgroup_mode == 1 && !c->lgroups.empty()) {
    for (const sv_ctx::lgroup &g : c->lgroups) {
      FilterArgs b = f;
      b.blist = g.blist;
      launch_filter_grid(c, b, g.nblk, g.hmax);
    }
    return;
  }
  launch_filter_grid(c, f, nb, c->L.hmax);
}

// ev (nullable): SV_NKERNELS+1 events recorded between the launches of one step
template <int FORM>
int step_form(sv_ctx *c, hipEvent_t *ev, double *const *tape) {
  const int nb = c->nblk;
  const size_t np = (size_t)nb * SPB;   // partial results of one kind
  double *pm = c->partial, *pe = pm + np, *pc = pm + 2 * np, *pv = pm + 3 * np;
  int ke = 0;
  auto mark = [&]() {
    if (ev) (void)hipEventRecord(ev[ke++], c->stream);
  };
  // small node sets: stage 1 makes the step's control values in the second
  // array and the last kernel the next ones in the first
  const bool small = c->L.halo && c->L.split && nb <= SMALL_BLOCKS;
  sv_ctrl *cs = small ? c->ctrl + c->nseg : c->ctrl;
  mark();
  if (!small) k_dt<<<c->nseg, 1024, 0, c->stream>>>(c->segk, pc, pv, c->ctrl);
  mark();
  StageArgs as[4] = {stage_args(c, 1, c->GA, c->GB), stage_args(c, 2, c->GB, c->GA),
                     stage_args(c, 3, c->GA, c->GB), stage_args(c, 4, c->GB, c->GA)};
  as[3].partial = pe;
  as[0].pcfl = pc;
  as[0].pvisc = pv;
  as[0].ctrl_out = cs;
  for (int k = 1; k < 4; k++) as[k].ctrl = cs;
  if (tape)
    for (int k = 0; k < 4; k++) { as[k].tapeG = tape[2 * k]; as[k].tapeD = tape[2 * k + 1]; }
  launch_stage<FORM, 1>(c, as[0], nb);
  mark();
  launch_stage<FORM, 2>(c, as[1], nb);
  mark();
  launch_stage<FORM, 3>(c, as[2], nb);
  mark();
  launch_stage<FORM, 4>(c, as[3], nb);
  mark();
  FilterArgs f{};
  f.blk_seg = c->blk_seg;
  f.seg = c->segk;
  f.off = c->L.off;
  f.kcnt = c->L.cnt;
  f.col = c->L.col;
  f.wh = c->L.wh;
  f.hsum = c->L.hsum;
  f.vol = c->L.vol;
  f.U = c->U;
  f.Uf = c->Uf;
  f.partial = pm;
  f.krange = c->L.krange;
  f.hoff = c->L.hoff;
  f.hidx = c->L.hidx;
  f.lcol = c->L.lcol;
  launch_filter(c, f, nb);
  mark();
  if (!small) k_reduce<<<c->nseg, 1024, 0, c->stream>>>(c->segk, pm, pe, c->ctrl);
  mark();
  ApplyArgs ap{};
  ap.blk_seg = c->blk_seg;
  ap.seg = c->segk;
  ap.Uf = c->Uf;
  ap.U = c->U;
  ap.G = c->GA;
  ap.s = c->L.s;
  ap.ctrl = cs;
  ap.pmass = pm;
  ap.perr = pe;
  ap.ctrl_out = c->ctrl;
  ap.pcfl = pc;
  ap.pvisc = pv;
  ap.bidx = c->L.bidx;
  ap.brec = c->L.brec;
  if (small) k_apply_state<FORM, true><<<nb, BS, 0, c->stream>>>(ap);
  else k_apply_state<FORM, false><<<nb, BS, 0, c->stream>>>(ap);
  mark();
  SV_HIP(c, hipGetLastError());
  return 0;
}

}  // namespace

int sv_dev_init_state(sv_ctx *c) {
  // gather records and the set_tstep partial minima of the current state (no
  // correction)
  const int nb = c->nblk;
  ApplyArgs ap{};
  ap.blk_seg = c->blk_seg;
  ap.seg = c->segk;
  ap.Uf = c->U;
  ap.U = c->U;
  ap.G = c->GA;
  ap.s = c->L.s;
  ap.ctrl = nullptr;
  ap.pcfl = c->partial + 2 * (size_t)nb * SPB;
  ap.pvisc = c->partial + 3 * (size_t)nb * SPB;
  ap.bidx = c->L.bidx;
  ap.brec = c->L.brec;
  if (c->cfg.form == SV_FORM_LC) k_apply_state<SV_FORM_LC, false><<<nb, BS, 0, c->stream>>>(ap);
  else k_apply_state<SV_FORM_DI, false><<<nb, BS, 0, c->stream>>>(ap);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}

int sv_dev_step(sv_ctx *c, hipEvent_t *ev) {
  return c->cfg.form == SV_FORM_LC ? step_form<SV_FORM_LC>(c, ev, nullptr)
                                   : step_form<SV_FORM_DI>(c, ev, nullptr);
}

int sv_dev_step_tape(sv_ctx *c, double *const tape[8]) {
  if (c->cfg.form != SV_FORM_DI) return sv_fail(c, SV_E_STATE, "the tape is DI-only");
  return step_form<SV_FORM_DI>(c, nullptr, tape);
}

// calc_all_rhs on the current state (interior nodes): the stage kernel in its
// right-hand-side-only form, written into the six arrays of out6 (npfb each).
int sv_dev_rhs(sv_ctx *c, int iRKstep, double *out6, double *tapeG, double *tapeD) {
  const int nb = c->nblk;
  StageArgs a = stage_args(c, 1, c->GA, c->GB);
  a.rk1 = (iRKstep == 1);
  a.rhs_out = out6;
  a.tapeG = tapeG;
  a.tapeD = tapeD;
  if (c->cfg.form == SV_FORM_LC) launch_stage<SV_FORM_LC, 0>(c, a, nb);
  else launch_stage<SV_FORM_DI, 0>(c, a, nb);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}

// Launch-group autotuning of an ensemble: the right-hand-side-only form of the
// stage sweep (it leaves the state untouched) timed over every block, one
// launch against one launch per group, reps times each after a warm-up; the
// faster mode is kept.
int sv_dev_tune_groups(sv_ctx *c, int reps) {
  if (c->lgroups.size() < 2) { c->lgroup_mode = 0; return 0; }
  DevTmp<double> out;
  SV_HIP(c, out.alloc(c, 6 * (size_t)c->ntot));
  EventTmp e0, e1;
  SV_HIP(c, e0.create());
  SV_HIP(c, e1.create());
  float ms[2] = {0.0f, 0.0f};
  for (int mode = 0; mode < 2; mode++) {
    c->lgroup_mode = mode;
    StageArgs a = stage_args(c, 1, c->GA, c->GB);
    a.rhs_stride = c->ntot;
    a.rhs_out = out;
    for (int r = -1; r < reps; r++) {
      if (r == 0) SV_HIP(c, hipEventRecord(e0, c->stream));
      if (c->cfg.form == SV_FORM_LC) launch_stage<SV_FORM_LC, 0>(c, a, c->nblk);
      else launch_stage<SV_FORM_DI, 0>(c, a, c->nblk);
    }
    SV_HIP(c, hipEventRecord(e1, c->stream));
    SV_HIP(c, hipGetLastError());
    SV_HIP(c, hipEventSynchronize(e1));
    SV_HIP(c, hipEventElapsedTime(&ms[mode], e0, e1));
  }
  c->lgroup_ms[0] = ms[0] / reps;
  c->lgroup_ms[1] = ms[1] / reps;
  c->lgroup_mode = ms[1] < ms[0] ? 1 : 0;
  return 0;
}

namespace {
__global__ void k_offset_int(int *dst, int64_t n, int add) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) dst[k] += add;
}
__global__ void k_offset_i64(int64_t *dst, int64_t n, int64_t add) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) dst[k] += add;
}
}  // namespace

int sv_dev_offset_int(sv_ctx *c, int *dst, int64_t n, int add) {
  if (n <= 0) return 0;
  k_offset_int<<<(unsigned)((n + 255) / 256), 256, 0, c->stream>>>(dst, n, add);
  SV_HIP(c, hipGetLastError());
  return 0;
}

int sv_dev_offset_i64(sv_ctx *c, int64_t *dst, int64_t n, int64_t add) {
  if (n <= 0) return 0;
  k_offset_i64<<<(unsigned)((n + 255) / 256), 256, 0, c->stream>>>(dst, n, add);
  SV_HIP(c, hipGetLastError());
  return 0;
}
