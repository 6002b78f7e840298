// k_stencil.hip -- the derivative operators of derivatives.F90 on the SELL-64
// stencil layout: one lane per node, links of a 64-node slice interleaved so a
// wavefront reads 64 consecutive indices / weights per link (coalesced), and
// the sum runs over k in the reference's order:
//   calc_gradient      :26-71    d_i = sum_k phi_j w_k - phi_i sum_k w_k
//   calc_laplacian     :73-116
//   calc_gradient_only :416-464
//   calc_filtered_var  :360-414  phi_i + (sum_k phi_j w_k - phi_i sum_k w_k)
//   calc_filter_term   :466-511
// Gradients and Laplacians run over the small stencil (ij_count_small), the
// filter over the full one (ij_count).
#include "sv_internal.h"

namespace {

// Fields of one launch: the links' columns and weights are read once for all of
// them.
constexpr int AP_NF = 4;
struct ApplyArgs {
  int npfb;
  const int64_t *off;
  const int *width;         // links per slice, padding included
  const int *kcnt;          // links per node for this operator
  const int *col;
  const double *w0, *w1;
  const double *s0, *s1;    // weight sums
  const double *phi[AP_NF];
  double *o0[AP_NF], *o1[AP_NF];
  const uint16_t *lcol;     // halos (k_apply_h)
  const int64_t *hoff;
  const int *hidx;
  int hmax;
};

// One lane per node, one wavefront per workgroup, links in batches of AP_U:
// every column and weight of a batch, then every gathered value, are requested
// before the first sum.  A batch past a node's own list reads the slice's
// padding (or its last link again) and leaves it out of the sums.
// 511x513 order 6, three fields: gradients 315 us in three launches of one field
// each, 152 so, Laplacians 200 and 122, filters 195 and 115 (the scattered reads
// of phi, up to 64 lines a wave, are what is left: see k_apply_h).
constexpr int AP_U = 4;
template <int OP, int NF>
__global__ __launch_bounds__(SV_WAVE) void k_apply(ApplyArgs a) {
  constexpr bool GRAD = OP == SV_OP_GRAD;
  const int s = sv_xcd_block();
  const int i = s * SV_WAVE + (int)threadIdx.x;
  const bool act = i < a.npfb;
  const int64_t b = a.off[s] + threadIdx.x;
  const int K = act ? a.kcnt[i] : 0, W = a.width[s];
  double t0[NF], t1[NF];
#pragma unroll
  for (int f = 0; f < NF; f++) t0[f] = t1[f] = 0.0;
  for (int k = 0; k < W; k += AP_U) {
    int j[AP_U];
    double w0[AP_U], w1[AP_U];
#pragma unroll
    for (int u = 0; u < AP_U; u++) {
      const int64_t e = b + (int64_t)min(k + u, W - 1) * SV_WAVE;
      j[u] = a.col[e];
      w0[u] = a.w0[e];
      if (GRAD) w1[u] = a.w1[e];
    }
    double p[AP_U][NF];
#pragma unroll
    for (int u = 0; u < AP_U; u++)
#pragma unroll
      for (int f = 0; f < NF; f++) p[u][f] = a.phi[f][j[u]];
#pragma unroll
    for (int u = 0; u < AP_U; u++)
      if (k + u < K) {
#pragma unroll
        for (int f = 0; f < NF; f++) {
          t0[f] = t0[f] + p[u][f] * w0[u];
          if (GRAD) t1[f] = t1[f] + p[u][f] * w1[u];
        }
      }
  }
  if (!act) return;
  const double s0 = a.s0[i], s1 = GRAD ? a.s1[i] : 0.0;
#pragma unroll
  for (int f = 0; f < NF; f++) {
    const double pi = a.phi[f][i];
    if (OP == SV_OP_FILTER) a.o0[f][i] = pi + (t0[f] - pi * s0);
    else a.o0[f][i] = t0[f] - pi * s0;
    if (GRAD) a.o1[f][i] = t1[f] - pi * s1;
  }
}

// k_apply with the slice's distinct neighbour values staged in LDS first (11 per
// node in row order, order 6): a wavefront per field stages and walks its own
// field, so every sum is k_apply's.  k_apply's scattered reads find little in the
// L1 and take ~100 clocks each.  511x513 order 6, three fields, gradients 152 ->
// 124 us, Laplacians 122 -> 73, filters 115 -> 71; what is left is the requests'
// latency at 24 wavefronts a CU.  Taken where no slice has more than 1024 distinct
// neighbours (not on the cylinder channel's order of nodes), on folded columns.
constexpr int AH_U = 8;     // values a lane stages, and links it reads, at once (12, 16: the
                            // same, 24: 8% slower)
template <int OP>
__global__ __launch_bounds__(SV_WAVE *AP_NF) void k_apply_h(ApplyArgs a) {
  extern __shared__ double hl[];
  constexpr bool GRAD = OP == SV_OP_GRAD;
  const int s = sv_xcd_block();
  const int lane = (int)threadIdx.x & (SV_WAVE - 1);
  const int f = __builtin_amdgcn_readfirstlane((int)threadIdx.x / SV_WAVE);
  const int i = s * SV_WAVE + lane;
  const bool act = i < a.npfb;
  const int64_t b = a.off[s] + lane;
  const int K = act ? a.kcnt[i] : 0, W = a.width[s];
  const int64_t h0 = a.hoff[s];
  const int nh = (int)(a.hoff[s + 1] - h0);
  const double *phi = a.phi[f];
  double *hf = hl + (size_t)f * a.hmax;
  for (int h = lane; h < nh; h += AH_U * SV_WAVE) {
    int j[AH_U];
#pragma unroll
    for (int u = 0; u < AH_U; u++) j[u] = a.hidx[h0 + min(h + u * SV_WAVE, nh - 1)];
    double v[AH_U];
#pragma unroll
    for (int u = 0; u < AH_U; u++) v[u] = phi[j[u]];
#pragma unroll
    for (int u = 0; u < AH_U; u++)
      if (h + u * SV_WAVE < nh) hf[h + u * SV_WAVE] = v[u];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // its own wavefront reads it
  double t0 = 0.0, t1 = 0.0;
  for (int k = 0; k < W; k += AH_U) {
    int j[AH_U];
    double w0[AH_U], w1[AH_U];
#pragma unroll
    for (int u = 0; u < AH_U; u++) {
      const int64_t e = b + (int64_t)min(k + u, W - 1) * SV_WAVE;
      j[u] = a.lcol[e];
      w0[u] = a.w0[e];
      if (GRAD) w1[u] = a.w1[e];
    }
#pragma unroll
    for (int u = 0; u < AH_U; u++)
      if (k + u < K) {
        const double p = hf[j[u]];
        t0 = t0 + p * w0[u];
        if (GRAD) t1 = t1 + p * w1[u];
      }
  }
  if (!act) return;
  const double pi = phi[i], s0 = a.s0[i];
  if (OP == SV_OP_FILTER) a.o0[f][i] = pi + (t0 - pi * s0);
  else a.o0[f][i] = t0 - pi * s0;
  if (GRAD) a.o1[f][i] = t1 - pi * a.s1[i];
}

template <int OP>
void launch_apply(const ApplyArgs &a, int nf, int ns, hipStream_t st) {
  if (a.hmax > 0) {
    k_apply_h<OP><<<ns, SV_WAVE * nf, sizeof(double) * (size_t)nf * a.hmax, st>>>(a);
    return;
  }
  switch (nf) {
  case 1: k_apply<OP, 1><<<ns, SV_WAVE, 0, st>>>(a); break;
  case 2: k_apply<OP, 2><<<ns, SV_WAVE, 0, st>>>(a); break;
  case 3: k_apply<OP, 3><<<ns, SV_WAVE, 0, st>>>(a); break;
  default: k_apply<OP, 4><<<ns, SV_WAVE, 0, st>>>(a); break;
  }
}

// Whether the fields of one call may share a launch: no output overlaps
// another field's input or output (a call may chain fields, one's output the
// next one's input, as the launches of the fields follow each other)
bool fields_apart(int n, int nf, const double *const *phi, double *const *out, size_t nout) {
  auto overlap = [](const double *p, size_t np, const double *q, size_t nq) {
    return p < q + nq && q < p + np;
  };
  for (int f = 0; f < nf; f++)
    for (int g = 0; g < nf; g++)
      if (f != g && (overlap(out[f], nout, phi[g], n) || overlap(out[f], nout, out[g], nout)))
        return false;
  return true;
}

}  // namespace

namespace {

// The mass correction of filter_variables (rhs_lc.F90:871-890, -Dmcorr):
// ro -= sum_i (ro_i - rho_char) vol_i / sum_i vol_i over the real nodes, with
// rho_char = 1 (load_data.F90:132).  One block: each thread sums a strided
// slice in node order, then a fixed-shape tree, so the result does not depend
// on scheduling.
__global__ __launch_bounds__(1024) void k_mass_correct(int n, const double *vol, double *ro) {
  __shared__ double sm[1024], sv[1024];
  const int t = threadIdx.x;
  double tm = 0.0, tv = 0.0;
  for (int i = t; i < n; i += 1024) {
    tm += (ro[i] - 1.0) * vol[i];
    tv += vol[i];
  }
  sm[t] = tm;
  sv[t] = tv;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (t < o) {
      sm[t] += sm[t + o];
      sv[t] += sv[t + o];
    }
    __syncthreads();
  }
  const double dro = sm[0] / sv[0];
  for (int i = t; i < n; i += 1024) ro[i] = ro[i] - dro;
}

}  // namespace

int sv_dev_mass_correct(sv_ctx *c, double *ro, hipStream_t st) {
  k_mass_correct<<<1, 1024, 0, st>>>(c->npfb, c->vol, ro);
  SV_HIP(c, hipGetLastError());
  return 0;
}

int sv_dev_apply(sv_ctx *c, int op, int nfields, const double *const *phi, double *const *out,
                 bool raw_cols, hipStream_t st) {
  ApplyArgs a{};
  a.npfb = c->npfb;
  a.off = c->sell_off;
  a.width = c->sell_w;
  a.col = raw_cols ? c->scol_raw : c->scol;
  if (!raw_cols) {   // the halos are of the folded columns
    a.lcol = c->slcol;
    a.hoff = c->shoff;
    a.hidx = c->shidx;
    a.hmax = c->shmax;
  }
  switch (op) {
  case SV_OP_GRAD: a.kcnt = c->cnt_small; a.w0 = c->swx; a.w1 = c->swy; a.s0 = c->gsx; a.s1 = c->gsy; break;
  case SV_OP_LAP:
  case SV_OP_LAP_TRANSVERSE: a.kcnt = c->cnt_small; a.w0 = c->swl; a.s0 = c->lsum; break;
  case SV_OP_GRAD_X: a.kcnt = c->cnt_small; a.w0 = c->swx; a.s0 = c->gsx; break;
  case SV_OP_GRAD_Y: a.kcnt = c->cnt_small; a.w0 = c->swy; a.s0 = c->gsy; break;
  case SV_OP_FILTER:
  case SV_OP_FILTER_TERM: a.kcnt = c->cnt; a.w0 = c->swh; a.s0 = c->hsum; break;
  default: return sv_fail(c, SV_E_ARG, "unknown operator %d", op);
  }
  const size_t nout = (op == SV_OP_GRAD ? 2 : 1) * (size_t)c->npfb;
  const size_t nin = raw_cols ? c->np : c->npfb;
  for (int f0 = 0; f0 < nfields;) {
    int nf = nfields - f0 < AP_NF ? nfields - f0 : AP_NF;
    if (!fields_apart(nin, nf, phi + f0, out + f0, nout)) nf = 1;
    for (int f = 0; f < nf; f++) {
      a.phi[f] = phi[f0 + f];
      a.o0[f] = out[f0 + f];
      a.o1[f] = out[f0 + f] + c->npfb;
    }
    switch (op) {
    case SV_OP_GRAD: launch_apply<SV_OP_GRAD>(a, nf, c->nslices, st); break;
    case SV_OP_FILTER: launch_apply<SV_OP_FILTER>(a, nf, c->nslices, st); break;
    default: launch_apply<SV_OP_LAP>(a, nf, c->nslices, st); break;
    }
    SV_HIP(c, hipGetLastError());
    // calc_laplacian_transverse_only_on_bound: the Laplacian on the internal
    // nodes (derivatives.F90:315-325), the boundary nodes overwritten with the
    // tangential part (:327-337)
    if (op == SV_OP_LAP_TRANSVERSE)
      for (int f = 0; f < nf; f++)
        if (int rc = sv_dev_boundary_tt_apply(c, phi[f0 + f], out[f0 + f], raw_cols, st))
          return rc;
    f0 += nf;
  }
  return 0;
}
