// k_nodes.hip -- ghost (mirror) creation, cell-list neighbour search and the
// SELL-64 layout of the stencils.
//
// Reference behaviour reproduced:
//  * create_mirror_particles (mirror_boundaries.F90:34-261): ghosts within
//    ss*h*2 of periodic/symmetric/no-slip edges, numbered node by node in the
//    order left/right, lower/upper, four corners; positions with the same
//    left-to-right arithmetic (contraction off) so distances are bit-identical.
//  * find_neighbours (neighbours.F90:32-341): every j with
//    |r_i - r_j|^2 <= (h_i*ss)^2 (self included), r^2 = dx*dx + dy*dy without
//    FMA contraction, lists sorted by (r^2, j); ij_count_small counts
//    r^2 <= (h_small_i*ss)^2.
// The cell grid is this library's own: cells of side ss*max(h) over the box
// padded by its size on each side, so a 3x3 block of cells covers every
// stencil whatever h_i is.
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "sv_internal.h"

#define SS 2.0

namespace {

struct GhostDom {
  double xmin, xmax, ymin, ymax;
  int xl, xu, yl, yu;
};

// Enumerate the ghosts of node i in reference order.  emit(gx, gy, vrel).
template <class F>
__device__ void ghost_enum(const GhostDom &g, double xi, double yi, double hi, F emit) {
#pragma clang fp contract(off)
  const double lim = SS * hi * 2.0;
  if (xi <= g.xmin + lim) {
    if (g.xl == 1) emit(xi + g.xmax - g.xmin, yi, 1);
    else if (g.xl == 2) emit(2.0 * g.xmin - xi, yi, 2);
  }
  if (xi >= g.xmax - lim) {
    if (g.xu == 1) emit(xi - g.xmax + g.xmin, yi, 1);
    else if (g.xu == 2) emit(2.0 * g.xmax - xi, yi, 2);
  }
  if (yi <= g.ymin + lim) {
    if (g.yl == 1) emit(xi, yi + g.ymax - g.ymin, 1);
    else if (g.yl == 2) emit(xi, 2.0 * g.ymin - yi, 3);
    else if (g.yl == 3) emit(xi, 2.0 * g.ymin - yi, 4);
  }
  if (yi >= g.ymax - lim) {
    if (g.yu == 1) emit(xi, yi - g.ymax + g.ymin, 1);
    else if (g.yu == 2) emit(xi, 2.0 * g.ymax - yi, 3);
    else if (g.yu == 3) emit(xi, 2.0 * g.ymax - yi, 4);
  }
  const double cx[4] = {g.xmin, g.xmax, g.xmin, g.xmax};
  const double cy[4] = {g.ymin, g.ymin, g.ymax, g.ymax};
  const int bx[4] = {g.xl, g.xu, g.xl, g.xu};
  const int by[4] = {g.yl, g.yl, g.yu, g.yu};
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const double dx = cx[c] - xi, dy = cy[c] - yi;
    const double cd = sqrt(dx * dx + dy * dy + 0.0 * 0.0);
    if (cd <= lim && bx[c] != 0 && by[c] != 0) {
      const bool perx = bx[c] == 1, pery = by[c] == 1;
      const bool symx = bx[c] == 2, symy = by[c] == 2;
      double px, py;
      if (c == 0 || c == 2) px = perx ? xi + g.xmax - g.xmin : 2.0 * g.xmin - xi;
      else px = perx ? xi - g.xmax + g.xmin : 2.0 * g.xmax - xi;
      if (c == 0 || c == 1) py = pery ? yi + g.ymax - g.ymin : 2.0 * g.ymin - yi;
      else py = pery ? yi - g.ymax + g.ymin : 2.0 * g.ymax - yi;
      int vr = 0;
      if (perx && pery) vr = 1;
      else if (symx && pery) vr = 2;
      else if (perx && symy) vr = 3;
      else if (symx && symy) vr = 4;
      if (vr) emit(px, py, vr);
      else emit(0.0, 0.0, 0);   // the reference counts the ghost but leaves rp = 0
    }
  }
}

__global__ void k_ghost_count(int npfb, GhostDom g, const double *x, const double *y,
                              const double *h, int *gcount) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npfb) return;
  int n = 0;
  ghost_enum(g, x[i], y[i], h[i], [&](double, double, int) { n++; });
  gcount[i] = n;
}

__global__ void k_ghost_write(int npfb, GhostDom g, double *x, double *y, double *h, double *hs,
                              double *s, int *nt, int *irel, int *vrel, const int *goff) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npfb) return;
  int k = npfb + goff[i];
  const double hi = h[i], hsi = hs[i], si = s[i];
  const int nti = nt[i];
  ghost_enum(g, x[i], y[i], hi, [&](double gx, double gy, int vr) {
    x[k] = gx; y[k] = gy; irel[k] = i; vrel[k] = vr;
    h[k] = hi; hs[k] = hsi; s[k] = si; nt[k] = nti;
    k++;
  });
  irel[i] = i;
  vrel[i] = 0;
}

struct Grid {
  double x0, y0, inv;
  int ncx, ncy;
  // the reference's cells (cell_generator, neighbours.F90:75-93): size
  // ss*h0 over the domain padded by its size on every side; a node sees the
  // 3x3 cells around its own (neighbour_cells, :95-157), which cuts the disc
  // of a node with h > h0
  double rx0, ry0, rinv, h0;
};

__device__ __forceinline__ int cell_of(const Grid &G, double x, double y, int *cx, int *cy) {
  int ix = (int)((x - G.x0) * G.inv);
  int iy = (int)((y - G.y0) * G.inv);
  ix = ix < 0 ? 0 : (ix >= G.ncx ? G.ncx - 1 : ix);
  iy = iy < 0 ? 0 : (iy >= G.ncy ? G.ncy - 1 : iy);
  *cx = ix;
  *cy = iy;
  return iy * G.ncx + ix;
}

__global__ void k_cell_count(int np, Grid G, const double *x, const double *y, int *cellof,
                             int *ccount) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= np) return;
  int cx, cy;
  const int c = cell_of(G, x[k], y[k], &cx, &cy);
  cellof[k] = c;
  atomicAdd(&ccount[c], 1);
}

__global__ void k_cell_fill(int np, const int *cellof, const int *cstart, int *cfill, int *ip) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= np) return;
  const int c = cellof[k];
  const int pos = atomicAdd(&cfill[c], 1);
  ip[cstart[c] + pos] = k;
}

__device__ __forceinline__ double dist2(double xi, double yi, double xj, double yj) {
#pragma clang fp contract(off)
  const double dx = xi - xj, dy = yi - yj;
  double t = dx * dx;
  t = t + dy * dy;
  return t;
}

// Wave-scope ordering of LDS traffic between the lanes of one wavefront.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int NW = 4;   // nodes (wavefronts) per block of the neighbour search

// One wavefront per node.  The cells within the node's own search radius
// 2 h_i (one cell of margin) are scanned row by row: a row of cells is one
// contiguous range of the cell-sorted node list, taken 64 candidates at a
// time, and matches are compacted with a ballot.  Pass 0 counts; pass 1
// collects (j, r^2) in LDS, ranks every entry by (r^2, j) -- the order of the
// reference's sorted lists (neighbours.F90:247-341) -- and writes the row in
// that order, with the count of entries inside 2 h_small.  The cell size is
// 2 h_min, so nodes of every size scan a few candidates per neighbour.  A node
// with h > h0 (boundary nodes at order 4: hovs_bound 2.1 > hovs 1.8,
// common_parameter.F90:46-47) keeps, as the reference does, only the
// candidates inside the 3x3 reference cells of size 2 h0 around it.
template <int PASS>
__global__ __launch_bounds__(NW * SV_WAVE) void k_neigh(
    int npfb, Grid G, const double *x, const double *y, const double *h, const double *hs,
    const int *cstart, const int *ip, int *cnt, int *cnt_small, const int64_t *row_ptr,
    int *col, int cap) {
#pragma clang fp contract(off)
  extern __shared__ double nb_lds[];
  const int wave = (int)threadIdx.x / SV_WAVE, lane = (int)threadIdx.x % SV_WAVE;
  const int i = (int)blockIdx.x * NW + wave;
  if (i >= npfb) return;   // whole wavefronts; no block-wide barrier follows
  double *r2s = nb_lds + (size_t)wave * cap;
  int *js = reinterpret_cast<int *>(nb_lds + (size_t)NW * cap) + (size_t)wave * cap;
  const double xi = x[i], yi = y[i];
  const double R = h[i] * SS;
  const double st2 = R * R;
  // only a node with h > h0 reaches past the reference's 3x3 cells
  const bool clip = h[i] > G.h0;
  const int rcx = (int)((xi - G.rx0) * G.rinv), rcy = (int)((yi - G.ry0) * G.rinv);
  int ix0 = (int)((xi - R - G.x0) * G.inv) - 1, ix1 = (int)((xi + R - G.x0) * G.inv) + 1;
  int iy0 = (int)((yi - R - G.y0) * G.inv) - 1, iy1 = (int)((yi + R - G.y0) * G.inv) + 1;
  ix0 = ix0 < 0 ? 0 : ix0;
  iy0 = iy0 < 0 ? 0 : iy0;
  ix1 = ix1 >= G.ncx ? G.ncx - 1 : ix1;
  iy1 = iy1 >= G.ncy ? G.ncy - 1 : iy1;
  int n = 0;
  for (int cy = iy0; cy <= iy1; cy++) {
    const int lo = cstart[cy * G.ncx + ix0], hi = cstart[cy * G.ncx + ix1 + 1];
    for (int b0 = lo; b0 < hi; b0 += SV_WAVE) {
      const int jj = b0 + lane;
      bool m = false;
      double r2 = 0.0;
      int j = 0;
      if (jj < hi) {
        j = ip[jj];
        r2 = dist2(xi, yi, x[j], y[j]);
        m = r2 <= st2;
        if (clip && m) {
          const int dcx = (int)((x[j] - G.rx0) * G.rinv) - rcx;
          const int dcy = (int)((y[j] - G.ry0) * G.rinv) - rcy;
          m = dcx >= -1 && dcx <= 1 && dcy >= -1 && dcy <= 1;
        }
      }
      const unsigned long long bal = __ballot(m);
      if (PASS == 1 && m) {
        const int pos = n + __popcll(bal & ((1ull << lane) - 1ull));
        if (pos < cap) {
          r2s[pos] = r2;
          js[pos] = j;
        }
      }
      n += __popcll(bal);
    }
  }
  if (PASS == 0) {
    if (lane == 0) cnt[i] = n;
    return;
  }
  wave_sync();
  // the same scan as pass 0, so n == cnt[i] <= cap; clamped all the same so
  // that a row can never spill into the next one
  n = n < cnt[i] ? n : cnt[i];
  const int64_t base = row_ptr[i];
  const double hsm = hs[i] * SS;
  const double st2s = hsm * hsm;
  int ks = 0;
  for (int a = lane; a < n; a += SV_WAVE) {
    const double ra = r2s[a];
    const int ja = js[a];
    int rank = 0;
    for (int b = 0; b < n; b++) {
      const double rb = r2s[b];
      const int jb = js[b];
      rank += (rb < ra || (rb == ra && jb < ja)) ? 1 : 0;
    }
    col[base + rank] = ja;
    ks += (ra <= st2s) ? 1 : 0;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) ks += __shfl_xor(ks, o);
  if (lane == 0) cnt_small[i] = ks;
}

// SELL packing of the drop-in operators.  One block per 64-row slice: the rows
// are read 16 links at a time and transposed through LDS into the slice's
// link-major columns.  (One 64-thread block per four links reading and writing
// the rows directly: 1726 us on a 511x513 order-6 lattice; 568 so.)
constexpr int SP_T = 256, SP_K = 16, SP_LD = SP_K + 1;
__global__ __launch_bounds__(SP_T) void k_sell_pack(
    int npfb, const int64_t *sell_off, const int *sell_w, const int64_t *row_ptr, const int *cnt,
    const int *col_raw, const int *irel, const double *wx, const double *wy, const double *wl,
    const double *wh, int *scol, int *scol_raw, double *swx, double *swy, double *swl,
    double *swh) {
  __shared__ double tw[4][SV_WAVE * SP_LD];
  __shared__ int tc[SV_WAVE * SP_LD], tr[SV_WAVE * SP_LD];
  __shared__ int64_t rbase[SV_WAVE];
  __shared__ int rcnt[SV_WAVE];
  const int s = blockIdx.x, t = threadIdx.x;
  if (t < SV_WAVE) {
    const int i = s * SV_WAVE + t;
    rbase[t] = i < npfb ? row_ptr[i] : 0;
    rcnt[t] = i < npfb ? cnt[i] : 0;
  }
  __syncthreads();
  const int W = sell_w[s];
  const int64_t off = sell_off[s];
  for (int k0 = 0; k0 < W; k0 += SP_K) {
    for (int p = t; p < SV_WAVE * SP_K; p += SP_T) {
      const int r = p / SP_K, kk = p % SP_K, k = k0 + kk, e = r * SP_LD + kk;
      const int i = s * SV_WAVE + r, self = i < npfb ? i : 0;
      if (k < rcnt[r]) {
        const int64_t q = rbase[r] + k;
        const int j = col_raw[q];
        tr[e] = j;
        tc[e] = irel[j];
        tw[0][e] = wx ? wx[q] : 0.0;
        tw[1][e] = wy ? wy[q] : 0.0;
        tw[2][e] = wl ? wl[q] : 0.0;
        tw[3][e] = wh ? wh[q] : 0.0;
      } else {
        tr[e] = tc[e] = self;
        tw[0][e] = tw[1][e] = tw[2][e] = tw[3][e] = 0.0;
      }
    }
    __syncthreads();
    for (int p = t; p < SV_WAVE * SP_K; p += SP_T) {
      const int kk = p / SV_WAVE, l = p % SV_WAVE, k = k0 + kk, e = l * SP_LD + kk;
      if (k >= W) break;
      const int64_t d = off + (int64_t)k * SV_WAVE + l;
      scol_raw[d] = tr[e];
      scol[d] = tc[e];
      swx[d] = tw[0][e];
      swy[d] = tw[1][e];
      swl[d] = tw[2][e];
      swh[d] = tw[3][e];
    }
    __syncthreads();
  }
}

}  // namespace

static int scan_int(sv_ctx *c, const int *in, int *out, int n) {
  size_t tb = 0;
  SV_HIP(c, hipcub::DeviceScan::ExclusiveSum(nullptr, tb, in, out, n, c->stream));
  DevTmp<char> tmp;
  SV_HIP(c, tmp.alloc(c, tb > 0 ? tb : 16));
  SV_HIP(c, hipcub::DeviceScan::ExclusiveSum((void *)tmp, tb, in, out, n, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}

int sv_dev_create_ghosts(sv_ctx *c) {
  const int n = c->npfb;
  GhostDom g{c->xmin, c->xmax, c->ymin, c->ymax, c->bc[0], c->bc[1], c->bc[2], c->bc[3]};
  DevTmp<int> gcount, goff;
  SV_HIP(c, gcount.alloc(c, n + 1));
  SV_HIP(c, goff.alloc(c, n + 1));
  SV_HIP(c, hipMemsetAsync(gcount, 0, sizeof(int) * (n + 1), c->stream));
  const int B = 256, nb = (n + B - 1) / B;
  k_ghost_count<<<nb, B, 0, c->stream>>>(n, g, c->x, c->y, c->h, gcount);
  SV_HIP(c, hipGetLastError());
  if (int rc = scan_int(c, gcount, goff, n + 1)) return rc;
  int ng = 0;
  SV_HIP(c, hipMemcpy(&ng, goff + n, sizeof(int), hipMemcpyDeviceToHost));
  if (n + ng > c->cap) {
    return sv_fail(c, SV_E_ARG, "ghost count %d exceeds node capacity %d", ng, c->cap - n);
  }
  k_ghost_write<<<nb, B, 0, c->stream>>>(n, g, c->x, c->y, c->h, c->hs, c->s, c->node_type,
                                         c->irel, c->vrel, goff);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipStreamSynchronize(c->stream));
  // symmetric (2) or no-slip (3) edges make mirror ghosts with sign flips
  c->has_mirror = false;
  for (int k = 0; k < 4; k++) c->has_mirror |= (c->bc[k] == 2 || c->bc[k] == 3) && ng > 0;
  c->np = n + ng;
  return 0;
}

int sv_dev_find_neighbours(sv_ctx *c) {
  EventTmp e0, e1;
  SV_HIP(c, e0.create());
  SV_HIP(c, e1.create());
  SV_HIP(c, hipEventRecord(e0, c->stream));
  const int np = c->np, npfb = c->npfb;
  const double Lx = c->xmax - c->xmin, Ly = c->ymax - c->ymin;
  double csz = SS * (c->hmin > 0.0 ? c->hmin : c->hmax);
  // keep the padded grid below ~64M cells
  const double area = 9.0 * Lx * Ly;
  if (area / (csz * csz) > 6.4e7) csz = sqrt(area / 6.4e7);
  Grid G;
  G.x0 = c->xmin - Lx;
  G.y0 = c->ymin - Ly;
  G.inv = 1.0 / csz;
  G.ncx = (int)(3.0 * Lx / csz) + 1;
  G.ncy = (int)(3.0 * Ly / csz) + 1;
  G.rx0 = c->xmin - Lx;
  G.ry0 = c->ymin - Ly;
  G.rinv = 1.0 / (1.0 * (SS * c->h0));
  G.h0 = c->h0;
  const int nct = G.ncx * G.ncy;
  DevTmp<int> cellof, ccount, cstart, ip;
  SV_HIP(c, cellof.alloc(c, np));
  SV_HIP(c, ccount.alloc(c, nct + 1));
  SV_HIP(c, cstart.alloc(c, nct + 1));
  SV_HIP(c, ip.alloc(c, np));
  SV_HIP(c, hipMemsetAsync(ccount, 0, sizeof(int) * (nct + 1), c->stream));
  const int B = 256;
  k_cell_count<<<(np + B - 1) / B, B, 0, c->stream>>>(np, G, c->x, c->y, cellof, ccount);
  SV_HIP(c, hipGetLastError());
  if (int rc = scan_int(c, ccount, cstart, nct + 1)) return rc;
  SV_HIP(c, hipMemsetAsync(ccount, 0, sizeof(int) * (nct + 1), c->stream));
  k_cell_fill<<<(np + B - 1) / B, B, 0, c->stream>>>(np, cellof, cstart, ccount, ip);
  SV_HIP(c, hipGetLastError());
  // counts
  if (!c->cnt)
    if (int rc = sv_alloc_all(c, {sv_want(&c->cnt, npfb), sv_want(&c->cnt_small, npfb),
                                  sv_want(&c->row_ptr, (size_t)npfb + 1)}))
      return rc;
  const int nb = (npfb + NW - 1) / NW;
  k_neigh<0><<<nb, NW * SV_WAVE, 0, c->stream>>>(npfb, G, c->x, c->y, c->h, c->hs, cstart, ip,
                                                 c->cnt, c->cnt_small, nullptr, nullptr, 0);
  SV_HIP(c, hipGetLastError());
  std::vector<int> hc(npfb);
  SV_HIP(c, hipMemcpyAsync(hc.data(), c->cnt, sizeof(int) * npfb, hipMemcpyDeviceToHost,
                           c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  std::vector<int64_t> rp(npfb + 1);
  rp[0] = 0;
  int maxk = 0;
  for (int i = 0; i < npfb; i++) {
    rp[i + 1] = rp[i] + hc[i];
    maxk = hc[i] > maxk ? hc[i] : maxk;
  }
  c->maxK = maxk;
  c->nnz = rp[npfb];
  SV_HIP(c, hipMemcpyAsync(c->row_ptr, rp.data(), sizeof(int64_t) * (npfb + 1),
                           hipMemcpyHostToDevice, c->stream));
  sv_free(c, c->col_raw);
  c->col_raw = nullptr;
  if (sv_alloc(c, (void **)&c->col_raw, sizeof(int) * (c->nnz + 1))) return SV_E_NOMEM;
  static_assert(NW * SV_LIST_MAX * (sizeof(double) + sizeof(int)) <= 64 * 1024,
                "the longest lists of a block's nodes fit LDS");
  const int cap = maxk > 0 ? maxk : 1;
  const size_t shm = (size_t)NW * cap * (sizeof(double) + sizeof(int));
  if (maxk > SV_LIST_MAX)
    return sv_fail(c, SV_E_OVERFLOW, "neighbour list of %d entries too long for the search", maxk);
  k_neigh<1><<<nb, NW * SV_WAVE, shm, c->stream>>>(npfb, G, c->x, c->y, c->h, c->hs, cstart, ip,
                                                   c->cnt, c->cnt_small, c->row_ptr, c->col_raw,
                                                   cap);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipEventRecord(e1, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  float ms = 0;
  SV_HIP(c, hipEventElapsedTime(&ms, e0, e1));
  c->t_neigh = ms;
  c->have_lists = true;
  c->sell_dirty = true;
  c->L.valid = false;
  return 0;
}

// links per slice, padding included
static __global__ void k_slice_links(int ns, const int64_t *off, int *w) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < ns) w[s] = (int)((off[s + 1] - off[s]) / SV_WAVE);
}

int sv_dev_build_sell(sv_ctx *c) {
  const int npfb = c->npfb;
  const int ns = (npfb + SV_WAVE - 1) / SV_WAVE;
  if (c->nslices != ns) {
    for (void *b : {(void *)c->sell_off, (void *)c->sell_w, (void *)c->shoff}) sv_free(c, b);
    c->sell_off = c->shoff = nullptr;
    c->sell_w = nullptr;
    if (sv_alloc(c, (void **)&c->sell_off, sizeof(int64_t) * (ns + 1)) ||
        sv_alloc(c, (void **)&c->sell_w, sizeof(int) * (ns + 1)))
      return SV_E_NOMEM;
  }
  int64_t nnz = 0;
  if (int rc = sv_dev_slice_offsets(c, npfb, c->cnt, c->sell_off, &nnz)) return rc;
  if (c->nslices != ns || c->sell_nnz != nnz) {
    for (void *b : {(void *)c->scol, (void *)c->scol_raw, (void *)c->swx, (void *)c->swy,
                    (void *)c->swl, (void *)c->swh, (void *)c->slcol})
      sv_free(c, b);
    c->scol = c->scol_raw = nullptr;
    c->slcol = nullptr;
    c->swx = c->swy = c->swl = c->swh = nullptr;
    c->nslices = ns;
    c->sell_nnz = nnz;
    const size_t L = (size_t)c->sell_nnz + 1;
    if (sv_alloc(c, (void **)&c->scol, sizeof(int) * L) ||
        sv_alloc(c, (void **)&c->scol_raw, sizeof(int) * L) ||
        sv_alloc(c, (void **)&c->swx, sizeof(double) * L) ||
        sv_alloc(c, (void **)&c->swy, sizeof(double) * L) ||
        sv_alloc(c, (void **)&c->swl, sizeof(double) * L) ||
        sv_alloc(c, (void **)&c->swh, sizeof(double) * L)) {
      c->nslices = 0;
      return SV_E_NOMEM;
    }
  }
  k_slice_links<<<(ns + 255) / 256, 256, 0, c->stream>>>(ns, c->sell_off, c->sell_w);
  k_sell_pack<<<ns, SP_T, 0, c->stream>>>(npfb, c->sell_off, c->sell_w, c->row_ptr, c->cnt,
                                          c->col_raw, c->irel, c->wx, c->wy, c->wl, c->wh,
                                          c->scol, c->scol_raw, c->swx, c->swy, c->swl, c->swh);
  SV_HIP(c, hipGetLastError());
  if (int rc = sv_dev_sell_halos(c)) return rc;
  SV_HIP(c, hipStreamSynchronize(c->stream));
  c->sell_dirty = false;
  return 0;
}
