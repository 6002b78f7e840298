// k_loop.hip -- the layout the RK sweeps run in: node order, SELL-64 stencils
// in that order, and per-block neighbour halos, all built on the device.
//
// Order.  The nodes are split recursively, each segment along the longer side
// of its box at a multiple of 64 nodes (of 256 while it holds more than 256),
// so every 64-node slice and every 256-node block is a compact rectangle of
// the domain whatever the node counts along its sides.  A Morton order of the
// positions does the same only on 2^k lattices: on a 301x283 order-8 lattice
// its 256-node halos reached 947 records (mean 787), more than the 819 that the
// sweeps' LDS budget holds; split, they are 694 at most (mean 667); on 260x260
// at order 6, 829 -> 617 records.
// One level of the split is a stable radix sort of (segment, coordinate)
// keys, 14 levels at 1M nodes.
//
// Halos.  One workgroup per halo block inserts the block's link targets into
// an LDS hash set, sorts the distinct ones and re-expresses every link as a
// 16-bit rank.  (On 16 host threads, with the columns copied down and up, the
// halo pass took most of sv_set_initial: 0.25 s at 1M nodes.)
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "sv_internal.h"

namespace {

// Loop-order SELL packing: block (s, y) fills links [16y, 16y+16) of the 64
// nodes of slice s.  The CSR rows are read 16 links at a time (one cache
// line of each array per row), transposed through LDS, and written as the
// slice's link-major columns (64 consecutive slots per link).  Links past a
// node's count, and slots past npfb, get the padding entry: the node's own
// slot (0 past npfb) with zero weights.
constexpr int PK_K = 16;           // links per block
constexpr int PK_T = 256;          // threads per block
constexpr int PK_LD = PK_K + 1;    // LDS row stride of the tiles
__global__ __launch_bounds__(PK_T) void k_loop_pack(
    int npfb, const int64_t *off, const int *perm, const int *iperm, const int64_t *row_ptr,
    const int *cnt, const int *col_raw, const int *irel, const int *vrel, const double *wx,
    const double *wy, const double *wl, const double *wh, int64_t nnz_max, int *lcol,
    double *lw3, double *lwh, uint8_t *lflip) {
  __shared__ double tx[SV_WAVE * PK_LD], ty[SV_WAVE * PK_LD], tl[SV_WAVE * PK_LD],
      th[SV_WAVE * PK_LD];
  __shared__ int tc[SV_WAVE * PK_LD];
  __shared__ uint8_t tf[SV_WAVE * PK_LD];
  __shared__ int rnode[SV_WAVE], rcnt[SV_WAVE];
  __shared__ int64_t rbase[SV_WAVE];
  const int s = blockIdx.x;
  const int t = threadIdx.x;
  const int64_t o = off[s];
  const int W = (int)((off[s + 1] - o) / SV_WAVE);
  const int k0 = blockIdx.y * PK_K;
  if (k0 >= W) return;
  if (t < SV_WAVE) {
    const int slot = s * SV_WAVE + t;
    const int i = slot < npfb ? perm[slot] : -1;
    rnode[t] = i;
    rcnt[t] = i >= 0 ? cnt[i] : 0;
    rbase[t] = i >= 0 ? row_ptr[i] : 0;
  }
  __syncthreads();
  // gather: 16 consecutive threads read 16 consecutive links of one row
  for (int p = t; p < SV_WAVE * PK_K; p += PK_T) {
    const int r = p / PK_K, kk = p % PK_K, k = k0 + kk;
    const int slot = s * SV_WAVE + r;
    const int e = r * PK_LD + kk;
    if (rnode[r] >= 0 && k < rcnt[r]) {
      const int64_t sidx = rbase[r] + k;
      const int raw = col_raw[sidx];
      tc[e] = iperm[irel[raw]];
      tx[e] = wx[sidx];
      ty[e] = wy[sidx];
      tl[e] = wl[sidx];
      th[e] = wh[sidx];
      const int vr = (lflip && raw >= npfb) ? vrel[raw] : 0;
      tf[e] = (uint8_t)(vr >= 2 ? vr - 1 : 0);
    } else {
      tc[e] = slot < npfb ? slot : 0;
      tx[e] = 0.0;
      ty[e] = 0.0;
      tl[e] = 0.0;
      th[e] = 0.0;
      tf[e] = 0;
    }
  }
  __syncthreads();
  // scatter: 64 consecutive threads write one link's column of the slice
  for (int p = t; p < SV_WAVE * PK_K; p += PK_T) {
    const int kk = p / SV_WAVE, l = p % SV_WAVE, k = k0 + kk;
    if (k >= W) break;
    const int64_t d = o + (int64_t)k * SV_WAVE + l;
    if (d >= nnz_max) break;
    const int e = l * PK_LD + kk;
    lcol[d] = tc[e];
    lw3[sv_w3(d, 0)] = tx[e];
    lw3[sv_w3(d, 1)] = ty[e];
    lw3[sv_w3(d, 2)] = tl[e];
    lwh[sv_pair(d)] = th[e];
    if (lflip) lflip[d] = tf[e];
  }
}

template <typename T>
__global__ void k_permute(int n, const int *perm, const T *src, T *dst) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) dst[k] = src[perm[k]];
}

__global__ void k_invert(int n, int np, const int *perm, int *iperm) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) iperm[perm[k]] = k;
  else if (k < np) iperm[k] = -1;   // ghosts are folded before lookup
}

__global__ void k_iota(int n, int *v) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) v[k] = k;
}

// ---- recursive splitting ---------------------------------------------------
constexpr int KD_BITS = 24;   // coordinate bits of a key

struct KdBox {
  double x0, x1, y0, y1;
};

// key of slot k: (its segment, the coordinate of its node along the longer
// side of the segment's box); segments that are not split any more keep their
// order (equal keys, stable sort)
__global__ void k_kd_key(int n, int nseg, const int *start, const int *left, const KdBox *box,
                         KdBox dom, const double *x, const double *y, const int *ids,
                         uint64_t *key) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  int lo = 0, hi = nseg;   // start[lo] <= k < start[hi]
  while (hi - lo > 1) {
    const int m = (lo + hi) >> 1;
    if (start[m] <= k) lo = m;
    else hi = m;
  }
  uint32_t q = 0;
  if (left[lo] > 0) {
    const KdBox b = box[lo];
    const int i = ids[k];
    const bool along_x = b.x1 - b.x0 >= b.y1 - b.y0;
    const double t = along_x ? (x[i] - dom.x0) / (dom.x1 - dom.x0)
                             : (y[i] - dom.y0) / (dom.y1 - dom.y0);
    const double top = (double)((1u << KD_BITS) - 1);
    q = (uint32_t)fmin(fmax(t * top, 0.0), top);
  }
  key[k] = ((uint64_t)lo << KD_BITS) | q;
}

// boxes of the next level's segments, cut at the first node of the right part
__global__ void k_kd_split(int nseg, const int *start, const int *left, const int *child,
                           const KdBox *box, const double *x, const double *y, const int *ids,
                           KdBox *out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  KdBox a = box[s], b = a;
  const int c = child[s];
  if (left[s] > 0) {
    const int i = ids[start[s] + left[s]];
    if (a.x1 - a.x0 >= a.y1 - a.y0) {
      const double cut = fmin(fmax(x[i], a.x0), a.x1);
      a.x1 = cut;
      b.x0 = cut;
    } else {
      const double cut = fmin(fmax(y[i], a.y0), a.y1);
      a.y1 = cut;
      b.y0 = cut;
    }
    out[c + 1] = b;
  }
  out[c] = a;
}

// ---- SELL offsets -------------------------------------------------------------
// entries of slice s: 64 times its longest list, made even
__global__ void k_slice_width(int n, const int *cnt, int even, int64_t *w) {
  const int s = blockIdx.x, slot = s * SV_WAVE + (int)threadIdx.x;
  int m = slot < n ? cnt[slot] : 0;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o));
  if (threadIdx.x == 0) w[s] = (int64_t)(even ? (m + 1) & ~1 : m) * SV_WAVE;
}

// fewest and most links of the slice's nodes, small and full lists
__global__ void k_slice_range(const int *cnt_small, const int *cnt, int4 *out) {
  const int s = blockIdx.x, slot = s * SV_WAVE + (int)threadIdx.x;
  int4 r{cnt_small[slot], cnt_small[slot], cnt[slot], cnt[slot]};
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    r.x = min(r.x, __shfl_xor(r.x, o));
    r.y = max(r.y, __shfl_xor(r.y, o));
    r.z = min(r.z, __shfl_xor(r.z, o));
    r.w = max(r.w, __shfl_xor(r.w, o));
  }
  if (threadIdx.x == 0) out[s] = r;
}

// ---- halos ----------------------------------------------------------------------
constexpr int HC = 1024;    // largest halo the builder handles (the LDS budget of
                            // the sweeps holds fewer records)
constexpr int HT = 4096;    // hash slots
constexpr int HTHREADS = 256;
constexpr int H_EMPTY = -1;

__device__ __forceinline__ int halo_hash(int key) {
  return (int)(((uint32_t)key * 2654435761u) >> 20);   // 12 bits: HT slots
}
static_assert(HT == 1 << 12, "halo_hash gives 12 bits");

// Distinct link targets of halo block b (slots [b * hb, (b + 1) * hb)), sorted,
// into list[b * HC ..), their number into hcnt[b] (HC + 1 when there are more
// than HC: such a layout has no halo sweeps), and every link's rank into lcol.
// Latency-bound LDS work: 28 KB per workgroup, five workgroups per CU.  PAIRS:
// lcol and the padding by pairs of links (the loop layout), else entry by entry.
template <bool PAIRS>
__global__ __launch_bounds__(HTHREADS) void k_halo(int hb, int nslot, const int64_t *off,
                                                   const int *cnt, const int *col,
                                                   const uint8_t *flip, int *hcnt, int *list,
                                                   uint16_t *lcol) {
  __shared__ int tab[HT];
  __shared__ uint16_t rank[HT];
  __shared__ int uniq[HC];
  __shared__ int nu, over;
  const int t = threadIdx.x, b = blockIdx.x;
  for (int k = t; k < HT; k += HTHREADS) tab[k] = H_EMPTY;
  if (t == 0) { nu = 0; over = 0; }
  __syncthreads();
  const int spb = hb / SV_WAVE, wave = t / SV_WAVE, lane = t % SV_WAVE;
  volatile int *vover = &over;
  for (int q = 0; q < spb; q++) {
    const int s = b * spb + q, slot = s * SV_WAVE + lane;
    if (s * SV_WAVE >= nslot) break;
    const int64_t o = off[s];
    const int K = slot < nslot ? cnt[slot] : 0;
    for (int k = wave; k < K; k += HTHREADS / SV_WAVE) {
      const int64_t e = o + (int64_t)k * SV_WAVE + lane;
      const int key = flip ? col[e] | (int)flip[e] << SV_FLIP_SHIFT : col[e];
      int h = halo_hash(key);
      // at most HT probes; every new key past HC raises the flag, so the
      // table never fills
      for (int p = 0; p < HT && !*vover; p++) {
        const int old = atomicCAS(&tab[h], H_EMPTY, key);
        if (old == key) break;
        if (old == H_EMPTY) {
          const int u = atomicAdd(&nu, 1);
          if (u < HC) uniq[u] = key;
          else *vover = 1;
          break;
        }
        h = (h + 1) & (HT - 1);
      }
    }
  }
  __syncthreads();
  if (over) {
    if (t == 0) hcnt[b] = HC + 1;
    return;
  }
  const int n = nu;
  int m = 2;
  while (m < n) m <<= 1;
  for (int k = n + t; k < m; k += HTHREADS) uniq[k] = INT32_MAX;
  for (int size = 2; size <= m; size <<= 1)      // bitonic, ascending
    for (int d = size >> 1; d > 0; d >>= 1) {
      __syncthreads();
      for (int k = t; k < m / 2; k += HTHREADS) {
        const int i = 2 * d * (k / d) + k % d, j = i + d;
        const int a = uniq[i], c = uniq[j];
        if ((a > c) == ((i & size) == 0)) { uniq[i] = c; uniq[j] = a; }
      }
    }
  __syncthreads();
  for (int k = t; k < n; k += HTHREADS) {
    int h = halo_hash(uniq[k]);
    while (tab[h] != uniq[k]) h = (h + 1) & (HT - 1);   // present: inserted above
    rank[h] = (uint16_t)k;
    list[(size_t)b * HC + k] = uniq[k];
  }
  if (t == 0) hcnt[b] = n;
  __syncthreads();
  for (int q = 0; q < spb; q++) {
    const int s = b * spb + q, slot = s * SV_WAVE + lane;
    if (s * SV_WAVE >= nslot) break;
    const int64_t o = off[s];
    const int K = slot < nslot ? cnt[slot] : 0;
    int W = K;   // the slice's padded length: padding entries get rank 0
#pragma unroll
    for (int o2 = 32; o2 >= 1; o2 >>= 1) W = max(W, __shfl_xor(W, o2));
    if (PAIRS) W = (W + 1) & ~1;
    for (int k = wave; k < W; k += HTHREADS / SV_WAVE) {
      const int64_t e = o + (int64_t)k * SV_WAVE + lane;
      if (k >= K) {
        lcol[PAIRS ? sv_pair(e) : e] = 0;
        continue;
      }
      const int key = flip ? col[e] | (int)flip[e] << SV_FLIP_SHIFT : col[e];
      int h = halo_hash(key);
      while (tab[h] != key) h = (h + 1) & (HT - 1);
      lcol[PAIRS ? sv_pair(e) : e] = rank[h];
    }
  }
}

__global__ void k_halo_compact(const int64_t *hoff, const int *list, int *hidx) {
  const int b = blockIdx.x;
  const int64_t o = hoff[b];
  const int n = (int)(hoff[b + 1] - o);
  for (int k = threadIdx.x; k < n; k += blockDim.x) hidx[o + k] = list[(size_t)b * HC + k];
}

// ---- transposed lists -------------------------------------------------------
// Links pointing at each slot; bad: a target outside the slots.
constexpr int TT = 256;
__global__ __launch_bounds__(TT) void k_t_count(int n, const int64_t *off, const int *cnt,
                                                const int *col, int *tc, int *bad) {
  const int lane = threadIdx.x % SV_WAVE, slot = blockIdx.x * SV_WAVE + lane;
  if (slot >= n) return;
  const int64_t o = off[blockIdx.x] + lane;
  for (int k = threadIdx.x / SV_WAVE; k < cnt[slot]; k += TT / SV_WAVE) {
    const int j = col[o + (int64_t)k * SV_WAVE];
    if ((unsigned)j < (unsigned)n) atomicAdd(&tc[j], 1);
    else *bad = 1;
  }
}

// the links of each target, (source slot, position in its list), in any order
__global__ __launch_bounds__(TT) void k_t_fill(int n, const int64_t *off, const int *cnt,
                                               const int *col, const int64_t *start, int *fill,
                                               uint64_t *key) {
  const int lane = threadIdx.x % SV_WAVE, slot = blockIdx.x * SV_WAVE + lane;
  if (slot >= n) return;
  const int64_t o = off[blockIdx.x] + lane;
  for (int k = threadIdx.x / SV_WAVE; k < cnt[slot]; k += TT / SV_WAVE) {
    const int j = col[o + (int64_t)k * SV_WAVE];
    key[start[j] + atomicAdd(&fill[j], 1)] = (uint64_t)slot << 32 | (uint64_t)k;
  }
}

// One wavefront per target: its links ranked by source slot (each link counts
// the smaller keys: lists are short), then written to the transposed layout.
// Stage weights past the source's small list are zero.
__global__ __launch_bounds__(TT) void k_t_emit(int n, const int64_t *off, const int *cnt_small,
                                               const double *w3, const double *wh,
                                               const int64_t *start, const int *tc,
                                               const uint64_t *key, const int64_t *toff, int *tcol,
                                               double *tw3, double *twh) {
  const int j = blockIdx.x * (TT / SV_WAVE) + threadIdx.x / SV_WAVE;
  if (j >= n) return;
  const int K = tc[j];
  const uint64_t *q = key + start[j];
  for (int a = threadIdx.x % SV_WAVE; a < K; a += SV_WAVE) {
    const uint64_t me = q[a];
    int rank = 0;
    for (int b = 0; b < K; b++) rank += q[b] < me;
    const int i = (int)(me >> 32), k = (int)(me & 0xffffffffu);
    const int64_t e = off[i >> 6] + (int64_t)k * SV_WAVE + (i & 63);
    const int64_t d = toff[j >> 6] + (int64_t)rank * SV_WAVE + (j & 63);
    const bool small = k < cnt_small[i];
    tcol[d] = i;
    for (int w = 0; w < 3; w++) tw3[sv_w3(d, w)] = small ? w3[sv_w3(e, w)] : 0.0;
    twh[sv_pair(d)] = wh[sv_pair(e)];
  }
}

// int -> int64 exclusive scan of n values (out[n - 1] is the sum of the first
// n - 1)
struct ToI64 {
  __device__ __host__ int64_t operator()(int v) const { return v; }
};

template <class In>
int scan_i64(sv_ctx *c, In in, int64_t *out, int n) {
  size_t tb = 0;
  SV_HIP(c, hipcub::DeviceScan::ExclusiveSum(nullptr, tb, in, out, n, c->stream));
  DevTmp<char> tmp;
  SV_HIP(c, tmp.alloc(c, tb > 0 ? tb : 16));
  SV_HIP(c, hipcub::DeviceScan::ExclusiveSum((void *)tmp, tb, in, out, n, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}

// nodes left of the split of a segment of `size` nodes (0: a single slice)
int kd_left(int size) {
  const int slices = (size + SV_WAVE - 1) / SV_WAVE;
  constexpr int SPB = SV_BLOCK / SV_WAVE;
  if (slices <= 1) return 0;
  if (slices <= SPB) return SV_WAVE * (slices / 2);
  return SV_BLOCK * (((slices + SPB - 1) / SPB) / 2);
}

// key of slot k: its block, then its node's links, most first
__global__ void k_len_key(int n, int hb, const int *ids, const int *cnt, uint64_t *key) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) key[k] = (uint64_t)(k / hb) << 16 | (uint64_t)(65535 - min(cnt[ids[k]], 65535));
}

// perm[k] = node in loop slot k; by_len: the nodes of each block sorted by
// their number of links
int kd_order(sv_ctx *c, int *perm, int by_len) {
  const int n = c->npfb, B = 256;
  // the tree's shape depends on n alone: starts, left sizes and first child
  // of every level, concatenated
  std::vector<int> starts, lefts, childs, first;
  std::vector<int> cur{0, n};   // segment bounds of the level
  size_t most = 1;
  for (;;) {
    std::vector<int> nxt;
    const int nseg = (int)cur.size() - 1;
    bool any = false;
    first.push_back((int)starts.size());
    for (int s = 0; s < nseg; s++) {
      const int l = kd_left(cur[s + 1] - cur[s]);
      starts.push_back(cur[s]);
      lefts.push_back(l);
      childs.push_back((int)nxt.size());
      nxt.push_back(cur[s]);
      if (l > 0) { nxt.push_back(cur[s] + l); any = true; }
    }
    most = std::max(most, nxt.size());
    nxt.push_back(n);
    if (!any) break;
    cur.swap(nxt);
  }
  first.push_back((int)starts.size());
  const int levels = (int)first.size() - 2;   // the last level splits nothing
  k_iota<<<(n + B - 1) / B, B, 0, c->stream>>>(n, perm);
  SV_HIP(c, hipGetLastError());
  DevTmp<int> plan, alt;
  DevTmp<uint64_t> key;
  DevTmp<KdBox> boxes;
  DevTmp<char> tmp;
  const size_t P = starts.size();
  size_t tb = 0;
  SV_HIP(c, plan.alloc(c, 3 * P));
  SV_HIP(c, alt.alloc(c, n));
  SV_HIP(c, key.alloc(c, 2 * (size_t)n));
  SV_HIP(c, boxes.alloc(c, 2 * most));
  hipcub::DoubleBuffer<uint64_t> kb(key.p, key.p + n);
  hipcub::DoubleBuffer<int> vb(perm, alt.p);
  SV_HIP(c, hipcub::DeviceRadixSort::SortPairs(nullptr, tb, kb, vb, n, 0, 64, c->stream));
  SV_HIP(c, tmp.alloc(c, tb > 0 ? tb : 16));
  const KdBox dom{c->xmin, c->xmax, c->ymin, c->ymax};
  std::vector<int> h(3 * P);
  std::copy(starts.begin(), starts.end(), h.begin());
  std::copy(lefts.begin(), lefts.end(), h.begin() + P);
  std::copy(childs.begin(), childs.end(), h.begin() + 2 * P);
  SV_HIP(c, hipMemcpyAsync(plan.p, h.data(), sizeof(int) * h.size(), hipMemcpyHostToDevice,
                           c->stream));
  SV_HIP(c, hipMemcpyAsync(boxes.p, &dom, sizeof(dom), hipMemcpyHostToDevice, c->stream));
  for (int l = 0; l < levels; l++) {
    const int nseg = first[l + 1] - first[l];
    const int *st = plan.p + first[l], *lf = plan.p + P + first[l],
              *ch = plan.p + 2 * P + first[l];
    KdBox *in = boxes.p + (l % 2) * most, *out = boxes.p + ((l + 1) % 2) * most;
    int bits = KD_BITS;
    while ((nseg - 1) >> (bits - KD_BITS)) bits++;
    k_kd_key<<<(n + B - 1) / B, B, 0, c->stream>>>(n, nseg, st, lf, in, dom, c->x, c->y,
                                                   vb.Current(), kb.Current());
    SV_HIP(c, hipGetLastError());
    SV_HIP(c, hipcub::DeviceRadixSort::SortPairs((void *)tmp, tb, kb, vb, n, 0, bits,
                                                 c->stream));
    k_kd_split<<<(nseg + B - 1) / B, B, 0, c->stream>>>(nseg, st, lf, ch, in, c->x, c->y,
                                                        vb.Current(), out);
    SV_HIP(c, hipGetLastError());
  }
  if (by_len) {
    int bits = 16;
    while ((n - 1) / by_len >> (bits - 16)) bits++;
    k_len_key<<<(n + B - 1) / B, B, 0, c->stream>>>(n, by_len, vb.Current(), c->cnt, kb.Current());
    SV_HIP(c, hipGetLastError());
    SV_HIP(c, hipcub::DeviceRadixSort::SortPairs((void *)tmp, tb, kb, vb, n, 0, bits,
                                                 c->stream));
  }
  if (vb.Current() != perm)
    SV_HIP(c, hipMemcpyAsync(perm, vb.Current(), sizeof(int) * n, hipMemcpyDeviceToDevice,
                             c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));   // the temporaries go out of scope
  return 0;
}

// Halos of hb slots per block, nslot slots in all.  L.halo stays false when a
// block's halo exceeds the LDS budget of the sweeps (of 64 slots: SV_HALO_MAX).
int build_halos(sv_ctx *c, sv_loopl &L, int hb, int nslot) {
  // whole node blocks, as the sweeps' grids cover them: the halo blocks past
  // the last slot are empty
  const int nb = (nslot + SV_BLOCK - 1) / SV_BLOCK * (SV_BLOCK / hb);
  DevTmp<int> hcnt, list;
  SV_HIP(c, hcnt.alloc(c, (size_t)nb + 1));
  SV_HIP(c, list.alloc(c, (size_t)nb * HC));
  if (!L.lcol) {
    const int nsl = (nslot + SV_BLOCK - 1) / SV_BLOCK * (SV_BLOCK / SV_WAVE);
    if (sv_alloc(c, (void **)&L.lcol, sizeof(uint16_t) * (L.nnz + 1)) ||
        sv_alloc(c, (void **)&L.krange, sizeof(int4) * (size_t)nsl))
      return SV_E_NOMEM;
    k_slice_range<<<nsl, SV_WAVE, 0, c->stream>>>(L.cnt_small, L.cnt, L.krange);
    SV_HIP(c, hipGetLastError());
  }
  k_halo<true><<<nb, HTHREADS, 0, c->stream>>>(hb, nslot, L.off, L.cnt, L.col, L.lflip, hcnt, list,
                                         L.lcol);
  SV_HIP(c, hipGetLastError());
  L.hcnt.resize(nb);
  SV_HIP(c, hipMemcpyAsync(L.hcnt.data(), hcnt.p, sizeof(int) * nb, hipMemcpyDeviceToHost,
                           c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  int64_t tot = 0;
  L.hmax = 0;
  for (int v : L.hcnt) {
    L.hmax = std::max(L.hmax, v);
    tot += v;
  }
  L.halo = L.hmax <= (hb == SV_WAVE ? SV_HALO_MAX : SV_HALO_LDS_MAX / SV_HALO_REC);
  if (!L.halo) return 0;
  L.hb = hb;
  SV_HIP(c, hipMemsetAsync(hcnt.p + nb, 0, sizeof(int), c->stream));
  hipcub::TransformInputIterator<int64_t, ToI64, const int *> in(hcnt.p, ToI64());
  if (sv_alloc(c, (void **)&L.hoff, sizeof(int64_t) * ((size_t)nb + 1)) ||
      sv_alloc(c, (void **)&L.hidx, sizeof(int) * ((size_t)tot + 1)))
    return SV_E_NOMEM;
  if (int rc = scan_i64(c, in, L.hoff, nb + 1)) return rc;
  k_halo_compact<<<nb, HTHREADS, 0, c->stream>>>(L.hoff, list, L.hidx);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}

}  // namespace

// Workgroup size of the sweeps and whether their weights stream past the
// caches, from the node count and the links.  One RK3 step, us, for workgroups
// of 64 / 128 with cached loads, 128 / 256 with non-temporal ones:
//   128^2 order 6 LC   73 /  79,   91 /  128   (few waves: one per workgroup)
//   200^2 order 6 LC   99 / 103,  115 /  142
//   260^2 order 6 LC  140 / 140,  150 /  171
//   301x283 order 8 DI 189 / 180, 192 /  206
//   360^2 order 6 LC  283 / 237,  233 /  232
//   512^2 order 6 LC  588 / 552,  457 /  498   (1024 blocks of 256 leave CUs idle)
//   700^2 order 6 LC    - /1014,  851 /  857
//   1024^2 order 6 LC   - /2082, 1916 / 1882   (fewer halo records per node)
// Cached loads win while a stage's weights and link targets (26 bytes a link)
// stay in the 256 MB Infinity Cache between stages.
// Up to 32768 nodes several wavefronts walk a slice's links, each for its own
// fields: with one, a CU has one or two waves, which wait for one request after
// another.  A step in us, one and several:
//   64^2 order 4 DI     44 / 41     150^2 order 6 LC    85 / 74
//   64^2 order 6 LC     62 / 54     165^2 order 8 DI    89 / 81
//   127^2 order 6 LC    74 / 65     180^2 order 6 LC    90 / 85
//   128^2 order 6 DI    63 / 57
// (Four waves with a quarter of the links each are faster still, 57 at 127^2,
// but then the order of the sums depends on the node count.)
struct Blocks {
  int hb;
  bool nt;
  bool split;
};
static Blocks choose_blocks(int nslot, int64_t links) {
  if (nslot <= 32768) return {64, false, true};
  if (26 * links <= (int64_t)256 << 20) return {128, false, false};
  return {nslot <= 500000 ? 128 : 256, true, false};
}

int sv_dev_build_halos(sv_ctx *c, int nslot) {
  const Blocks b = choose_blocks(nslot, c->L.nnz);
  c->L.nt = b.nt;
  c->L.split = b.split;
  if (int rc = build_halos(c, c->L, b.hb, nslot)) return rc;
  return c->L.halo || b.hb == SV_WAVE ? 0 : build_halos(c, c->L, SV_WAVE, nslot);
}

void sv_free_layout(sv_ctx *c, sv_loopl &L) {
  if (L.cnt_small == L.cnt) L.cnt_small = nullptr;   // transposed lists have the one
  void *old[] = {L.off, L.col, L.w3, L.wh, L.cnt, L.cnt_small, L.gsx, L.gsy,
                 L.lsum, L.hsum, L.vol, L.s, L.perm, L.iperm, L.hoff, L.hidx, L.lcol,
                 L.bidx, L.brec, L.lflip, L.krange};
  for (void *b : old) sv_free(c, b);
  L = sv_loopl{};
}

static int build_layout(sv_ctx *c, int hb) {
  const int n = c->npfb;
  sv_loopl &L = c->L;
  sv_free_layout(c, L);
  const int ns = (n + SV_WAVE - 1) / SV_WAVE;
  L.nslices = ns;
  const size_t D = sizeof(double), I = sizeof(int);
  // whole blocks of counts and slice offsets: no links past the last node
  const int nslot = (n + SV_BLOCK - 1) / SV_BLOCK * SV_BLOCK;
  if (sv_alloc(c, (void **)&L.off, sizeof(int64_t) * (nslot / SV_WAVE + 1)) ||
      sv_alloc(c, (void **)&L.cnt, I * nslot) || sv_alloc(c, (void **)&L.cnt_small, I * nslot) ||
      sv_alloc(c, (void **)&L.gsx, D * n) || sv_alloc(c, (void **)&L.gsy, D * n) ||
      sv_alloc(c, (void **)&L.lsum, D * n) || sv_alloc(c, (void **)&L.hsum, D * n) ||
      sv_alloc(c, (void **)&L.vol, D * n) || sv_alloc(c, (void **)&L.s, D * n) ||
      sv_alloc(c, (void **)&L.perm, I * n) || sv_alloc(c, (void **)&L.iperm, I * c->np))
    return SV_E_NOMEM;
  SV_HIP(c, hipMemsetAsync(L.off, 0, sizeof(int64_t) * (nslot / SV_WAVE + 1), c->stream));
  SV_HIP(c, hipMemsetAsync(L.cnt, 0, I * nslot, c->stream));
  SV_HIP(c, hipMemsetAsync(L.cnt_small, 0, I * nslot, c->stream));
  const int B = 256, nb = (n + B - 1) / B;
  if (c->loop_order) {
    if (int rc = kd_order(c, L.perm, hb == SV_WAVE ? 0 : hb)) return rc;
  } else {
    k_iota<<<nb, B, 0, c->stream>>>(n, L.perm);
    SV_HIP(c, hipGetLastError());
  }
  L.hperm.resize(n);
  SV_HIP(c, hipMemcpyAsync(L.hperm.data(), L.perm, I * n, hipMemcpyDeviceToHost, c->stream));
  k_invert<<<(c->np + B - 1) / B, B, 0, c->stream>>>(n, c->np, L.perm, L.iperm);
  k_permute<int><<<nb, B, 0, c->stream>>>(n, L.perm, c->cnt, L.cnt);
  k_permute<int><<<nb, B, 0, c->stream>>>(n, L.perm, c->cnt_small, L.cnt_small);
  const double *src[6] = {c->gsx, c->gsy, c->lsum, c->hsum, c->vol, c->s};
  double *dst[6] = {L.gsx, L.gsy, L.lsum, L.hsum, L.vol, L.s};
  for (int k = 0; k < 6; k++) k_permute<double><<<nb, B, 0, c->stream>>>(n, L.perm, src[k], dst[k]);
  SV_HIP(c, hipGetLastError());
  {
    DevTmp<int64_t> w;
    SV_HIP(c, w.alloc(c, (size_t)ns + 1));
    SV_HIP(c, hipMemsetAsync(w.p + ns, 0, sizeof(int64_t), c->stream));
    k_slice_width<<<ns, SV_WAVE, 0, c->stream>>>(n, L.cnt, 1, w);
    SV_HIP(c, hipGetLastError());
    if (int rc = scan_i64(c, (const int64_t *)w.p, L.off, ns + 1)) return rc;
  }
  SV_HIP(c, hipMemcpy(&L.nnz, L.off + ns, sizeof(int64_t), hipMemcpyDeviceToHost));
  const size_t E = (size_t)L.nnz + 1;
  if (sv_alloc(c, (void **)&L.col, I * E) || sv_alloc(c, (void **)&L.w3, 3 * D * E) ||
      sv_alloc(c, (void **)&L.wh, D * E))
    return SV_E_NOMEM;
  if (c->has_mirror && sv_alloc(c, (void **)&L.lflip, E)) return SV_E_NOMEM;
  if (c->maxK > 0) {
    dim3 grid(ns, (c->maxK + 1 + PK_K - 1) / PK_K);
    k_loop_pack<<<grid, PK_T, 0, c->stream>>>(n, L.off, L.perm, L.iperm, c->row_ptr, c->cnt,
                                              c->col_raw, c->irel, c->vrel, c->wx, c->wy, c->wl,
                                              c->wh, L.nnz, L.col, L.w3, L.wh, L.lflip);
    SV_HIP(c, hipGetLastError());
  }
  if (c->halo_sweeps)
    if (int rc = build_halos(c, L, hb, n)) return rc;
  SV_HIP(c, hipStreamSynchronize(c->stream));
  L.valid = true;
  return 0;
}

int sv_dev_build_loop(sv_ctx *c) {
  const Blocks b = choose_blocks(c->npfb, c->nnz);
  if (int rc = build_layout(c, b.hb)) return rc;
  if (!c->L.halo && c->halo_sweeps && b.hb != SV_WAVE) {
    c->L.valid = false;   // halos too large: the smallest blocks
    if (int rc = build_layout(c, SV_WAVE)) return rc;
  }
  c->L.nt = b.nt && c->L.hb != SV_WAVE;
  c->L.split = b.split;
  return 0;
}

// The transposed lists of the loop layout: for each slot j the links (i, k) that
// point at it, by ascending i, with the halos of 64-slot blocks.  (On the host
// this was 30 ms of a 16k-node gradient's first 48.)
int sv_dev_build_transpose(sv_ctx *c, sv_loopl &T) {
  const sv_loopl &L = c->L;
  const int n = c->npfb, ns = L.nslices;
  const int nslot = (n + SV_BLOCK - 1) / SV_BLOCK * SV_BLOCK;
  T.nslices = ns;
  if (sv_alloc(c, (void **)&T.off, sizeof(int64_t) * (nslot / SV_WAVE + 1)) ||
      sv_alloc(c, (void **)&T.cnt, sizeof(int) * nslot))
    return SV_E_NOMEM;
  T.cnt_small = T.cnt;
  DevTmp<int> fill, bad;
  DevTmp<int64_t> start, w;
  SV_HIP(c, fill.alloc(c, n));
  SV_HIP(c, bad.alloc(c, 1));
  SV_HIP(c, start.alloc(c, (size_t)n + 1));
  SV_HIP(c, w.alloc(c, (size_t)ns + 1));
  SV_HIP(c, hipMemsetAsync(T.off, 0, sizeof(int64_t) * (nslot / SV_WAVE + 1), c->stream));
  SV_HIP(c, hipMemsetAsync(T.cnt, 0, sizeof(int) * nslot, c->stream));
  SV_HIP(c, hipMemsetAsync(fill, 0, sizeof(int) * n, c->stream));
  SV_HIP(c, hipMemsetAsync(bad, 0, sizeof(int), c->stream));
  SV_HIP(c, hipMemsetAsync(w.p + ns, 0, sizeof(int64_t), c->stream));
  k_t_count<<<ns, TT, 0, c->stream>>>(n, L.off, L.cnt, L.col, T.cnt, bad);
  k_slice_width<<<ns, SV_WAVE, 0, c->stream>>>(n, T.cnt, 1, w);
  SV_HIP(c, hipGetLastError());
  if (int rc = scan_i64(c, (const int64_t *)w.p, T.off, ns + 1)) return rc;
  int64_t links = 0;
  {
    DevTmp<int> one;   // the counts and a last zero, for an exclusive scan of n + 1
    SV_HIP(c, one.alloc(c, (size_t)n + 1));
    SV_HIP(c, hipMemcpyAsync(one, T.cnt, sizeof(int) * n, hipMemcpyDeviceToDevice, c->stream));
    SV_HIP(c, hipMemsetAsync(one.p + n, 0, sizeof(int), c->stream));
    hipcub::TransformInputIterator<int64_t, ToI64, const int *> in(one.p, ToI64());
    if (int rc = scan_i64(c, in, start, n + 1)) return rc;   // synchronises
  }
  int hbad = 0;
  SV_HIP(c, hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipMemcpyAsync(&links, start.p + n, sizeof(int64_t), hipMemcpyDeviceToHost,
                           c->stream));
  SV_HIP(c, hipMemcpyAsync(&T.nnz, T.off + ns, sizeof(int64_t), hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  if (hbad) return sv_fail(c, SV_E_STATE, "stencil column out of range");
  const size_t E = (size_t)T.nnz + 1;
  DevTmp<uint64_t> key;
  SV_HIP(c, key.alloc(c, (size_t)links));
  if (sv_alloc(c, (void **)&T.col, sizeof(int) * E) ||
      sv_alloc(c, (void **)&T.w3, 3 * sizeof(double) * E) ||
      sv_alloc(c, (void **)&T.wh, sizeof(double) * E))
    return SV_E_NOMEM;
  k_t_fill<<<ns, TT, 0, c->stream>>>(n, L.off, L.cnt, L.col, start, fill, key);
  k_t_emit<<<(n + TT / SV_WAVE - 1) / (TT / SV_WAVE), TT, 0, c->stream>>>(
      n, L.off, L.cnt_small, L.w3, L.wh, start, T.cnt, key, T.off, T.col, T.w3, T.wh);
  SV_HIP(c, hipGetLastError());
  if (int rc = build_halos(c, T, SV_WAVE, n)) return rc;
  SV_HIP(c, hipStreamSynchronize(c->stream));   // the temporaries go out of scope
  return 0;
}

// Slice offsets of lists of cnt[n] links (exact widths), on the device
int sv_dev_slice_offsets(sv_ctx *c, int n, const int *cnt, int64_t *off, int64_t *total) {
  const int ns = (n + SV_WAVE - 1) / SV_WAVE;
  DevTmp<int64_t> w;
  SV_HIP(c, w.alloc(c, (size_t)ns + 1));
  SV_HIP(c, hipMemsetAsync(w.p + ns, 0, sizeof(int64_t), c->stream));
  k_slice_width<<<ns, SV_WAVE, 0, c->stream>>>(n, cnt, 0, w);
  SV_HIP(c, hipGetLastError());
  if (int rc = scan_i64(c, (const int64_t *)w.p, off, ns + 1)) return rc;
  SV_HIP(c, hipMemcpyAsync(total, off + ns, sizeof(int64_t), hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}

// Halos of the drop-in layout's slices (folded columns), for the operators.
// shmax 0: none (a slice has more than HC distinct neighbours, or no memory).
int sv_dev_sell_halos(sv_ctx *c) {
  const int n = c->npfb, ns = c->nslices;
  c->shmax = 0;
  DevTmp<int> hcnt, list;
  SV_HIP(c, hcnt.alloc(c, (size_t)ns + 1));
  if (list.alloc(c, (size_t)ns * HC) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  if ((!c->slcol && sv_alloc(c, (void **)&c->slcol, sizeof(uint16_t) * ((size_t)c->sell_nnz + 1))) ||
      (!c->shoff && sv_alloc(c, (void **)&c->shoff, sizeof(int64_t) * ((size_t)ns + 1)))) {
    (void)hipGetLastError();
    return 0;
  }
  k_halo<false><<<ns, HTHREADS, 0, c->stream>>>(SV_WAVE, n, c->sell_off, c->cnt, c->scol, nullptr,
                                                hcnt, list, c->slcol);
  SV_HIP(c, hipGetLastError());
  std::vector<int> hc(ns);
  SV_HIP(c, hipMemcpyAsync(hc.data(), hcnt.p, sizeof(int) * ns, hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  int most = 0;
  int64_t tot = 0;
  for (int v : hc) {
    most = std::max(most, v);
    tot += v;
  }
  if (most > HC) return 0;
  if (tot > c->shcap) {
    sv_free(c, c->shidx);
    c->shidx = nullptr;
    c->shcap = 0;
    if (sv_alloc(c, (void **)&c->shidx, sizeof(int) * ((size_t)tot + 1))) {
      (void)hipGetLastError();
      return 0;
    }
    c->shcap = tot;
  }
  SV_HIP(c, hipMemsetAsync(hcnt.p + ns, 0, sizeof(int), c->stream));
  hipcub::TransformInputIterator<int64_t, ToI64, const int *> in(hcnt.p, ToI64());
  if (int rc = scan_i64(c, in, c->shoff, ns + 1)) return rc;
  k_halo_compact<<<ns, HTHREADS, 0, c->stream>>>(c->shoff, list, c->shidx);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipStreamSynchronize(c->stream));
  c->shmax = most;
  return 0;
}
