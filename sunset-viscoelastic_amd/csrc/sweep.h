// sweep.h -- what the halo-staged sweeps over the loop layout share (the RK
// stages and the filter, k_step.hip; their transposes, k_adjoint.hip): staging
// of a block's neighbour records in LDS, the streamed link arrays, and the walk
// over a slice's links.
#ifndef SV_SWEEP_H
#define SV_SWEEP_H
#include "sv_internal.h"

namespace {

typedef double dbl2 __attribute__((ext_vector_type(2)));

// Reductions over a wavefront in a fixed order (every lane ends with the
// result).  The partial results of the node kernels are per 64-slot slice, so
// they do not depend on the workgroup size a sweep runs with.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}

// Records a thread stages at once: a usual halo (~600 records per 256 slots,
// ~270 per 64) in one round of requests, since a round costs two dependent
// trips to memory (key, record).
// NB slots per workgroup, NT threads.
template <int NB, int NT>
struct HaloC {
  static constexpr int C = NB < NT ? (NT == 128 ? 3 : 2) : NB == SV_WAVE ? 5 : NB == 128 ? 4 : 3;
};

// The halo keys of this thread's records h, h + NT, ... of a round; past the
// end the last key (a valid record, not stored)
template <int NB, int NT>
struct HaloKeys {
  static constexpr int C = HaloC<NB, NT>::C;
  int key[C];
  __device__ __forceinline__ void get(const int *hx, int h, int nh) {
#pragma unroll
    for (int c = 0; c < C; c++) key[c] = hx[min(h + c * NT, nh - 1)];
  }
};

// The block's halo to LDS: load(key) reads a record, put(h, key, record)
// stores it as record h.  keys holds the first round's keys.
template <int NB, int NT, class Load, class Put>
__device__ __forceinline__ void halo_stage(const int *hx, int nh, HaloKeys<NB, NT> &keys,
                                           Load load, Put put) {
  constexpr int C = HaloC<NB, NT>::C;
  auto round = [&](int h) {
    decltype(load(0)) r[C];
#pragma unroll
    for (int c = 0; c < C; c++) r[c] = load(keys.key[c] & SV_FLIP_MASK);
#pragma unroll
    for (int c = 0; c < C; c++)
      if (h + c * NT < nh) put(h + c * NT, keys.key[c] >> SV_FLIP_SHIFT, r[c]);
  };
  // the first round apart: its requests wait for the keys only, not for the
  // links requested after them
  if (nh > 0) round(threadIdx.x);
  for (int h = threadIdx.x + C * NT; h < nh; h += C * NT) {
    keys.get(hx, h, nh);
    round(h);
  }
}

// One streamed array of a wavefront's slice (W groups of 64 values of 4 or 16
// bytes per pair of links), read through a buffer descriptor of exactly the
// slice's pairs: a batch costs one address addition (the pairs within it are
// immediate offsets), and entries past them read as 0 by the hardware's range
// check, which covers the vector and immediate offsets used here (it leaves
// out the scalar one, kept 0), so the requests need no guards.
template <typename T, int W, bool NT>
struct Stream {
  __amdgpu_buffer_rsrc_t r;
  // n: links of the slice's longest list
  __device__ __forceinline__ Stream(const void *base, int n)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0,
                                            (n + 1) / 2 * W * SV_WAVE * (int)sizeof(T),
                                            0x00020000)) {}
  // group c of the u-th pair from position p (entry_at)
  __device__ __forceinline__ T at(int p, int u, int c) const {
    const int vo = p * W * (int)sizeof(T) + (int)(threadIdx.x & (SV_WAVE - 1)) * (int)sizeof(T) +
                   (u * W + c) * SV_WAVE * (int)sizeof(T);
    constexpr int aux = NT ? 2 : 0;   // nt
    if constexpr (sizeof(T) == 16)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, vo, 0, aux));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, vo, 0, aux));
  }
};

// Position of link pair k / 2 in its slice (64 per pair), kept opaque so that
// the pairs after it stay immediate offsets (the loop's strength reduction
// would otherwise carry one address per pair)
__device__ __forceinline__ int entry_at(int k) {
  int p = k / 2 * SV_WAVE;
  asm volatile("" : "+v"(p));
  return p;
}

// The links of one wavefront's slice, walked in batches of U pairs with the
// next batch's global streams in flight while a batch is consumed (two register
// sets, no copies between them), and each link's LDS record requested before
// the link before it is summed.  Batches that reach past the shortest list of
// the slice send the requests of lanes past their own list out of range (no
// memory traffic for the padding; they read record 0) and guard the sums.
//   load(set, u, p)  requests the u-th pair from position p into entry u
//   fetch(set, l)    the LDS record of link l of the set's 2U
//   link(r, set, l)  adds it, with its record r
// The share of a slice's links that one of NW wavefronts walks: whole pairs,
// the same for all lanes; k0 its first link.
template <int NW>
struct Share {
  int k0, K, KF, KM;   // first link; this lane's, fewest and most links of the share
  __device__ __forceinline__ Share(int w, int k, int kf, int km) {
    const int n = 2 * (((km + 1) / 2 + NW - 1) / NW);
    k0 = w * n;
    auto part = [&](int v) { return min(max(v - k0, 0), n); };
    K = part(k);
    KF = part(kf);
    KM = part(km);
  }
};

constexpr int OUT_OF_RANGE = 1 << 22;   // past every list, in pairs times 64
template <int U, class Rec, class Load, class Fetch, class Link>
__device__ __forceinline__ void walk_links(int K, int KF, int KM, Load load, Fetch fetch,
                                           Link link) {
  constexpr int V = 2 * U;   // links of a batch
  auto fill = [&](int s, int k0) {
    const int p = entry_at(k0);
#pragma unroll
    for (int u = 0; u < U; u++) load(s, u, p);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto fill_guarded = [&](int s, int k0) {
    const int p = entry_at(k0);
#pragma unroll
    for (int u = 0; u < U; u++) load(s, u, k0 + 2 * u < K ? p : OUT_OF_RANGE);
    __builtin_amdgcn_sched_barrier(0);
  };
  int k = 0;
  Rec r = fetch(0, 0);
  for (; k + 3 * V <= KF; k += 2 * V) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      fill(1 - s, k + (1 + s) * V);
#pragma unroll
      for (int l = 0; l < V; l++) {
        const Rec n = l + 1 < V ? fetch(s, l + 1) : fetch(1 - s, 0);
        __builtin_amdgcn_sched_barrier(0);
        link(r, s, l);
        r = n;
      }
    }
  }
  for (; k < KM; k += 2 * V) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      fill_guarded(1 - s, k + (1 + s) * V);
#pragma unroll
      for (int l = 0; l < V; l++) {
        const Rec n = l + 1 < V ? fetch(s, l + 1) : fetch(1 - s, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (k + s * V + l < K) link(r, s, l);
        r = n;
      }
    }
  }
}

// The sums that wave w of a workgroup made for the slice of wave 0, through LDS
// (which may be the halo's area): give by the waves that made them, take by wave
// 0, between them a barrier.  each(f) calls f on every sum.
constexpr size_t part_doubles(int n) { return (size_t)n * SV_WAVE; }

template <class Each>
__device__ __forceinline__ void give_sums(double *lds, Each each) {
  double *p = lds + ((int)threadIdx.x & (SV_WAVE - 1));
  each([&](double &v) { *p = v; p += SV_WAVE; });
}
template <class Each>
__device__ __forceinline__ void take_sums(const double *lds, Each each) {
  const double *p = lds + ((int)threadIdx.x & (SV_WAVE - 1));
  each([&](double &v) { v = *p; p += SV_WAVE; });
}

}  // namespace

#endif
