// sv_mem.hip -- device memory of a context (host code only).
#include <algorithm>

#include "sv_internal.h"

// A new node set takes over the blocks of the one before it that fit (spare, at
// most a quarter larger than asked for): hipFree and hipMalloc of ~60 blocks were
// 14 of the 24 ms of a 262k-node start-up.  What is left of them is given back
// once the set-up is complete or has got as far as a caller takes it (a first
// state or operator, the weights copied out, adapted stencils), when an
// allocation of this context fails, temporaries included, with the next node
// set, and with the context; more than SV_SPARE_MAX is given back at once (a
// set-up of that size takes 0.1 s).
hipError_t sv_dev_malloc(sv_ctx *c, void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess && !c->spare.empty()) {
    (void)hipGetLastError();
    sv_release_spare(c);
    e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();   // told here: not to the check of a later launch
  }
  return e;
}

int sv_alloc(sv_ctx *c, void **p, size_t bytes) {
  if (bytes == 0) bytes = 16;
  size_t best = c->spare.size();
  for (size_t k = 0; k < c->spare.size(); k++) {
    const size_t have = c->spare[k].bytes;
    if (have >= bytes && have - bytes <= bytes / 4 &&
        (best == c->spare.size() || have < c->spare[best].bytes))
      best = k;
  }
  if (best < c->spare.size()) {
    c->allocs.push_back(c->spare[best]);
    c->spare.erase(c->spare.begin() + best);
    *p = c->allocs.back().p;
    return 0;
  }
  const hipError_t e = sv_dev_malloc(c, p, bytes);
  if (e != hipSuccess)
    return sv_fail(c, SV_E_NOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
  c->allocs.push_back(sv_blk{*p, bytes});
  return 0;
}

int sv_alloc_all(sv_ctx *c, std::initializer_list<sv_req> reqs) {
  for (const sv_req &r : reqs) *r.p = nullptr;
  for (const sv_req &r : reqs)
    if (int rc = sv_alloc(c, r.p, r.bytes)) {
      for (const sv_req &q : reqs) {
        sv_free(c, *q.p);
        *q.p = nullptr;
      }
      return rc;
    }
  return 0;
}

size_t sv_spare_bytes(const sv_ctx *c) {
  size_t n = 0;
  for (const sv_blk &b : c->spare) n += b.bytes;
  return n;
}

void sv_release_spare(sv_ctx *c) {
  for (const sv_blk &b : c->spare) (void)hipFree(b.p);
  c->spare.clear();
}

void sv_free(sv_ctx *c, void *p) {
  if (!p) return;
  auto it = std::find_if(c->allocs.begin(), c->allocs.end(),
                         [p](const sv_blk &b) { return b.p == p; });
  if (it != c->allocs.end()) c->allocs.erase(it);
  (void)hipFree(p);
}
