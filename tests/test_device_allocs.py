"""Device arrays that are allocated together (sv_alloc_all): all of them or none, so
that a call refused for want of memory can be made again and finds no half of what
it needs.  As test_device_memory.py, over a hipMalloc of 100 bytes."""
import os
import subprocess

import pytest

from test_device_memory import CSRC, HIPCC, PROGRAM

STUBS, _ = PROGRAM.split("// 80 of the 100 bytes")
MAIN = r"""
int main() {
  sv_ctx c;
  int *a = nullptr;
  double *b = nullptr, *d = nullptr;
  CHECK(sv_alloc_all(&c, {sv_want(&a, 5), sv_want(&b, 5), sv_want(&d, 6)}) == SV_E_NOMEM);
  CHECK(!a && !b && !d && total == 0 && c.allocs.empty());       // 20 + 40 + 48
  CHECK(hipGetLastError() == hipSuccess);
  CHECK(sv_alloc_all(&c, {sv_want(&a, 5), sv_want(&b, 5), sv_want(&d, 5)}) == 0);
  CHECK(a && b && d && total == 100 && c.allocs.size() == 3);
  int *e = a;                                                    // beside others
  CHECK(sv_alloc_all(&c, {sv_want(&e, 1)}) == SV_E_NOMEM && !e && total == 100);
  sv_free(&c, a);
  sv_free(&c, b);
  sv_free(&c, d);
  {
    void *p;                                                     // blocks of a set before count
    CHECK(sv_alloc(&c, &p, 60) == 0);
    c.spare.swap(c.allocs);
    CHECK(sv_alloc_all(&c, {sv_want(&b, 7), sv_want(&d, 7)}) == SV_E_NOMEM);   // 56 in 60, 56
    CHECK(!b && !d && total == 0 && c.spare.empty() && c.allocs.empty());
    CHECK(sv_alloc_all(&c, {sv_want(&b, 6), sv_want(&d, 6)}) == 0 && total == 96);
  }
  return failures != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_all_or_none(tmp_path):
    src, exe = tmp_path / "allocs.hip", tmp_path / "allocs"
    src.write_text(STUBS + MAIN)
    r = subprocess.run([HIPCC, "-std=c++17", "-O1", "--offload-host-only", "-x", "hip",
                        f"-I{CSRC}", str(src), os.path.join(CSRC, "sv_mem.hip"), "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
