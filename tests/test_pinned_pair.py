"""The pinned buffers of the closure's inference when an allocation fails:
after a failure at any point, the next call completes the pair (a null second
buffer would be written by the first call of more than one chunk), nothing is
made twice and nothing is left behind.  CPU: the header against counting
stand-ins of the HIP calls."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <stdlib.h>
typedef int hipError_t;
typedef void *hipEvent_t;
enum { hipSuccess = 0, hipHostMallocDefault = 0, hipEventDisableTiming = 0 };
inline int &calls() { static int n = 0; return n; }
inline int &fail_at() { static int n = -1; return n; }
inline int &live() { static int n = 0; return n; }
inline hipError_t take(void **p) {
  if (calls()++ == fail_at()) return 2;
  *p = malloc(8);
  ++live();
  return hipSuccess;
}
inline hipError_t give(void *p) { free(p); --live(); return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t, unsigned) { return take(p); }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return take(e); }
inline hipError_t hipHostFree(void *p) { return give(p); }
inline hipError_t hipEventDestroy(hipEvent_t e) { return give(e); }
"""

MAIN = r"""
#include "ibg_pinned.h"
int main() {
  for (int f = -1; f < 4; ++f) {
    ibg::PinnedPair p;
    calls() = 0;
    fail_at() = f;
    if (p.make(8) != (f < 0)) return 1;
    if (f >= 0 && !p.make(8)) return 2;
    if (!p.make(8)) return 3;
    for (int b = 0; b < 2; ++b)
      if (!p.buf[b] || !p.done[b]) return 4;
    if (live() != 4) return 5;
    p.release();
    if (live() != 0) return 6;
  }
  return 0;
}
"""


def test_a_failed_allocation_is_made_up_for(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    dev = os.path.join(ROOT, "immsered-boundary_amd", "csrc", "device")
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", f"-I{tmp_path}", f"-I{dev}", str(tmp_path / "main.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe]).returncode == 0
