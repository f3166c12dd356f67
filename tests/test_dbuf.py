"""Device arrays of a recall handle (dbuf.h) when an allocation fails, compiled
for the host on a stand-in for the runtime whose allocations fail on demand: a
failed array is empty, and the next use of the handle makes it anew."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#pragma once
#include <stdlib.h>
#include <string.h>
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipMemcpyHostToDevice = 1 };
extern int fail_next, live, sticky;
template <typename T> hipError_t hipMalloc(T** p, size_t n) {
  if (fail_next > 0) { --fail_next; sticky = hipErrorOutOfMemory; return hipErrorOutOfMemory; }
  *p = (T*)malloc(n); ++live; return hipSuccess;
}
inline hipError_t hipFree(void* p) { free(p); --live; return hipSuccess; }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipGetLastError() { int e = sticky; sticky = 0; return e; }
"""

SOURCE = r"""
#include <stdio.h>
#include "dbuf.h"
int fail_next, live, sticky, released;
extern "C" int gsbn_memory_release(void) { ++released; return 0; }
#define CHECK(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }
int main() {
  {
    DBuf<int> b;
    CHECK(b.alloc(10) == hipSuccess && b.n == 10 && b.p && live == 1);
    fail_next = 1;  /* the second try is without the kept memory */
    CHECK(b.alloc(100) == hipSuccess && b.n == 100 && b.p && released == 1 && sticky == 0);
    fail_next = 2;
    CHECK(b.alloc(1000) == hipErrorOutOfMemory && released == 2);
    CHECK(b.n == 0 && !b.p && live == 0 && sticky == 0);
    CHECK(b.n < 50);  /* a use that needs less than the failed one makes it */
    CHECK(b.alloc(50) == hipSuccess && b.n == 50 && b.p);
    const int v[3] = {1, 2, 3};
    fail_next = 2;
    CHECK(b.upload(v, 3) == hipErrorOutOfMemory && b.n == 0 && !b.p);
    CHECK(b.upload(v, 3) == hipSuccess && b.n == 3 && b.p[2] == 3);
    CHECK(b.alloc(0) == hipSuccess && b.n == 0 && !b.p && live == 0);
    CHECK(b.alloc(7) == hipSuccess);
  }
  CHECK(live == 0);
  printf("ok\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_a_failed_allocation_leaves_an_empty_array(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    src = tmp_path / "t.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "gsbn_amd", "csrc"), "-o", exe, str(src)], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
