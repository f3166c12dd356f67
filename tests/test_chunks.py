"""Arrays carved from few allocations (chunks.h), compiled for the host with a
source that only counts: what is left over for the arrays of batches and single
networks, alignment, no overlap, reuse of released arrays, and memory that runs
out."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdint.h>
#include <stdio.h>
#include "chunks.h"
struct Device { size_t at = (size_t)1 << 40, room = (size_t)1 << 50, taken = 0; int calls = 0; };
struct Source {
  Device* d;
  char* take(size_t size, size_t most, size_t* got) {
    if (most < size || size > d->room) return nullptr;
    ++d->calls;
    d->room -= size;
    d->taken += size;
    *got = size;
    char* p = (char*)d->at;
    d->at += (size + 4095) / 4096 * 4096 + 4096; /* never adjacent */
    return p;
  }
};
typedef gsbn::Chunks<Source> Arrays;
#define CHECK(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }
static uint64_t s = 88172645463325252ull;
static uint64_t rnd() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s >> 11; }
int main() {
  const size_t mb = 1000000;
  { /* 40 equal networks of a large array and smaller ones */
    Device d; Arrays a(Source{&d}); size_t live = 0;
    for (int i = 0; i < 40; ++i) {
      auto add = [&](size_t n) { live += n; return a.alloc(n) != nullptr; };
      CHECK(add(540 * mb));
      for (int k = 0; k < 8; ++k) CHECK(add(12 * mb));
      for (int k = 0; k < 30; ++k) CHECK(add(40000));
    }
    CHECK(d.taken < live + live / 20 && d.calls < 80);
  }
  { /* one network of 100 x 100 */
    Device d; Arrays a(Source{&d}); size_t live = 0;
    for (size_t n : {2376 * mb, 16 * mb, 4 * mb, 4 * mb, 4 * mb, 99 * mb, 8 * mb}) live += n, a.alloc(n);
    for (int k = 0; k < 40; ++k) live += 40000, a.alloc(40000);
    CHECK(d.taken < live + live / 20 && d.calls < 8);
  }
  for (int nets : {128, 512}) { /* batches of 8-64 hypercolumns of 16-128 units */
    Device d; Arrays a(Source{&d}); size_t live = 0;
    for (int i = 0; i < nets; ++i) {
      const size_t H = 8 + rnd() % 57, M = 16 + rnd() % 113, C = (1 + 4 * (rnd() % 3)) * (H - 1) * M / 10;
      for (size_t n : {H * C * M * 24, H * C * M, H * C * 16, H * C * 4, H * C * 4, 8 * H * C, H * M * 256})
        live += n, a.alloc(n);
      for (int k = 0; k < 30; ++k) live += H * M * 4, a.alloc(H * M * 4);
    }
    CHECK(d.taken < live + live / 20 && d.calls < nets);
  }
  { /* placed apart and aligned; a released array serves one of about its size */
    Device d; Arrays a(Source{&d});
    std::map<char*, size_t> live;
    for (int i = 0; i < 20000; ++i) {
      if (live.size() > 300 || (live.size() > 3 && rnd() % 3 == 0)) {
        auto it = live.begin();
        for (size_t k = rnd() % live.size(); k; --k) ++it;
        a.release(it->first);
        live.erase(it);
        continue;
      }
      const size_t n = 1 + rnd() % ((size_t)1 << (4 + rnd() % 24));
      char* p = (char*)a.alloc(n);
      CHECK(p && ((uintptr_t)p & 255) == 0);
      auto next = live.lower_bound(p);
      CHECK(next == live.end() || p + n <= next->first);
      CHECK(next == live.begin() || std::prev(next)->first + std::prev(next)->second <= p);
      bool in = false;
      for (auto& c : a.chunks()) in = in || (p >= c.base && p + n <= c.base + c.used && c.used <= c.size);
      CHECK(in);
      live[p] = n;
    }
    a.release((char*)8); /* not one of them */
    CHECK(a.alloc(0) != nullptr);
  }
  {
    Device d; Arrays a(Source{&d});
    void* p = a.alloc(5000);
    a.release(p);
    CHECK(a.alloc(2000) != p); /* less than half of it */
    CHECK(a.alloc(4000) == p);
  }
  { /* out of memory: exactly what is asked for is tried, then null, and the rest goes on */
    Device d; Arrays a(Source{&d});
    d.room = 1 << 20;
    CHECK(a.alloc(100 << 10) && d.taken < (1 << 20));
    CHECK(a.alloc(2 << 20) == nullptr);
    CHECK(a.alloc(100 << 10));
  }
  printf("ok\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_arrays_from_chunks(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "gsbn_amd", "csrc"),
                    "-o", exe, str(src)], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
