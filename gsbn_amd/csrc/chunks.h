/*
 * chunks.h -- arrays carved from a few large allocations.
 *
 * Source::take(size, most, &got) allocates at least `size` bytes (`most`: what
 * a kept allocation may have at most) and returns null when there are none.
 */
#ifndef GSBN_CHUNKS_H
#define GSBN_CHUNKS_H

#include <algorithm>
#include <cstddef>
#include <map>
#include <vector>

namespace gsbn {

template <class Source>
class Chunks {
 public:
  struct Chunk {
    char* base;
    size_t size, used;
  };
  explicit Chunks(Source s) : _source(s) {}
  const std::vector<Chunk>& chunks() const { return _chunks; }

  /* 256-byte aligned; null when memory is out */
  void* alloc(size_t bytes) {
    const size_t need = (std::max<size_t>(bytes, 1) + 255) & ~(size_t)255;
    /* a released array of at most twice the size */
    auto f = _free.lower_bound(need);
    if (f != _free.end() && f->first <= 2 * need) {
      void* p = f->second;
      _live[p] = f->first;
      _free.erase(f);
      return p;
    }
    /* the chunk with the smallest tail that holds it */
    Chunk* at = nullptr;
    for (auto& c : _chunks)
      if (c.size - c.used >= need && (!at || c.size - c.used < at->size - at->used)) at = &c;
    if (!at) at = add(need);
    if (!at) return nullptr;
    void* p = at->base + at->used;
    _live[p] = need;
    at->used += need;
    return p;
  }

  void release(void* p) {
    auto it = _live.find(p);
    if (it == _live.end()) return;
    _free.emplace(it->second, p);
    _live.erase(it);
  }

 private:
  /* Shared chunks have half of what there is in shared ones already, or a
   * sixteenth of everything, from 4 MB to 1 GB, so that there are few of them.
   * An array above a quarter of that has a chunk of its own, with nothing left
   * over.  (With all arrays in shared chunks, none of several large equal ones
   * fits another's tail: 40 networks of 540 MB and eight arrays of 12 MB left
   * 39 % of their memory unused, a network of 100 x 100 27 %; now 1 % in 55
   * allocations, and 0.5 % in 2.  128 networks of 8-64 hypercolumns 1.7 % in
   * 44, 512 0.2 % in 115.) */
  Chunk* add(size_t need) {
    const size_t mb = (size_t)1 << 20;
    const size_t shared = std::min(std::max(std::max(_shared / 2, _total / 16), 4 * mb), 1024 * mb);
    const bool own = need > shared / 4;
    const size_t unit = own ? (size_t)4096 : 2 * mb;
    const size_t want = ((own ? need : shared) + unit - 1) / unit * unit;
    size_t got = 0;
    char* base = _source.take(want, own ? want + want / 16 : 2 * want, &got);
    if (!base && want > need) base = _source.take(need, need, &got);
    if (!base) return nullptr;
    _chunks.push_back({base, got, 0});
    _total += got;
    if (!own) _shared += got;
    return &_chunks.back();
  }

  Source _source;
  std::vector<Chunk> _chunks;
  std::map<void*, size_t> _live;
  std::multimap<size_t, void*> _free; /* released arrays by size */
  size_t _shared = 0, _total = 0;     /* bytes of the shared chunks, of all */
};

}  // namespace gsbn

#endif /* GSBN_CHUNKS_H */
