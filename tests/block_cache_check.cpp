// Checks thg::BlockCache (thea_amd/csrc/block_cache.hpp) over a model of a driver with a fixed amount of
// memory on each of two devices. Prints the name of each check that fails; exit status = their number.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <new>

#include "block_cache.hpp"

static bool no_memory = false;  // host allocations fail
void *operator new(std::size_t n) {
  void *p = no_memory ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

struct Model {
  size_t capacity = 1000, used[2] = {0, 0}, pooled[2] = {0, 0};
  int current = 0, allocs = 0, asyncs = 0;
  bool idle = true;
  uintptr_t next = 4096;
  std::map<void *, std::pair<size_t, int>> live;  // bytes, device
};

struct ModelDriver {
  using Error = int;
  using Stream = int;
  Model *m;
  static Error success() { return 0; }
  static bool out_of_memory(Error e) { return e == 2; }
  Error alloc(void **p, size_t n) {
    ++m->allocs;
    if (m->used[m->current] + m->pooled[m->current] + n > m->capacity) return 2;
    *p = (void *)(m->next += 4096);
    m->live[*p] = {n, m->current};
    m->used[m->current] += n;
    return 0;
  }
  Error alloc_async(void **p, size_t n, Stream) {
    ++m->asyncs;
    return alloc(p, n);
  }
  void free(void *p) {
    m->used[m->live.at(p).second] -= m->live.at(p).first;
    m->live.erase(p);
  }
  bool wait(int) { return m->idle; }
  void trim(int device) { m->pooled[device] = 0; }
};

static int bad = 0;
static void check(bool ok, const char *what) {
  if (!ok) { std::puts(what); ++bad; }
}

using Cache = thg::BlockCache<ModelDriver>;

int main() {
  void *p = nullptr, *q = nullptr;
  size_t b = 0, c = 0;
  {
    Model m;
    Cache k(ModelDriver{&m}, 600);
    k.alloc(&p, 100, 0, &b);
    k.free(p, b, 0);
    check(k.alloc(&q, 90, 0, &c) == 0 && q == p && c == 100 && m.allocs == 1, "a freed block serves a slightly smaller request");
    k.free(q, c, 0);
    check(k.alloc(&q, 79, 0, &c) == 0 && q != p && c == 79, "a block more than a quarter too large is left");
    void *r = nullptr;
    size_t d = 0;
    check(k.alloc(&r, 101, 0, &d) == 0 && r != p, "a block too small is left");
    m.current = 1;
    check(k.alloc(&r, 100, 1, &d) == 0 && r != p && m.live[r].second == 1, "a block of another device is left");
  }
  {
    Model m;
    Cache k(ModelDriver{&m}, 600);
    k.alloc(&p, 500, 0, &b);
    k.free(p, b, 0);
    check(m.used[0] == 500, "the block is kept");
    check(k.alloc(&q, 700, 0, &c) == 0, "kept blocks are given back before an allocation fails");
    check(k.alloc(&p, 400, 0, &b) == 2, "an allocation that cannot fit fails");
  }
  {
    Model m;
    Cache k(ModelDriver{&m}, 600);
    k.alloc(&p, 500, 0, &b);
    k.free(p, b, 0);
    check(k.alloc_async(&q, 700, 0, 0) == 0 && m.asyncs == 2, "kept blocks are given back before a stream-ordered one fails");
    check(k.alloc_async(&p, 400, 0, 0) == 2, "a stream-ordered allocation that cannot fit fails");
  }
  {
    Model m;
    m.pooled[0] = m.pooled[1] = 600;
    Cache k(ModelDriver{&m}, 600);
    check(k.alloc(&q, 700, 0, &c) == 0 && m.pooled[1] == 600, "the idle pool of the device is given back before an allocation fails");
  }
  {
    Model m;
    Cache k(ModelDriver{&m}, 600);
    void *x[4];
    size_t n[4];
    for (int i = 0; i < 4; ++i) k.alloc(&x[i], 220, i == 1 ? 1 : 0, &n[i]);
    for (int i = 0; i < 4; ++i) k.free(x[i], n[i], i == 1 ? 1 : 0);
    check(!m.live.count(x[0]) && m.live.count(x[1]) && m.live.count(x[2]) && m.live.count(x[3]),
          "beyond the limit the device's oldest block is given back");
    k.release(0);
    check(m.live.size() == 1 && m.live.count(x[1]), "release gives back the blocks of one device");
    k.reclaim(1);
    check(m.live.empty(), "reclaim gives back the blocks");
  }
  {
    Model m;
    Cache k(ModelDriver{&m}, 600);
    k.alloc(&p, 700, 0, &b);
    k.free(p, b, 0);
    check(m.live.empty(), "a block beyond the limit is not kept");
    k.alloc(&p, 100, 0, &b);
    m.idle = false;
    k.free(p, b, 0);
    check(m.live.empty(), "a block whose device could not be waited for is not kept");
  }
  {
    Model m;
    Cache k(ModelDriver{&m}, 600);
    k.alloc(&p, 100, 0, &b);
    no_memory = true;
    bool threw = false;
    try {
      k.free(p, b, 0);
    } catch (const std::bad_alloc &) {
      threw = true;
    }
    no_memory = false;
    check(!threw && m.live.empty(), "without host memory to note a block, it is given back");
  }
  return bad;
}
