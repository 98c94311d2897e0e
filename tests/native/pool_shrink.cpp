// The caching allocator's in-place shrink: random allocations, shrinks and
// frees over fake memory; every live block's bytes stay its own, freed tails are
// handed out again, and everything returns at the end.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>

#include "pool_core.h"

static char *g_next = reinterpret_cast<char *>(size_t(1) << 40);
static void *fake_alloc(size_t n, void *) {
  char *p = g_next;
  g_next += n + (size_t(1) << 20);
  return p;
}
static void fake_release(void *, void *) {}

#define CHECK(x)                              \
  do {                                        \
    if (!(x)) {                               \
      std::printf("line %d: %s\n", __LINE__, #x); \
      return 1;                               \
    }                                         \
  } while (0)

int main() {
  const size_t big = size_t(1) << 20, unit = size_t(64) << 10, seg = size_t(256) << 20;
  gemh::PoolCore pool(gemh::PoolBacking{fake_alloc, fake_release, nullptr, nullptr}, big, unit, seg);
  const int dummy = 0;
  const void *s = &dummy;
  size_t cls = 0;
  // below the carved size, and a shrink that gives nothing back
  void *p = pool.alloc(1000, s, &cls);
  CHECK(pool.shrink(p, cls, 10, s) == cls);
  pool.free(p, cls, s);
  p = pool.alloc(big, s, &cls);
  CHECK(pool.shrink(p, cls, 1, s) == cls);
  pool.free(p, cls, s);
  // the whole segment, shrunk: its tail serves the next request at once
  p = pool.alloc(seg, s, &cls);
  cls = pool.shrink(p, cls, 3 * big + 1, s);
  CHECK(cls == 3 * big + unit && pool.stats().in_use == cls);
  size_t c2 = 0;
  void *q = pool.alloc(seg - 4 * big, s, &c2);
  CHECK(static_cast<char *>(q) == static_cast<char *>(p) + cls && pool.stats().segments == 1);
  pool.free(p, cls, s);
  pool.free(q, c2, s);
  std::mt19937_64 rng(5);
  std::map<char *, size_t> live;  // base -> block size
  for (int i = 0; i < 20000; ++i) {
    const unsigned op = rng() % 4;
    if (op < 2 || live.empty()) {
      const size_t n = big / 2 + rng() % (24 * big);
      char *b = static_cast<char *>(pool.alloc(n, s, &cls));
      auto nx = live.upper_bound(b);
      CHECK(nx == live.end() || b + cls <= nx->first);
      if (nx != live.begin()) {
        --nx;
        CHECK(nx->first + nx->second <= b);
      }
      live[b] = cls;
    } else {
      auto it = live.lower_bound(static_cast<char *>(static_cast<void *>(live.begin()->first)) + rng() % (seg * 2));
      if (it == live.end()) it = live.begin();
      if (op == 2) {
        it->second = pool.shrink(it->first, it->second, 1 + rng() % it->second, s);
      } else {
        pool.free(it->first, it->second, s);
        live.erase(it);
      }
    }
    size_t sum = 0;
    for (auto &kv : live) sum += kv.second;
    CHECK(pool.stats().in_use == sum);
    while (live.size() > 60) {
      pool.free(live.begin()->first, live.begin()->second, s);
      live.erase(live.begin());
    }
  }
  for (auto &kv : live) pool.free(kv.first, kv.second, s);
  CHECK(pool.stats().in_use == 0);
  pool.trim();
  CHECK(pool.stats().held == 0);
  std::printf("ok\n");
  return 0;
}
