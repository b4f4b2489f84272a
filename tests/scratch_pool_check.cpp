// scratch_pool.hpp on counted blocks: `budget` bytes in all, every block freed once.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "scratch_pool.hpp"

using namespace sbfs;

static std::map<void*, size_t> g_live;
static size_t g_used = 0, g_budget = 0;
static char* g_next = (char*)4096;

struct Blocks {
  static int alloc(void** p, size_t bytes) {
    *p = nullptr;
    if (g_used + bytes > g_budget) return 2;
    *p = g_next;
    g_next += 4096;
    g_live[*p] = bytes;
    g_used += bytes;
    return 0;
  }
  static void free(void* p) {
    if (!p) return;
    if (!g_live.count(p)) {
      printf("freed twice\n");
      exit(1);
    }
    g_used -= g_live[p];
    g_live.erase(p);
  }
  static int zero(void*, size_t) { return 0; }
};

#define CHECK(x)                                 \
  do {                                           \
    if (!(x)) {                                  \
      printf("line %d: %s\n", __LINE__, #x);     \
      return 1;                                  \
    }                                            \
  } while (0)

int main() {
  using Pool = ScratchPool<Blocks>;
  constexpr size_t G = 1ull << 30, M = 1ull << 20;
  const auto sizes = [](size_t n, size_t field) { return ScratchSizes{n, n, field, field, field, field}; };
  FusedScratch a, b, c;

  // all six fields or none: the fifth does not fit
  {
    Pool pool;
    g_budget = 4 * M + M / 2;
    CHECK(pool.get(sizes(1, M), false, &a) != 0);
    CHECK(a.vof == nullptr && g_used == 0 && g_live.empty());
  }
  // a set comes back for the next domain of its size, with the learned buffers where they are wanted
  {
    Pool pool;
    g_budget = 100 * M;
    CHECK(pool.get(sizes(1, M), true, &a) == 0 && g_used == 6 * M && a.bytes == 6 * M);
    CHECK(pool.get(sizes(1, M), false, &b) == 0 && g_used == 12 * M);
    CHECK(Blocks::alloc((void**)&a.cut, M) == 0);
    a.bytes += M;
    double *const va = a.vof, *const vb = b.vof;
    pool.put(a);
    pool.put(b);
    CHECK(a.vof == nullptr && b.vof == nullptr && pool.bytes() == 13 * M);
    CHECK(pool.get(sizes(1, M), true, &a) == 0 && a.vof == va && a.cut);
    CHECK(pool.get(sizes(1, M), true, &b) == 0 && b.vof == vb && !b.cut && pool.bytes() == 0);
    pool.put(a);
    pool.put(b);
    // the last allocation that fits without them, and one that needs their memory
    void *p = nullptr, *q = nullptr;
    CHECK(pool.alloc(&p, 87 * M) == 0 && pool.bytes() == 13 * M);
    CHECK(pool.alloc(&q, M) == 0 && pool.bytes() == 0 && g_used == 88 * M);
    CHECK(pool.alloc(&q, 100 * M) != 0 && q == nullptr);
    g_budget = 1000 * G;
    Blocks::free(p);
  }
  g_live.clear();
  g_used = 0;
  // a domain of another size leaves kIdle at most: a large set goes, small ones stay
  {
    Pool pool;
    CHECK(pool.get(sizes(1, M), false, &a) == 0);
    CHECK(pool.get(sizes(2, G), false, &b) == 0);
    pool.put(a);
    pool.put(b);
    CHECK(pool.bytes() == 6 * G + 6 * M && g_used == pool.bytes());
    CHECK(pool.get(sizes(3, M), false, &c) == 0);
    CHECK(pool.bytes() == 6 * M && g_used == pool.bytes() + 6 * M);
    pool.put(c);
    // also where the pool has a set of the size
    CHECK(pool.get(sizes(2, G), false, &b) == 0);
    pool.put(b);
    CHECK(pool.get(sizes(3, M), false, &c) == 0);
    CHECK(pool.bytes() == 6 * M);
    pool.put(c);
    CHECK(g_used == pool.bytes());
  }
  g_live.clear();
  g_used = 0;
  // kMost, with the last one whatever its size
  {
    Pool pool;
    FusedScratch s[4];
    for (int k = 0; k < 4; k++) CHECK(pool.get(sizes(1, G / 2), false, &s[k]) == 0);  // 3 GiB each
    double* const last = s[3].vof;
    for (auto& x : s) pool.put(x);
    CHECK(pool.bytes() == 6 * G && g_used == 6 * G);
    CHECK(pool.get(sizes(1, G / 2), false, &a) == 0 && a.vof == last);
    CHECK(pool.get(sizes(2, 2 * G), false, &b) == 0);  // 12 GiB
    pool.put(a);
    pool.put(b);
    CHECK(pool.bytes() == 12 * G && g_used == 12 * G);
  }
  printf("ok\n");
  return 0;
}
