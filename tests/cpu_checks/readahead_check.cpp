// CPU check of the read-ahead window of solution vectors (built with g++ and
// AddressSanitizer/UBSan by tests/test_readahead_cpu.py): reads in every order return
// what the memory holds, windows stay within their bounds, and a window that another
// reader opened while the vectors were being written is not served afterwards.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../gaga_amd/csrc/xcs_readahead.h"

static int fails = 0;
#define CHECK(c, ...)               \
  do {                              \
    if (!(c)) {                     \
      fprintf(stderr, __VA_ARGS__); \
      fprintf(stderr, "\n");        \
      if (++fails > 20) exit(1);    \
    }                               \
  } while (0)

static bool no_memory = false;
static float *take(size_t bytes) { return no_memory ? nullptr : (float *)malloc(bytes); }
static void give(float *p) { free(p); }

struct Handle {
  std::vector<std::vector<float>> a, b;
  ReadAhead ahead{take, give};
  int fetches = 0, rows = 0;
  Handle(int count, int na, int nb) {
    for (int i = 0; i < count; i++) {
      a.emplace_back((size_t)(na + i % 5), (float)i);
      b.emplace_back((size_t)nb, (float)-i);
    }
  }
  void write(float v) {
    for (auto &r : a)
      for (float &x : r) x += v;
  }
  // false: the caller has to copy by itself
  bool read(int i, std::vector<float> &x, std::vector<float> &y, bool run_fails = false) {
    x.assign(a[(size_t)i].size(), -1.f);
    y.assign(b[(size_t)i].size(), -1.f);
    struct Move {
      const float *s;
      float *d;
      long n;
    };
    std::vector<Move> list;
    float *const out[2] = {x.data(), y.data()};
    return ahead.get(
        i, (int)a.size(), 2,
        [&](int r, int p, const float **s, long *n) {
          const std::vector<float> &v = p ? b[(size_t)r] : a[(size_t)r];
          *s = v.data();
          *n = (long)v.size();
        },
        out, [&](const float *s, float *d, long n) { list.push_back({s, d, n}); },
        [&] {
          if (run_fails) return false;
          for (const Move &m : list) memcpy(m.d, m.s, sizeof(float) * (size_t)m.n);
          fetches++;
          rows += (int)list.size() / 2;
          CHECK((int)list.size() <= 2 * READ_ROWS, "%zu pieces in a window", list.size());
          return true;
        });
  }
  void check(int i) {
    std::vector<float> x, y;
    if (read(i, x, y)) CHECK(x == a[(size_t)i] && y == b[(size_t)i], "row %d is not what the memory holds", i);
  }
};

int main() {
  for (int count : {1, 2, 3, 5, 64, 65, 300}) {
    Handle h(count, 100, 7);
    for (int i = 0; i < count; i++) h.check(i);
    for (int i = count - 1; i >= 0; i -= 3) h.check(i);
    for (int i = 0; i < 4 * count; i++) h.check((i * 7) % count);
    h.write(0.5f);  // outside a Writing nothing is promised; inside one everything is
    {
      ReadAhead::Writing w(h.ahead);
      h.write(1.f);
    }
    for (int i = 0; i < count; i++) h.check(i);
  }
  {  // in order: few fetches, rows beyond READ_BYTES alone
    Handle h(300, 1000, 10);
    for (int i = 0; i < 300; i++) h.check(i);
    CHECK(h.fetches <= 12 && h.rows == 299, "%d fetches of %d rows", h.fetches, h.rows);
    Handle big(3, (int)(READ_BYTES / 4), 1);
    for (int i = 0; i < 3; i++) big.check(i);
    CHECK(big.fetches == 0, "a row that does not fit was fetched");
  }
  {  // a second reader opens a window while the vectors are written
    Handle h(40, 50, 3);
    {
      ReadAhead::Writing w(h.ahead);
      std::vector<float> x, y;
      for (int i = 0; i < 5; i++) (void)h.read(i, x, y);
      CHECK(h.fetches > 0, "no window was opened");
      h.write(2.f);
    }
    for (int i = 2; i < 40; i++) h.check(i);  // row 2 lies in that window
    for (int i = 0; i < 9; i++) h.check(i);
  }
  {  // a failed transfer or no memory: the caller copies, and later reads recover
    Handle h(20, 50, 3);
    std::vector<float> x, y;
    h.check(0);
    CHECK(!h.read(1, x, y, true), "a failed transfer was served");
    for (int i = 2; i < 20; i++) h.check(i);
    no_memory = true;
    Handle g(20, 50, 3);
    for (int i = 0; i < 20; i++) CHECK(!g.read(i, x, y), "served without memory");
    no_memory = false;
  }
  if (fails) return 1;
  printf("read-ahead checks passed\n");
  return 0;
}
