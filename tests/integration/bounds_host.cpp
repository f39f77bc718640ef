// bounds_host.cpp -- the library's host checks (xt_bounds.hpp) at the edges of
// what they accept, built and run by tests/test_bounds.py.  Each argument names a
// group of checks; exit status 0 when all of them hold.
#include <cstdio>
#include <cstring>
#include <vector>

#include "xt_bounds.hpp"

#define CHECK(c)                                                           \
  do {                                                                     \
    if (!(c)) {                                                            \
      std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
      return 1;                                                            \
    }                                                                      \
  } while (0)

static const char* check(const std::vector<int64_t>& off, int64_t* most = nullptr) {
  return xt::check_offsets((int64_t)off.size() - 1, off.back(), off.data(), most);
}

static int offsets() {
  constexpr int64_t big = int64_t(1) << 62, low = INT64_MIN;
  int64_t most = -1;
  CHECK(!check({0, 2, 2, 9}, &most) && most == 7);
  CHECK(!check({0}, &most) && most == 0);
  CHECK(!check({0, INT64_MAX}, &most) && most == INT64_MAX);
  CHECK(!check({0, big, big, INT64_MAX}, &most) && most == big);
  most = -1;
  CHECK(check({0, 4, 2, 6}, &most) && most == -1);
  CHECK(check({1, 2, 6}) && check({-1, 2, 6}));
  // Steps down whose difference wraps to a step up.
  CHECK(check({0, big, low, -big, 6}));
  CHECK(check({0, 3, low, 6}) && check({0, INT64_MAX, -2, 6}) && check({0, INT64_MAX, low, 6}));
  const std::vector<int64_t> off = {0, 2, 4, 6};
  CHECK(xt::check_offsets(3, 7, off.data(), nullptr) && !xt::check_offsets(3, 6, off.data(), nullptr));
  return 0;
}

// The walk of k_rank_count over a row's items [is, ie), as its 32-bit arithmetic has
// it: a wave's 64 lanes at a time, each index compared with the end.  -1 where it
// visits an entry that is not the row's or does not end.
static int64_t walk(uint32_t is, uint32_t ie) {
  int64_t visited = 0, rounds = 0;
  for (uint32_t e = is; rounds == 0 || e < ie; e += 64) {
    if (++rounds > 64) return -1;
    for (uint32_t lane = 0; lane < 64; lane++)
      if (e + lane < ie) {
        if (e + lane < is) return -1;
        visited++;
      }
  }
  return visited;
}

static int index32() {
  constexpr int64_t top = int64_t(1) << 32;
  // 2^24 vertices leave room for the lists at any number of entries.
  constexpr int64_t nv = int64_t(1) << 24;
  for (int64_t ne = xt::kIndex32Entries - 128; ne < top; ne++) {
    bool ends = true;
    for (int64_t items = 1; items <= 300 && ends; items++) ends = walk((uint32_t)(ne - items), (uint32_t)ne) == items;
    for (bool by_label : {false, true}) {
      const bool fits = xt::rank_space_fits(256, by_label ? 250000 : nv, ne, by_label);
      CHECK(!fits || ends);
      CHECK(by_label || fits == (ne < xt::kIndex32Entries));
    }
    CHECK(ends || ne >= xt::kIndex32Entries);
  }
  CHECK(walk((uint32_t)(top - 110), (uint32_t)(top - 10)) == -1);  // what the limit keeps out
  CHECK(!xt::rank_space_fits(256, nv, top, false) && !xt::rank_space_fits(256, nv, top + 5, false));
  return 0;
}

int main(int argc, char** argv) {
  const struct {
    const char* name;
    int (*run)();
  } groups[] = {{"offsets", offsets}, {"index32", index32}};
  if (argc != 2) return 2;
  for (const auto& g : groups)
    if (std::strcmp(argv[1], g.name) == 0) {
      const int rc = g.run();
      if (rc == 0) std::printf("%s hold\n", g.name);
      return rc;
    }
  return 2;
}
