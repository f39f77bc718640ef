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
      const bool fits = xt::rank_space_fits(256, by_label ? 250000 : nv, ne, by_label ? 256 : -1);
      CHECK(!fits || ends);
      CHECK(by_label || fits == (ne < xt::kIndex32Entries));
    }
    CHECK(ends || ne >= xt::kIndex32Entries);
  }
  CHECK(walk((uint32_t)(top - 110), (uint32_t)(top - 10)) == -1);  // what the limit keeps out
  CHECK(!xt::rank_space_fits(256, nv, top, -1) && !xt::rank_space_fits(256, nv, top + 5, -1));
  return 0;
}

// Chunks a list of d ids is given, at most: eight hot ids or four cold ones to a
// chunk, each part rounded up, then in full, half, quarter or eighth lines.  The
// worst split has one id in every part but the last, cold one.
static int64_t most_chunks(int64_t d, int parts) {
  if (d < 2) return 0;  // no pair, no list
  const int64_t others = parts - 1 < d - 1 ? parts - 1 : d - 1;
  const int64_t t = others + (d - others + 3) / 4;
  return t <= 2 ? t : t <= 4 ? 4 : (t + 7) / 8 * 8;
}

static int lists() {
  for (int cus : {64, 256, 304})
    for (int64_t nv : {64, 1000, 20001, 100000, 262139})
      for (int64_t d : {1, 2, 31, 32, 33, 100, 255, 256}) {
        if (d >= nv) continue;
        const int64_t ne = nv * d;
        for (int parts : {2, 4}) {
          int64_t lines = 0;
          const xt::ListRoom r = xt::rank_list_room(cus, nv, ne, d, parts, &lines);
          // Room for every vertex's list of half its row and for a wave of whole rows in each region ...
          CHECK(lines * 8 >= nv * most_chunks(d / 2, parts));
          CHECK((int64_t)r.region * 8 >= r.rows * most_chunks(d, parts));
          // ... but of that order: 6 bytes an entry, 500 a vertex and, for the waves' draws, 4 MB.
          CHECK(lines * 128 <= 6 * ne + 500 * nv + (int64_t(4) << 20) * cus / 256 + (int64_t(1) << 20));
        }
      }
  return 0;
}

int main(int argc, char** argv) {
  const struct {
    const char* name;
    int (*run)();
  } groups[] = {{"offsets", offsets}, {"index32", index32}, {"lists", lists}};
  if (argc != 2) return 2;
  for (const auto& g : groups)
    if (std::strcmp(argv[1], g.name) == 0) {
      const int rc = g.run();
      if (rc == 0) std::printf("%s hold\n", g.name);
      return rc;
    }
  return 2;
}
