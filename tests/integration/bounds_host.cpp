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

int main(int argc, char** argv) {
  const struct {
    const char* name;
    int (*run)();
  } groups[] = {{"offsets", offsets}};
  if (argc != 2) return 2;
  for (const auto& g : groups)
    if (std::strcmp(argv[1], g.name) == 0) {
      const int rc = g.run();
      if (rc == 0) std::printf("%s hold\n", g.name);
      return rc;
    }
  return 2;
}
