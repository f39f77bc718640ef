// xt_bounds.hpp -- host checks that decide what the kernels are given.  Plain
// C++, so that they can be built and tested without a GPU.
#pragma once

#include <cstdint>

namespace xt {

// nullptr where off[0 .. nv] is the index of ne entries, else what is wrong.
// max_degree (nullable) gets the longest row.  Neighbouring offsets are compared:
// the sign of their difference tells nothing where it does not fit 64 bits.
inline const char* check_offsets(int64_t nv, int64_t ne, const int64_t* off, int64_t* max_degree) {
  if (off[0] != 0 || off[nv] != ne) return "offsets must start at 0 and end at ne";
  uint64_t most = 0, down = 0;
  for (int64_t i = 0; i < nv; i++) {
    const uint64_t d = (uint64_t)off[i + 1] - (uint64_t)off[i];
    down |= (uint64_t)(off[i + 1] < off[i]);
    most = d > most ? d : most;
  }
  if (down) return "offsets are not monotone";
  if (max_degree) *max_degree = (int64_t)most;
  return nullptr;
}

}  // namespace xt
