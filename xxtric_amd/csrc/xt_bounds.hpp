// xt_bounds.hpp -- host checks and sizes that decide what the kernels are given.
// Plain C++, so that they can be built and tested without a GPU.
#pragma once

#include <cmath>
#include <cstdint>

namespace xt {

// The counts in rank space and of batches of small graphs index entries in 32 bits.
// A wave forms the index of each lane's entry, and of its next step, before it
// compares them with the end of a row, so up to 64 past the last entry: below this
// many none of these wraps to the front of the array.
constexpr int64_t kIndex32Entries = (int64_t(1) << 32) - 64;

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

// ---- lists of the count in rank space (rank.hip) ----------------------------
constexpr int kListShards = 16;

struct ListRoom {
  uint64_t region, grant;  // lines of a shard's region; lines drawn at once
  int rows;                // vertices of a wave: 16, 32 or 64
  int together;            // log2 of the neighbouring vertices it takes at a time
  int64_t nbatch;
};

// Room for the lists of a simple graph, in 128-byte lines: |E+| = ne / 2 ids; a
// list of d >= 2 ids is given at most min(d, d / 4 + 9.25) chunks (hot and cold
// parts rounded up to chunks, then to list_room; two parts each: d / 4 + 11.5), a wave's lists at a time
// rounded up to a line.  Grants but a wave's last are used to three quarters.
// A region is left for the next when a request does not fit, so each may lose
// one request: a grant, or 64 of the longest lists.  Ranked by degree these have at
// most 1.02 sqrt(ne) ids, since out-neighbours have about the vertex's degree or
// more; ranked by label (max_degree >= 0) a list is at most its row.
inline ListRoom rank_list_room(int num_cus, int64_t nv, int64_t ne, int64_t max_degree, int parts, int64_t* lines) {
  ListRoom r;
  const int64_t waves = (int64_t)num_cus * 16;
  r.rows = 64;
  while (r.rows > 16 && nv / r.rows < waves) r.rows >>= 1;
  // Four neighbours read a quarter of a line of each vertex array: all right
  // while these stay in the 256 MB cache (20 bytes a vertex).
  r.together = nv <= (1ll << 22) ? 2 : 4;
  r.nbatch = (nv + r.rows - 1) / r.rows;
  const int64_t nlists = nv < ne / 4 ? nv : ne / 4;
  const int64_t chunks = parts == 4 ? ne / 8 + 12 * nlists
                         : ne / 8 + 10 * nlists < ne / 2 ? ne / 8 + 10 * nlists : ne / 2;
  const int64_t need = chunks / 8 + r.nbatch + 1;
  const int64_t grant = need / (waves * 32) < 8 ? 8 : need / (waves * 32);
  const int64_t used = need + need / 3 + (r.nbatch < waves ? r.nbatch : waves) * grant;
  const double longest = max_degree >= 0 ? (double)max_degree : 1.05 * std::sqrt((double)ne) + 64.0;
  const int64_t most = grant + (int64_t)(64.0 * (longest / 4 + 12) / 8) + 1;
  r.grant = (uint64_t)grant;
  r.region = (uint64_t)(used / kListShards + most + 1);
  *lines = (int64_t)r.region * kListShards;
  return r;
}

// Ranked by label a list may hold every vertex: a record's 16 bits of cold
// chunks hold the lists of this many vertices.
constexpr int64_t kLabelRankMax = 4 * 65535;

// Ranks, chunk starts of lists and entry indices fit their 32 bits (entries also a
// wave past the last).  max_degree: the longest row where vertices are ranked by
// label, -1 where by degree.
inline bool rank_space_fits(int num_cus, int64_t nv, int64_t ne, int64_t max_degree) {
  if (nv >= (max_degree >= 0 ? kLabelRankMax : 1ll << 30) || ne >= kIndex32Entries) return false;
  int64_t lines;
  rank_list_room(num_cus, nv, ne, max_degree, 4, &lines);
  return lines < (1ll << 29);
}

}  // namespace xt
