// rank.hip -- the count of one graph in rank space (gfx950): totals, per-vertex
// counts and owned ranges.
//
// Vertices are ranked by descending degree (rank 0 = the largest hub) and
// every triangle w < v < u (ranks) is counted once, at its edge (u, v), as an
// id common to N(v) and to the part of N(u) below v, N(x) holding x's
// neighbours of smaller rank.  Three things follow from ranks that labels do
// not give:
//  * only the ids of N(u) below v can close the edge (u, v), a prefix when
//    N(u) is in rank order: sum of prefixes against the sum of
//    min(d+(u), d+(v)) that the edge tiles of count.hip stream: 0.62 of it
//    (R-MAT s20, 1.97e9 -> 1.23e9 ids);
//  * the ids that occur in lists are small: those below 65535 ("hot") are
//    stored in 16 bits, and are nearly all that is streamed (s20: 0.9998), so
//    an id costs two bytes instead of four;
//  * N(v)'s hot ids are a 65536-bit map, 8 KB of LDS: one 4-byte LDS read and
//    a bit test per streamed id instead of a 16-byte hash bucket and four
//    compares, and a table per wave instead of one per workgroup.
// Ids from 65535 on ("cold") only matter when v is cold too: then u's cold
// list is streamed through a hash of N(v)'s cold ids.
//
// Both passes that gather or stream are bound by the lines that miss L2 (about
// 52-55 G lines of 128 bytes a second on this GPU, from HBM or from the 256 MB
// cache).  R-MAT s26: 353 ms with edge tiles, 182-188 here: k_rank_split 40-42,
// k_rank_lists 10-11, k_rank_count 131-135 (949 GB of such lines, 55 G/s).
//
// Six kernels, no scan over the vertices and no item list:
//  k_rank_clear   counters and class histogram cleared
//  k_rank_prep    degree classes counted, first and last row of every chunk
//  k_rank_assign  ranks: counting sort of the vertices by degree class
//  k_rank_split   per row, in place of the labels: ranks, smaller ones first
//  k_rank_lists   per vertex: the smaller ranks as a list (hot ascending
//                 16-bit, then cold 32-bit) and a 32-byte record
//  k_rank_count   per chunk of entries, one wave: v's map, the lists of its
//                 larger neighbours u streamed through it
#include <type_traits>

#include "xt_bounds.hpp"
#include "xt_device.hpp"
#include "xt_hash.hpp"
#include "xt_internal.hpp"

namespace xt {

// What is counted: the total; per vertex (each triangle credited to its smallest
// label); or, for an owned label range [lo, hi), the triangles whose smallest
// label is owned and, of those, the ones whose middle label is owned too.  With
// labels below lo left out, these are the triangles with one, and with two, of
// their vertices owned.
constexpr int kTotal = 0;
constexpr int kPerVertex = 1;
constexpr int kRange = 2;

constexpr uint32_t kHot = 65535;       // ranks below are hot; 65535 itself pads 16-bit lists
constexpr uint32_t kNoRank = ~0u;      // a self-loop or an id out of range; pads cold lists
constexpr int kRankClasses = 896;      // degree classes: exact below 64, then 32 per octave
constexpr int kRankMarks = 12;         // ids kept per list for finding prefixes
constexpr int kRankMarksPv = 10;       // the same beside the vertex's label (per-vertex counts)
constexpr int kMarksOwned = 3;         // owned-range counts: of the owned ids
constexpr int kMarksRest = 7;          // ... and of the others
constexpr uint32_t kOwnedBit = 1u << 31;  // on a rank: its label is owned (ranks are below 2^30)
constexpr int kAssignRun = 8;          // vertices per thread of k_rank_assign
constexpr int kLaneList = 32;          // lists of up to this many ids are written by one lane, unsorted
constexpr int kTinyRow = 8;            // rows of up to this many ids and 64 items: a lane per item

__device__ __forceinline__ int degree_class(int64_t d) {
  if (d < 64) return d < 0 ? 0 : (int)d;
  const uint32_t x = d > 0x7fffffff ? 0x7fffffffu : (uint32_t)d;
  const int e = 31 - __clz((int)x);
  return 64 + (e - 6) * 32 + (int)((x >> (e - 5)) & 31u);
}

// Record of the vertex of one rank: where its list starts (16-byte units), the
// 16-byte chunks of its hot part (ascending ids) and of its cold part, and the
// first id of every segment of ceil(hot / 12) hot chunks: the segments that
// start below v hold every id below v.  (Eight cuts at the same ranks for every
// list, in 16 bytes, streamed 1.26 times the ids below v at R-MAT s22.)
struct alignas(16) RankRec {
  uint32_t start;
  uint32_t len;  // hot chunks | cold chunks << 16
  uint32_t mark[kRankMarks / 2];
};
static_assert(sizeof(RankRec) == 32, "two 16-byte loads");

// A per-vertex count keeps ten marks, and the vertex's label in the last word.
// An owned-range count has four parts, each with its own chunks: owned hot ids,
// other hot ids, owned cold ids, other cold ids; its record holds {start,
// chunks 0 | 1 << 16, chunks 2 | 3 << 16, three marks of part 0 and seven of part 1}.
template <int MODE>
constexpr uint32_t hot_marks() {
  return MODE == kPerVertex ? kRankMarksPv : kRankMarks;
}
__device__ __forceinline__ uint32_t mark_step(uint32_t hot, uint32_t marks) { return (hot + marks - 1) / marks; }

// 16-byte chunks a list of t chunks is given: it starts on a multiple of its size up
// to eight chunks (a 128-byte line), so no list crosses more lines than it
// fills.
__device__ __forceinline__ uint32_t list_room(uint32_t t) {
  return t <= 2 ? t : t <= 4 ? 4 : (t + 7) & ~7u;
}

// The counters and both halves of the class histogram cleared in one launch (a
// launch is 5 to 8 us of a small count's 90).
__global__ __launch_bounds__(256) void k_rank_clear(uint64_t* __restrict__ counters, uint32_t* __restrict__ hist) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < kNumCounters) counters[i] = 0;
  if (i < kRankClasses) hist[i] = hist[kRankClasses + i] = 0;
}
static_assert(kNumCounters >= kRankClasses, "the grid covers both");

// ---------------------------------------------------------------------------
// Degree classes counted (one histogram per workgroup in LDS), per-row
// counters cleared, and the first and last row of every chunk of 2^log2 entries
// (crows[2c], crows[2c + 1]), each written by the row that holds the boundary.
__global__ __launch_bounds__(256) void k_rank_prep(int64_t nv, int64_t ne, const int64_t* __restrict__ off, int log2,
                                                   int32_t* __restrict__ crows, uint64_t* __restrict__ oc,
                                                   uint32_t* __restrict__ ic, uint32_t* __restrict__ hist,
                                                   unsigned long long* __restrict__ pv, uint64_t* __restrict__ oc1) {
  __shared__ uint32_t s_h[kRankClasses];
  for (int k = threadIdx.x; k < kRankClasses; k += 256) s_h[k] = 0;
  __syncthreads();
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t u0 = (int64_t)blockIdx.x * blockDim.x; u0 < nv; u0 += stride) {  // uniform
    const int64_t u = u0 + threadIdx.x;
    int64_t a = 0, b = 0;
    if (u < nv) {
      a = off[u];
      b = off[u + 1];
      oc[u] = 0;
      ic[u] = 0;
      if (pv) pv[u] = 0;
      if (oc1) oc1[u] = 0;
      atomicAdd(&s_h[degree_class(b - a)], 1u);
    }
    mark_chunks(u, a, b, ne, log2, crows);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kRankClasses; k += 256)
    if (s_h[k]) atomicAdd(&hist[k], s_h[k]);
}

// rank[u]: the number of vertices of larger classes, plus u's place among its
// class (workgroups take places by one atomic per class they hold; any order
// inside a class is a valid total order).
__global__ __launch_bounds__(256) void k_rank_assign(int64_t nv, const int64_t* __restrict__ off,
                                                     const uint32_t* __restrict__ hist, uint32_t* __restrict__ taken,
                                                     uint32_t* __restrict__ rank, uint32_t* __restrict__ orig) {
  __shared__ uint32_t s_base[kRankClasses], s_n[kRankClasses];
  __shared__ int64_t s_scan[256 / kWave];
  constexpr int kPer = (kRankClasses + 255) / 256;
  uint32_t h[kPer];
  int64_t sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; j++) {  // descending classes
    const int k = kRankClasses - 1 - ((int)threadIdx.x * kPer + j);
    h[j] = k >= 0 ? hist[k] : 0u;
    sum += h[j];
  }
  int64_t total;
  int64_t at = block_excl_scan_i64<256>(sum, s_scan, &total);
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int k = kRankClasses - 1 - ((int)threadIdx.x * kPer + j);
    if (k >= 0) {
      s_base[k] = (uint32_t)at;
      s_n[k] = 0;
    }
    at += h[j];
  }
  __syncthreads();
  const int64_t u0 = (int64_t)blockIdx.x * (256 * kAssignRun) + threadIdx.x;
  int cls[kAssignRun];
  uint32_t loc[kAssignRun];
#pragma unroll
  for (int j = 0; j < kAssignRun; j++) {
    const int64_t u = u0 + 256 * j;
    cls[j] = -1;
    if (u < nv) {
      cls[j] = degree_class(off[u + 1] - off[u]);
      loc[j] = atomicAdd(&s_n[cls[j]], 1u);
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kRankClasses; k += 256)
    if (s_n[k]) s_base[k] += atomicAdd(&taken[k], s_n[k]);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kAssignRun; j++)
    if (cls[j] >= 0) {
      const uint32_t r = s_base[cls[j]] + loc[j];
      rank[u0 + 256 * j] = r;
      if (orig) orig[r] = (uint32_t)(u0 + 256 * j);
    }
}

// Ranks by descending label: u -> v iff u < v, the reference's rule.
__global__ __launch_bounds__(256) void k_rank_by_label(int64_t nv, uint32_t* __restrict__ rank,
                                                       uint32_t* __restrict__ orig) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; u < nv; u += stride) {
    const uint32_t r = (uint32_t)(nv - 1 - u);
    rank[u] = r;
    if (orig) orig[u] = r;  // its own inverse
  }
}

// ---------------------------------------------------------------------------
// Row u's entries as ranks, the smaller ones (N(u)) at the front of the row's
// own range of `part` and the larger ones at its back; oc[u] = |N(u)| | hot
// ones << 32.  One workgroup per 2048 entries, eight per thread.  Every row
// that starts in the chunk marks its first entry with its end and its rank, so
// a thread meets its rows in LDS whatever empty rows lie between them.  A row
// inside the chunk is placed by a block scan, through LDS; the chunk's first
// and last row, which may continue in another chunk, take their places by
// atomics.  Entries that are no edge (self-loops, ids out of range) go to the
// back as kNoRank.
//
// RANGE: labels below rlo are left out (their rows are empty, entries of them no
// edges); ranks of owned labels carry kOwnedBit, and oc1[u] counts the owned ones
// of N(u) as oc[u] counts all.
template <typename T, bool RANGE>
__global__ __launch_bounds__(kBlock) void k_rank_split(int64_t nv, int64_t ne, const int64_t* __restrict__ off,
                                                       const T* __restrict__ tails, const uint32_t* __restrict__ rank,
                                                       const int32_t* __restrict__ crows, int per,
                                                       uint32_t* __restrict__ part, uint64_t* __restrict__ oc,
                                                       uint32_t* __restrict__ ic, uint64_t* __restrict__ counters,
                                                       uint64_t* __restrict__ oc1, int64_t rlo, int64_t rhi) {
  // Of the entries before each entry: smaller ranks | hot ones << 16 and, RANGE,
  // owned ones << 32 | owned hot ones << 48.
  using Pre = typename std::conditional<RANGE, uint64_t, uint32_t>::type;
  __shared__ alignas(16) int16_t s_end[kChunk];       // first entry of a row: where the row ends (clamped); 0 elsewhere
  __shared__ uint32_t s_rk[kChunk];       // and its rank; later the chunk's entries in their new order
  __shared__ Pre s_pre[kChunk + 1];
  __shared__ int64_t s_scan[kBlock / kWave];
  __shared__ int s_last[kBlock / kWave];
  __shared__ uint32_t s_ob[2], s_ib[2];   // places taken by the first and the last row
  __shared__ int s_rng[3];                // the inner rows' range; whether the first row starts before the chunk
  uint32_t* s_part = s_rk;
  const int64_t nchunks = (ne + kChunk - 1) / kChunk;
  const int64_t c = xcd_block(nchunks);
  if (c >= nchunks) return;  // whole workgroup
  const int64_t eb = c * kChunk;
  const int n = (int)min((int64_t)kChunk, ne - eb);
  const int64_t nsub = 2 * ((ne + (int64_t)kChunk / per - 1) / ((int64_t)kChunk / per));
  int64_t ulo = crows[2 * c * per], uhi = crows[min(2 * (c * per + per) - 1, nsub - 1)];
  ulo = ulo < 0 ? 0 : (ulo > nv - 1 ? nv - 1 : ulo);
  uhi = uhi < ulo ? ulo : (uhi > nv - 1 ? nv - 1 : uhi);
  const int64_t span = uhi - ulo + 1;
  auto rel = [&](int64_t o) -> int {  // an offset relative to the chunk, clamped to [-1, kChunk + 1]
    const int64_t d = o - eb;
    return (int)(d < -1 ? -1 : (d > kChunk + 1 ? kChunk + 1 : d));
  };
  const int tid = (int)threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const int i0 = tid * kPerThread;
  const bool live = i0 < n;
  *reinterpret_cast<int4*>(&s_end[i0]) = make_int4(0, 0, 0, 0);
  uint32_t rv[kPerThread];
  uint32_t bad = 0, own = 0, out = 0;  // RANGE: entries of owned labels, of labels left out
  if (live) {
    int64_t vals[kPerThread];
    load_run<T>(tails, eb + i0, eb + n, vals);
#pragma unroll
    for (int j = 0; j < kPerThread; j++) {  // eight gathers in flight
      const bool in = i0 + j < n, ok = in && vals[j] >= 0 && vals[j] < nv;
      if (in && !ok) bad++;
      const uint32_t r = rank[ok ? vals[j] : 0];
      rv[j] = ok ? r : kNoRank;
      if constexpr (RANGE) {
        own |= (ok && vals[j] >= rlo && vals[j] < rhi ? 1u : 0u) << j;
        out |= (ok && vals[j] < rlo ? 1u : 0u) << j;
      }
    }
  }
  if (bad) atomicAdd((unsigned long long*)&counters[kBadIds], (unsigned long long)bad);
  __syncthreads();
  for (int64_t k = tid; k < span; k += kBlock) {
    const int64_t o0 = off[ulo + k], o1 = off[ulo + k + 1];
    const int ro = rel(o0), re = rel(o1);
    if (re > 0 && ro < n && o1 > o0) {
      s_end[max(ro, 0)] = (int16_t)re;
      s_rk[max(ro, 0)] = rank[ulo + k] | (RANGE && ulo + k < rlo ? kOwnedBit : 0u);  // RANGE: a row left out
    }
    if (k == 0) {
      s_rng[0] = ro < 0 || re > n ? min(re, n) : 0;
      s_rng[2] = ro < 0;
    }
    if (k == span - 1) s_rng[1] = re > n || ro < 0 ? max(ro, 0) : n;
  }
  __syncthreads();
  // The row of this thread's first entry: the last mark up to it.
  int ends[kPerThread];
  int last = -1;
  {
    const int4 q = *reinterpret_cast<const int4*>(&s_end[i0]);
    const int w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      ends[2 * j] = (int16_t)(w[j] & 0xffff);
      ends[2 * j + 1] = w[j] >> 16;
    }
#pragma unroll
    for (int j = 0; j < kPerThread; j++)
      if (ends[j]) last = i0 + j;
  }
  int upto = last;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int y = __shfl_up(upto, o, kWave);
    if (lane >= o) upto = max(upto, y);
  }
  if (lane == kWave - 1) s_last[wv] = upto;
  int at = __shfl_up(upto, 1, kWave);
  if (lane == 0) at = -1;
  __syncthreads();
  for (int w = 0; w < wv; w++) at = max(at, s_last[w]);
  if (ends[0]) at = i0;
  at = max(at, 0);  // entry 0 is marked whenever the offsets are an index
  uint32_t small = 0, hot = 0;
  uint64_t edges = 0;  // RANGE: all of them, as other counts report
  if (live) {
    uint32_t ru = s_rk[at];
#pragma unroll
    for (int j = 0; j < kPerThread; j++) {
      if (i0 + j < n) {
        if (ends[j]) ru = s_rk[i0 + j];
        if constexpr (RANGE) {
          edges += rv[j] < (ru & ~kOwnedBit) ? 1u : 0u;
          if ((out >> j & 1u) || (ru & kOwnedBit)) rv[j] = kNoRank;
        }
        if (rv[j] < ru) {
          small |= 1u << j;
          if (rv[j] < kHot) hot |= 1u << j;
        } else if (rv[j] == ru) {
          rv[j] = kNoRank;  // self-loop
        }
      }
    }
  }
  auto counts = [&](uint32_t m) -> Pre {  // of the entries in m; a chunk's fields stay below 2^16
    Pre p = (Pre)(uint32_t)(__popc(small & m) | (__popc(hot & m) << 16));
    if constexpr (RANGE)
      p |= (Pre)(uint32_t)(__popc(small & own & m) | (__popc(hot & own & m) << 16)) << 32;
    return p;
  };
  int64_t total;
  const int64_t pre = block_excl_scan_i64<kBlock>((int64_t)counts(~0u), s_scan, &total);
  if (live) {
#pragma unroll
    for (int j = 0; j < kPerThread; j++)
      if (i0 + j < n) s_pre[i0 + j] = (Pre)pre + counts((1u << j) - 1u);
  }
  if constexpr (RANGE) {
    edges = wave_sum_u64(edges);
    if (lane == 0) add_sum(counters, kSumEdges, edges);
#pragma unroll
    for (int j = 0; j < kPerThread; j++)
      if (own >> j & 1u && rv[j] != kNoRank) rv[j] |= kOwnedBit;
  }
  if (tid == 0) s_pre[n] = (Pre)total;
  __syncthreads();  // s_rk is read: its place takes the new order
  for (int64_t k = tid; k < span; k += kBlock) {
    const int64_t o0 = off[ulo + k], o1 = off[ulo + k + 1];
    const int ro = rel(o0), re = rel(o1);
    if (re <= 0 || ro >= n || o1 <= o0) continue;
    const int a = max(ro, 0), b = min(re, n);
    const Pre q = s_pre[b] - s_pre[a];
    const uint32_t outs = (uint32_t)q & 0xffffu, hots = (uint32_t)q >> 16;
    uint32_t q1 = 0;
    if constexpr (RANGE) q1 = (uint32_t)(q >> 32);
    if (ro >= 0 && re <= n) {
      oc[ulo + k] = (uint64_t)outs | ((uint64_t)hots << 32);
      if constexpr (RANGE) oc1[ulo + k] = (uint64_t)(q1 & 0xffffu) | ((uint64_t)(q1 >> 16) << 32);
    } else {
      const int s = k == 0 ? 0 : 1;
      const uint32_t ins = (uint32_t)(b - a) - outs;
      s_ob[s] = outs ? (uint32_t)atomicAdd((unsigned long long*)&oc[ulo + k],
                                           (unsigned long long)outs | ((unsigned long long)hots << 32))
                     : 0u;
      if constexpr (RANGE)
        if (q1)
          atomicAdd((unsigned long long*)&oc1[ulo + k],
                    (unsigned long long)(q1 & 0xffffu) | ((unsigned long long)(q1 >> 16) << 32));
      s_ib[s] = ins ? atomicAdd(&ic[ulo + k], ins) : 0u;
    }
  }
  __syncthreads();
  if (live) {
    int cur = at, nxt = s_end[at];
#pragma unroll
    for (int j = 0; j < kPerThread; j++) {
      const int i = i0 + j;
      if (i < n) {
        if (ends[j]) {
          cur = i;
          nxt = ends[j];
        }
        const bool first = cur == 0 && s_rng[2];  // continues from an earlier chunk
        const uint32_t before = (uint32_t)(s_pre[i] - s_pre[cur]) & 0xffffu;
        const bool front = (small >> j) & 1u;
        if (!first && nxt <= n) {
          s_part[front ? cur + (int)before : nxt - 1 - (i - cur - (int)before)] = rv[j];
        } else {
          const int s = first || uhi == ulo ? 0 : 1;
          const int64_t u = s == 0 ? ulo : uhi;
          part[front ? off[u] + (int64_t)s_ob[s] + before
                     : off[u + 1] - 1 - (int64_t)s_ib[s] - (int64_t)(i - cur - (int)before)] = rv[j];
        }
      }
    }
  }
  __syncthreads();
  for (int i = s_rng[0] + tid; i < s_rng[1]; i += kBlock) part[eb + i] = s_part[i];  // the inner rows
}

// ---------------------------------------------------------------------------
// f(id) for the ids of a row, in order.  Beyond a wave's worth four loads are in
// flight instead of one after another: a hub's 1,500 ids are read twice for its list
// and by the wave of each of its chunks (R-MAT s22 6.35 -> 6.21 ms, per vertex with
// the generator's labels 17.0 -> 16.3; rows of up to 64 ids as before).
template <typename I, typename F>
__device__ __forceinline__ void each_id(uint32_t n, I&& id, F&& f) {
  if (n <= kWave) {
    f(id(0u));
    return;
  }
  for (uint32_t i = 0; i < n; i += 4 * kWave) {
    uint32_t y[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) y[k] = id(i + k * kWave);
#pragma unroll
    for (uint32_t k = 0; k < 4; k++)
      if (i + k * kWave < n) f(y[k]);
  }
}

// Lists and records, by independent waves.  A wave takes `rows` vertices at a
// time, one per lane, few neighbouring ones from all over the graph (labels that
// bring vertices of large degree together do not load one wave).  Their lists lie
// together, those of whole lines first, then of four, two and one chunk,
// placed by one scan over the four counts, in room that the wave draws
// `grant` lines at a time from one of kListShards regions (one atomic per 128
// vertices on one address made 9 of 19 ms at R-MAT s26).  Lists of up to
// kLaneList ids are written by their lane, unsorted: they fill a line at most.
// Longer ones are written by the whole wave, one after another: up to 64 ids
// are ranked by counting the smaller ones, more are sorted by a bit map of
// their hot ids in LDS with running counts (an id's place is the count before
// its word plus the bits below it).  Cold ids keep the row's order.
template <int MODE>
__global__ __launch_bounds__(64) void k_rank_lists(int64_t nv, const int64_t* __restrict__ off,
                                                   const uint64_t* __restrict__ oc, const uint64_t* __restrict__ oc1,
                                                   const uint32_t* __restrict__ rank,
                                                   const uint32_t* __restrict__ part, ListRoom lr,
                                                   uint4* __restrict__ lists, RankRec* __restrict__ rec,
                                                   uint64_t* __restrict__ counters) {
  constexpr int kGroups = 8;  // pairs of 64-bit words per lane
  __shared__ ulonglong2 s_bits[kGroups * kWave];
  __shared__ uint16_t s_pre[kGroups * kWave];
  constexpr bool PV = MODE == kPerVertex, RANGE = MODE == kRange;
  constexpr int kParts = RANGE ? 2 : 1;  // hot parts (and as many cold ones)
  __shared__ uint16_t s_mark[kRankMarks];
  const int lane = threadIdx.x;
  unsigned long long* bits = reinterpret_cast<unsigned long long*>(s_bits);
#pragma unroll
  for (int i = 0; i < kGroups; i++) s_bits[i * kWave + lane] = make_ulonglong2(0, 0);
  uint64_t room_at = 0, room_end = 0;  // lines drawn, not yet used (lane 0)
  int shard = (int)(blockIdx.x & (kListShards - 1));
  auto draw = [&](uint64_t lines) -> uint64_t {
    if (lines <= room_end - room_at) {
      room_at += lines;
      return room_at - lines;
    }
    const uint64_t ask = lines * 4 > lr.grant ? lines : lr.grant;  // leaves less than a quarter of a grant
    for (int k = 0; k < kListShards; k++) {  // a full region: the next one
      const uint64_t b = atomicAdd((unsigned long long*)&counters[kNumSlots + shard * kNumSums + kSumLists],
                                   (unsigned long long)ask);
      if (b + ask <= lr.region) {
        const uint64_t at = (uint64_t)shard * lr.region + b;
        if (ask > lines) {
          room_at = at + lines;
          room_end = at + ask;
        }
        return at;
      }
      shard = (shard + 1) & (kListShards - 1);
    }
    // Only for input that is no simple graph: the caller counts it with edge tiles.
    atomicAdd((unsigned long long*)&counters[kNoListRoom], 1ull);
    return kNoRank;
  };
  uint64_t edges = 0;
  for (int64_t batch = blockIdx.x; batch < lr.nbatch; batch += gridDim.x) {  // uniform
    // Group g of the wave's is group (g * a prime) mod the number of groups.
    const uint64_t groups = ((uint64_t)nv + (1u << lr.together) - 1) >> lr.together;
    const uint64_t g = (uint64_t)batch * (uint64_t)(lr.rows >> lr.together) + (uint64_t)(lane >> lr.together);
    const int64_t u = g < groups && lane < lr.rows ? (int64_t)((g * 2654435761ull % groups) << lr.together) | (lane & ((1 << lr.together) - 1)) : nv;
    const bool live = u < nv;
    uint32_t d = 0, h = 0, a0 = 0, ru = 0;
    uint32_t hc = 0, cc = 0;  // hot and cold chunks; RANGE: two parts each, part 1 << 16
    if (live) {
      const uint64_t q = oc[u];
      d = (uint32_t)q;
      h = (uint32_t)(q >> 32);
      a0 = (uint32_t)off[u];
      ru = rank[u];
      if (d >= 2) {  // a list of one id has no pair
        auto hot_chunks = [](uint32_t n) { return min((n + 7) >> 3, 8192u); };  // (the clamps hold for
        auto cold_chunks = [](uint32_t n) { return min((n + 3) >> 2, 65535u); };  // any simple graph)
        if constexpr (RANGE) {
          const uint64_t q1 = oc1[u];
          const uint32_t d1 = (uint32_t)q1, h1 = (uint32_t)(q1 >> 32);
          hc = hot_chunks(h1) | hot_chunks(h - h1) << 16;
          cc = cold_chunks(d1 - h1) | cold_chunks((d - d1) - (h - h1)) << 16;
        } else {
          hc = hot_chunks(h);
          cc = cold_chunks(d - h);
        }
      }
    }
    if constexpr (!RANGE) edges += d;
    auto both = [](uint32_t c) -> uint32_t { return RANGE ? (c & 0xffffu) + (c >> 16) : c; };
    const uint32_t room = list_room(both(hc) + both(cc));
    // lines: bits 0-31; lists of four, two, one chunk: 10 bits each from 32 on
    const int64_t mine = room >= 8 ? (int64_t)(room >> 3) : room == 4 ? 1ll << 32 : room == 2 ? 1ll << 42 : room == 1 ? 1ll << 52 : 0ll;
    const int64_t inc = wave_incl_scan_i64(mine), at = inc - mine, total = readlane64(inc, kWave - 1);
    auto field = [](int64_t v, int sh) -> uint32_t { return (uint32_t)(v >> sh) & 1023u; };
    const uint32_t n8 = (uint32_t)total, n4 = field(total, 32), n2 = field(total, 42), n1 = field(total, 52);
    const uint32_t chunks = 8 * n8 + 4 * n4 + 2 * n2 + n1;
    uint32_t base = 0;
    if (chunks) {  // uniform
      if (lane == 0) base = (uint32_t)draw((chunks + 7) >> 3);
      base = __builtin_amdgcn_readfirstlane(base);
    }
    uint32_t start = 0;
    if (room) {
      if (base == kNoRank) {
        d = hc = cc = 0;
      } else {
        const uint32_t b4 = 8 * n8, b2 = b4 + 4 * n4, b1 = b2 + 2 * n2;
        start = 8 * base + (room >= 8   ? 8 * (uint32_t)at
                            : room == 4 ? b4 + 4 * field(at, 32)
                            : room == 2 ? b2 + 2 * field(at, 42)
                                        : b1 + field(at, 52));
      }
    }
    const bool alone = live && d <= kLaneList;
    if (alone && d < 2) {
      uint4* to = reinterpret_cast<uint4*>(rec + ru);
      to[0] = make_uint4(0, 0, 0, 0);
      to[1] = make_uint4(0, 0, 0, PV ? (uint32_t)u : 0u);
    }
    if constexpr (RANGE) {
      if (alone && d >= 2) {  // part by part: hot ids, padding, cold ids, padding
        uint16_t* hot[2] = {reinterpret_cast<uint16_t*>(lists + start),
                            reinterpret_cast<uint16_t*>(lists + start + (hc & 0xffffu))};
        uint32_t* cold[2] = {reinterpret_cast<uint32_t*>(lists + start + both(hc)),
                             reinterpret_cast<uint32_t*>(lists + start + both(hc) + (cc & 0xffffu))};
        uint32_t nh[2] = {0, 0}, nc[2] = {0, 0}, least[2] = {kHot, kHot};
        for (uint32_t i = 0; i < d; i++) {
          const uint32_t w = part[a0 + i], r = w & ~kOwnedBit;
          const bool rest = !(w & kOwnedBit);
#pragma unroll
          for (int p = 0; p < 2; p++) {
            if (rest != (p == 1)) continue;
            if (r < kHot) {
              hot[p][nh[p]++] = (uint16_t)r;
              least[p] = min(least[p], r);
            } else {
              cold[p][nc[p]++] = r;
            }
          }
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
          for (; nh[p] & 7; nh[p]++) hot[p][nh[p]] = 0xffff;
          for (; nc[p] & 3; nc[p]++) cold[p][nc[p]] = kNoRank;
        }
        // Not sorted: all of a part or nothing of it is below v.
        uint4* to = reinterpret_cast<uint4*>(rec + ru);
        to[0] = make_uint4(start, hc, cc, least[0] | (least[0] << 16));
        to[1] = make_uint4(least[0] | (least[1] << 16), least[1] | (least[1] << 16), least[1] | 0xffff0000u, ~0u);
      }
    } else if (__builtin_amdgcn_ballot_w64(alone && d >= 2)) {  // uniform
      uint64_t lo = ~0ull, hi = ~0ull;
      uint32_t least = kHot, nh = 0, nc = 0;
      uint4* hot = lists + start;
      uint32_t* cold = reinterpret_cast<uint32_t*>(lists + start + hc);
      const uint32_t n = alone && d >= 2 ? d : 0;
      for (uint32_t i0 = 0; __builtin_amdgcn_ballot_w64(i0 < n); i0 += 8) {
        uint32_t w[8];
#pragma unroll
        for (int i = 0; i < 8; i++) w[i] = i0 + i < n ? part[a0 + i0 + i] : kNoRank;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          if (w[i] < kHot) {
            hi = (hi << 16) | (lo >> 48);
            lo = (lo << 16) | w[i];
            least = min(least, w[i]);
            if ((++nh & 7) == 0) {
              hot[(nh >> 3) - 1] = make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
              lo = hi = ~0ull;
            }
          } else if (i0 + i < n) {
            cold[nc++] = w[i];
          }
        }
      }
      if (n) {
        if (nh & 7) hot[nh >> 3] = make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
        for (; nc & 3; nc++) cold[nc] = kNoRank;
        static_assert(kLaneList <= 32, "four marks");
        const uint32_t m = least | (least << 16);  // not sorted: all of it or nothing is below v
        uint4* to = reinterpret_cast<uint4*>(rec + ru);
        to[0] = make_uint4(start, hc | (cc << 16), m, m);
        to[1] = make_uint4(~0u, ~0u, ~0u, PV ? (uint32_t)u : ~0u);
      }
    }
    uint64_t todo = __builtin_amdgcn_ballot_w64(live && d > kLaneList);
    // The next row: first entry, ids, list, rank, label, chunks; its first ids.
    uint32_t ra = 0, rd = 0, rs = 0, rr = 0, ro = 0, rhc = 0, rcc = 0, rw = kNoRank;
    auto pop = [&]() {
      const int src = __builtin_ctzll(todo);
      todo &= todo - 1;
      ra = __builtin_amdgcn_readlane(a0, src);
      rd = __builtin_amdgcn_readlane(d, src);
      rs = __builtin_amdgcn_readlane(start, src);
      rr = __builtin_amdgcn_readlane(ru, src);
      if constexpr (PV) ro = __builtin_amdgcn_readlane((uint32_t)u, src);
      rhc = __builtin_amdgcn_readlane(hc, src);
      rcc = __builtin_amdgcn_readlane(cc, src);
      rw = part[ra + lane];  // more than 32 ids and, in a simple graph, as many behind; the array is padded
    };
    bool more = todo != 0;
    if (more) pop();
    while (more) {  // uniform
      const uint32_t dd = rd, st = rs, rk = rr, label = ro, hcs = rhc, ccs = rcc, w0 = (uint32_t)lane < rd ? rw : kNoRank;
      const uint32_t* ids = part + ra;
      more = todo != 0;
      if (more) pop();  // the next row's ids fly while this one is written
      auto raw = [&](uint32_t i) -> uint32_t { return i == 0 ? w0 : i + lane < dd ? ids[i + lane] : kNoRank; };
      if (lane < kRankMarks) s_mark[lane] = 0xffff;
      uint32_t mark0 = 0, hot0 = 0, cold0 = both(hcs);  // where the part's marks and chunks start
#pragma unroll
      for (int part_no = 0; part_no < kParts; part_no++) {
        const uint32_t hcc = RANGE ? (hcs >> (16 * part_no)) & 0xffffu : hcs;
        const uint32_t ccc = RANGE ? (ccs >> (16 * part_no)) & 0xffffu : ccs;
        const uint32_t marks = !RANGE ? hot_marks<MODE>() : part_no == 0 ? kMarksOwned : kMarksRest;
        // The part's rank at i + lane, kNoRank where it has none.
        auto id = [&](uint32_t i) -> uint32_t {
          const uint32_t w = raw(i);
          if constexpr (RANGE)
            return w != kNoRank && (w & kOwnedBit ? 0 : 1) == part_no ? w & ~kOwnedBit : kNoRank;
          else
            return w;
        };
        uint32_t hh = 0, place = 0;
        if (dd <= kWave) {
          const uint32_t w = id(0);
          const uint64_t hm = __builtin_amdgcn_ballot_w64(w < kHot);
          hh = (uint32_t)__popcll(hm);
          for (uint64_t m = hm; m; m &= m - 1)
            place += (uint32_t)__builtin_amdgcn_readlane((int)w, __builtin_ctzll(m)) < w ? 1u : 0u;
        } else {
          uint32_t top = 0;  // groups in use
          each_id(dd, id, [&](uint32_t w) {
            if (w < kHot) {
              atomicOr(&bits[w >> 6], 1ull << (w & 63));
              top = max(top, (w >> 13) + 1);
            }
          });
          wave_lds_fence();
#pragma unroll 1
          for (uint32_t k = 0; k < (uint32_t)kGroups; k++) {
            if (__builtin_amdgcn_ballot_w64(top > k) == 0) break;
            const ulonglong2 t = s_bits[k * kWave + lane];
            const uint32_t n = (uint32_t)(__popcll(t.x) + __popcll(t.y));
            const uint32_t upto = wave_incl_scan_u32(n);
            s_pre[k * kWave + lane] = (uint16_t)(hh + upto - n);
            hh += __builtin_amdgcn_readlane(upto, kWave - 1);
          }
        }
        wave_lds_fence();
        const uint32_t seg = 8 * max(mark_step(hcc, marks), 1u);          // ids per segment
        const uint32_t inv = (uint32_t)(((1ull << 32) + seg - 1) / seg);  // r / seg for r < 2^16
        uint16_t* hl = reinterpret_cast<uint16_t*>(lists + st + hot0);
        uint32_t* cl = reinterpret_cast<uint32_t*>(lists + st + cold0);
        uint32_t ncold = 0;
        each_id(dd, id, [&](uint32_t w) {
          const bool cold = w >= kHot && w != kNoRank;
          const uint64_t cm = __builtin_amdgcn_ballot_w64(cold);
          if (w < kHot) {
            uint32_t r = place;
            if (dd > kWave) {
              const ulonglong2 t = s_bits[w >> 7];
              const uint64_t below = (1ull << (w & 63)) - 1ull;
              r = s_pre[w >> 7] + (uint32_t)((w & 64) ? __popcll(t.x) + __popcll(t.y & below) : __popcll(t.x & below));
            }
            if (r < 8 * hcc) hl[r] = (uint16_t)w;
            const uint32_t k = __umulhi(r, inv);
            if (k * seg == r && k < marks) s_mark[mark0 + k] = (uint16_t)w;
          } else if (cold) {
            const uint32_t r = ncold + lanes_below(cm);
            if (r < 4 * ccc) cl[r] = w;
          }
          ncold += (uint32_t)__popcll(cm);
        });
        wave_lds_fence();
        if (dd > kWave) {  // uniform
#pragma unroll
          for (int k = 0; k < kGroups; k++) s_bits[k * kWave + lane] = make_ulonglong2(0, 0);
        }
        if ((uint32_t)lane < 8 * hcc - min(hh, 8 * hcc)) hl[hh + lane] = 0xffff;
        if ((uint32_t)lane < 4 * ccc - min(ncold, 4 * ccc)) cl[ncold + lane] = kNoRank;
        mark0 += marks;
        hot0 += hcc;
        cold0 += ccc;
        wave_lds_fence();
      }
      if (lane < 8) {
        constexpr int kFirst = RANGE ? 3 : 2;  // words before the marks
        const uint32_t m = lane >= kFirst ? (uint32_t)s_mark[2 * (lane - kFirst)] | ((uint32_t)s_mark[2 * (lane - kFirst) + 1] << 16) : 0u;
        reinterpret_cast<uint32_t*>(rec + rk)[lane] = lane == 0   ? st
                                                      : lane == 1 ? (RANGE ? hcs : hcs | (ccs << 16))
                                                      : RANGE && lane == 2 ? ccs
                                                      : PV && lane == 7    ? label
                                                                           : m;
      }
      wave_lds_fence();
    }
  }
  if constexpr (!RANGE) {
    edges = wave_sum_u64(edges);
    if (lane == 0) add_sum(counters, kSumEdges, edges);
  }
}

// ---------------------------------------------------------------------------
// One wave per chunk of S entries.  For every row v with N(v) not empty and
// larger neighbours u in the chunk: N(v)'s hot ids become a bit map in LDS and
// the u's hot prefixes are streamed through it; a cold v with cold ids hashes
// these in the same LDS and streams the u's cold lists.
//
// 64 items (u's) are taken at once, one per lane, their 16-byte chunks numbered
// through and dealt out one per lane and step, so every lane has a chunk
// whatever the lists' lengths (a list per group of 4-16 lanes left 62 % of the
// lanes without one at R-MAT s24: 27.4 ms against 21.9).  Chunk c belongs to item (number of items that
// start at 1 .. c): lane b keeps the bits of the starts in chunks 64 b + 1 ..
// 64 b + 64, so a step needs two readlanes and a masked bit count.
constexpr int kStreamBlocks = kWave;  // 64-chunk blocks that the bits cover

// LDS of one wave's streaming.
struct StreamLds {
  unsigned long long bit[kStreamBlocks];
  uint32_t adj[kWave];  // per item with chunks: its list's start less its first chunk
};
// Per item: u's label and the hits credited to u (per-vertex counts), or a mask
// of the hits that count as local (owned ranges).
struct ItemLds {
  uint32_t label[kWave];
  uint32_t hits[kWave];
};

// probe(chunk, item): item is the chunk's index among the items with chunks.
// kPerVertex: `label` is u's label; the hits that probe adds to items are added
// to pv, after done(), which ends what probe has put off.  kRange: `label` is
// kept for probe.
template <int MODE, typename F, typename G>
__device__ __forceinline__ void stream_lists(uint32_t start, uint32_t n, uint32_t label, StreamLds& s, ItemLds* s_items,
                                             int lane, const uint4* __restrict__ lists, uint32_t pad,
                                             unsigned long long* __restrict__ pv, F&& probe, G&& done) {
  const uint32_t inc = wave_incl_scan_u32(n);
  const uint32_t all = __builtin_amdgcn_readlane(inc, kWave - 1);
  if (all == 0) return;  // uniform
  auto load = [&](uint32_t at, bool on) -> uint4 {
    uint4 v = make_uint4(pad, pad, pad, pad);
    if (on) v = lists[at];
    return v;
  };
  const uint64_t some = __builtin_amdgcn_ballot_w64(n > 0);
  if constexpr (MODE != kTotal) {
    wave_lds_fence();
    if (n > 0) s_items->label[lanes_below(some)] = label;
    if constexpr (MODE == kPerVertex) s_items->hits[lane] = 0;
    wave_lds_fence();
  }
  if (all <= kStreamBlocks * kWave) {
    const uint32_t p = inc - n;
    wave_lds_fence();
    s.bit[lane] = 0ull;
    if (n > 0) s.adj[lanes_below(some)] = start - p;
    wave_lds_fence();
    if (n > 0 && p > 0) atomicOr(&s.bit[(p - 1) >> 6], 1ull << ((p - 1) & 63));
    wave_lds_fence();
    const int64_t my = (int64_t)s.bit[lane];
    const int steps = (int)((all + kWave - 1) / kWave);
    uint32_t before = 0;
    auto next = [&](int b, uint32_t& item) -> uint4 {
      const uint64_t m = (uint64_t)readlane64(my, b);
      const uint32_t c = (uint32_t)b * kWave + lane;
      item = before + lanes_below(m);
      const uint32_t at = s.adj[item] + c;
      before += (uint32_t)__popcll(m);
      return load(at, c < all);
    };
    // Two buffers by hand: the next step's loads are in flight while one is probed.
    uint32_t ia = 0, ib = 0;
    uint4 va = next(0, ia), vb;
    for (int b = 1;; b += 2) {
      if (b < steps) vb = next(b, ib);
      probe(va, ia);
      if (b >= steps) break;
      if (b + 1 < steps) va = next(b + 1, ia);
      probe(vb, ib);
      if (b + 1 >= steps) break;
    }
  } else {  // long lists: the whole wave on one item at a time
    uint32_t item = 0;
    for (uint64_t left = some; left; left &= left - 1, item++) {
      const int k = __builtin_ctzll(left);
      const uint32_t s0 = __builtin_amdgcn_readlane(start, k), nk = __builtin_amdgcn_readlane(n, k);
      uint4 va = load(s0 + lane, (uint32_t)lane < nk), vb;
      for (uint32_t c = kWave;; c += 2 * kWave) {
        if (c < nk) vb = load(s0 + c + lane, c + lane < nk);
        probe(va, item);
        if (c >= nk) break;
        if (c + kWave < nk) va = load(s0 + c + kWave + lane, c + kWave + lane < nk);
        probe(vb, item);
        if (c + kWave >= nk) break;
      }
    }
  }
  if constexpr (MODE == kPerVertex) {
    done();
    wave_lds_fence();
    const uint32_t t = s_items->hits[lane];
    if (t) atomicAdd(&pv[s_items->label[lane]], (unsigned long long)t);
    wave_lds_fence();
  }
}

template <int LOGB>
__device__ __forceinline__ void cold_table_clear(int4* tab, int lane) {
#pragma unroll
  for (int i = 0; i < (1 << LOGB) / kWave; i++) tab[lane + kWave * i] = make_int4(kEmpty, kEmpty, kEmpty, kEmpty);
  wave_lds_fence();
}

struct Head {  // a record
  uint4 a, b;
};

// PV: every triangle is credited to its smallest label (xxtric.hpp:165).  A hit
// w of the item u in v's map: with its place p among N(v)'s hot ids (count
// before its word plus the bits below it) s_label[p] is w's label; if it is the
// smallest, slot p counts it (added to pv when the row ends), otherwise u's item
// counter or v's register does.  Places from kSlots on, cold hits and the rows of
// few ids look labels up and add to pv directly.
// A lane has 0 to 8 hits of a chunk (2 on average at R-MAT s22), so the hits of a
// step are put into a queue first and taken from it 128 at a time, two a lane
// (R-MAT s22, this kernel: 20.5 ms with every lane its own hits one after another,
// 15.2 with 64 at a time, 14.6 with 128).  What bounds it is the wait for LDS at
// eight waves a compute unit, and the slots: with the generator's labels, where
// hubs are credited, 512 take 27.9 ms, 1024 14.3, and 2048, with fewer waves, 21.7.
constexpr int kSlots = 1024;
constexpr int kQueue = 10 * kWave;  // a step's hits behind up to 127 older ones
struct PvLds {
  uint32_t queue[kQueue];  // hit | item << 16
  uint16_t pre[1024];  // hot ids of N(v) before each 64-bit word of the map
  uint32_t label[kSlots];
  uint32_t hits[kSlots / 2];  // 16 bits each: a row's items in a chunk hit a place once each
  static_assert(kChunk < 65536, "hits of a place");
  ItemLds items;
};
struct RangeLds {
  ItemLds items;
};
struct NoLds {};

// kRange: a triangle with its labels above rlo counts as owned when one of its
// vertices is owned, as local when two are.  Of u's list the owned ids are
// streamed for every item, the others only where u or v is owned (rank 0 of 8
// of R-MAT s23: 20.3 ms in edge tiles, 12.3 here, 6.0 of them in this kernel
// against 9.2 for the total).
template <int MODE>
__global__ __launch_bounds__(64) void k_rank_count(int64_t nv, int64_t ne, const int64_t* __restrict__ off,
                                                   const uint32_t* __restrict__ rank, const uint64_t* __restrict__ oc,
                                                   const uint32_t* __restrict__ part, const RankRec* __restrict__ rec,
                                                   const uint4* __restrict__ lists, const int32_t* __restrict__ crows,
                                                   int64_t S, uint64_t* __restrict__ counters,
                                                   const uint32_t* __restrict__ orig,
                                                   unsigned long long* __restrict__ pv, int64_t rlo, int64_t rhi) {
  constexpr bool PV = MODE == kPerVertex, RANGE = MODE == kRange;
  constexpr int kWords = 2048;
  constexpr int kColdSmall = 6, kColdBig = 9;  // hash buckets (log2) for up to 128 and up to 1024 cold ids
  __shared__ uint4 s_mem[kWords / 4];
  __shared__ StreamLds s_stream;
  __shared__ typename std::conditional<PV, PvLds, typename std::conditional<RANGE, RangeLds, NoLds>::type>::type s_pv;
  ItemLds* s_items = nullptr;
  if constexpr (MODE != kTotal) s_items = &s_pv.items;
  uint32_t* s_bm = reinterpret_cast<uint32_t*>(s_mem);
  int4* s_tab = reinterpret_cast<int4*>(s_mem);
  const int lane = threadIdx.x;
  const int64_t c = blockIdx.x;
  const int64_t eb = c * S, ee = min(ne, eb + S);
  int64_t row_lo = crows[2 * c], row_hi = crows[2 * c + 1];
  row_lo = row_lo < 0 ? 0 : (row_lo > nv - 1 ? nv - 1 : row_lo);
  row_hi = row_hi < row_lo ? row_lo : (row_hi > nv - 1 ? nv - 1 : row_hi);
  auto clear_words = [&](int quads) {  // 16-byte pieces from the front
    for (int i = lane; i < quads; i += kWave) s_mem[i] = make_uint4(0, 0, 0, 0);
  };
  clear_words(kWords / 4);
  if constexpr (PV)
    for (int i = lane; i < kSlots / 2; i += kWave) s_pv.hits[i] = 0;
  wave_lds_fence();
  uint64_t hits = 0, local = 0;  // local: kRange
  auto strip = [](uint32_t w) -> uint32_t { return RANGE && w != kNoRank ? w & ~kOwnedBit : w; };
  auto owned = [&](uint32_t label) -> bool { return (int64_t)label >= rlo && (int64_t)label < rhi; };
  auto tiny_rows = [&](bool tiny, uint32_t a0, uint32_t is, uint32_t items, uint32_t d, uint32_t row0) -> uint32_t {
    const uint32_t n = tiny ? items : 0;
    const uint32_t inc = wave_incl_scan_u32(n), p = inc - n;
    const uint32_t all = __builtin_amdgcn_readlane(inc, kWave - 1);
    const uint64_t some = __builtin_amdgcn_ballot_w64(n > 0);
    wave_lds_fence();
    s_stream.bit[lane] = 0ull;
    if (n > 0) s_stream.adj[lanes_below(some)] = (uint32_t)lane;
    wave_lds_fence();
    if (n > 0 && p > 0) atomicOr(&s_stream.bit[(p - 1) >> 6], 1ull << ((p - 1) & 63));
    wave_lds_fence();
    const int64_t my = (int64_t)s_stream.bit[lane];
    uint32_t before = 0, acc = 0;
    for (uint32_t b = 0; b * kWave < all; b++) {
      const uint64_t m = (uint64_t)readlane64(my, (int)b);
      const uint32_t c = b * kWave + lane;
      const int row = (int)s_stream.adj[before + lanes_below(m)];
      before += (uint32_t)__popcll(m);
      const uint32_t entry = (uint32_t)__shfl((int)(is - p), row, kWave) + c;
      const uint32_t first = (uint32_t)__shfl((int)a0, row, kWave), nd = (uint32_t)__shfl((int)d, row, kWave);
      uint32_t x[kTinyRow];
      uint2 r = make_uint2(0, 0);
      uint32_t two = 0;  // PV: the smaller of u's and v's label; RANGE: how many of the two are owned
      uint32_t cold2 = 0;  // RANGE: the cold parts' chunks
#pragma unroll
      for (int i = 0; i < kTinyRow; i++) x[i] = kNoRank - 1;  // matches no id and no padding
      if (c < all) {
        const uint32_t ur = part[entry];
#pragma unroll
        for (int i = 0; i < kTinyRow; i++)
          if ((uint32_t)i < nd) x[i] = strip(part[first + i]);
        if (ur != kNoRank) {
          const RankRec* q = rec + strip(ur);
          r = *reinterpret_cast<const uint2*>(q);
          if constexpr (PV) two = min(q->mark[5], row0 + (uint32_t)row);
          if constexpr (RANGE) {
            cold2 = q->mark[0];
            two = (ur & kOwnedBit ? 1u : 0u) + (owned(row0 + (uint32_t)row) ? 1u : 0u);
          }
        }
      }
      // PV: the ids w of a chunk that N(v) holds (bit j: id j), one credit each.
      auto credit = [&](uint32_t found, auto&& w) {
        acc += (uint32_t)__popc(found);
        while (found) {
          const int j = __builtin_ctz(found);
          found &= found - 1;
          atomicAdd(&pv[min(two, orig[w(j)])], 1ull);
        }
      };
      // One hot and one cold part: cnt chunks from `from`, every id compared with
      // every id of N(v); every lane its own item's.
      auto hot_part = [&](uint32_t from, uint32_t cnt) -> uint32_t {
        uint32_t acc = 0;
        for (uint32_t k = 0; __builtin_amdgcn_ballot_w64(k < cnt); k++) {
          if (k < cnt) {
            const uint4 q = lists[from + k];
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
            uint32_t found = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
              const uint32_t lo = w[j] & 0xffffu, hi = w[j] >> 16;
              const uint32_t lo2 = lo < kHot ? lo : kNoRank, hi2 = hi < kHot ? hi : kNoRank;
              bool in_lo = false, in_hi = false;
#pragma unroll
              for (int i = 0; i < kTinyRow; i++) {
                if constexpr (PV) {
                  in_lo |= x[i] == lo2;
                  in_hi |= x[i] == hi2;
                } else {
                  acc += (x[i] == lo2 ? 1u : 0u) + (x[i] == hi2 ? 1u : 0u);
                }
              }
              found |= (in_lo ? 1u : 0u) << (2 * j) | (in_hi ? 1u : 0u) << (2 * j + 1);
            }
            if constexpr (PV)
              credit(found, [&](int j) { return ((j & 4) ? (j & 2 ? w[3] : w[2]) : (j & 2 ? w[1] : w[0])) >> (16 * (j & 1)) & 0xffffu; });
          }
        }
        return acc;
      };
      auto cold_part = [&](uint32_t from, uint32_t cnt) -> uint32_t {
        uint32_t acc = 0;
        for (uint32_t k = 0; __builtin_amdgcn_ballot_w64(k < cnt); k++) {
          if (k < cnt) {
            const uint4 q = lists[from + k];
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
            uint32_t found = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
              bool in = false;
#pragma unroll
              for (int i = 0; i < kTinyRow; i++) {
                if constexpr (PV)
                  in |= x[i] == w[j];
                else
                  acc += x[i] == w[j] ? 1u : 0u;
              }
              found |= (in ? 1u : 0u) << j;
            }
            if constexpr (PV) credit(found, [&](int j) { return (j & 2) ? (j & 1 ? w[3] : w[2]) : (j & 1 ? w[1] : w[0]); });
          }
        }
        return acc;
      };
      if constexpr (RANGE) {
        const uint32_t h0 = r.y & 0xffffu, h1 = r.y >> 16, c0 = cold2 & 0xffffu, c1 = cold2 >> 16;
        const uint32_t a = hot_part(r.x, h0) + cold_part(r.x + h0 + h1, c0);  // owned ids
        const uint32_t o = hot_part(r.x + h0, two ? h1 : 0) + cold_part(r.x + h0 + h1 + c0, two ? c1 : 0);
        acc += a + o;
        local += (two ? a : 0) + (two == 2 ? o : 0);
      } else {
        const uint32_t hc = r.y & 0xffffu, cc = r.y >> 16;
        acc += hot_part(r.x, hc) + cold_part(r.x + hc, cc);
      }
    }
    return acc;
  };
  for (int64_t rb = row_lo; rb <= row_hi; rb += kWave) {
    const int64_t r = rb + lane;
    int64_t a0 = 0, is = 0, ie = 0;
    uint32_t d = 0, h = 0, v = 0;
    if (r <= row_hi) {
      const uint64_t q = oc[r];
      a0 = off[r];
      ie = min(off[r + 1], ee);
      v = rank[r];
      d = (uint32_t)q;
      h = (uint32_t)(q >> 32);
      is = max(a0 + (int64_t)d, eb);
    }
    const bool work = d > 0 && is < ie;
    // Rows of few ids and few items: their items are taken together, one lane
    // per item, every id of N(v) compared with every id of u's list.
    const bool tiny = work && d <= kTinyRow && ie - is <= kWave;
    if (__builtin_amdgcn_ballot_w64(tiny)) 
      hits += tiny_rows(tiny, (uint32_t)a0, (uint32_t)is, (uint32_t)(ie - is), d, (uint32_t)rb);
    uint64_t todo = __builtin_amdgcn_ballot_w64(work && !tiny);
    // Row by row; the next row's ids and items are loaded before the current
    // row's map is built, its items' records before the current lists stream.
    uint32_t b0 = 0, s0 = 0, s1 = 0, dd = 0, hh = 0, vv = 0, vo = 0;
    auto pop = [&]() {
      const int src = __builtin_ctzll(todo);
      todo &= todo - 1;
      b0 = __builtin_amdgcn_readlane((uint32_t)a0, src);
      s0 = __builtin_amdgcn_readlane((uint32_t)is, src);
      s1 = __builtin_amdgcn_readlane((uint32_t)ie, src);
      dd = __builtin_amdgcn_readlane(d, src);
      hh = __builtin_amdgcn_readlane(h, src);
      vv = __builtin_amdgcn_readlane(v, src);
      vo = (uint32_t)rb + (uint32_t)src;
    };
    auto item = [&](uint32_t e) -> uint32_t { return e + lane < s1 ? part[e + lane] : kNoRank; };
    auto head = [&](uint32_t ur) -> Head {
      Head x{make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
      if (ur != kNoRank) {
        const uint4* q = reinterpret_cast<const uint4*>(rec + strip(ur));
        x.a = q[0];
        x.b = q[1];
      }
      return x;
    };
    if (todo == 0) continue;  // uniform
    pop();
    uint32_t w0 = (uint32_t)lane < dd ? strip(part[b0 + lane]) : kNoRank;
    uint32_t xu = item(s0);
    Head x = head(xu);
    for (;;) {  // uniform
      const uint32_t cb = b0, cs0 = s0, cs1 = s1, cd = dd, ch = hh, cv = vv, cl = vo, w = w0;
      const bool more = todo != 0;
      uint32_t un = kNoRank;
      if (more) {
        pop();
        w0 = (uint32_t)lane < dd ? strip(part[b0 + lane]) : kNoRank;
        un = item(s0);
      }
      auto id = [&](uint32_t i) -> uint32_t { return i == 0 ? w : i + lane < cd ? strip(part[cb + i + lane]) : kNoRank; };
      // Hot chunks of the item whose record is h that hold every id below v.
      auto prefix = [&](const Head& h) -> uint32_t {
        const uint32_t hot = h.a.y & 0xffffu;
        const uint32_t mk[kRankMarks / 2] = {h.a.z, h.a.w, h.b.x, h.b.y, h.b.z, h.b.w};
        uint32_t segs = 0;  // segments that start below v
#pragma unroll
        for (int t = 0; t < (int)hot_marks<MODE>() / 2; t++) segs += ((mk[t] & 0xffffu) < cv ? 1u : 0u) + ((mk[t] >> 16) < cv ? 1u : 0u);
        return min(segs * mark_step(hot, hot_marks<MODE>()), hot);
      };
      // kRange: the same of the owned ids and of the others.
      auto prefix_owned = [&](const Head& h) -> uint32_t {
        const uint32_t hot = h.a.y & 0xffffu;
        const uint32_t segs = ((h.a.w & 0xffffu) < cv ? 1u : 0u) + ((h.a.w >> 16) < cv ? 1u : 0u) + ((h.b.x & 0xffffu) < cv ? 1u : 0u);
        return min(segs * mark_step(hot, kMarksOwned), hot);
      };
      auto prefix_rest = [&](const Head& h) -> uint32_t {
        const uint32_t hot = h.a.y >> 16;
        const uint32_t mk[3] = {h.b.y, h.b.z, h.b.w};
        uint32_t segs = (h.b.x >> 16) < cv ? 1u : 0u;
#pragma unroll
        for (int t = 0; t < 3; t++) segs += ((mk[t] & 0xffffu) < cv ? 1u : 0u) + ((mk[t] >> 16) < cv ? 1u : 0u);
        return min(segs * mark_step(hot, kMarksRest), hot);
      };
      const bool v_own = RANGE && owned(cl);  // uniform
      const bool cold = ch < cd && cv > kHot;  // cold ids below a cold v
      const uint32_t st = x.a.x, len = x.a.y, len2 = x.a.z, label = x.b.w, u0 = xu;  // the first 64 items
      const uint32_t n = RANGE ? prefix_owned(x) : prefix(x);
      const uint32_t n_rest = RANGE && (v_own || (u0 & kOwnedBit && u0 != kNoRank)) ? prefix_rest(x) : 0;
      uint32_t at_v = 0;  // PV: hits credited to v
      if (ch > 0)
        each_id(cd, id, [&](uint32_t y) {
          if (y < kHot) atomicOr(&s_bm[y >> 5], 1u << (y & 31));
        });
      unsigned long long* s_map = reinterpret_cast<unsigned long long*>(s_mem);
      auto place = [&](uint32_t y) -> uint32_t {  // of hot id y of N(v)
        if constexpr (PV)
          return s_pv.pre[y >> 6] + (uint32_t)__popcll(s_map[y >> 6] & ((1ull << (y & 63)) - 1ull));
        else
          return 0;
      };
      if constexpr (PV) {
        if (ch > 0) {
          wave_lds_fence();
          if (cd <= kWave) {  // counts at the words in use, by comparing the ids
            uint32_t less = 0;
            for (uint64_t m = __builtin_amdgcn_ballot_w64(w < kHot); m; m &= m - 1)
              less += ((uint32_t)__builtin_amdgcn_readlane((int)w, __builtin_ctzll(m)) >> 6) < (w >> 6) ? 1u : 0u;
            if (w < kHot) s_pv.pre[w >> 6] = (uint16_t)less;
          } else {
            uint32_t base = 0;
            for (int g = 0; g < 1024 / kWave && base < ch; g++) {
              const uint32_t t = (uint32_t)__popcll(s_map[g * kWave + lane]);
              const uint32_t upto = wave_incl_scan_u32(t);
              s_pv.pre[g * kWave + lane] = (uint16_t)(base + upto - t);
              base += __builtin_amdgcn_readlane(upto, kWave - 1);
            }
          }
          wave_lds_fence();
          each_id(cd, id, [&](uint32_t y) {
            if (y < kHot) {
              const uint32_t p = place(y);
              if (p < kSlots) s_pv.label[p] = orig[y];
            }
          });
          wave_lds_fence();
        }
      }
      if (more) {
        x = head(un);
        xu = un;
      }
      auto items = [&](uint32_t e) -> uint32_t { return e + lane < cs1 ? part[e + lane] : kNoRank; };
      if (ch > 0) {
        uint32_t acc = 0, acc_local = 0;
        uint32_t queued = 0;  // PV, uniform
        // K queue entries a lane (kNoRank: none), their chains of LDS reads side by side.
        auto credit = [&](const auto& e) {
          if constexpr (PV) {
            constexpr int K = sizeof(e) / sizeof(e[0]);
            uint32_t lu[K], p[K], lw[K];
#pragma unroll
            for (int k = 0; k < K; k++) {
              lu[k] = s_pv.items.label[(e[k] >> 16) & 63u];
              p[k] = place(e[k] & 0xffffu);
            }
#pragma unroll
            for (int k = 0; k < K; k++) lw[k] = s_pv.label[min(p[k], (uint32_t)kSlots - 1)];
#pragma unroll
            for (int k = 0; k < K; k++) {
              if (e[k] == kNoRank) continue;
              if (p[k] >= kSlots) lw[k] = orig[e[k] & 0xffffu];
              if (lw[k] > min(lu[k], cl)) {
                if (cl < lu[k])
                  at_v++;
                else
                  atomicAdd(&s_pv.items.hits[e[k] >> 16], 1u);
              } else if (p[k] < kSlots) {
                atomicAdd(&s_pv.hits[p[k] >> 1], 1u << (16 * (p[k] & 1)));
              } else {
                atomicAdd(&pv[lw[k]], 1ull);
              }
            }
          }
        };
        auto probe = [&](const uint4 q, uint32_t item) {
          const uint32_t y[4] = {q.x, q.y, q.z, q.w};
          uint32_t found = 0;
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const uint32_t lo = s_bm[(y[j] >> 5) & 2047u], hi = s_bm[y[j] >> 21];
            const uint32_t t0 = (lo >> (y[j] & 31)) & 1u, t1 = (hi >> ((y[j] >> 16) & 31)) & 1u;
            if constexpr (PV)
              found |= t0 << (2 * j) | t1 << (2 * j + 1);
            else if constexpr (RANGE)
              found += t0 + t1;
            else
              acc += t0 + t1;
          }
          if constexpr (RANGE) {
            acc += found;
            acc_local += found & s_pv.items.label[item];
          }
          if constexpr (PV) {
            const uint32_t n = (uint32_t)__popc(found), inc = wave_incl_scan_u32(n);
            acc += n;
            uint32_t at = queued + inc - n;
#pragma unroll
            for (int j = 0; j < 8; j++) {
              if ((found >> j) & 1u) {
                s_pv.queue[at] = (j & 1 ? y[j / 2] >> 16 : y[j / 2] & 0xffffu) | (item << 16);
                at++;
              }
            }
            queued += __builtin_amdgcn_readlane(inc, kWave - 1);
            wave_lds_fence();
            while (queued >= 2 * kWave) {  // uniform
              queued -= 2 * kWave;
              const uint32_t e[2] = {s_pv.queue[queued + lane], s_pv.queue[queued + kWave + lane]};
              credit(e);
            }
            wave_lds_fence();
          }
        };
        auto done = [&]() {
          if constexpr (PV) {
            if (queued == 0) return;  // uniform
            const uint32_t e[2] = {(uint32_t)lane < queued ? s_pv.queue[lane] : kNoRank,
                                   kWave + lane < queued ? s_pv.queue[kWave + lane] : kNoRank};
            credit(e);
            queued = 0;
          }
        };
        // kRange: hits of owned ids are local where u or v is owned, those of the
        // others (streamed only there) where both are.
        auto stream = [&](uint32_t ss, uint32_t nn, uint32_t nr, uint32_t hot2, uint32_t ll, uint32_t ur) {
          if constexpr (RANGE) {
            const bool u_own = ur != kNoRank && (ur & kOwnedBit);
            stream_lists<MODE>(ss, nn, v_own || u_own ? ~0u : 0u, s_stream, s_items, lane, lists, 0xffffffffu, pv, probe, done);
            stream_lists<MODE>(ss + (hot2 & 0xffffu), nr, v_own && u_own ? ~0u : 0u, s_stream, s_items, lane, lists,
                               0xffffffffu, pv, probe, done);
          } else {
            stream_lists<MODE>(ss, nn, ll, s_stream, s_items, lane, lists, 0xffffffffu, pv, probe, done);
          }
        };
        uint32_t yu = kNoRank;
        if (cs0 + kWave < cs1) yu = items(cs0 + kWave);
        Head y = head(yu);
        stream(st, n, n_rest, len, label, u0);
        for (uint32_t e = cs0 + kWave; e < cs1; e += kWave) {
          const uint32_t sty = y.a.x, leny = y.a.y, ly = y.b.w, uy = yu;
          const uint32_t ny = RANGE ? prefix_owned(y) : prefix(y);
          const uint32_t nry = RANGE && (v_own || (uy & kOwnedBit && uy != kNoRank)) ? prefix_rest(y) : 0;
          if (e + kWave < cs1) {
            yu = items(e + kWave);
            y = head(yu);
          }
          stream(sty, ny, nry, leny, ly, uy);
        }
        local += acc_local;
        hits += acc;
        wave_lds_fence();
        if constexpr (PV)
          for (uint32_t p = lane; 2 * p < min(ch, (uint32_t)kSlots); p += kWave) {
            const uint32_t t = s_pv.hits[p];
            if (t & 0xffffu) atomicAdd(&pv[s_pv.label[2 * p]], (unsigned long long)(t & 0xffffu));
            if (t >> 16) atomicAdd(&pv[s_pv.label[2 * p + 1]], (unsigned long long)(t >> 16));
            if (t) s_pv.hits[p] = 0;
          }
        if (cd <= kWave) {
          if (w < kHot) s_bm[w >> 5] = 0;
        } else {
          clear_words(kWords / 4);
        }
        wave_lds_fence();
      }
      if (cold) {
        uint32_t acc = 0, acc_local = 0;
        // Cold ids [first, first + room) of N(v), in row order, hashed.
        auto pass = [&](auto logb, uint32_t first, uint32_t room) {
          constexpr int L = decltype(logb)::value;
          cold_table_clear<L>(s_tab, lane);
          bool passed = false;
          uint32_t seen = 0;
          for (uint32_t i = 0; i < cd; i += kWave) {
            const uint32_t y = id(i);
            const bool in = i + lane < cd && y >= kHot;
            const uint64_t m = __builtin_amdgcn_ballot_w64(in);
            const uint32_t at = seen + lanes_below(m);
            if (in && at >= first && at - first < room) passed |= wave_tab_insert<L>(s_tab, (int32_t)y);
            seen += (uint32_t)__popcll(m);
          }
          const bool spl = __builtin_amdgcn_ballot_w64(passed) != 0;
          wave_lds_fence();
          auto probe = [&](const uint4 q, uint32_t item) {
            const int32_t y[4] = {(int32_t)q.x, (int32_t)q.y, (int32_t)q.z, (int32_t)q.w};
            int4 t[4];
#pragma unroll
            for (int j = 0; j < 4; j++) t[j] = s_tab[wave_bucket<L>(y[j])];
#pragma unroll
            for (int j = 0; j < 4; j++) {
              bool hit = bucket_miss(t[j], y[j]) == 0;
              if (spl && !hit && bucket_spilled(t[j]) && y[j] != -1)
                hit = wave_tab_continue<L>(s_tab, wave_bucket<L>(y[j]), y[j]);
              acc += hit ? 1u : 0u;
              if constexpr (RANGE) acc_local += hit ? s_pv.items.label[item] & 1u : 0u;
              if constexpr (PV) {
                if (hit) {
                  const uint32_t lu = s_pv.items.label[item], lw = orig[y[j]];
                  if (lw < min(lu, cl))
                    atomicAdd(&pv[lw], 1ull);
                  else if (cl < lu)
                    at_v++;
                  else
                    atomicAdd(&s_pv.items.hits[item], 1u);
                }
              }
            }
          };
          auto stream = [&](uint32_t ss, uint32_t l1, uint32_t l2, uint32_t ll, uint32_t ur) {
            if constexpr (RANGE) {
              const bool u_own = ur != kNoRank && (ur & kOwnedBit);
              const uint32_t c0 = ss + (l1 & 0xffffu) + (l1 >> 16);  // behind both hot parts
              stream_lists<MODE>(c0, l2 & 0xffffu, v_own || u_own ? ~0u : 0u, s_stream, s_items, lane, lists, kNoRank, pv, probe, [] {});
              stream_lists<MODE>(c0 + (l2 & 0xffffu), v_own || u_own ? l2 >> 16 : 0, v_own && u_own ? ~0u : 0u, s_stream,
                                 s_items, lane, lists, kNoRank, pv, probe, [] {});
            } else {
              stream_lists<MODE>(ss + (l1 & 0xffffu), l1 >> 16, ll, s_stream, s_items, lane, lists, kNoRank, pv, probe, [] {});
            }
          };
          stream(st, len, len2, label, u0);
          for (uint32_t e = cs0 + kWave; e < cs1; e += kWave) {
            const uint32_t ur = items(e);
            uint4 y = make_uint4(0, 0, 0, 0);
            uint32_t ly = 0;
            if (ur != kNoRank) {
              const RankRec* q = rec + strip(ur);
              y = *reinterpret_cast<const uint4*>(q);
              if constexpr (PV) ly = q->mark[5];
            }
            stream(y.x, y.y, y.z, ly, ur);
          }
          wave_lds_fence();
          clear_words(1 << L);
          wave_lds_fence();
        };
        const uint32_t ncold = cd - ch;
        if (ncold <= (2u << kColdSmall)) {
          pass(std::integral_constant<int, kColdSmall>{}, 0u, ncold);
        } else {
          for (uint32_t f = 0; f < ncold; f += 2u << kColdBig) pass(std::integral_constant<int, kColdBig>{}, f, 2u << kColdBig);
        }
        hits += acc;
        local += acc_local;
      }
      if constexpr (PV) {
        const uint64_t t = wave_sum_u64(at_v);
        if (lane == 0 && t) atomicAdd(&pv[cl], (unsigned long long)t);
      }
      if (!more) break;
    }
  }
  hits = wave_sum_u64(hits);
  if (lane == 0) add_sum(counters, RANGE ? kSumOwned : kSumTotal, hits);
  if constexpr (RANGE) {
    local = wave_sum_u64(local);
    if (lane == 0) add_sum(counters, kSumLocal, local);
  }
}

// ---------------------------------------------------------------------------
static unsigned rank_grid(int64_t n, int per, int64_t cap) {
  int64_t g = (n + per - 1) / per;
  g = g < 1 ? 1 : g > cap ? cap : g;
  return (unsigned)g;
}

bool rank_fits(const xt_ctx* ctx, int64_t nv, int64_t ne, int mode, int64_t max_degree) {
  return rank_space_fits(ctx->num_cus, nv, ne, mode == kOrientId ? max_degree : -1);
}

// Entries per wave of k_rank_count.
static int64_t rank_chunk(const xt_ctx* ctx, int64_t ne) {
  int64_t S = kChunk;
  while (S > 256 && ne / S < (int64_t)ctx->num_cus * 18 * 8) S >>= 1;
  return S;
}

// The list memory of a count, cut short for tests.
static ListRoom list_room(const xt_ctx* ctx, int64_t nv, int64_t ne, int mode, int64_t max_degree, bool range,
                          int64_t* lines) {
  ListRoom lr = rank_list_room(ctx->num_cus, nv, ne, mode == kOrientId ? max_degree : -1, range ? 4 : 2, lines);
  if (ctx->list_lines > 0 && ctx->list_lines < *lines) lr.region = (uint64_t)ctx->list_lines / kListShards;
  return lr;
}

int rank_reserve(xt_ctx* ctx, Scratch& s, int64_t nv, int64_t ne, int mode, int64_t max_degree, bool per_vertex,
                 bool range) {
  struct Ranking {  // what an allocation that fails may free meanwhile
    xt_ctx* ctx;
    ~Ranking() { ctx->ranking = false; }
  } ranking{ctx};
  ctx->ranking = true;
  const int64_t S = rank_chunk(ctx, ne);
  XT_TRY(ensure(ctx, s.crows, (size_t)(2 * ((ne + S - 1) / S)) * sizeof(int32_t)));
  XT_TRY(ensure(ctx, s.rank, (size_t)nv * sizeof(uint32_t)));
  XT_TRY(ensure(ctx, s.ocount, (size_t)nv * sizeof(uint64_t)));
  XT_TRY(ensure(ctx, s.itcnt, (size_t)nv * sizeof(uint32_t)));
  XT_TRY(ensure(ctx, s.rpart, (size_t)(ne + kWave) * sizeof(uint32_t)));  // a wave reads past a short row
  int64_t lines;
  list_room(ctx, nv, ne, mode, max_degree, range, &lines);
  XT_TRY(ensure(ctx, s.rlists, (size_t)lines * 128));
  XT_TRY(ensure(ctx, s.rrec, (size_t)nv * sizeof(RankRec)));
  XT_TRY(ensure(ctx, s.rhist, (size_t)(2 * kRankClasses) * sizeof(uint32_t)));
  if (range) XT_TRY(ensure(ctx, s.vrec, (size_t)nv * sizeof(uint64_t)));
  if (per_vertex) XT_TRY(ensure(ctx, s.rorig, (size_t)nv * sizeof(uint32_t)));
  return XT_OK;
}

template <typename T>
int rank_count(xt_ctx* ctx, Scratch& s, int64_t nv, int64_t ne, const int64_t* off, const T* tails, int mode,
               int64_t max_degree, uint64_t* pv, const OwnedRange* range, hipStream_t st, hipEvent_t split_done) {
  const int64_t S = rank_chunk(ctx, ne);
  const int64_t nch = (ne + S - 1) / S, nchunks = (ne + kChunk - 1) / kChunk;
  int64_t lines;
  const ListRoom lr = list_room(ctx, nv, ne, mode, max_degree, range != nullptr, &lines);
  uint64_t* oc1 = range ? s.vrec.as<uint64_t>() : nullptr;
  const int64_t rlo = range ? range->lo : 0, rhi = range ? range->hi : 0;
  uint32_t* orig = pv ? s.rorig.as<uint32_t>() : nullptr;
  unsigned long long* pvp = reinterpret_cast<unsigned long long*>(pv);
  uint64_t* counters = s.counters.as<uint64_t>();
  uint32_t* hist = s.rhist.as<uint32_t>();
  int32_t* crows = s.crows.as<int32_t>();
  uint32_t* rank = s.rank.as<uint32_t>();
  uint64_t* oc = s.ocount.as<uint64_t>();
  uint32_t* part = s.rpart.as<uint32_t>();
  uint4* lists = s.rlists.as<uint4>();
  RankRec* rec = s.rrec.as<RankRec>();
  hipLaunchKernelGGL(k_rank_clear, dim3((kNumCounters + 255) / 256), dim3(256), 0, st, counters, hist);
  XT_HIP(ctx, hipGetLastError());
  hipLaunchKernelGGL(k_rank_prep, dim3(rank_grid(nv, 1024, 8192)), dim3(256), 0, st, nv, ne, off,
                     __builtin_ctzll((uint64_t)S), crows, oc,
                     s.itcnt.as<uint32_t>(), hist, pvp, oc1);
  XT_HIP(ctx, hipGetLastError());
  if (mode == kOrientId)
    hipLaunchKernelGGL(k_rank_by_label, dim3(rank_grid(nv, 256, 8192)), dim3(256), 0, st, nv, rank, orig);
  else
    hipLaunchKernelGGL(k_rank_assign, dim3(rank_grid(nv, 256 * kAssignRun, 1ll << 31)), dim3(256), 0, st, nv, off,
                       (const uint32_t*)hist, hist + kRankClasses, rank, orig);
  XT_HIP(ctx, hipGetLastError());
#define XT_RANK_SPLIT(R)                                                                                             \
  hipLaunchKernelGGL((k_rank_split<T, R>), dim3(xcd_grid(nchunks)), dim3(kBlock), 0, st, nv, ne, off, tails,            \
                     (const uint32_t*)rank, (const int32_t*)crows, (int)(kChunk / S), part, oc,                       \
                     s.itcnt.as<uint32_t>(), counters, oc1, rlo, rhi)
  if (range)
    XT_RANK_SPLIT(true);
  else
    XT_RANK_SPLIT(false);
#undef XT_RANK_SPLIT
  XT_HIP(ctx, hipGetLastError());
  const dim3 lgrid(rank_grid(lr.nbatch, 1, (int64_t)ctx->num_cus * 16));
#define XT_RANK_LISTS(M)                                                                                             \
  hipLaunchKernelGGL((k_rank_lists<M>), lgrid, dim3(64), 0, st, nv, off, (const uint64_t*)oc, (const uint64_t*)oc1,     \
                     (const uint32_t*)rank, (const uint32_t*)part, lr, lists, rec, counters)
  if (pv)
    XT_RANK_LISTS(kPerVertex);
  else if (range)
    XT_RANK_LISTS(kRange);
  else
    XT_RANK_LISTS(kTotal);
#undef XT_RANK_LISTS
  XT_HIP(ctx, hipGetLastError());
  if (split_done) XT_HIP(ctx, hipEventRecord(split_done, st));
#define XT_RANK_COUNT(M)                                                                                             \
  hipLaunchKernelGGL((k_rank_count<M>), dim3((unsigned)nch), dim3(64), 0, st, nv, ne, off, (const uint32_t*)rank,       \
                     (const uint64_t*)oc, (const uint32_t*)part, (const RankRec*)rec, (const uint4*)lists,            \
                     (const int32_t*)crows, S, counters, (const uint32_t*)orig, pvp, rlo, rhi)
  if (pv)
    XT_RANK_COUNT(kPerVertex);
  else if (range)
    XT_RANK_COUNT(kRange);
  else
    XT_RANK_COUNT(kTotal);
#undef XT_RANK_COUNT
  XT_HIP(ctx, hipGetLastError());
  ctx->rank_chunks = nch;
  return XT_OK;
}

template int rank_count<int32_t>(xt_ctx*, Scratch&, int64_t, int64_t, const int64_t*, const int32_t*, int, int64_t, uint64_t*,
                                 const OwnedRange*, hipStream_t, hipEvent_t);
template int rank_count<int64_t>(xt_ctx*, Scratch&, int64_t, int64_t, const int64_t*, const int64_t*, int, int64_t, uint64_t*,
                                 const OwnedRange*, hipStream_t, hipEvent_t);

}  // namespace xt
