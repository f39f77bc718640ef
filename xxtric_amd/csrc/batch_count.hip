// batch_count.hip -- the count of a batch of graphs of up to 65,535 vertices
// each (gfx950).
//
// The graphs of a batch lie behind each other in one CSR (batch.hip).  Their ids
// are consecutive, so the low 16 bits of a vertex number tell the vertices of
// one graph apart: lists and items are 16-bit, a record per vertex ({first
// entry, out-degree}) finds a list, and every triangle is counted at the edge
// (u, v), u -> v, as an id common to N+(u) and N+(v).  Three kernels:
//  k_batch_prep   degrees, chunk table, records and totals cleared
//  k_batch_split  each row in 16 bits: its out-neighbours first, then its
//                 in-neighbours (one gather of a degree per entry)
//  k_batch_count  per chunk of entries, one wave: the in-neighbours u of its rows v
// A row v of up to kTinyRow ids has them in registers, a lane per item.  The other
// rows have bit maps side by side in LDS, as many as fit 8 KB (vertices / 8 bytes
// each) and as one step's 64 items and 64 ids allow; the lists N+(u) of the items
// are numbered through in chunks of eight ids, one chunk per lane and step.
// What bounds it: k_batch_count by vector instructions (0.58 of 0.92 ms for 1024
// graphs) and the wait for its three dependent loads (item, record, list; all from
// L2) at the 17 waves a compute unit has LDS for; k_batch_split by latency (two
// block scans and a returning atomic per chunk; 0.36 ms where the bytes take 0.09).
// 1024 graphs, 43.6 M edges: 1.28 ms; 3.13 ms with edge tiles, which gather an
// 8-byte record and write a 16-byte item per entry in about 20 launches.  Every row
// a lane per item (up to 72 ids compared in registers): 2.46 ms; every row through
// bit maps: 1.38 ms; tiny rows of up to 16 ids: 1.45 ms.
#include "xt_bounds.hpp"
#include "xt_device.hpp"
#include "xt_internal.hpp"

namespace xt {

typedef uint32_t v4u_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef const __attribute__((address_space(1))) v4u_a2 gv4u_a2;

// Eight 16-bit ids from a 2-byte aligned address.
__device__ __forceinline__ uint4 load_ids8(const uint16_t* p) {
  const v4u_a2 t = *reinterpret_cast<gv4u_a2*>(reinterpret_cast<uint64_t>(p));
  return make_uint4(t.x, t.y, t.z, t.w);
}

// The vertex with low bits x in the graph that starts at base.
__device__ __forceinline__ int64_t vertex_of(uint32_t x, int32_t base, int64_t nv) {
  return min(base + (int64_t)((x - (uint32_t)base) & 0xffffu), nv - 1);
}

__global__ __launch_bounds__(256) void k_batch_prep(int64_t nv, int64_t ne, int64_t ng, const int64_t* __restrict__ off,
                                                    int64_t S, int32_t* __restrict__ crows, uint16_t* __restrict__ deg,
                                                    uint64_t* __restrict__ rec, uint32_t* __restrict__ ic,
                                                    unsigned long long* __restrict__ gtotal) {
  const int64_t nchunks = (ne + S - 1) / S;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t g = t0; g < ng; g += stride) gtotal[g] = 0;
  for (int64_t u = t0; u < nv; u += stride) {
    const int64_t a = off[u], b = off[u + 1];
    deg[u] = (uint16_t)min(b - a, (int64_t)65535);
    rec[u] = (uint64_t)(uint32_t)a;
    ic[u] = 0;
    if (a < 0 || b > ne || a >= b) continue;
    for (int64_t c = (a + S - 1) / S; c * S < b; c++) crows[2 * c] = (int32_t)u;
    for (int64_t c1 = a / S + 1; c1 * S <= b; c1++) crows[2 * c1 - 1] = (int32_t)u;
    if (b == ne) crows[2 * nchunks - 1] = (int32_t)u;
  }
}

// As k_rank_split: rows marked at their first entry in LDS, inner rows placed by
// a block scan, the chunk's first and last row by atomics.  Entries that are no
// edge (self-loops) go to the back as the row's own id.
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_batch_split(int64_t nv, int64_t ne, const int64_t* __restrict__ off,
                                                        const int32_t* __restrict__ tails,
                                                        const uint16_t* __restrict__ deg,
                                                        const int32_t* __restrict__ crows, int per,
                                                        uint16_t* __restrict__ part, uint64_t* __restrict__ rec,
                                                        uint32_t* __restrict__ ic) {
  __shared__ alignas(16) int16_t s_end[kChunk];  // first entry of a row: where the row ends (clamped); 0 elsewhere
  __shared__ uint32_t s_row[kChunk];             // and the row
  __shared__ uint16_t s_deg[kChunk];             // and its degree; later the chunk's entries in their new order
  __shared__ uint16_t s_pre[kChunk + 2];         // out-neighbours before each entry
  __shared__ uint32_t s_scan[kBlock / kWave];
  __shared__ int s_last[kBlock / kWave];
  __shared__ uint32_t s_ob[2], s_ib[2];          // places taken by the first and the last row
  __shared__ int s_rng[3];                       // the inner rows' range; whether the first row starts before the chunk
  uint16_t* s_part = s_deg;
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
  int32_t v[kPerThread];
  uint16_t dv[kPerThread];
  if (live) {
    int64_t vals[kPerThread];
    load_run<int32_t>(tails, eb + i0, eb + n, vals);
#pragma unroll
    for (int j = 0; j < kPerThread; j++) {  // eight gathers in flight
      v[j] = i0 + j < n && vals[j] >= 0 && vals[j] < nv ? (int32_t)vals[j] : -1;
      dv[j] = MODE == kOrientDegree ? deg[v[j] < 0 ? 0 : v[j]] : 0;
    }
  }
  __syncthreads();
  for (int64_t k = tid; k < span; k += kBlock) {
    const int64_t o0 = off[ulo + k], o1 = off[ulo + k + 1];
    const int ro = rel(o0), re = rel(o1);
    if (re > 0 && ro < n && o1 > o0) {
      s_end[max(ro, 0)] = (int16_t)re;
      s_row[max(ro, 0)] = (uint32_t)(ulo + k);
      s_deg[max(ro, 0)] = (uint16_t)min(o1 - o0, (int64_t)65535);
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
  const int upto = wave_incl_max_i32(last);
  if (lane == kWave - 1) s_last[wv] = upto;
  int at = __shfl_up(upto, 1, kWave);
  if (lane == 0) at = -1;
  __syncthreads();
  for (int w = 0; w < wv; w++) at = max(at, s_last[w]);
  if (ends[0]) at = i0;
  at = max(at, 0);  // entry 0 is marked whenever the offsets are an index
  uint32_t outs = 0;
  uint16_t id[kPerThread];
  if (live) {
    uint32_t u = s_row[at], du = s_deg[at];
#pragma unroll
    for (int j = 0; j < kPerThread; j++) {
      if (i0 + j < n) {
        if (ends[j]) {
          u = s_row[i0 + j];
          du = s_deg[i0 + j];
        }
        const bool up = (uint32_t)v[j] > u;
        const bool out = MODE == kOrientDegree ? dv[j] > du || (dv[j] == du && up) : up;
        if (v[j] >= 0 && out) outs |= 1u << j;
        id[j] = v[j] < 0 ? (uint16_t)u : (uint16_t)v[j];
      }
    }
  }
  const uint32_t cnts = (uint32_t)__popc(outs), upto_n = wave_incl_scan_u32(cnts);
  if (lane == kWave - 1) s_scan[wv] = upto_n;
  __syncthreads();
  uint32_t pre = upto_n - cnts, total = 0;
#pragma unroll
  for (int w = 0; w < kBlock / kWave; w++) {
    if (w < wv) pre += s_scan[w];
    total += s_scan[w];
  }
  if (live) {
#pragma unroll
    for (int j = 0; j < kPerThread; j++)
      if (i0 + j < n) s_pre[i0 + j] = (uint16_t)(pre + __popc(outs & ((1u << j) - 1u)));
  }
  if (tid == 0) s_pre[n] = (uint16_t)total;
  __syncthreads();  // s_deg is read: its place takes the new order
  for (int64_t k = tid; k < span; k += kBlock) {
    const int64_t o0 = off[ulo + k], o1 = off[ulo + k + 1];
    const int ro = rel(o0), re = rel(o1);
    if (re <= 0 || ro >= n || o1 <= o0) continue;
    const int a = max(ro, 0), b = min(re, n);
    const uint32_t cnt = (uint32_t)s_pre[b] - s_pre[a];
    if (ro >= 0 && re <= n) {
      rec[ulo + k] = (uint64_t)(uint32_t)o0 | ((uint64_t)cnt << 32);
    } else {
      const int s = k == 0 ? 0 : 1;
      const uint32_t ins = (uint32_t)(b - a) - cnt;
      s_ob[s] = cnt ? (uint32_t)(atomicAdd((unsigned long long*)&rec[ulo + k], (unsigned long long)cnt << 32) >> 32) : 0u;
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
        const int before = (int)s_pre[i] - (int)s_pre[cur];
        const bool front = (outs >> j) & 1u;
        if (!first && nxt <= n) {
          s_part[front ? cur + before : nxt - 1 - (i - cur - before)] = id[j];
        } else {
          const int s = first || uhi == ulo ? 0 : 1;
          const int64_t u = s == 0 ? ulo : uhi;
          part[front ? off[u] + (int64_t)s_ob[s] + before : off[u + 1] - 1 - (int64_t)s_ib[s] - (int64_t)(i - cur - before)] = id[j];
        }
      }
    }
  }
  __syncthreads();
  // The inner rows, two ids to a word where the range starts on one.
  const int a = s_rng[0], b = s_rng[1], a2 = (a + 1) & ~1, b2 = b & ~1;
  if (tid == 0 && a < b && a2 != a) part[eb + a] = s_part[a];
  if (tid == 0 && a < b && b2 != b && b2 >= a2) part[eb + b2] = s_part[b2];
  for (int i = a2 / 2 + tid; i < b2 / 2; i += kBlock)
    reinterpret_cast<uint32_t*>(part + eb)[i] = reinterpret_cast<const uint32_t*>(s_part)[i];
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kTinyRow = 8;      // rows of up to this many ids: a lane per item
constexpr uint32_t kMapWords = 2048;  // of the bit maps of a wave's rows

struct CountLds {
  uint4 map[kMapWords / 4];
  uint4 tail[9];                  // the first 0..8 halves of a chunk set
  unsigned long long bit[kWave];
  uint2 list[kWave];              // lists of a step: {first entry - 8 * first chunk, end | map << 16}
  uint8_t row[kWave];             // lanes whose rows have items
};

__device__ __forceinline__ void lds_turn() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Consecutive pieces (of the lanes where on) that start at p <= 4096 of a line:
// word w of the result (lane w's) has a bit at place i where one starts at
// 64 w + i + 1.  So the bits below place i, counted from the first piece's start,
// number the piece that place i lies in.
__device__ __forceinline__ uint64_t start_bits(CountLds& s, bool on, uint32_t p) {
  lds_turn();
  s.bit[threadIdx.x] = 0ull;
  lds_turn();
  if (on && p > 0) atomicOr(&s.bit[(p - 1) >> 6], 1ull << ((p - 1) & 63));
  lds_turn();
  return s.bit[threadIdx.x];
}

// 64 bits of it from place p on (uniform).
__device__ __forceinline__ uint64_t bits_from(uint64_t mine, uint32_t p) {
  const int w = (int)(p >> 6), sh = (int)(p & 63);
  const uint64_t lo = (uint64_t)readlane64((int64_t)mine, w & 63);
  const uint64_t hi = (uint64_t)readlane64((int64_t)mine, (w + 1) & 63);
  return sh ? (lo >> sh) | (hi << (64 - sh)) : lo;
}

__device__ __forceinline__ uint32_t min_u16x2(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// Ids common to two lists, by lane: the one of up to kTinyRow ids at av in
// registers (each id in both halves of a word, filled up with an id the graph does
// not have), two ids of the other against one of them by an exclusive-or and a
// packed minimum.
__device__ __forceinline__ uint32_t common_tiny(const CountLds& s, const uint16_t* __restrict__ part, uint32_t av,
                                                uint32_t m, uint32_t fill, uint32_t au, uint32_t n) {
  uint32_t x[kTinyRow];
#pragma unroll
  for (uint32_t c = 0; c < kTinyRow; c += 8) {
    uint4 q = make_uint4(0, 0, 0, 0);
    if (m > c) q = load_ids8(part + av + c);
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t lo = c + 2 * j < m ? w[j] & 0xffffu : fill, hi = c + 2 * j + 1 < m ? w[j] >> 16 : fill;
      x[c + 2 * j] = lo | (lo << 16);
      x[c + 2 * j + 1] = hi | (hi << 16);
    }
  }
  uint32_t h = 0;
  for (uint32_t k = 0; k < n; k += 8) {
    const uint4 q = load_ids8(part + au + k);
    const uint4 t = s.tail[min(n - k, 8u)];
    const uint32_t w[4] = {q.x, q.y, q.z, q.w}, ts[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      uint32_t z = ~0u;  // a half ends as zero where its id is in the other list
#pragma unroll
      for (uint32_t i = 0; i < kTinyRow; i++) z = min_u16x2(z, w[j] ^ x[i]);
      z |= ~ts[j];
      h += ((z & 0xffffu) == 0 ? 1u : 0u) + ((z >> 16) == 0 ? 1u : 0u);
    }
  }
  return h;
}

__global__ __launch_bounds__(64) void k_batch_count(int64_t nv, int64_t ne, int64_t ng,
                                                    const int64_t* __restrict__ off,
                                                    const uint64_t* __restrict__ rec, const uint16_t* __restrict__ part,
                                                    const int32_t* __restrict__ gid, const int32_t* __restrict__ gbase,
                                                    const int32_t* __restrict__ crows, int64_t S,
                                                    unsigned long long* __restrict__ gtotal) {
  __shared__ CountLds s;
  uint32_t* s_map = reinterpret_cast<uint32_t*>(s.map);
  const int lane = threadIdx.x;
  const int64_t nch = (ne + S - 1) / S;
  const int64_t c = xcd_block(nch);
  if (c >= nch) return;
  const int64_t eb = c * S, ee = min(ne, eb + S);
  int64_t row_lo = crows[2 * c], row_hi = crows[2 * c + 1];
  row_lo = row_lo < 0 ? 0 : (row_lo > nv - 1 ? nv - 1 : row_lo);
  row_hi = row_hi < row_lo ? row_lo : (row_hi > nv - 1 ? nv - 1 : row_hi);
  for (uint32_t i = lane; i < kMapWords / 4; i += kWave) s.map[i] = make_uint4(0, 0, 0, 0);
  if (lane < 9 * 4) {
    const int k = lane / 4, j = lane % 4;
    reinterpret_cast<uint32_t*>(s.tail)[lane] = k > 2 * j + 1 ? ~0u : (k > 2 * j ? 0xffffu : 0u);
  }
  int32_t gcur = -1;  // graph of acc
  uint32_t acc = 0;
  auto flush = [&]() {
    const uint64_t t = wave_sum_u64(acc);
    if (lane == 0 && t) atomicAdd(&gtotal[gcur], (unsigned long long)t);
    acc = 0;
  };
  for (int64_t rb = row_lo; rb <= row_hi; rb += kWave) {
    const int64_t r = rb + lane;
    uint32_t a0 = 0, d = 0, is = 0, ie = 0;
    int32_t g = -1;
    if (r <= row_hi) {
      const uint64_t q = rec[r];
      a0 = (uint32_t)q;
      d = (uint32_t)(q >> 32);
      g = gid[r];
      is = (uint32_t)max((int64_t)a0 + d, eb);
      ie = (uint32_t)min(off[r + 1], ee);
    }
    const uint32_t n_row = d > 0 && is < ie ? ie - is : 0;
    const uint64_t tiny = __builtin_amdgcn_ballot_w64(n_row > 0 && d <= kTinyRow);
    if (tiny) {  // uniform
      const uint32_t ni = d <= kTinyRow ? n_row : 0;
      const uint32_t inc = wave_incl_scan_u32(ni), p = inc - ni;
      const uint32_t all = __builtin_amdgcn_readlane(inc, kWave - 1);
      const uint64_t bits = start_bits(s, ni > 0, p);
      if (ni > 0) s.row[lanes_below(tiny)] = (uint8_t)lane;
      lds_turn();
      const int32_t gq = __builtin_amdgcn_readlane(g, __builtin_ctzll(tiny));
      if (gq != gcur) {
        if (gcur >= 0) flush();
        gcur = gq;
      }
      uint32_t past = 0;
      for (uint32_t b = 0; b * kWave < all; b++) {
        const uint64_t m = (uint64_t)readlane64((int64_t)bits, (int)b);
        const int row = (int)s.row[(past + lanes_below(m)) & 63u];
        past += (uint32_t)__popcll(m);
        const uint32_t entry = (uint32_t)__shfl((int)(is - p), row, kWave) + b * kWave + lane;
        const uint32_t av = (uint32_t)__shfl((int)a0, row, kWave), dv = (uint32_t)__shfl((int)d, row, kWave);
        const int32_t gr = __shfl(g, row, kWave);
        if (b * kWave + lane < all) {
          const uint32_t x = part[entry];
          if (x != ((uint32_t)(rb + row) & 0xffffu)) {
            const int32_t base = gbase[gr];
            const uint64_t q = rec[vertex_of(x, base, nv)];
            const uint32_t n = (uint32_t)(q >> 32);
            if (n >= 2) {
              const uint32_t h = common_tiny(s, part, av, dv, (uint32_t)(base - 1) & 0xffffu, (uint32_t)q, n);
              if (gr == gcur)
                acc += h;
              else if (h)
                atomicAdd(&gtotal[gr], (unsigned long long)h);
            }
          }
        }
      }
    }
    const uint32_t ni = d > kTinyRow ? n_row : 0;
    const uint32_t inc = wave_incl_scan_u32(ni), p = inc - ni;
    const uint64_t work = __builtin_amdgcn_ballot_w64(ni > 0);
    if (work == 0) continue;  // uniform
    // The rows' ids, as many of each as fit one step: a longer row is alone in its step.
    const uint32_t di = ni > 0 ? min(d, (uint32_t)kWave) : 0;
    const uint32_t dinc = wave_incl_scan_u32(di), dp = dinc - di;
    const uint32_t nth = lanes_below(work);
    const uint64_t item_bits = start_bits(s, ni > 0, p), id_bits = start_bits(s, ni > 0, dp);
    if (ni > 0) s.row[nth] = (uint8_t)lane;
    lds_turn();
    for (uint64_t todo = work; todo;) {
      // Rows of one graph whose bit maps fit side by side and whose ids and items
      // a step holds.
      const int head = __builtin_ctzll(todo);
      const int32_t gq = __builtin_amdgcn_readlane(g, head);
      const uint32_t pb = __builtin_amdgcn_readlane(p, head), dpb = __builtin_amdgcn_readlane(dp, head);
      const uint32_t nb = __builtin_amdgcn_readlane(nth, head), dh = __builtin_amdgcn_readlane(d, head);
      if (gq != gcur) {
        if (gcur >= 0) flush();
        gcur = gq;
      }
      // Ids count from 1 within a graph: no bit 0, so a zero stands for no id.
      const int32_t base = gbase[gq];
      const uint32_t vg = (uint32_t)((gq + 1 < ng ? gbase[gq + 1] : (int32_t)nv) - base);
      const uint32_t w = min((vg >> 5) + 1, kMapWords);
      const bool take = ((todo >> lane) & 1u) &&
                        (lane == head || (g == gq && (nth - nb + 1) * w <= kMapWords && inc - pb <= kWave &&
                                          dinc - dpb <= kWave));
      const uint64_t taken = __builtin_amdgcn_ballot_w64(take);
      todo &= ~taken;
      const int last = 63 - __builtin_clzll(taken);
      const uint32_t items = __builtin_amdgcn_readlane(inc, last) - pb;
      const uint32_t before = (uint32_t)(base - 1) & 0xffffu;
      const uint64_t rows = bits_from(item_bits, pb);
      uint32_t k = 0, au = 0, n = 0;  // this lane's item: its row's place and its list
      auto item = [&](uint32_t e) {
        k = e ? 0u : lanes_below(rows);
        const int row = (int)s.row[(nb + k) & 63u];
        const uint32_t entry = (uint32_t)__shfl((int)(is - p), row, kWave) + pb + e + lane;
        au = n = 0;
        if (e + lane < items) {
          const uint32_t x = part[entry];
          if (x != ((uint32_t)(rb + row) & 0xffffu)) {
            const uint64_t q = rec[vertex_of(x, base, nv)];
            au = (uint32_t)q;
            n = (uint32_t)(q >> 32);
          }
        }
      };
      // The bit maps; the items' loads are on their way meanwhile.
      const uint32_t ids = __builtin_amdgcn_readlane(dinc, last) - dpb;
      const uint32_t ki = dh > kWave ? 0u : lanes_below(bits_from(id_bits, dpb));
      const int irow = (int)s.row[(nb + ki) & 63u];
      const uint32_t at = (uint32_t)__shfl((int)(a0 - dp), irow, kWave) + dpb + lane;
      const uint32_t yi = (uint32_t)lane < ids ? (part[at] - before) & 0xffffu : 0u;
      item(0);
      uint32_t* mapped = &s_map[min(ki * w + (yi >> 5), kMapWords - 1)];
      if (yi) atomicOr(mapped, 1u << (yi & 31));
      if (dh > kWave) {  // uniform
        const uint32_t ah = __builtin_amdgcn_readlane(a0, head);
        for (uint32_t i = kWave + lane; i < dh; i += kWave) {
          const uint32_t y = (part[ah + i] - before) & 0xffffu;
          atomicOr(&s_map[y >> 5], 1u << (y & 31));
        }
      }
      for (uint32_t e = 0; e < items; e += kWave) {
        if (e) item(e);
        if (n < 2) n = 0;  // u has no neighbour besides v
        // The lists in chunks of eight ids, numbered through; at most 64 chunks of
        // a list at a time.
        for (uint32_t from = 0; __builtin_amdgcn_ballot_w64(from < n); from += 8 * kWave) {
          const uint32_t left = from < n ? min(n - from, 8u * kWave) : 0, nc = (left + 7) >> 3;
          const uint32_t cinc = wave_incl_scan_u32(nc), cp = cinc - nc;
          const uint32_t chunks = __builtin_amdgcn_readlane(cinc, kWave - 1);
          const uint32_t ln = lanes_below(__builtin_amdgcn_ballot_w64(nc > 0));
          const uint64_t list_bits = start_bits(s, nc > 0, cp);
          if (nc > 0) s.list[ln] = make_uint2(au + from - 8 * cp, (left + 8 * cp) | ((k * w) << 16));
          lds_turn();
          uint32_t past = 0;
          for (uint32_t b = 0; b * kWave < chunks; b++) {
            const uint64_t m = (uint64_t)readlane64((int64_t)list_bits, (int)b);
            const uint32_t ch = b * kWave + lane;
            const uint2 l = s.list[(past + lanes_below(m)) & 63u];
            past += (uint32_t)__popcll(m);
            if (ch < chunks) {
              const uint4 q = load_ids8(part + (uint32_t)(l.x + 8 * ch));  // summed in 32 bits: l.x may lie below zero
              const uint4 t = s.tail[min((l.y & 0xffffu) - 8 * ch, 8u)];
              const uint32_t* bm = s_map + (l.y >> 16);
              const uint32_t xs[4] = {q.x, q.y, q.z, q.w}, ts[4] = {t.x, t.y, t.z, t.w};
              const u16x2 b2 = {(unsigned short)before, (unsigned short)before};
#pragma unroll
              for (int j = 0; j < 4; j++) {
                const uint32_t y = __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, xs[j]) - b2)) & ts[j];
                acc += (bm[(y >> 5) & 2047u] >> (y & 31)) & 1u;
                acc += (bm[y >> 21] >> ((y >> 16) & 31)) & 1u;
              }
            }
          }
        }
      }
      lds_turn();
      if (dh > kWave) {  // uniform
        for (uint32_t i = lane; i < (w + 3) / 4; i += kWave) s.map[i] = make_uint4(0, 0, 0, 0);
      } else if (yi) {
        *mapped = 0;
      }
      lds_turn();
    }
  }
  if (gcur >= 0) flush();
}

// ---------------------------------------------------------------------------
constexpr int64_t kBatchChunkMin = 256;

// Entries per wave of k_batch_count: fewer where the chip's waves (18 a compute
// unit, by the LDS they use) would get less than four chunks each.  1024 graphs:
// 1.40, 1.38 and 1.38 ms with 512, 1024 and 2048 entries; a chunk has at most 4096
// (start_bits).
static int64_t batch_chunk(const xt_ctx* ctx, int64_t ne) {
  int64_t S = 1024;
  while (S > kBatchChunkMin && ne / S < (int64_t)ctx->num_cus * 18 * 4) S >>= 1;
  return S;
}

bool batch_small_fits(int64_t max_graph_vertices, int64_t ne) {
  return max_graph_vertices <= 65535 && ne < kIndex32Entries;
}

int batch_small_reserve(xt_ctx* ctx, Scratch& s, int64_t nv, int64_t ne) {
  const int64_t e = ne > 0 ? ne : 1, v = nv > 0 ? nv : 1;
  XT_TRY(ensure(ctx, s.crows, (size_t)(2 * ((e + kBatchChunkMin - 1) / kBatchChunkMin)) * sizeof(int32_t)));
  XT_TRY(ensure(ctx, s.deg, (size_t)v * sizeof(uint16_t)));
  XT_TRY(ensure(ctx, s.vrec, (size_t)v * sizeof(uint64_t)));
  XT_TRY(ensure(ctx, s.itcnt, (size_t)v * sizeof(uint32_t)));
  return ensure(ctx, s.otails, (size_t)(e + 32) * sizeof(uint16_t));  // lists are read eight ids at a time
}

int batch_small_count(xt_ctx* ctx, Scratch& s, int64_t nv, int64_t ne, int64_t ng, const int64_t* off,
                      const int32_t* tails, const int32_t* gid, const int32_t* gbase, uint64_t* gtotal, int mode,
                      hipStream_t st) {
  if (nv <= 0 || ne <= 0) return fill_u64(ctx, gtotal, ng, 0, st);
  XT_TRY(batch_small_reserve(ctx, s, nv, ne));
  const int64_t S = batch_chunk(ctx, ne), nch = (ne + S - 1) / S, nchunks = (ne + kChunk - 1) / kChunk;
  int32_t* crows = s.crows.as<int32_t>();
  uint16_t* deg = s.deg.as<uint16_t>();
  uint16_t* part = s.otails.as<uint16_t>();
  uint64_t* rec = s.vrec.as<uint64_t>();
  const int64_t pg = ((nv > ng ? nv : ng) + 1023) / 1024;
  hipLaunchKernelGGL(k_batch_prep, dim3((unsigned)(pg > 8192 ? 8192 : pg)), dim3(256), 0, st, nv, ne, ng, off, S, crows,
                     deg, rec, s.itcnt.as<uint32_t>(), (unsigned long long*)gtotal);
  XT_HIP(ctx, hipGetLastError());
#define XT_BATCH_SPLIT(M)                                                                                            \
  hipLaunchKernelGGL((k_batch_split<M>), dim3(xcd_grid(nchunks)), dim3(kBlock), 0, st, nv, ne, off, tails,              \
                     (const uint16_t*)deg, (const int32_t*)crows, (int)(kChunk / S), part, rec, s.itcnt.as<uint32_t>())
  if (mode == kOrientId)
    XT_BATCH_SPLIT(kOrientId);
  else
    XT_BATCH_SPLIT(kOrientDegree);
#undef XT_BATCH_SPLIT
  XT_HIP(ctx, hipGetLastError());
  hipLaunchKernelGGL(k_batch_count, dim3(xcd_grid(nch)), dim3(64), 0, st, nv, ne, ng, off, (const uint64_t*)rec,
                     (const uint16_t*)part, gid, gbase, (const int32_t*)crows, S, (unsigned long long*)gtotal);
  XT_HIP(ctx, hipGetLastError());
  return XT_OK;
}

}  // namespace xt
