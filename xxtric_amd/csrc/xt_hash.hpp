// xt_hash.hpp -- per-wave LDS hash tables of vertex ids (gfx950).
//
// Buckets of four ids; empty slots hold kEmpty = 2^31 - 1.  A bucket that was
// full when a later key hashed to it has the top bit of its last slot set
// ("spilled"); that key went to the next bucket (linear probing by bucket).  A
// lookup reads its home bucket with one 16-byte LDS read and stops at the
// first bucket that holds the id or has not spilled.  Ids are below 2^31 - 1,
// so neither an empty nor a marked slot equals an id, and the padding id -1
// matches nothing.
#pragma once

#include "xt_device.hpp"

namespace xt {

constexpr int32_t kEmpty = 0x7fffffff;

// 0 when the bucket holds w (slot values xor w, minimum over the four slots).
__device__ __forceinline__ uint32_t bucket_miss(const int4 t, int32_t w) {
  const uint32_t x = (uint32_t)(t.x ^ w), y = (uint32_t)(t.y ^ w), z = (uint32_t)(t.z ^ w);
  const uint32_t q = (uint32_t)((t.w & 0x7fffffff) ^ w);
  return min(min(x, y), min(z, q));
}

__device__ __forceinline__ bool bucket_spilled(const int4 t) { return t.w < 0; }

// Home bucket of w among 2^LOGB: a multiplicative hash, so ids sharing their
// low bits (strided or clustered labels) still spread.
template <int LOGB>
__device__ __forceinline__ uint32_t wave_bucket(int32_t w) {
  return ((uint32_t)w * 0x9E3779B1u) >> (32 - LOGB);
}

// Inserts key; returns whether a full bucket had to be passed (and was
// marked spilled).
template <int LOGB>
__device__ __forceinline__ bool wave_tab_insert(int4* tab, int32_t key) {
  uint32_t b = wave_bucket<LOGB>(key);
  bool passed = false;
  for (;;) {
    int* s = reinterpret_cast<int*>(tab + b);
    if (atomicCAS(s, kEmpty, key) == kEmpty) return passed;
    if (atomicCAS(s + 1, kEmpty, key) == kEmpty) return passed;
    if (atomicCAS(s + 2, kEmpty, key) == kEmpty) return passed;
    if (atomicCAS(s + 3, kEmpty, key) == kEmpty) return passed;
    atomicOr(s + 3, (int)0x80000000);
    passed = true;
    b = (b + 1) & ((1u << LOGB) - 1);
  }
}

// Continues a lookup past the spilled home bucket b; ends because at most half
// the slots are used, so some bucket is not full and therefore not spilled.
template <int LOGB>
__device__ __forceinline__ bool wave_tab_continue(const int4* tab, uint32_t b, int32_t w) {
  for (;;) {
    b = (b + 1) & ((1u << LOGB) - 1);
    const int4 t = tab[b];
    if (bucket_miss(t, w) == 0) return true;
    if (!bucket_spilled(t)) return false;
  }
}

// Orders this wave's LDS accesses before and after it (one wave owns the
// table; LDS instructions of a wave execute in order).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace xt
