// yk_wsel.h -- per-query sorts and selections of 64-bit keys by one wave,
// shared by the FP32 and the precision form.
#ifndef YK_WSEL_H_INCLUDED
#define YK_WSEL_H_INCLUDED

#include <hip/hip_runtime.h>

#include "yk_dev.h"

// ---------------------------------------------------------------------------
// One wave per query, keys in registers: E keys per lane (64 E keys), the
// lane's keys being elements lane * E .. lane * E + E - 1 of the sequence.
// Bitonic network (ascending): strides below E are compare-exchanges inside
// the lane, strides of E and more exchange with lane ^ (stride / E) by a
// shuffle, each lane keeping the min or the max of its pair.  No LDS and no
// barrier: the per-query sorts of the filtered pass's candidates (a few
// hundred keys) measured ~4x faster than the workgroup LDS network.

__device__ __forceinline__ uint64_t yk_shfl_xor64(uint64_t x, int m) {
  const uint32_t lo = __shfl_xor((uint32_t)x, m), hi = __shfl_xor((uint32_t)(x >> 32), m);
  return ((uint64_t)hi << 32) | lo;
}

template <int E>
__device__ __forceinline__ void yk_wave_sort(uint64_t (&v)[E], int lane) {
#pragma unroll
  for (int size = 2; size <= 64 * E; size <<= 1) {
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= E) {
#pragma unroll
        for (int i = 0; i < E; i++) {
          const int e = lane * E + i;
          const uint64_t o = yk_shfl_xor64(v[i], stride / E);
          const bool keep_min = ((e & stride) == 0) == ((e & size) == 0);
          v[i] = keep_min ? (v[i] < o ? v[i] : o) : (v[i] < o ? o : v[i]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < E; i++) {
          if (i & stride) continue;
          const int j = i | stride;
          const bool up = ((lane * E + i) & size) == 0;
          const uint64_t x = v[i], y = v[j];
          if ((x > y) == up) {
            v[i] = y;
            v[j] = x;
          }
        }
      }
    }
  }
}

// the m (<= 64 E) keys at src, sorted; the kp smallest to dst (kp <= 64 E),
// or only the kp-th smallest to *kth
template <int E>
__device__ __forceinline__ void yk_wave_select(const uint64_t *src, int m, int kp, int lane,
                                               uint64_t *dst, uint64_t *kth) {
  uint64_t v[E];
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int e = lane * E + i;
    v[i] = e < m ? src[e] : YK_KEY_NONE;
  }
  yk_wave_sort<E>(v, lane);
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int e = lane * E + i;
    if (dst && e < kp) dst[e] = v[i];
    if (kth && e == kp - 1) *kth = v[i];
  }
}

// ---------------------------------------------------------------------------
// Selection without a full sort: one wave per query holds the query's m keys
// E per lane (element i * 64 + lane, so the loads are coalesced; padding
// YK_KEY_NONE) and finds the kp-th smallest key bit by bit, top bit first:
// with X the bits fixed so far, the candidate C = X with the current bit 0
// and every lower bit 1 counts the keys <= C by one compare per held key
// and a ballot popcount; fewer than kp means the bit is 1.  After the last
// bit X is the least value with at least kp keys <= it: the kp-th smallest
// key itself.  With lo_const (the sketch's keys, whose low word is always
// 0xffffffff) only the 32 high bits are searched.  The search starts below
// the bits every real key shares (the highest bit where the least and the
// greatest real key differ: distances of one magnitude share sign and
// exponent), and once the high word is fixed, a high word held by a single
// key makes that key the answer without searching the index bits.

template <int E>
__device__ __forceinline__ void yk_wave_load(const uint64_t *src, int m, int lane,
                                             uint64_t (&v)[E]) {
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int e = i * 64 + lane;
    v[i] = e < m ? src[e] : YK_KEY_NONE;
  }
}

__device__ __forceinline__ uint64_t yk_wave_min64(uint64_t a) {
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)a, o), hi = __shfl_xor((uint32_t)(a >> 32), o);
    const uint64_t b = ((uint64_t)hi << 32) | lo;
    a = b < a ? b : a;
  }
  return a;
}

// keys <= c among the held keys
template <int E>
__device__ __forceinline__ int yk_wave_count_le(const uint64_t (&v)[E], uint64_t c) {
  int n = 0;
#pragma unroll
  for (int i = 0; i < E; i++) n += __popcll(__builtin_amdgcn_ballot_w64(v[i] <= c));
  return n;
}

template <int E>
__device__ __forceinline__ uint64_t yk_wave_kth(const uint64_t (&v)[E], int kp, bool lo_const) {
  uint64_t x = 0;
  int top = 63;
  if (E <= 16) {  // (with more keys per lane the bookkeeping costs occupancy)
    // the least and the greatest real key (the greatest as the least of the
    // complements), and the real key count
    uint64_t mn = YK_KEY_NONE, cmx = YK_KEY_NONE;
    int nreal = 0;
#pragma unroll
    for (int i = 0; i < E; i++) {
      const bool real = v[i] != YK_KEY_NONE;
      nreal += __popcll(__builtin_amdgcn_ballot_w64(real));
      mn = v[i] < mn ? v[i] : mn;
      cmx = real && ~v[i] < cmx ? ~v[i] : cmx;
    }
    if (nreal < kp) return YK_KEY_NONE;
    mn = yk_wave_min64(mn);
    const uint64_t diff = mn ^ ~yk_wave_min64(cmx);
    if (diff == 0) return mn;
    top = 63 - __builtin_clzll(diff);  // the bits above it: every real key's
    x = top == 63 ? 0 : (mn >> (top + 1)) << (top + 1);
  }
  // the high word
  for (int bit = top; bit >= 32; bit--)
    if (yk_wave_count_le<E>(v, x | ((1ull << bit) - 1)) < kp) x |= 1ull << bit;
  if (lo_const) return x | 0xffffffffull;
  if (E <= 16 && top >= 32) {
    // the high word is fixed: if one key holds it, that key is the answer
    const uint64_t xh = x >> 32;
    int eq = 0;
    uint64_t keq = YK_KEY_NONE;
#pragma unroll
    for (int i = 0; i < E; i++) {
      const bool in = (v[i] >> 32) == xh && v[i] != YK_KEY_NONE;
      eq += __popcll(__builtin_amdgcn_ballot_w64(in));
      keq = in && v[i] < keq ? v[i] : keq;
    }
    if (eq == 1) return yk_wave_min64(keq);
  }
  // the index bits
  for (int bit = top < 31 ? top : 31; bit >= 0; bit--)
    if (yk_wave_count_le<E>(v, x | ((1ull << bit) - 1)) < kp) x |= 1ull << bit;
  return x;
}

// the kp (<= 64 E2) smallest of the keys held in v (keys are distinct;
// fewer than kp real keys: padded with YK_KEY_NONE), ascending, as w (element
// lane * E2 + i): the keys <= the kp-th are compacted into the wave's LDS
// slice (ballot ranks), then sorted in registers
template <int E, int E2>
__device__ __forceinline__ void yk_wave_topk_reg(const uint64_t (&v)[E], int kp, int lane,
                                                 uint64_t *lds, uint64_t (&w)[E2]) {
  const uint64_t kth = yk_wave_kth<E>(v, kp, false);
  int base = 0;
#pragma unroll
  for (int i = 0; i < E; i++) {
    const bool take = v[i] <= kth && v[i] != YK_KEY_NONE;
    const uint64_t m = __builtin_amdgcn_ballot_w64(take);
    const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                               __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    if (take) lds[base + rank] = v[i];
    base += __popcll(m);
  }
  // (base <= kp <= 64 E2: the LDS slice holds 64 E2 keys)
  for (int e = base + lane; e < 64 * E2; e += 64) lds[e] = YK_KEY_NONE;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int i = 0; i < E2; i++) w[i] = lds[lane * E2 + i];
  yk_wave_sort<E2>(w, lane);
}

// the same, written to dst[0 .. kp)
template <int E, int E2>
__device__ __forceinline__ void yk_wave_topk(const uint64_t (&v)[E], int kp, int lane,
                                             uint64_t *lds, uint64_t *dst) {
  uint64_t w[E2];
  yk_wave_topk_reg<E, E2>(v, kp, lane, lds, w);
#pragma unroll
  for (int i = 0; i < E2; i++) {
    const int e = lane * E2 + i;
    if (e < kp) dst[e] = w[i];
  }
}

#endif
