// Order statistics by radix selection: the float <-> key encoding and the byte
// passes shared by the quantile kernels.
#pragma once
#include "common.hpp"

namespace wgbm {

constexpr int kSelMaxTargets = 256;   // 2 * 126 ranks at most (num_bins <= 127)
constexpr int kSelGroup = 32;         // distinct prefixes histogrammed per scan

__device__ inline uint32_t float_to_key(float x) {
  uint32_t u = __float_as_uint(x);
  if (x != x) return 0xffffffffu;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
// the key of a value's bits, the value not a NaN
__device__ inline uint32_t bits_to_key(uint32_t u) {
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float key_to_float(uint32_t k) {
  const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(u);
}

// Radix selection, four byte passes over a multiset of keys: target t's rank
// trank[t] in it becomes its key, tprefix[t].  for_src(fn) calls fn(key) for
// every key, the keys spread over the workgroup's NT threads; every thread
// calls this.  Workgroup (LDS) scratch: hist, dist, tfirst, s_nd.  The caller
// has written trank and synchronised.
template <int NT, typename ForSrc>
__device__ inline void radix_select(ForSrc&& for_src, int nt, uint32_t* tprefix, int64_t* trank,
                                    uint32_t (*hist)[256], uint32_t* dist, uint32_t* tfirst,
                                    int* s_nd) {
  constexpr int nwaves = NT / 64;
  static_assert(nwaves < kSelGroup, "a row per wave and one for their sum");
  const int tid = threadIdx.x;
  // a 256-bin row of counts -> inclusive prefix, in place (one wave, 4 bins
  // a lane)
  auto row_prefix = [&](uint32_t* row) {
    const int ln = tid & 63;
    uint32_t v[4];
    uint32_t t = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      t += row[4 * ln + j];
      v[j] = t;
    }
    const uint32_t base = (uint32_t)(wgbm_wave_incl_scan_i64((int64_t)t) - t);
#pragma unroll
    for (int j = 0; j < 4; ++j) row[4 * ln + j] = base + v[j];
  };
  // first bin whose inclusive prefix exceeds r (bins 0..255; 255 when none
  // below does), and r made relative to that bin
  auto pick_bin = [&](const uint32_t* P, int64_t& r) {
    int a = 0, b = 255;
    while (a < b) {
      const int mid = (a + b) >> 1;
      if ((int64_t)P[mid] > r) b = mid; else a = mid + 1;
    }
    if (a > 0) r -= P[a - 1];
    return a;
  };
  for (int i = tid; i < nwaves * 256; i += NT) (&hist[0][0])[i] = 0;
  __syncthreads();
  {
    const int w = tid >> 6;
    for_src([&](uint32_t k) { atomicAdd(&hist[w][k >> 24], 1u); });
  }
  __syncthreads();
  for (int b = tid; b < 256; b += NT) {
    uint32_t sum = 0;
    for (int w = 0; w < nwaves; ++w) sum += hist[w][b];
    hist[nwaves][b] = sum;
  }
  __syncthreads();
  if (tid < 64) row_prefix(hist[nwaves]);
  __syncthreads();
  for (int t = tid; t < nt; t += NT) {
    int64_t r = trank[t];
    const int b = pick_bin(hist[nwaves], r);
    tprefix[t] = (uint32_t)b;
    trank[t] = r;
  }
  __syncthreads();
  // index of prefix pre in the sorted dist[lo..hi] (or where it would be)
  auto find = [&](uint32_t pre, int a, int b) {
    while (a < b) {
      const int mid = (a + b) >> 1;
      if (dist[mid] < pre) a = mid + 1; else b = mid;
    }
    return a;
  };
  // passes 2..4: next byte of the keys that share a target's prefix
  for (int pass = 1; pass < 4; ++pass) {
    const int sh = 32 - 8 * pass;  // prefix = key >> sh
    // sorted distinct prefixes, in parallel (a serial sort on one thread
    // waits on every LDS access behind the other waves' atomics): thread
    // t marks whether it holds the first occurrence of its value, then a
    // first occurrence stores its value at the count of distinct values
    // below it
    if (tid == 0) *s_nd = 0;
    if (tid < nt) {
      const uint32_t v = tprefix[tid];
      bool first = true;
      for (int u = 0; u < tid; ++u) first = first && tprefix[u] != v;
      tfirst[tid] = first ? 1u : 0u;
    }
    __syncthreads();
    if (tid < nt && tfirst[tid]) {
      const uint32_t v = tprefix[tid];
      int below = 0;
      for (int u = 0; u < nt; ++u) below += (tfirst[u] && tprefix[u] < v) ? 1 : 0;
      dist[below] = v;
      atomicAdd(s_nd, 1);
    }
    __syncthreads();
    const int nd = *s_nd;
    // highest group first: a finished target's longer prefix is above every
    // prefix of this pass that is still to come (0 is in the last group)
    for (int g0 = (nd - 1) / kSelGroup * kSelGroup; g0 >= 0; g0 -= kSelGroup) {
      const int gn = nd - g0 < kSelGroup ? nd - g0 : kSelGroup;
      for (int i = tid; i < gn * 256; i += NT) (&hist[0][0])[i] = 0;
      __syncthreads();
      const uint32_t lo_p = dist[g0], hi_p = dist[g0 + gn - 1];
      for_src([&](uint32_t k) {
        const uint32_t pre = k >> sh;
        if (pre < lo_p || pre > hi_p) return;
        const int g = find(pre, g0, g0 + gn - 1);
        if (dist[g] == pre) atomicAdd(&hist[g - g0][(k >> (sh - 8)) & 255u], 1u);
      });
      __syncthreads();
      for (int g = tid >> 6; g < gn; g += nwaves) row_prefix(hist[g]);
      __syncthreads();
      for (int t = tid; t < nt; t += NT) {
        const uint32_t pre = tprefix[t];
        if (pre < dist[g0] || pre > dist[g0 + gn - 1]) continue;
        const int g = find(pre, g0, g0 + gn - 1);
        int64_t r = trank[t];
        const int b = pick_bin(hist[g - g0], r);
        tprefix[t] = (pre << 8) | (uint32_t)b;
        trank[t] = r;
      }
      __syncthreads();
    }
  }
}

}  // namespace wgbm
