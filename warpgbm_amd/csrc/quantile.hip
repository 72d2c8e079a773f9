// Quantile edges of a resident row-major matrix in two reads of it.
//
// The order statistics torch.quantile interpolates between (warpgbm/core.py:
// 529-534; ranks and interpolation as in quantile_select_kernel) are found
// per feature without a transposed copy of the matrix:
//   1. sample   1024 values of the column fix the value buckets: kQBuckets
//               equal-width buckets over a range just wider than the targets'
//               (sample order statistics below the lowest and above the
//               highest rank), the two end buckets open, so that neither
//               outliers nor a long tail stretch them;
//   2. count    the first read: values per bucket, 16-bit counters in LDS,
//               one lane per feature (a lane's counters all lie in its own
//               bank: no conflicts), one partial table per row block, then
//               their sum;
//   3. targets  the bucket of every target rank, numbered (slots), and a
//               reference value for every slot in which several sample values
//               are equal;
//   4. gather   the second read: the values of those buckets, except those
//               equal to the slot's reference (their number is the bucket's
//               count less what is gathered), so that a heavily tied column
//               gathers next to nothing;
//   5. pick     each slot split into sub-buckets, the target's sub-bucket
//               copied to LDS and its rank found by counting; a feature whose
//               sub-buckets do not fit runs radix passes over its gathered
//               values instead.
// bucket(v) = clamp(int(fma(v, scale, offset))) is non-decreasing in v, so
// every bucket (and sub-bucket) is a contiguous run of the sorted column:
// the result is exact whatever the sample was.
//
// What bounds it: the count walks 4 GB (1M x 1000) in 0.71 ms = 5.6 TB/s; the
// gather takes 0.75 ms where nothing is gathered and 1.02 ms for smooth columns
// (5% of the values at 32 bins: ring stores); the pick is LDS-bound on the
// gathered values (0.18 ms at 5%).  Against the transposed copy and its two
// scans (quantile_select_kernel), all edges of 1M x 1000 at 32 bins: smooth
// columns 3.43 -> 1.95 ms, with a seventh of the columns lognormal and a tenth
// rounded to whole numbers 7.6 -> 2.3 ms; at 127 bins 5.6 -> 3.3 ms.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "quantile_radix.hpp"

namespace wgbm {

constexpr int kQNone = 255;   // slot / reference byte of a bucket that holds no target
constexpr int kQRefs = 127;   // references per feature; row 127: none (a NaN, equal to nothing)
constexpr int kQRing = 15;    // values a lane holds back before it stores eight of them
static_assert(kSelMaxTargets >= 2 * 126 && kQNone >= 2 * 126, "a slot per target at most");

__device__ __forceinline__ float q_pos(float v, float2 m) { return __builtin_fmaf(v, m.x, m.y); }
// (the conversion saturates: negative and NaN to 0)
__device__ __forceinline__ uint32_t q_bucket(float x) {
  uint32_t b;
  __asm__("v_cvt_u32_f32 %0, %1" : "=v"(b) : "v"(x));
  return b < kQBuckets - 1 ? b : kQBuckets - 1;
}
// byte address of a lane's entry for bucket b in a [256][64] word table (byte
// b >> 8 of word (b & 255) * 64 + lane): a byte permute and a bitwise or
__device__ __forceinline__ uint32_t q_slot_addr(uint32_t b, uint32_t lane4) {
  return __builtin_amdgcn_perm(0u, b, 0x0c0c0001u) | lane4;
}

// ---------------------------------------------------------------------------
// 1. sample: a wave per feature
// ---------------------------------------------------------------------------
// Latency-bound (one strided gather, then 32 rounds of counting): the two
// order statistics are found bit by bit, both in the same round.
__global__ __launch_bounds__(256) void quantile_sample_kernel(
    const float* __restrict__ X, int64_t n, int32_t F, int64_t xs, const float* __restrict__ q,
    int32_t nq, float* __restrict__ sample, float2* __restrict__ map,
    uint32_t* __restrict__ nan_flag, uint32_t* __restrict__ negz) {
  constexpr int PER = kQSample / 64;
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (f >= F) return;
  // evenly spread rows, shifted inside their stratum so that a period of the
  // rows does not alias with the stride
  float v[PER];
  uint32_t key[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = k * 64 + lane;
    const int64_t r0 = (int64_t)i * n / kQSample, r1 = (int64_t)(i + 1) * n / kQSample;
    const uint32_t h = ((uint32_t)i * 2654435761u) >> 8;
    const int64_t r = r0 + (r1 > r0 ? (int64_t)(h % (uint32_t)(r1 - r0)) : 0);
    v[k] = X[(r < n ? r : n - 1) * xs + f];
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    key[k] = float_to_key(v[k]);
    sample[(int64_t)f * kQSample + k * 64 + lane] = v[k];
  }
  float ql = 1.0f, qh = 0.0f;
  for (int j = lane; j < nq; j += 64) {
    ql = fminf(ql, q[j]);
    qh = fmaxf(qh, q[j]);
  }
  for (int o = 32; o > 0; o >>= 1) {
    ql = fminf(ql, __shfl_xor(ql, o, 64));
    qh = fmaxf(qh, __shfl_xor(qh, o, 64));
  }
  // sample ranks about five standard deviations outside the targets'
  const float el = fmaxf(ql, 0.0f) * kQSample, eh = fmaxf(1.0f - qh, 0.0f) * kQSample;
  const int il = (int)fmaxf(el - 5.0f * sqrtf(el) - 2.0f, 0.0f);
  const int ih = kQSample - 1 - (int)fmaxf(eh - 5.0f * sqrtf(eh) - 2.0f, 0.0f);
  // the largest key with at most il (ih) keys below it is the order statistic
  uint32_t a = 0, b = 0;
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t ta = a | (1u << bit), tb = b | (1u << bit);
    int ca = 0, cb = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      ca += __builtin_popcountll(__ballot(key[k] < ta));
      cb += __builtin_popcountll(__ballot(key[k] < tb));
    }
    if (ca <= il) a = ta;
    if (cb <= ih) b = tb;
  }
  if (lane == 0) {
    float lo = key_to_float(a), hi = key_to_float(b);
    // a rank below every sample value: an open end bucket that holds a target
    // costs that column radix passes (2 ms), a wider range a sixteenth more
    // gathered values
    const float ext = (hi - lo) * 0.0625f;
    if (il == 0) lo -= ext;
    if (ih == kQSample - 1) hi += ext;
    float scale = (float)kQBuckets / (hi - lo);
    float off = -lo * scale;
    // one value, a NaN or an infinite end in the sample: a single bucket
    if (!(scale > 0.0f && scale < __builtin_inff() && fabsf(off) < __builtin_inff())) {
      scale = 0.0f;
      off = 0.0f;
    }
    map[f] = float2{scale, off};
    nan_flag[f] = 0u;
    negz[f] = 0u;
  }
}

// ---------------------------------------------------------------------------
// 2. count: workgroup (row block, 64 features), lane l owns feature 64c + l
// ---------------------------------------------------------------------------
// Counters [kQBuckets / 2][64] words of two 16-bit counts: 128 KB, one
// workgroup per CU; a row block has fewer than 65536 rows.  Each wave takes
// groups of U rows, two groups alternating (the loads of one in flight while
// the other is counted).
// add(group, rows): rows = U (a compile-time constant of the instance) but for
// the last group of the block.
template <int U, typename Add>
__device__ __forceinline__ void q_walk_rows(const float* __restrict__ src, int64_t xs, int nrows,
                                            int wave, Add&& add) {
  constexpr int step = (kQThreads / 64) * U;
  float ga[U], gb[U];
  auto issue = [&](float (&g)[U], int i0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u < nrows ? i0 + u : nrows - 1;
      g[u] = src[(int64_t)i * xs];
    }
  };
  auto last = [&](float (&g)[U], int i0) {
    if (i0 + U <= nrows) add(g, U); else add(g, nrows - i0);
  };
  int i = wave * U;
  if (i >= nrows) return;
  issue(ga, i);
  while (i + 2 * step < nrows) {
    issue(gb, i + step);
    add(ga, U);
    issue(ga, i + 2 * step);
    add(gb, U);
    i += 2 * step;
  }
  if (i + step < nrows) {
    issue(gb, i + step);
    add(ga, U);
    last(gb, i + step);
  } else {
    last(ga, i);
  }
}

__global__ __launch_bounds__(kQThreads) void quantile_count_kernel(
    const float* __restrict__ X, int64_t n, int32_t F, int64_t xs, int32_t rows_per, int32_t nrb,
    const float2* __restrict__ map, uint32_t* __restrict__ part,
    uint32_t* __restrict__ nan_flag, uint32_t* __restrict__ negz) {
  extern __shared__ uint32_t qsm[];
  const int nc = (F + 63) / 64;
  // a row block's chunks on one XCD: rows are not line-aligned, and chunks
  // that share a line then share it through that XCD's L2
  const int64_t w = wgbm_xcd_work(blockIdx.x, (int64_t)nrb * nc);
  if (w >= (int64_t)nrb * nc) return;  // uniform over the workgroup
  const int rb = (int)(w / nc), chunk = (int)(w - (int64_t)rb * nc);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int W = kQBuckets / 2 * 64;
  for (int i = threadIdx.x; i < W; i += kQThreads) qsm[i] = 0u;
  __syncthreads();
  const int64_t r0 = (int64_t)rb * rows_per;
  const int nrows = (int)(n - r0 < rows_per ? n - r0 : rows_per);
  const int f = chunk * 64 + lane < F ? chunk * 64 + lane : F - 1;
  const float2 m = map[f];
  bool nan = false;
  uint32_t nz = 0;  // -0.0 values: they compare equal to a reference of +0.0
  constexpr int U = 16;
  q_walk_rows<U>(X + r0 * xs + f, xs, nrows, wave, [&](const float(&g)[U], int rows) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float v = g[u];
      const bool in = u < rows;  // (rows: a constant but for the last group)
      nan = nan || v != v;
      nz += __float_as_uint(v) == 0x80000000u && in ? 1u : 0u;
      const uint32_t b = q_bucket(q_pos(v, m));
      const uint32_t inc = in ? 1u << ((b & 1u) * 16u) : 0u;
      atomicAdd(&qsm[(b >> 1) * 64u + (uint32_t)lane], inc);
    }
  });
  __syncthreads();
  if (nan) nan_flag[f] = 1u;  // (every writer stores the same value)
  if (nz && chunk * 64 + lane < F) atomicAdd(&negz[f], nz);
  uint32_t* out = part + w * W;
  for (int i = threadIdx.x; i < W; i += kQThreads) out[i] = qsm[i];
}

// ---------------------------------------------------------------------------
// the row blocks' counts added up: workgroup = 64 words of a chunk, a quarter of
// the row blocks a wave
// ---------------------------------------------------------------------------
// Its own launch, over all CUs: added up by the few workgroups of the targets, 64
// .. 196 tables one after the other took 61 .. 86 us of a call of 150 .. 230 (131k x
// 1, 200k x 100), here 3 .. 6 us and 14 .. 16 for the targets.  Counts
// [chunk][kQBuckets][64].
__global__ __launch_bounds__(256) void quantile_sum_kernel(const uint32_t* __restrict__ part,
                                                           int32_t nrb, int32_t nc,
                                                           uint32_t* __restrict__ cnt) {
  constexpr int W = kQBuckets / 2 * 64;
  __shared__ uint32_t los[4][64], his[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chunk = blockIdx.x / (W / 64), wd = blockIdx.x - chunk * (W / 64);
  const uint32_t* p = part + (int64_t)chunk * W + wd * 64 + lane;
  uint32_t lo = 0u, hi = 0u;
  constexpr int RU = 16;  // row blocks in flight
  for (int r0 = wave; r0 < nrb; r0 += 4 * RU) {
    uint32_t x[RU];
#pragma unroll
    for (int k = 0; k < RU; ++k) {
      const int r = r0 + 4 * k;
      x[k] = p[(int64_t)(r < nrb ? r : nrb - 1) * nc * W];
    }
#pragma unroll
    for (int k = 0; k < RU; ++k) {
      const uint32_t v = r0 + 4 * k < nrb ? x[k] : 0u;
      lo += v & 0xffffu;
      hi += v >> 16;
    }
  }
  los[wave][lane] = lo;
  his[wave][lane] = hi;
  __syncthreads();
  if (wave < 2) {
    const uint32_t(*s)[64] = wave ? his : los;
    cnt[((int64_t)chunk * kQBuckets + 2 * wd + wave) * 64 + lane] =
        s[0][lane] + s[1][lane] + s[2][lane] + s[3][lane];
  }
}

// ---------------------------------------------------------------------------
// 3. targets: workgroup = 16 features of a chunk
// ---------------------------------------------------------------------------
// A wave each after the loads: its words are its own, so nothing past them is a
// barrier (each waited for the stores before it, a memory round trip: 23 us of
// few features with 25 of them).
__global__ __launch_bounds__(kQThreads) void quantile_targets_kernel(
    const uint32_t* __restrict__ counts, int64_t n, int32_t F, const float* __restrict__ q,
    int32_t nq, const float2* __restrict__ map, const float* __restrict__ sample,
    uint32_t* __restrict__ slot_map, uint32_t* __restrict__ row_map, uint32_t* __restrict__ refs,
    uint32_t* __restrict__ slot_size, uint32_t* __restrict__ slot_ref,
    uint8_t* __restrict__ tslot, int32_t* __restrict__ trank, int32_t* __restrict__ nslots) {
  constexpr int CS = kQBuckets + 1;  // odd row stride: the features' rows start in other banks
  __shared__ uint32_t cnt[16][CS];
  __shared__ uint8_t mark[16][kQBuckets];
  const int chunk = blockIdx.x >> 2, l0 = (blockIdx.x & 3) * 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fl = wave;
  const int f = chunk * 64 + l0 + fl;
  const bool on = f < F;
  constexpr int SPER = kQSample / 64;
  uint32_t sv[SPER];
  const float2 m = map[on ? f : F - 1];
#pragma unroll
  for (int k = 0; k < SPER; ++k)
    sv[k] = __float_as_uint(sample[(int64_t)(on ? f : F - 1) * kQSample + k * 64 + lane]);
  {
    // counts of 16 features: thread (lane l0 + tid % 16, buckets tid / 16 ..)
    const int l = tid & 15, b0 = tid >> 4;
    constexpr int STEP = kQThreads / 16, NB = kQBuckets / STEP;
    uint32_t x[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k)
      x[k] = counts[((int64_t)chunk * kQBuckets + b0 + k * STEP) * 64 + l0 + l];
#pragma unroll
    for (int k = 0; k < NB; ++k) cnt[l][b0 + k * STEP] = x[k];
    for (int i = tid; i < 16 * kQBuckets / 4; i += kQThreads)
      reinterpret_cast<uint32_t*>(&mark[0][0])[i] = 0u;
  }
  __syncthreads();
  // from here on a wave owns feature f; its lane holds buckets 64 k + lane
  constexpr int PER = kQBuckets / 64;
  uint32_t c[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) c[k] = cnt[fl][64 * k + lane];
  {
    uint32_t base = 0u;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const uint32_t incl = wgbm_wave_incl_scan_u32(c[k]);
      cnt[fl][64 * k + lane] = base + incl - c[k];  // exclusive prefix
      base += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    }
  }
  wgbm_wave_lds_order();
  const int nt = 2 * nq;
  const int64_t last = n - 1;
  constexpr int TPL = kSelMaxTargets / 64;  // targets per lane
  int tb[TPL];
#pragma unroll
  for (int j = 0; j < TPL; ++j) {
    const int t = j * 64 + lane;
    tb[j] = -1;
    if (t >= nt) continue;
    const float rank = q[t >> 1] * (float)last;
    int64_t r = (t & 1) ? (int64_t)ceilf(rank) : (int64_t)rank;
    r = r < 0 ? 0 : (r > last ? last : r);
    int a = 0, b = kQBuckets - 1;  // last bucket whose prefix is <= r
    while (a < b) {
      const int mid = (a + b + 1) >> 1;
      if ((int64_t)cnt[fl][mid] <= r) a = mid; else b = mid - 1;
    }
    mark[fl][a] = 1;
    tb[j] = a;
    if (on) trank[(int64_t)f * kSelMaxTargets + t] = (int32_t)(r - (int64_t)cnt[fl][a]);
  }
  wgbm_wave_lds_order();
  // slots: the marked buckets in order
  int slots = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const bool mk = mark[fl][64 * k + lane] != 0;
    const uint64_t bal = __ballot(mk);
    const int s = slots + __builtin_popcountll(bal & ((1ull << lane) - 1ull));
    mark[fl][64 * k + lane] = mk ? (uint8_t)s : (uint8_t)kQNone;
    if (mk && on) slot_size[(int64_t)f * 256 + s] = c[k];
    slots += __builtin_popcountll(bal);
  }
  if (lane == 0 && on) nslots[f] = slots;
  // four candidates a slot, each the last of a quarter of its sample values;
  // the one that most of the slot's sample values equal is its reference,
  // if any other does (a slot of distinct values needs none)
  __shared__ uint32_t ref[16][256], cand[16][256], votes[16][256];
  uint32_t best[4] = {1u, 1u, 1u, 1u}, bref[4];  // of slots lane, lane + 64, ...
#pragma unroll
  for (int j = 0; j < 4; ++j) bref[j] = 0xffffffffu;
  int ss[SPER];
  for (int i = lane; i < 256; i += 64) votes[fl][i] = 0u;
  wgbm_wave_lds_order();
#pragma unroll
  for (int j = 0; j < TPL; ++j)
    if (tb[j] >= 0 && on)
      tslot[(int64_t)f * kSelMaxTargets + j * 64 + lane] = mark[fl][tb[j]];
  for (int wd = lane; wd < 256; wd += 64) {
    const uint32_t x = (uint32_t)mark[fl][wd] | (uint32_t)mark[fl][wd + 256] << 8 |
                       (uint32_t)mark[fl][wd + 512] << 16 | (uint32_t)mark[fl][wd + 768] << 24;
    slot_map[((int64_t)chunk * 256 + wd) * 64 + l0 + fl] = x;
  }
#pragma unroll
  for (int k = 0; k < SPER; ++k) {
    if (sv[k] == 0x80000000u) sv[k] = 0u;  // references compare as floats
    ss[k] = mark[fl][q_bucket(q_pos(__uint_as_float(sv[k]), m))];
  }
  for (int round = 0; round < 4; ++round) {
#pragma unroll
    for (int k = 0; k < SPER; ++k)
      if (ss[k] != kQNone && k % 4 == round) cand[fl][ss[k]] = sv[k];
    wgbm_wave_lds_order();
#pragma unroll
    for (int k = 0; k < SPER; ++k)
      if (ss[k] != kQNone && cand[fl][ss[k]] == sv[k]) atomicAdd(&votes[fl][ss[k]], 1u);
    wgbm_wave_lds_order();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = j * 64 + lane;
      const uint32_t v = votes[fl][i];
      votes[fl][i] = 0u;
      if (v > best[j]) {
        best[j] = v;
        bref[j] = cand[fl][i];
      }
    }
    wgbm_wave_lds_order();
  }
  // rows of the references: slot order within each quarter of the slots
  int row0 = 0;
  for (int i = lane; i < 256; i += 64) ref[fl][i] = 0xffffffffu;
  wgbm_wave_lds_order();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint64_t has = __ballot(bref[j] != 0xffffffffu);
    const int row = row0 + __builtin_popcountll(has & ((1ull << lane) - 1ull));
    const bool kept = bref[j] != 0xffffffffu && row < kQRefs;
    if (kept) ref[fl][row] = bref[j];
    cand[fl][j * 64 + lane] = kept ? (uint32_t)row : (uint32_t)kQRefs;  // row of slot
    if (on) slot_ref[(int64_t)f * 256 + j * 64 + lane] = kept ? bref[j] : 0xffffffffu;
    row0 += __builtin_popcountll(has);
  }
  wgbm_wave_lds_order();
  // the gather's tables: the reference row of every bucket, and the rows
  for (int wd = lane; wd < 256; wd += 64) {
    uint32_t x = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int sl = mark[fl][wd + 256 * k];
      x |= (sl == kQNone || !on ? (uint32_t)kQNone : cand[fl][sl]) << (8 * k);
    }
    row_map[((int64_t)chunk * 256 + wd) * 64 + l0 + fl] = x;
  }
  for (int i = lane; i < 128; i += 64)
    refs[((int64_t)chunk * 128 + i) * 64 + l0 + fl] = ref[fl][i];
}

// ---------------------------------------------------------------------------
// 4. gather: the same walk as the count
// ---------------------------------------------------------------------------
// Tables in LDS: a reference-row byte per bucket [256][64] words and the
// references [128][64] words; every lane reads its own bank.  A bucket of no
// target (or of no feature) has row byte 255, a slot without reference row 127.
// A workgroup's values of feature f go to its own part of the feature's
// column of buf (rows_per words), their number to gcount.  A lane keeps its
// values in a ring of its own in LDS and stores eight at a time: single-word
// stores of 64 features are 64 lines each, and took 1.9 ms instead of 1.0 ms
// where an eighth of the values is gathered (1M x 1000, 127 bins).
__global__ __launch_bounds__(kQThreads) void quantile_gather_kernel(
    const float* __restrict__ X, int64_t n, int32_t F, int64_t xs, int32_t rows_per, int32_t nrb,
    const float2* __restrict__ map, const uint32_t* __restrict__ row_map,
    const uint32_t* __restrict__ refs, uint32_t* __restrict__ buf, int64_t ks,
    uint32_t* __restrict__ gcount) {
  extern __shared__ uint32_t qsm[];
  const int nc = (F + 63) / 64;
  const int64_t w = wgbm_xcd_work(blockIdx.x, (int64_t)nrb * nc);
  if (w >= (int64_t)nrb * nc) return;  // uniform over the workgroup
  const int rb = (int)(w / nc), chunk = (int)(w - (int64_t)rb * nc);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int T = 256 * 64, R = 128 * 64;
  float* ref_s = reinterpret_cast<float*>(qsm + T);
  uint32_t* cursor = qsm + T + R;  // [64]
  uint32_t* ring = qsm + T + R + 64 + wave * kQRing * 64 + lane;  // [kQRing] at stride 64
  for (int i = threadIdx.x; i < T; i += kQThreads) qsm[i] = row_map[(int64_t)chunk * T + i];
  for (int i = threadIdx.x; i < R; i += kQThreads) qsm[T + i] = refs[(int64_t)chunk * R + i];
  if (threadIdx.x < 64) cursor[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t r0 = (int64_t)rb * rows_per;
  const int nrows = (int)(n - r0 < rows_per ? n - r0 : rows_per);
  const bool real = chunk * 64 + lane < F;
  const int f = real ? chunk * 64 + lane : F - 1;
  const float2 m = map[f];
  uint32_t* dst = buf + (int64_t)f * ks + r0;
  const uint8_t* rows = reinterpret_cast<const uint8_t*>(qsm);
  uint32_t held = 0;  // values in the ring, < 8 between half groups
  constexpr int U = 16;
  q_walk_rows<U>(X + r0 * xs + f, xs, nrows, wave, [&](const float(&g)[U], int rows_in) {
    uint32_t rw[U];
    float rf[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      rw[u] = rows[q_slot_addr(q_bucket(q_pos(g[u], m)), (uint32_t)lane * 4u)];
    // (row 255, past the references, is some word of the ring: not used)
#pragma unroll
    for (int u = 0; u < U; ++u) rf[u] = ref_s[rw[u] * 64u + (uint32_t)lane];
#pragma unroll
    for (int h = 0; h < U; h += 8) {
#pragma unroll
      for (int u = h; u < h + 8; ++u) {
        // written whether it is kept or not (held <= 14 here): no branch
        ring[held * 64] = __float_as_uint(g[u]);
        held += (rw[u] != kQNone && g[u] != rf[u] && u < rows_in) ? 1u : 0u;
      }
      if (held >= 8) {
        // (every reserved word is written: fewer than nrows values in all)
        uint32_t* d = dst + atomicAdd(&cursor[lane], 8u);
        uint32_t x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = ring[k * 64];
#pragma unroll
        for (int k = 0; k < 8; ++k) d[k] = x[k];
        held -= 8;
#pragma unroll
        for (int k = 0; k < kQRing - 8; ++k) ring[k * 64] = ring[(k + 8) * 64];
      }
    }
  });
  if (held) {
    uint32_t* d = dst + atomicAdd(&cursor[lane], held);
    for (uint32_t k = 0; k < held; ++k) d[k] = ring[k * 64];
  }
  __syncthreads();
  if (threadIdx.x < 64 && real) gcount[(int64_t)f * nrb + rb] = cursor[threadIdx.x];
}

// ---------------------------------------------------------------------------
// 5. pick: a workgroup per feature
// ---------------------------------------------------------------------------
constexpr int kPickThreads = 512;
constexpr int kPickSub = 8192;    // (slot, sub-bucket) counters, then the sorted lists
constexpr int kPickList = 8192;   // values of the targets' sub-buckets
constexpr int kPickListMax = 4096;  // of one sub-bucket (its ranks are found by counting)
constexpr int kPickListWide = 256;  // more: the whole workgroup counts

__global__ __launch_bounds__(kPickThreads) void quantile_pick_kernel(
    const uint32_t* __restrict__ buf, int64_t ks, int64_t n, int32_t rows_per, int32_t nrb,
    const uint32_t* __restrict__ gcount, const float* __restrict__ q, int32_t nq,
    const float2* __restrict__ map, const uint32_t* __restrict__ slot_map,
    const uint32_t* __restrict__ slot_size, const uint32_t* __restrict__ slot_ref,
    const uint8_t* __restrict__ tslot, const int32_t* __restrict__ trank_in,
    const int32_t* __restrict__ nslots, const uint32_t* __restrict__ nan_flag,
    const uint32_t* __restrict__ negz, float* __restrict__ edges) {
  __shared__ uint32_t sub_n[kPickSub];    // counts, then the list cursors
  __shared__ uint32_t list[kPickList];    // also the radix passes' counters
  __shared__ uint8_t slot_of[kQBuckets];
  __shared__ float ref[256];
  __shared__ uint32_t got[256], less[256], lpos[kSelMaxTargets], llen[kSelMaxTargets];
  __shared__ uint32_t tkey[kSelMaxTargets], tlist[kSelMaxTargets];
  __shared__ uint32_t dist[kSelMaxTargets], tfirst[kSelMaxTargets];
  __shared__ int64_t trank[kSelMaxTargets];
  __shared__ int s_nd;
  __shared__ uint32_t s_total, s_big, s_rounds;
  static_assert(kPickList >= kSelGroup * 256, "the radix counters use the list's words");
  static_assert(kPickSub >= kPickList, "the lists are sorted into the counters' words");
  static_assert(kPickThreads >= kSelMaxTargets, "a thread per target, a thread per slot");
  const int f = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float* out = edges + (int64_t)f * nq;
  if (nan_flag[f]) {  // a NaN anywhere makes every quantile NaN
    for (int j = tid; j < nq; j += kPickThreads) out[j] = __builtin_nanf("");
    return;
  }
  const int nt = 2 * nq;
  const int ns = nslots[f];
  const float2 m = map[f];
  const int chunk = f >> 6, fl = f & 63;
  // sub-buckets per slot: a power of two, ns * subs <= kPickSub
  int lg = 0;
  while (lg < 7 && (ns << (lg + 1)) <= kPickSub) ++lg;
  const int subs = 1 << lg;
  if (tid < 256) {
    const uint32_t x = slot_map[((int64_t)chunk * 256 + tid) * 64 + fl];
    slot_of[tid] = (uint8_t)x;
    slot_of[tid + 256] = (uint8_t)(x >> 8);
    slot_of[tid + 512] = (uint8_t)(x >> 16);
    slot_of[tid + 768] = (uint8_t)(x >> 24);
    ref[tid] = __uint_as_float(slot_ref[(int64_t)f * 256 + tid]);
    less[tid] = 0u;
  }
  for (int i = tid; i < ns * subs; i += kPickThreads) sub_n[i] = 0u;
  if (tid == 0) s_total = s_big = 0u;
  __syncthreads();
  // every gathered value: a wave per row block's run
  auto for_vals = [&](auto fn) {
    for (int s = wave; s < nrb; s += kPickThreads / 64) {
      const uint32_t c = gcount[(int64_t)f * nrb + s];
      const uint32_t* p = buf + (int64_t)f * ks + (int64_t)s * rows_per;
      constexpr uint32_t U = 8;
      for (uint32_t i0 = lane; i0 < c; i0 += 64 * U) {
        uint32_t x[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) x[u] = p[i0 + 64 * u < c ? i0 + 64 * u : c - 1];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
          if (i0 + 64 * u < c) fn(x[u]);
      }
    }
  };
  // (slot, sub-bucket) of a value: the position inside its bucket, the open
  // end buckets clamped; non-decreasing in the value
  auto cell = [&](uint32_t bits, uint32_t& s) {
    const float x = q_pos(__uint_as_float(bits), m);
    const uint32_t b = q_bucket(x);
    s = slot_of[b];
    const float y = (x - (float)b) * (float)subs;
    const uint32_t k = (uint32_t)fminf(fmaxf(y, 0.0f), (float)(subs - 1));
    return (s << lg) + k;
  };
  for_vals([&](uint32_t bits) {
    uint32_t s;
    const uint32_t k = cell(bits, s);
    atomicAdd(&sub_n[k], 1u);
    // (false for a slot without reference, whose ref is a NaN)
    if (__uint_as_float(bits) < ref[s]) atomicAdd(&less[s], 1u);
  });
  __syncthreads();
  if (tid < ns) {
    uint32_t g = 0;
    for (int k = 0; k < subs; ++k) g += sub_n[(tid << lg) + ((k + tid) & (subs - 1))];
    got[tid] = g;
  }
  __syncthreads();
  // targets: the reference itself, or a rank among the slot's gathered values
  const int t0 = tid;
  if (t0 < nt) {
    const int s = tslot[(int64_t)f * kSelMaxTargets + t0];
    uint32_t r = (uint32_t)trank_in[(int64_t)f * kSelMaxTargets + t0];
    const uint32_t eq = slot_size[(int64_t)f * 256 + s] - got[s];
    const bool is_ref = r >= less[s] && r < less[s] + eq;
    tlist[t0] = 0xffffffffu;
    tfirst[t0] = 0u;
    if (is_ref) {
      // a reference of zero stands for both zeros, -0.0 first
      const bool neg = ref[s] == 0.0f && r - less[s] < negz[f];
      tkey[t0] = bits_to_key(neg ? 0x80000000u : __float_as_uint(ref[s]));
    } else {
      if (r >= less[s] + eq) r -= eq;
      trank[t0] = (int64_t)r;  // among the slot's gathered values
      uint32_t k = (uint32_t)s << lg;
      const uint32_t end = k + subs - 1;
      uint32_t rr = r;
      while (k < end && rr >= sub_n[k]) rr -= sub_n[k++];
      tlist[t0] = k;
      lpos[t0] = rr;
    }
  }
  __syncthreads();
  // a list per distinct target sub-bucket: its first target marks the count
  constexpr uint32_t kOwned = 0x80000000u;
  if (t0 < nt && tlist[t0] != 0xffffffffu) {
    const uint32_t old = atomicOr(&sub_n[tlist[t0]], kOwned);
    const uint32_t len = old & ~kOwned;
    llen[t0] = len;
    if (!(old & kOwned)) {
      tfirst[t0] = 1u;
      dist[t0] = atomicAdd(&s_total, len);
      if (len > kPickListMax) s_big = 1u;
    }
  }
  __syncthreads();
  if (!s_big) {
    // the lists in rounds of at most kPickList values (one round but for a
    // column whose values crowd into few buckets): a pass over the gathered
    // values each, against the radix passes' four and their conflicts
    if (tid == 0) {
      uint32_t at = 0, rd = 0;
      if (s_total > kPickList) {
        for (int t = 0; t < nt; ++t) {
          if (!tfirst[t]) continue;
          if (at + llen[t] > kPickList) {
            at = 0;
            ++rd;
          }
          dist[t] = at;
          tfirst[t] = 1u + rd;
          at += llen[t];
        }
      }
      s_rounds = rd + 1;
    }
    __syncthreads();
    const uint32_t rounds = s_rounds;
    for (uint32_t rd = 1; rd <= rounds; ++rd) {
      // sub_n becomes the cursor of a list of this round, or none
      for (int i = tid; i < ns * subs; i += kPickThreads) sub_n[i] = 0xffffffffu;
      __syncthreads();
      if (t0 < nt && tfirst[t0] == rd) sub_n[tlist[t0]] = dist[t0];
      __syncthreads();
      uint32_t l0 = 0xffffffffu;  // this target's list in this round
      if (t0 < nt && tlist[t0] != 0xffffffffu) l0 = sub_n[tlist[t0]];
      __syncthreads();
      for_vals([&](uint32_t bits) {
        uint32_t s;
        const uint32_t k = cell(bits, s);
        if (sub_n[k] != 0xffffffffu) list[atomicAdd(&sub_n[k], 1u)] = bits_to_key(bits);
      });
      __syncthreads();
      // every list sorted into sub_n by counting (equal values in list
      // order): 16 threads a list, all threads a long one
      auto place = [&](int t, uint32_t i) {
        const uint32_t len = llen[t], o = dist[t];
        const uint32_t k = list[o + i];
        uint32_t before = 0;
#pragma unroll 4
        for (uint32_t j = 0; j < len; ++j) {
          const uint32_t y = list[o + j];
          before += (y < k || (y == k && j < i)) ? 1u : 0u;
        }
        sub_n[o + before] = k;
      };
      for (int t = tid >> 4; t < nt; t += kPickThreads / 16)
        if (tfirst[t] == rd && llen[t] <= kPickListWide)
          for (uint32_t i = tid & 15; i < llen[t]; i += 16) place(t, i);
      for (int t = 0; t < nt; ++t)
        if (tfirst[t] == rd && llen[t] > kPickListWide)  // uniform over the workgroup
          for (uint32_t i = tid; i < llen[t]; i += kPickThreads) place(t, i);
      __syncthreads();
      if (l0 != 0xffffffffu) tkey[t0] = sub_n[l0 + lpos[t0]];
      __syncthreads();
    }
  } else {
    // radix passes over all gathered values: ranks among all of them
    const bool by_rank = t0 < nt && tlist[t0] != 0xffffffffu;
    const uint32_t own_key = t0 < nt ? tkey[t0] : 0u;
    if (t0 < nt) {
      int64_t r = 0;
      if (by_rank) {
        const int s = tslot[(int64_t)f * kSelMaxTargets + t0];
        r = trank[t0];
        for (int u = 0; u < s; ++u) r += got[u];
      }
      trank[t0] = r;
    }
    __syncthreads();
    radix_select<kPickThreads>(
        [&](auto fn) { for_vals([&](uint32_t bits) { fn(bits_to_key(bits)); }); }, nt, tkey, trank,
        reinterpret_cast<uint32_t(*)[256]>(list), dist, tfirst, &s_nd);
    __syncthreads();
    if (t0 < nt && !by_rank) tkey[t0] = own_key;
    __syncthreads();
  }
  // interpolate (torch.quantile, linear): see quantile_edges_kernel
  const int64_t last = n - 1;
  for (int j = tid; j < nq; j += kPickThreads) {
    const float rank = q[j] * (float)last;
    const int64_t lo_r = (int64_t)rank;
    const float wt = rank - (float)lo_r;
    const float a = key_to_float(tkey[2 * j]);
    const float b = key_to_float(tkey[2 * j + 1]);
    const float d = b - a;
    out[j] = wt < 0.5f ? fmaf(wt, d, a) : fmaf(wt - 1.0f, d, b);
  }
}

// Host: X [n, F] -> edges [F][nq]; buf is ks words per feature.
int launch_quantile_two_reads(const float* X, int64_t n, int32_t F, int64_t xs, const float* q,
                              int32_t nq, float* edges, uint32_t* buf, int64_t ks,
                              hipStream_t st) {
  const int64_t nc = (F + 63) / 64;
  // one workgroup per CU in one round where the rows allow it
  int64_t nrb = std::max<int64_t>(1, 256 / nc);
  int64_t rows_per = std::max<int64_t>((n + nrb - 1) / nrb, 2048);
  rows_per = std::min<int64_t>((rows_per + 15) / 16 * 16, kQMaxRows);
  nrb = (n + rows_per - 1) / rows_per;
  const size_t part_b = (size_t)(nrb * nc) * (kQBuckets / 2 * 64) * 4;
  // small arrays, each a multiple of 16 bytes
  size_t off = 0;
  auto take = [&](size_t b) {
    const size_t o = off;
    off += (b + 255) / 256 * 256;
    return o;
  };
  const size_t o_sample = take((size_t)F * kQSample * 4), o_map = take((size_t)F * 8),
               o_nan = take((size_t)F * 4), o_negz = take((size_t)F * 4),
               o_smap = take((size_t)nc * 256 * 64 * 4),
               o_rmap = take((size_t)nc * 256 * 64 * 4), o_refs = take((size_t)nc * 128 * 64 * 4),
               o_size = take((size_t)F * 256 * 4), o_sref = take((size_t)F * 256 * 4),
               o_tslot = take((size_t)F * kSelMaxTargets),
               o_trank = take((size_t)F * kSelMaxTargets * 4), o_ns = take((size_t)F * 4),
               o_gc = take((size_t)F * nrb * 4), o_cnt = take((size_t)nc * kQBuckets * 64 * 4);
  uint32_t* part = (uint32_t*)scratch_get(st, part_b, 19);
  char* sm = (char*)scratch_get(st, off, 20);
  WGBM_REQUIRE(part && sm, "scratch allocation failed");
  float2* map = (float2*)(sm + o_map);
  uint32_t *nanf = (uint32_t*)(sm + o_nan), *smap = (uint32_t*)(sm + o_smap),
           *refs = (uint32_t*)(sm + o_refs), *ssize = (uint32_t*)(sm + o_size),
           *gc = (uint32_t*)(sm + o_gc), *negz = (uint32_t*)(sm + o_negz),
           *rmap = (uint32_t*)(sm + o_rmap), *sref = (uint32_t*)(sm + o_sref);
  uint8_t* tslot = (uint8_t*)(sm + o_tslot);
  int32_t *trank = (int32_t*)(sm + o_trank), *ns = (int32_t*)(sm + o_ns);
  float* sample = (float*)(sm + o_sample);
  const size_t lds_count = (size_t)kQBuckets / 2 * 64 * 4;
  const size_t lds_gather =
      (size_t)(256 * 64 + 128 * 64 + 64 + kQThreads / 64 * kQRing * 64) * 4;  // 156.25 KB of 160
  static_assert(kQBuckets == 1024, "slot bytes: four per word, 256 words per lane");
  WGBM_CHECK(hipFuncSetAttribute((const void*)quantile_count_kernel,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_count));
  WGBM_CHECK(hipFuncSetAttribute((const void*)quantile_gather_kernel,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_gather));
  const dim3 grid((unsigned)wgbm_xcd_grid(nrb * nc));
  hipLaunchKernelGGL(quantile_sample_kernel, dim3((unsigned)((F + 3) / 4)), dim3(256), 0, st, X, n,
                     F, xs, q, nq, sample, map, nanf, negz);
  WGBM_LAUNCH_CHECK();
  hipLaunchKernelGGL(quantile_count_kernel, grid, dim3(kQThreads), lds_count, st, X, n, F, xs,
                     (int32_t)rows_per, (int32_t)nrb, map, part, nanf, negz);
  WGBM_LAUNCH_CHECK();
  uint32_t* cnt = (uint32_t*)(sm + o_cnt);
  hipLaunchKernelGGL(quantile_sum_kernel, dim3((unsigned)(nc * (kQBuckets / 2))), dim3(256), 0, st,
                     part, (int32_t)nrb, (int32_t)nc, cnt);
  WGBM_LAUNCH_CHECK();
  hipLaunchKernelGGL(quantile_targets_kernel, dim3((unsigned)(nc * 4)), dim3(kQThreads), 0, st, cnt,
                     n, F, q, nq, map, sample, smap, rmap, refs, ssize, sref, tslot, trank, ns);
  WGBM_LAUNCH_CHECK();
  hipLaunchKernelGGL(quantile_gather_kernel, grid, dim3(kQThreads), lds_gather, st, X, n, F, xs,
                     (int32_t)rows_per, (int32_t)nrb, map, rmap, refs, buf, ks, gc);
  WGBM_LAUNCH_CHECK();
  hipLaunchKernelGGL(quantile_pick_kernel, dim3((unsigned)F), dim3(kPickThreads), 0, st, buf, ks,
                     n, (int32_t)rows_per, (int32_t)nrb, gc, q, nq, map, smap, ssize, sref, tslot,
                     trank, ns, nanf, negz, edges);
  WGBM_LAUNCH_CHECK();
  return 0;
}

}  // namespace wgbm
