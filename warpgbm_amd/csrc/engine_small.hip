// One-era rounds of few rows: one launch per level.
//
// The level chain (histogram tiles, finalize, split search, partition, level
// scan) is five dependent launches a level, each a few microseconds of latency
// whatever the data: 10000 rows x 50 features took 180 us a tree of depth 5,
// 33 us a level.  With few rows a workgroup can hold all of them, so here
// workgroup (feature, tree) of a level's launch
//   * routes every row through the previous level's picks itself (no rows are
//     moved: a row carries its heap index) and finds the nodes' largest
//     |residual| and so their histogram shifts,
//   * histograms its own feature of every node of the level (LDS, copies per
//     lane group against conflicts),
//   * scans it and adds its best candidate of each node to the level's picks
//     (atomicMax on the packed key of the level chain).
// One more workgroup per tree keeps the rows' new indices, the nodes' shifts,
// exact totals and the previous level's record.  Every sum is an exact integer
// and every scan the sequential float32 one, so the trees are those of the
// level chain bit for bit.  A level is bound by its chain of dependent loads
// and barriers, about 8 us.
#include <algorithm>

#include "common.hpp"
#include "engine.hpp"
#include "kernels.hpp"
#include "split_scan.hpp"

namespace wgbm {

constexpr int kSmThreads = 1024;

// fn(k) for the 2^rl copies of a cell, from a start that differs by thread (the
// threads of a wave then read different banks), eight reads in flight
template <typename Fn>
__device__ __forceinline__ void for_copies(int rl, int start, Fn&& fn) {
  const int R = 1 << rl;
  if (R >= 8) {
    for (int k = 0; k < R; k += 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) fn((k + j + start) & (R - 1));
    }
  } else {
    for (int k = 0; k < R; ++k) fn((k + start) & (R - 1));
  }
}

// RPT: rows per thread (n <= RPT * 1024); row u * 1024 + tid is the thread's
template <int RPT>
__global__ __launch_bounds__(kSmThreads) void small_level_kernel(SmallArgs a) {
  extern __shared__ unsigned long long sm[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int t = blockIdx.y, d = a.depth;
  const bool keeper = (int)blockIdx.x == a.n_feat_wg;  // the tree's bookkeeping workgroup
  const int nodes = 1 << d, first = nodes - 1;          // this level's heap range
  const int pnodes = nodes >> 1, pfirst = pnodes - 1;   // the previous level's (d > 0)
  const int B = a.B, Bp = B | 1;
  const int64_t n = a.n, hb = (int64_t)t * a.H;
  // LDS: parents' picks and this level's words, then the histogram copies (or
  // the keeper's totals copies)
  int32_t* dec_col = reinterpret_cast<int32_t*>(sm);  // [pnodes] column, -1: no split
  int32_t* dec_bin = dec_col + nodes;
  int32_t* shift_s = dec_bin + nodes;                 // [nodes]
  int32_t* pres_s = shift_s + nodes;
  unsigned long long* pick_s = sm + 2 * nodes;        // [nodes]
  unsigned long long* work = sm + 3 * nodes;
  __shared__ uint32_t s_root;

  // ---- rows: everything that does not depend on the picks.  Loads are
  // unconditional throughout (a row past the end repeats the last one and
  // belongs to no node): a load under a condition is a branch and a wait of
  // its own.  Offsets fit 32 bits (small_round_fits).
  float rv[RPT];
  int id[RPT], code[RPT];
  const int nn = (int)n;
  const float* resid_t = a.resid + (int64_t)t * n;
  const uint16_t* ids_t = a.ids_in + (int64_t)t * n;
  const int l = blockIdx.x;  // feature (index in the round's subset)
  const int8_t* col_own = nullptr;
  if (!keeper) col_own = a.codes_cm + (int64_t)a.feat_sel[l] * n;
  uint32_t rc[RPT];
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    const int r = u * kSmThreads + tid;
    rc[u] = (uint32_t)(r < nn ? r : nn - 1);
    code[u] = 0;
    id[u] = 0;
  }
  if (a.from_target) {  // (one tree: the residual as residual_regression_kernel)
#pragma unroll
    for (int u = 0; u < RPT; ++u) rv[u] = a.target[rc[u]] - a.pred[rc[u]];
  } else {
#pragma unroll
    for (int u = 0; u < RPT; ++u) rv[u] = resid_t[rc[u]];
  }
  if (d > 1) {
#pragma unroll
    for (int u = 0; u < RPT; ++u) id[u] = (int)ids_t[rc[u]];
  }
  if (!keeper) {
#pragma unroll
    for (int u = 0; u < RPT; ++u) code[u] = (int)col_own[rc[u]];
  }
#pragma unroll
  for (int u = 0; u < RPT; ++u)
    if (u * kSmThreads + tid >= nn) id[u] = 0xffff;  // no row: below no node
  // ---- the previous level's picks
  for (int p = tid; p < pnodes; p += kSmThreads) {
    const int64_t h = hb + pfirst + p;
    const unsigned long long k = a.best[h];
    const bool sp = a.present[h] && k != 0ull;
    const int idx = (int)(0xffffffffu - (uint32_t)(k & 0xffffffffull));
    const int pl = sp ? idx / (B - 1) : 0;
    const int pb = sp ? idx - pl * (B - 1) : 0;
    const int col = sp ? a.feat_sel[pl] : -1;
    dec_col[p] = col;
    dec_bin[p] = pb;
    // the children's presence, and their parent's shift until the rule below
    const int32_t ps = a.node_shift[h];
    shift_s[2 * p] = shift_s[2 * p + 1] = ps;
    pres_s[2 * p] = pres_s[2 * p + 1] = sp ? 1 : 0;
    if (keeper) {
      // the record of the previous level (finish_node)
      const int64_t cnt = a.tot_c[h];
      if (!a.present[h]) {
        a.rec.feat[h] = -2;
        a.rec.bin[h] = -1;
        a.rec.leaf[h] = 0.0f;
        a.rec.count[h] = 0;
      } else if (sp) {
        a.rec.feat[h] = col;
        a.rec.bin[h] = pb;
        a.rec.leaf[h] = 0.0f;
        a.rec.count[h] = cnt;
        a.rec.gain[h] = gain_from_key((uint32_t)(k >> 32));
      } else {
        a.rec.feat[h] = -1;
        a.rec.bin[h] = -1;
        a.rec.leaf[h] = leaf_mean(a.tot_qh[h], a.tot_ql[h], cnt, a.shifts[t] + a.s63_add);
        a.rec.count[h] = cnt;
      }
    }
  }
  if (d == 0) {
    uint32_t m = 0;
    if (a.from_target) {
#pragma unroll
      for (int u = 0; u < RPT; ++u) {
        const uint32_t b = wgbm_abs_bits(rv[u]);  // (a repeated last row changes no maximum)
        m = b > m ? b : m;
      }
    } else {
      for (int i = tid; i < a.n_part; i += kSmThreads) {
        const uint32_t b = a.abs_part[(int64_t)t * a.n_part + i];
        m = b > m ? b : m;
      }
    }
    m = wgbm_block_max_u32(m);
    if (tid == 0) {
      s_root = m;
      shift_s[0] = m >= 0x7f800000u ? 0 : wgbm_shift_from_absmax(__uint_as_float(m), a.qbits);
      pres_s[0] = 1;
    }
  }
  __syncthreads();
  // ---- route
  if (d > 0) {
    int c[RPT];
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      const uint32_t p = (uint32_t)(id[u] - pfirst);
      const int col = dec_col[p < (uint32_t)pnodes ? p : 0];
      c[u] = (int)a.codes_cm[(uint32_t)(col > 0 ? col : 0) * (uint32_t)nn + rc[u]];
    }
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      const uint32_t p = (uint32_t)(id[u] - pfirst);
      const uint32_t pc = p < (uint32_t)pnodes ? p : 0;
      const bool sp = p < (uint32_t)pnodes && dec_col[pc] >= 0;
      id[u] = sp ? 2 * id[u] + 1 + (c[u] > dec_bin[pc] ? 1 : 0) : id[u];
    }
  }
  // the row's node on this level, or the spare one past them
  uint32_t nd[RPT];
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    const uint32_t p = (uint32_t)(id[u] - first);
    nd[u] = p < (uint32_t)nodes ? p : (uint32_t)nodes;
  }
  // ---- the nodes' shifts (a level whose nodes are histogrammed)
  if (d > 0 && d < a.max_depth) {
    const int rl = a.max_copies_log2;
    uint32_t* mx = reinterpret_cast<uint32_t*>(work);
    for (int i = tid; i < nodes << rl; i += kSmThreads) mx[i] = 0u;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < RPT; ++u)
      atomicMax(mx + (nd[u] << rl) + (lane & ((1 << rl) - 1)), wgbm_abs_bits(rv[u]));
    __syncthreads();
    for (int p = tid; p < nodes; p += kSmThreads) {
      uint32_t m = 0;
      for_copies(rl, p, [&](int k) {
        const uint32_t v = mx[(p << rl) + k];
        m = v > m ? v : m;
      });
      shift_s[p] = node_shift_rule(m, shift_s[p], a.qbits);
    }
    __syncthreads();
  }
  if (keeper) {
    // ---- totals of this level's nodes: exact sums of the wide quantisation
    const int s63 = (d == 0 ? shift_s[0] : a.shifts[t]) + a.s63_add;
    const int rl = a.tot_copies_log2, R = 1 << rl;
    // (q >> 32) * 2^kCnt + 1 and q mod 2^32: |q >> 32| <= 2^30 a row
    constexpr int kCnt = 15;
    static_assert(kSmallMaxRows < (1 << kCnt) && 30 + 2 * kCnt < 63, "sum and count in one word");
    unsigned long long* qh_s = work;
    unsigned long long* ql_s = qh_s + ((nodes + 1) << rl);
    for (int i = tid; i < nodes << rl; i += kSmThreads) qh_s[i] = ql_s[i] = 0ull;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      const int64_t q = (int64_t)rintf(ldexpf(rv[u], s63));
      const uint32_t i = (nd[u] << rl) + (uint32_t)(lane & (R - 1));
      atomicAdd(qh_s + i, (unsigned long long)((q >> 32) * (int64_t)(1 << kCnt) + 1));
      atomicAdd(ql_s + i, (unsigned long long)(q & 0xffffffffll));
    }
    if (d > 0 && d < a.max_depth) {
#pragma unroll
      for (int u = 0; u < RPT; ++u)
        if (u * kSmThreads + tid < nn) a.ids_out[(int64_t)t * n + rc[u]] = (uint16_t)id[u];
    }
    if (a.from_target) {
#pragma unroll
      for (int u = 0; u < RPT; ++u)
        if (u * kSmThreads + tid < nn) a.resid_out[rc[u]] = rv[u];
    }
    __syncthreads();
    if (d == 0 && tid == 0) {
      a.shifts[t] = shift_s[0];
      a.absmax[t] = s_root;
    }
    for (int p = tid; p < nodes; p += kSmThreads) {
      int64_t qh = 0, ql = 0, c = 0;
      for_copies(rl, p, [&](int k) {
        const int i = (p << rl) + k;
        const int64_t w = (int64_t)qh_s[i];
        qh += w >> kCnt;
        c += w & ((1 << kCnt) - 1);
        ql += (int64_t)ql_s[i];
      });
      const int64_t h = hb + first + p;
      if (d < a.max_depth) {
        a.tot_qh[h] = qh;
        a.tot_ql[h] = ql;
        a.tot_c[h] = c;
        a.present[h] = pres_s[p];
        a.node_shift[h] = shift_s[p];
      } else {
        const bool pr = pres_s[p] != 0;
        a.rec.feat[h] = pr ? -1 : -2;
        a.rec.bin[h] = -1;
        a.rec.leaf[h] = pr ? leaf_mean(qh, ql, c, s63) : 0.0f;
        a.rec.count[h] = pr ? c : 0;
      }
    }
    // the next level's picks start empty (after the last level: the root's)
    if (d + 1 < a.max_depth) {
      for (int p = tid; p < 2 * nodes; p += kSmThreads) a.best[hb + 2 * nodes - 1 + p] = 0ull;
    } else if (d == a.max_depth && tid == 0) {
      a.best[hb] = 0ull;
    }
    if (d < a.max_depth) return;
    // ---- predictions: every row's leaf, in the record (written above and by
    // the earlier levels' launches)
    __syncthreads();
    float* pred_t = a.pred + (int64_t)t * a.pcol;
    const float* leaf_t = a.rec.leaf + hb;
    float pv[RPT], lv[RPT];
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      pv[u] = pred_t[rc[u]];
      lv[u] = leaf_t[id[u] < a.H ? id[u] : 0];
    }
#pragma unroll
    for (int u = 0; u < RPT; ++u)
      if (u * kSmThreads + tid < nn) pred_t[rc[u]] = pv[u] + a.lr * lv[u];
    return;
  }
  // ---- the feature's histogram of every node: cell (node, bin), R copies
  const int cells = nodes * B;
  const int rl = a.hist_copies_log2, R = 1 << rl;
  for (int i = tid; i < cells << rl; i += kSmThreads) work[i] = 0ull;
  __syncthreads();
  // (a row of no node, or a code outside the bins, adds to the spare cell)
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    const bool in = nd[u] < (uint32_t)nodes && (uint32_t)code[u] < (uint32_t)B;
    const int64_t q = (int64_t)wgbm_quantise(rv[u], shift_s[in ? nd[u] : 0]);
    const uint32_t cell = in ? nd[u] * (uint32_t)B + (uint32_t)code[u] : (uint32_t)cells;
    atomicAdd(work + (cell << rl) + (uint32_t)(lane & (R - 1)),
              (unsigned long long)(q * (int64_t)(1 << WGBM_CBITS) + 1));
  }
  __syncthreads();
  // ---- each cell's float sum and count (the copies read from a start that
  // differs by lane), then each node's prefixes in place, in bin order
  float* gf = reinterpret_cast<float*>(work + ((cells + 1) << rl));  // [nodes][Bp]
  float* hf = gf + nodes * Bp;
  for (int c = tid; c < cells; c += kSmThreads) {
    int64_t Q = 0, C = 0;
    for_copies(rl, c, [&](int k) {
      const unsigned long long P = work[(c << rl) + k];
      C += (int64_t)(P & (unsigned long long)WGBM_CMASK);
      Q += (int64_t)P >> WGBM_CBITS;
    });
    const int p = c / B, b = c - p * B;
    gf[p * Bp + b] = wgbm_dequantise(Q, shift_s[p]);
    hf[p * Bp + b] = (float)C;
  }
  for (int p = tid; p < nodes; p += kSmThreads) pick_s[p] = 0ull;
  __syncthreads();
  for (int p = tid; p < nodes; p += kSmThreads) {
    float G = 0.0f, H = 0.0f;
    float* g = gf + p * Bp;
    float* h = hf + p * Bp;
    constexpr int U = 8;  // words read together
    for (int b0 = 0; b0 < B; b0 += U) {
      float x[U], y[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        x[k] = g[b0 + k < B ? b0 + k : B - 1];
        y[k] = h[b0 + k < B ? b0 + k : B - 1];
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        if (b0 + k >= B) break;  // uniform
        G = G + x[k];
        H = H + y[k];
        g[b0 + k] = G;
        h[b0 + k] = H;
      }
    }
  }
  __syncthreads();
  for (int c = tid; c < nodes * (B - 1); c += kSmThreads) {
    const int p = c / (B - 1), b = c - p * (B - 1);
    if (!pres_s[p]) continue;
    float g, w;
    split_candidate(gf[p * Bp + b], hf[p * Bp + b], gf[p * Bp + B - 1], hf[p * Bp + B - 1], a.mcw,
                    a.eps, g, w);
    if (g > a.msg)
      atomicMax(pick_s + p, ((unsigned long long)gain_key(g) << 32) |
                                (unsigned long long)(0xffffffffu - (uint32_t)(l * (B - 1) + b)));
  }
  __syncthreads();
  for (int p = tid; p < nodes; p += kSmThreads)
    if (pick_s[p]) atomicMax(a.best + hb + first + p, pick_s[p]);
}

// LDS bytes of a level's launch and its copy counts (set in a)
static size_t small_lds(SmallArgs& a) {
  const int64_t nodes = int64_t(1) << a.depth, Bp = a.B | 1;
  // at most 16 copies (more take longer to add up than they save in
  // conflicts) within 48 KB (of what clearing and adding them up costs; a level
  // whose cells alone take more has one copy)
  auto copies = [](int64_t words, int64_t bytes) {
    int lg = 4;
    while (lg > 0 && (words << lg) * bytes > 48 * 1024) --lg;
    return lg;
  };
  a.hist_copies_log2 = copies(nodes * a.B, 8);
  a.max_copies_log2 = copies(nodes, 4);
  a.tot_copies_log2 = copies(nodes, 16);
  const int64_t hist = ((nodes * a.B + 1) << a.hist_copies_log2) * 8 + nodes * Bp * 8;
  const int64_t most = std::max(std::max(hist, ((nodes + 1) << a.max_copies_log2) * 4),
                                ((nodes + 1) << a.tot_copies_log2) * 16);
  return (size_t)(nodes * 24 + most);
}

bool small_round_fits(int64_t n, int32_t F, int32_t B, int32_t max_depth) {
  if (n > kSmallMaxRows || max_depth > 13 || F * n > (int64_t(1) << 31)) return false;
  SmallArgs a{};
  a.B = B;
  a.depth = max_depth - 1;
  const size_t h = small_lds(a);
  // (the last level's launch holds totals of 2^max_depth nodes, and no histogram)
  return h <= 128 * 1024 && ((int64_t(1) << max_depth) + 1) * 40 <= 128 * 1024;
}

// Whether one launch per level is faster than the level chain.  The chain's
// launches take longer with more bins, and with more trees hardly longer; a
// turn of these workgroups takes longer with more rows.  Level chain / one launch
// per level, us per round of depth 5: up to 12288 rows it wins wherever it is
// allowed (12288 x 51, 10 classes, 5 bins: 1.04 times); then at most two turns
// (20480 x 400, 32 bins 1.3 times), but for few bins and a second turn of few
// workgroups (20480 x 107, 3 classes, 5 bins 160 / 169; 128, 2 classes 158 / 165),
// or three turns where bins or rows make up for them (20480 x 512, 63 bins 1.35
// times, 32 bins 0.89; 16384 x 512, 32 bins 1.07, 10 classes 0.94).
bool small_round_pays(int64_t n, int32_t B, int32_t T, int32_t n_sel) {
  if ((int64_t)T * n_sel > kSmallMaxWork) return false;
  const int64_t wgs = (int64_t)T * (n_sel + 1);
  if (n <= 12288 || wgs <= 256) return true;
  if (wgs <= 512) return !(n > 16384 && T > 1 && B <= 10 && wgs <= 384);
  return B > 48 || (n <= 16384 && T <= 3 && B >= 32);
}

template <int RPT>
static int launch_small(const SmallArgs& a, int T, size_t lds, hipStream_t st) {
  static bool attr = false;
  if (!attr) {
    WGBM_CHECK(hipFuncSetAttribute((const void*)small_level_kernel<RPT>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 144 * 1024));
    attr = true;
  }
  hipLaunchKernelGGL(small_level_kernel<RPT>, dim3((unsigned)(a.n_feat_wg + 1), (unsigned)T),
                     dim3(kSmThreads), lds, st, a);
  WGBM_LAUNCH_CHECK();
  return 0;
}

int launch_small_level(SmallArgs a, int T, hipStream_t st) {
  const size_t lds = [&] {
    if (a.depth < a.max_depth) return small_lds(a);
    SmallArgs last = a;  // no histogram: the totals only
    last.B = 1;
    const size_t b = small_lds(last);
    a.tot_copies_log2 = last.tot_copies_log2;
    a.max_copies_log2 = last.max_copies_log2;
    return b;
  }();
  if (a.n <= 1 * kSmThreads) return launch_small<1>(a, T, lds, st);
  if (a.n <= 2 * kSmThreads) return launch_small<2>(a, T, lds, st);
  if (a.n <= 4 * kSmThreads) return launch_small<4>(a, T, lds, st);
  if (a.n <= 8 * kSmThreads) return launch_small<8>(a, T, lds, st);
  if (a.n <= 12 * kSmThreads) return launch_small<12>(a, T, lds, st);
  if (a.n <= 16 * kSmThreads) return launch_small<16>(a, T, lds, st);
  // (20: 128 registers and four spilled; 24 rows a thread took 2.4 ms for 0.1 ms)
  static_assert(kSmallMaxRows <= 20 * kSmThreads, "rows per thread");
  return launch_small<20>(a, T, lds, st);
}

}  // namespace wgbm
