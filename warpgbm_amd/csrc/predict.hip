// Tree-ensemble inference on int8 bin codes.
//
// Reference (warpgbm/cuda/predict.cu:13-44): thread (row i, tree t) starts at
// node 0 of the flattened table [T, M, 6] = (feature, bin, left, right,
// is_leaf, leaf_value); while !(is_leaf > 0.5): go left if code <= bin;
// at the leaf: atomicAdd(out[i], lr * leaf_value).
//
// Here one lane owns a row (or a (row, class) pair) and adds the trees in tree
// order, so out[i] = ((out[i] + lr*v_0) + lr*v_1) + ... is deterministic; it is
// one of the orders the reference's atomics may produce.  Each product lr*v is
// rounded to float32 before the add, as in the reference.
#include <algorithm>

#include "common.hpp"
#include "engine.hpp"
#include "kernels.hpp"

namespace wgbm {

// reference table format, walk bounded by M steps (malformed tables cannot
// loop forever; a walk that leaves the table contributes NaN)
// run_if (optional): the walk runs only when *run_if is nonzero (the fallback
// of wgbm_predict_forest's heap path, decided on the device)
__global__ void predict_table_kernel(const int8_t* __restrict__ codes, int64_t n, int64_t F,
                                     const float* __restrict__ table, int64_t T, int64_t M,
                                     float lr, float* __restrict__ out,
                                     const int32_t* __restrict__ run_if) {
  if (run_if && *run_if == 0) return;  // uniform
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int8_t* row = codes + i * F;
  float acc = out[i];
  for (int64_t t = 0; t < T; ++t) {
    const float* tree = table + t * M * 6;
    int64_t node = 0;
    float v = __builtin_nanf("");
    for (int64_t step = 0; step <= M; ++step) {
      const float* nd = tree + node * 6;
      if (nd[4] > 0.5f) {
        v = nd[5];
        break;
      }
      const int feat = (int)nd[0];
      const int sb = (int)nd[1];
      if (feat < 0 || feat >= F) break;
      const int nxt = (int)row[feat] <= sb ? (int)nd[2] : (int)nd[3];
      if (nxt < 0 || nxt >= M) break;
      node = nxt;
    }
    acc = acc + lr * v;
  }
  out[i] = acc;
}

// The reference's flat tables [T, M, 6] as heap tables of depth D (H =
// 2^(D+1) - 1 slots per tree), for wgbm_predict_forest's heap path: one
// thread per (tree, heap node h) walks from node 0 along h's path and
// writes what the flat walk of predict_table_kernel meets there: a leaf
// (feat -1, its value), a split (feature, bin), an absent node (-2, under a
// leaf) or -- where that walk would stop with NaN (a feature outside [0, F),
// a child index outside [0, M)) -- a leaf of value NaN, so the heap walk
// returns the same value.  A split on the last heap level (a deeper tree), a
// negative bin or a feature >= 65536 cannot be held: then *fallback is set
// and the caller's flat walk runs instead.  Bins of 127 and above hold as
// 255: every int8 code is <= such a bin, and every code byte of the native
// copy (127 and 128 included) is <= 255.
__global__ void flat_to_heap_kernel(const float* __restrict__ table, int64_t T, int64_t M,
                                    int64_t F, int32_t D, int32_t* __restrict__ feat,
                                    int32_t* __restrict__ bin, float* __restrict__ leaf,
                                    int32_t* __restrict__ fallback) {
  const int64_t H = (int64_t(2) << D) - 1;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= T * H) return;
  const int64_t t = gid / H;
  const int h = (int)(gid - t * H);
  const float* tree = table + t * M * 6;
  const int d = 31 - __builtin_clz((unsigned)(h + 1));  // depth of heap node h
  int32_t f_out = -2, b_out = 0;
  float v_out = 0.0f;
  int64_t node = 0;
  bool reached = true;
  for (int k = 0; k < d && reached; ++k) {
    const float* nd = tree + node * 6;
    if (nd[4] > 0.5f) {  // a leaf above h: h is absent
      reached = false;
      break;
    }
    const int f = (int)nd[0];
    if (f < 0 || f >= F) {  // the walk stops here (NaN): h is absent
      reached = false;
      break;
    }
    const int right = ((h + 1) >> (d - 1 - k)) & 1;
    const int nxt = right ? (int)nd[3] : (int)nd[2];
    if (nxt < 0 || nxt >= M) {
      // the walk stops (NaN) on this edge: a NaN leaf if it leads to h
      if (k == d - 1) {
        f_out = -1;
        v_out = __builtin_nanf("");
      }
      reached = false;
      break;
    }
    node = nxt;
  }
  if (reached) {
    const float* nd = tree + node * 6;
    if (nd[4] > 0.5f) {
      f_out = -1;
      v_out = nd[5];
    } else {
      const int f = (int)nd[0];
      const int sb = (int)nd[1];
      if (f < 0 || f >= F) {
        f_out = -1;
        v_out = __builtin_nanf("");
      } else if (d == D || sb < 0 || f > 65535) {
        *fallback = 1;
        f_out = -1;
      } else {
        f_out = f;
        b_out = sb < 127 ? sb : 255;
      }
    }
  }
  feat[gid] = f_out;
  bin[gid] = b_out;
  leaf[gid] = v_out;
}

// compact heap tables written by the engine: node h has children 2h+1, 2h+2.
//   feat[t][h] >= 0 split feature, -1 leaf; bin[t][h]; leaf[t][h]
// trees are ordered (round, class); out is [n, K] row-major, pre-initialised.
// codes are native (bytes in [0, B + 1], B = num_bins): the byte B stands for
// a negative code, which goes left at every split (a raw int8 code <= bin
// with bin >= 0), and B + 1 for a code >= B, which goes right; the other
// bytes are the codes themselves.
__global__ void predict_heap_kernel(const int8_t* __restrict__ codes, int64_t n, int64_t S,
                                    int32_t num_bins, const int32_t* __restrict__ feat,
                                    const int32_t* __restrict__ bin,
                                    const float* __restrict__ leaf, int32_t n_rounds, int32_t K,
                                    int32_t H, int32_t max_depth, float lr,
                                    float* __restrict__ out, const int32_t* __restrict__ skip) {
  if (skip && *skip) return;  // uniform: the caller's fallback runs instead
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= n * K) return;
  const int64_t i = gid / K;
  const int k = (int)(gid - i * K);
  const int8_t* row = codes + i * S;
  float acc = out[gid];
  for (int r = 0; r < n_rounds; ++r) {
    const int64_t t = (int64_t)r * K + k;
    const int32_t* ft = feat + t * H;
    const int32_t* bt = bin + t * H;
    int h = 0;
    for (int d = 0; d < max_depth; ++d) {
      const int f = ft[h];
      if (f < 0) break;
      const int c = (int)(uint8_t)row[f];
      h = 2 * h + ((c <= bt[h] || c == num_bins) ? 1 : 2);
    }
    acc = acc + lr * leaf[t * H + h];
  }
  out[gid] = acc;
}

// Complete-tree tables for the LDS predictors.  Per tree: (2^D - 1) node
// words for the levels above the last, feature << 16 | bin for a split whose
// ancestors are all splits, else (a leaf, an absent node, or any position
// under one) the always-left word 255 (every code byte is <= 255); and 2^D
// last-level values, slot s = lr times the leaf value of the first node on
// the path from the root to heap node 2^D - 1 + s that is not a split (or of
// that node itself), rounded to float32 as the walkers' per-tree products
// are.  A walk then takes exactly D steps with no leaf test and reaches
// the value the heap walk stops at.  Features are clamped into the row
// (S - 1 < 65536), as the walkers clamp them.
__global__ void complete_tables_kernel(const int32_t* __restrict__ feat,
                                       const int32_t* __restrict__ bin,
                                       const float* __restrict__ leaf, int64_t T, int32_t D,
                                       int64_t S, float lr, uint32_t* __restrict__ cnode,
                                       float* __restrict__ cleaf) {
  const int Hi = (1 << D) - 1, L = 1 << D, H = 2 * L - 1;
  const int64_t per = (int64_t)Hi + L;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= T * per) return;
  const int64_t t = gid / per;
  const int j = (int)(gid - t * per);
  const int32_t* ft = feat + t * H;
  if (j < Hi) {
    const int dj = 31 - __builtin_clz((unsigned)(j + 1));  // depth of node j
    bool split = true;
    for (int k = 0; k <= dj && split; ++k) split = ft[((j + 1) >> (dj - k)) - 1] >= 0;
    uint32_t w = 255u;
    if (split) {
      const int64_t f = ft[j] < S ? ft[j] : S - 1;
      w = ((uint32_t)f << 16) | ((uint32_t)bin[t * H + j] & 0xffu);
    }
    cnode[t * Hi + j] = w;
  } else {
    const int sl = j - Hi;
    const int h = Hi + sl;  // heap node at depth D
    int a = h;
    for (int k = 0; k < D; ++k) {
      const int ak = ((h + 1) >> (D - k)) - 1;
      if (ft[ak] < 0) {
        a = ak;
        break;
      }
    }
    cleaf[t * L + sl] = lr * leaf[t * H + a];
  }
}

// Code bytes as the LDS walkers read them: a native byte equal to num_bins (a
// negative code, left at every split) becomes 0, which also goes left at
// every split (split bins are >= 0), so a walk step is one compare: right iff
// code > bin.  bb = num_bins * 0x01010101.
__device__ __forceinline__ uint32_t walk_bytes(uint32_t x, uint32_t bb) {
  const uint32_t t = x ^ bb;  // zero bytes where x has num_bins
  // 0x80 in every byte of t that is not zero (no carries between bytes)
  const uint32_t nz = (((t & 0x7f7f7f7fu) + 0x7f7f7f7fu) | t) & 0x80808080u;
  return x & ((nz >> 7) * 0xffu);
}

// A walk over a complete table held in LDS, stepped by LDS byte address: the
// tree's node words start at `base`, node g (1-based heap index, children 2g
// and 2g + 1) sits at a = base + 4 (g - 1), so the step to child 2g + x is
// a' = 2a + 4 + 4x - base (mod 2^32): one compare, one select, one shift-add
// and the row byte's address per step.
typedef __attribute__((address_space(3))) uint32_t lds_u32_t;
typedef __attribute__((address_space(3))) uint8_t lds_u8_t;
typedef __attribute__((address_space(3))) int8_t lds_i8_t;

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const lds_u8_t*)p;
}

struct Walk {
  uint32_t a, k0, k1;  // node address; step offsets for left / right
  __device__ __forceinline__ void start(uint32_t base) {
    a = base;
    k0 = 4u - base;
    k1 = 8u - base;
    // opaque to the optimiser, which would otherwise fold the select back into
    // select(4, 8) - base, one more instruction per step
    __asm__("" : "+v"(k0), "+v"(k1));
  }
  // row: LDS address of the row's first code byte.  RAW: a raw int8 code (the
  // reference's bin_indices, any value), read signed: a negative one goes left
  // at every split as the reference's signed `code <= bin` sends it (split
  // bins are 0..126, or 255)
  template <bool RAW>
  __device__ __forceinline__ void step(uint32_t row) {
    const uint32_t w = *(const lds_u32_t*)(uintptr_t)a;
    const uintptr_t at = row + (w >> 16);
    const int c = RAW ? (int)*(const lds_i8_t*)at : (int)*(const lds_u8_t*)at;
    a = 2u * a + (c > (int)(w & 0xffu) ? k1 : k0);
  }
};

typedef __attribute__((address_space(3))) float lds_f32_t;

// Walks the trees j = j_first, j_first + G, ... (j < n_trees) of one row, NW
// in lock-step, and stores each tree's value at out_a + 4j.  LDS byte
// addresses: row_a = the row's code bytes, nodes_a = tree 0's node words (Hi
// per tree), values_a = tree 0's last-level values (Hi + 1 per tree).  After
// D steps a walk of tree j sits at a = nodes_a + 4 (j Hi + g - 1) with g =
// 2^D + slot, so its value is at a + c0 + 4j, c0 = values_a - nodes_a + 4 -
// 4 (Hi + 1): every address is an add, and the trees' node words advance by
// a uniform stride.  An idle walk (past n_trees, or row_on false) walks tree
// 0 and stores nothing.
template <int NW, bool RAW>
__device__ __forceinline__ void walk_trees(int j_first, int n_trees, int G, bool row_on,
                                           uint32_t row_a, uint32_t nodes_a, uint32_t values_a,
                                           int Hi, int D, uint32_t out_a) {
  const uint32_t hi4 = 4u * (uint32_t)Hi, nstep = hi4 * (uint32_t)G;
  const uint32_t c0 = values_a - nodes_a + 4u - 4u * (uint32_t)(Hi + 1);
  uint32_t nb = nodes_a + hi4 * (uint32_t)j_first;  // node words of tree j0
  for (int j0 = j_first; j0 < n_trees; j0 += NW * G, nb += NW * nstep) {
    Walk wk[NW];
    uint32_t t4[NW];
    bool on[NW];
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      on[k] = row_on && j0 + k * G < n_trees;
      t4[k] = on[k] ? 4u * (uint32_t)(j0 + k * G) : 0u;
      wk[k].start(on[k] ? nb + (uint32_t)k * nstep : nodes_a);
    }
    for (int d = 0; d < D; ++d) {
#pragma unroll
      for (int k = 0; k < NW; ++k) wk[k].template step<RAW>(row_a);
    }
#pragma unroll
    for (int k = 0; k < NW; ++k)
      if (on[k])
        *(lds_f32_t*)(uintptr_t)(out_a + t4[k]) =
            *(const lds_f32_t*)(uintptr_t)(wk[k].a + c0 + t4[k]);
  }
}

// Row-block inference (same results as predict_heap_kernel): a workgroup of
// 1024 threads stages a block of RB rows of codes in LDS (one coalesced read
// of the rows instead of a dependent byte gather per tree level) and walks
// the trees a chunk of TC at a time: the chunk's complete-tree tables
// (complete_tables_kernel) are staged in LDS, every (row, tree) pair of the
// chunk is walked by its own thread (all walks independent: D dependent LDS
// reads each instead of D per tree in sequence), the products lr * leaf (the
// tables hold them) go to an LDS table [row][tree], and one thread per (row,
// class) adds them in tree order.  TC is a multiple of K, so tree t0 + j belongs to class j % K.
//   LDS: rows [RB][S + 4] bytes (a 4-byte pad per row spreads the rows of
//   one wave over the banks), node words [TC][2^D - 1], last-level values
//   [TC][2^D], vals [RB][TC + 1] (odd row stride: no bank conflicts).
constexpr int kPredThreads = 1024;
constexpr int kPredMaxAcc = 4;  // (row, class) accumulators per thread
constexpr int kPredWalks = 2;   // walks a thread advances in lock-step

__global__ __launch_bounds__(kPredThreads) void predict_rows_kernel(
    const int8_t* __restrict__ codes, int64_t n, int64_t S, int32_t num_bins,
    const uint32_t* __restrict__ cnode, const float* __restrict__ cleaf, int32_t n_rounds,
    int32_t K, int32_t max_depth, int32_t RB, int32_t TC, float* __restrict__ out,
    const int32_t* __restrict__ skip) {
  if (skip && *skip) return;  // uniform: the caller's fallback runs instead
  extern __shared__ uint32_t psm[];
  const int Sp = (int)S + 4;
  const int Hi = (1 << max_depth) - 1, L = 1 << max_depth;  // complete-table widths
  uint8_t* rows_s = reinterpret_cast<uint8_t*>(psm);
  uint32_t* nodes_s = psm + (RB * Sp) / 4;
  float* leaves_s = reinterpret_cast<float*>(nodes_s + TC * Hi);
  float* vals_s = leaves_s + TC * L;
  const int64_t row0 = (int64_t)blockIdx.x * RB;
  const int nr = (int)(n - row0 < RB ? n - row0 : RB);
  const int tid = threadIdx.x;
  const uint32_t bb = (uint32_t)num_bins * 0x01010101u;
  // stage the row block: 16-byte global loads, 4-byte LDS stores
  {
    const int q_per_row = (int)(S / 16);
    const int nq = nr * q_per_row;
    for (int q = tid; q < nq; q += kPredThreads) {
      const int r = q / q_per_row, c = q - r * q_per_row;
      typedef uint32_t u4 __attribute__((ext_vector_type(4)));
      const u4 v = __builtin_nontemporal_load(
          reinterpret_cast<const u4*>(codes + (row0 + r) * S) + c);
      uint32_t* dst = reinterpret_cast<uint32_t*>(rows_s + r * Sp + c * 16);
      dst[0] = walk_bytes(v.x, bb);
      dst[1] = walk_bytes(v.y, bb);
      dst[2] = walk_bytes(v.z, bb);
      dst[3] = walk_bytes(v.w, bb);
    }
  }
  // accumulators: pair m*1024 + tid = (row, class) = (p % RB, p / RB)
  float acc[kPredMaxAcc];
#pragma unroll
  for (int m = 0; m < kPredMaxAcc; ++m) {
    const int p = m * kPredThreads + tid;
    const int r = p % RB, k = p / RB;
    acc[m] = (k < K && r < nr) ? out[(row0 + r) * K + k] : 0.0f;
  }
  const int T = n_rounds * K;
  const int G = kPredThreads / RB;  // RB <= 256: G >= 4
  const bool walker = tid < G * RB;
  const int wr = walker ? tid % RB : 0;
  const int wt0 = walker ? tid / RB : 0;
  for (int t0 = 0; t0 < T; t0 += TC) {
    const int tc = T - t0 < TC ? T - t0 : TC;
    __syncthreads();  // rows staged / previous chunk's vals consumed
    for (int i = tid; i < tc * Hi; i += kPredThreads) nodes_s[i] = cnode[(int64_t)t0 * Hi + i];
    for (int i = tid; i < tc * L; i += kPredThreads) leaves_s[i] = cleaf[(int64_t)t0 * L + i];
    __syncthreads();
    // walks: thread w < G * RB owns row wr = w % RB and the chunk's trees
    // wt0, wt0 + G, ... (G = threads / RB row groups, no division per walk),
    // two in lock-step so that the LDS reads of one overlap those of the
    // other; max_depth steps on the complete tables (no leaf test)
    if (walker)
      walk_trees<kPredWalks, false>(wt0, tc, G, wr < nr, lds_addr(rows_s + wr * Sp),
                                    lds_addr(nodes_s), lds_addr(leaves_s), Hi, max_depth,
                                    lds_addr(vals_s + wr * (TC + 1)));
    __syncthreads();
    // ordered sums: trees t0 + j of class k are j = k, k + K, ... (t0 % K == 0)
#pragma unroll
    for (int m = 0; m < kPredMaxAcc; ++m) {
      const int p = m * kPredThreads + tid;
      const int r = p % RB, k = p / RB;
      if (k < K && r < nr) {
        float a = acc[m];
        for (int j = k; j < tc; j += K) a = a + vals_s[r * (TC + 1) + j];
        acc[m] = a;
      }
    }
  }
#pragma unroll
  for (int m = 0; m < kPredMaxAcc; ++m) {
    const int p = m * kPredThreads + tid;
    const int r = p % RB, k = p / RB;
    if (k < K && r < nr) out[(row0 + r) * K + k] = acc[m];
  }
}

// ---------------------------------------------------------------------------
// Resident-tree inference, for ensembles whose complete-tree tables fit in
// LDS next to a row block (same results as predict_rows_kernel).  Persistent
// workgroups (one per CU) load every tree once, then stride over blocks of RB
// rows:
//   * the next block's codes are loaded into registers while the current one
//     is walked (QPT 16-byte loads per thread), then stored to the LDS row
//     buffer after the walks;
//   * waves 1..15 walk the (row, tree) pairs of the block, two per thread
//     in lock-step, and write lr * leaf (from the tables) to a per-block value
//     table [RB][T + 1];
//   * wave 0 meanwhile adds the previous block's table to `out` in tree
//     order (one lane per (row, class)), so the ordered sums run beside the
//     walks; the value tables alternate between two buffers.
// Bound by VALU work about as much as by the walks' LDS reads (four or seven
// walks in lock-step are no faster than two), so a load's address is its place
// in the block's run of bytes (no division by the row length, no row test: the
// buffer's size ends the block), its place in LDS is found once, and raw codes
// are compared as signed bytes instead of being mapped when stored.  100 trees of
// depth 5, us before / now: 1M x 1000 raw codes 335 / 272; 300k rows of 1000, 696,
// 400 raw codes 123 / 101, 100 / 90, 90 / 82, of 1000 and 500 native ones 97 /
// 93, 82 / 76.
// ---------------------------------------------------------------------------
constexpr int kResThreads = 1024;
constexpr int kResMaxQ = 4;  // 16-byte row loads per thread and block
constexpr int kResWalks = 2;  // walks a walker thread advances in lock-step

// RAW: the rows are raw int8 codes of stride S (a multiple of 8, read with
// 8-byte loads, twice as many per thread) and walked as signed bytes, instead
// of native codes (S a multiple of 16) mapped by walk_bytes.
template <bool RAW>
__global__ __launch_bounds__(kResThreads) void predict_resident_kernel(
    const int8_t* __restrict__ codes, int64_t n, int64_t S, int32_t num_bins,
    const uint32_t* __restrict__ cnode, const float* __restrict__ cleaf, int32_t T, int32_t K,
    int32_t max_depth, int32_t RB, float* __restrict__ out,
    const int32_t* __restrict__ skip) {
  if (skip && *skip) return;  // uniform: the caller's fallback runs instead
  extern __shared__ uint32_t psm[];
  const int Sp = (int)S + 4;
  const int TV = T + 1;  // value-table row stride (odd or even, see below)
  const int Hi = (1 << max_depth) - 1, L = 1 << max_depth;  // complete-table widths
  uint32_t* nodes_s = psm;
  float* leaves_s = reinterpret_cast<float*>(nodes_s + T * Hi);
  uint8_t* rows_s = reinterpret_cast<uint8_t*>(leaves_s + T * L);
  float* vals_s = reinterpret_cast<float*>(rows_s + RB * Sp);  // 2 x [RB][TV]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t bb = (uint32_t)num_bins * 0x01010101u;
  for (int i = tid; i < T * Hi; i += kResThreads) nodes_s[i] = cnode[i];
  for (int i = tid; i < T * L; i += kResThreads) leaves_s[i] = cleaf[i];
  const int64_t nblk = (n + RB - 1) / RB;
  constexpr int QW = RAW ? 2 : 4;            // 32-bit words per load
  constexpr int NQ = kResMaxQ * 4 / QW;      // loads per thread and block
  const int qpr = (int)(S / (4 * QW));       // loads per row
  const int nq = RB * qpr;
  typedef uint32_t uq __attribute__((ext_vector_type(QW)));
  uq pre[NQ];
  // a block's rows are one run of bytes (past the last row: zeros, no access);
  // in LDS load q of row r moves by r pads
  auto prefetch = [&](int64_t b) {
    const int64_t left = n - b * RB;
    const __amdgpu_buffer_rsrc_t rs =
        wgbm_rsrc(codes + b * RB * S, (uint32_t)((left < RB ? left : RB) * S));
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      const int at = (u * kResThreads + tid) * (4 * QW);
      if (u * kResThreads + wave * 64 >= nq) break;  // uniform over the wave
      if constexpr (RAW)
        pre[u] = __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, kAuxStream);
      else
        pre[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, kAuxStream);
    }
  };
  uint32_t to[NQ];  // the load's place in LDS
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int q = u * kResThreads + tid;
    to[u] = (uint32_t)(q * (4 * QW) + q / qpr * 4);
  }
  auto stash = [&]() {
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      if (u * kResThreads + tid < nq) {
        uint32_t* dst = reinterpret_cast<uint32_t*>(rows_s + to[u]);
#pragma unroll
        for (int k = 0; k < QW; ++k) dst[k] = RAW ? pre[u][k] : walk_bytes(pre[u][k], bb);
      }
    }
  };
  // ordered sums of a finished block (wave 0): lane per (row, class)
  auto sums = [&](int64_t b, const float* vt) {
    const int64_t row0 = b * RB;
    const int nr = (int)(n - row0 < RB ? n - row0 : RB);
    for (int p = lane; p < RB * K; p += 64) {
      const int r = p % RB, k = p / RB;
      if (r >= nr) continue;
      float* o = out + (row0 + r) * K + k;
      const float* v = vt + r * TV;
      float a = *o;
      // tree order; eight loads issued ahead of their sequential adds
      int j = k;
      // (one wave runs this loop, bound by its instruction fetch: starting at
      // 28 of 32 bytes it took 4% more of a call of 16 classes than at 4 .. 16)
      __asm__ volatile(".p2align 6");
      for (; j + 7 * K < T; j += 8 * K) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = v[j + u * K];
#pragma unroll
        for (int u = 0; u < 8; ++u) a = a + x[u];
      }
      for (; j < T; j += K) a = a + v[j];
      *o = a;
    }
  };
  // walkers (waves 1..15): thread w owns row wr = w % RB of every block and
  // the trees wt0, wt0 + G, ... (G = walkers / RB row groups), so no walk
  // divides; the kWalkers - G * RB threads left over idle
  constexpr int kWalkers = kResThreads - 64;
  const int G = kWalkers / RB;  // RB <= 256: G >= 3
  const int wid = tid - 64;
  const bool walker = wid >= 0 && wid < G * RB;
  const int wr = walker ? wid % RB : 0;
  const int wt0 = walker ? wid / RB : 0;
  int64_t b = blockIdx.x;
  if (b < nblk) prefetch(b);
  int64_t prev = -1;
  for (int it = 0; b < nblk; b += gridDim.x, ++it) {
    stash();
    __syncthreads();  // rows of block b (and the tables) in LDS; last walks done
    if (b + gridDim.x < nblk) prefetch(b + gridDim.x);
    float* vt = vals_s + (it & 1) * RB * TV;
    if (tid < 64) {
      if (prev >= 0) sums(prev, vals_s + ((it & 1) ^ 1) * RB * TV);
    } else if (walker) {
      const int64_t row0 = b * RB;
      const int nr = (int)(n - row0 < RB ? n - row0 : RB);
      walk_trees<kResWalks, RAW>(wt0, T, G, wr < nr, lds_addr(rows_s + wr * Sp),
                                 lds_addr(nodes_s), lds_addr(leaves_s), Hi, max_depth,
                                 lds_addr(vt + wr * TV));
    }
    prev = b;
    __syncthreads();  // the walks are done: the row buffer can be refilled
  }
  if (prev >= 0 && tid < 64) {
    // the last block: its table is the one the last iteration wrote
    int it_last = 0;
    for (int64_t bb = blockIdx.x; bb + gridDim.x < nblk; bb += gridDim.x) ++it_last;
    sums(prev, vals_s + (it_last & 1) * RB * TV);
  }
}

template __global__ void predict_resident_kernel<false>(const int8_t*, int64_t, int64_t, int32_t,
                                                        const uint32_t*, const float*, int32_t,
                                                        int32_t, int32_t, int32_t, float*,
                                                        const int32_t*);
template __global__ void predict_resident_kernel<true>(const int8_t*, int64_t, int64_t, int32_t,
                                                       const uint32_t*, const float*, int32_t,
                                                       int32_t, int32_t, int32_t, float*,
                                                       const int32_t*);

// block shape of predict_resident_kernel: 0 when the trees do not fit (raw:
// rows of raw codes, S a multiple of 8; else native rows, S a multiple of 16)
int predict_resident_plan(int64_t n, int64_t S, int32_t K, int32_t H, int32_t n_rounds,
                          int32_t* RB_out, size_t* lds_out, bool raw) {
  constexpr int64_t kBudget = 150 * 1024;
  const int64_t T = (int64_t)n_rounds * K;
  // complete tables: (H - 1) / 2 node words and (H + 1) / 2 values per tree
  if (S % (raw ? 8 : 16) != 0 || S > (1 << 16) || T * H * 4 > 64 * 1024) return 0;
  const int64_t Sp = S + 4;
  // RB rows: the row buffer, two value tables and at most kResMaxQ loads per thread
  int64_t RB = (kBudget - 4 * T * H) / (Sp + 8 * (T + 1));
  RB = std::min<int64_t>(RB, (int64_t)kResMaxQ * kResThreads * 16 / S);
  RB = std::min<int64_t>(RB, 256);
  // whole waves of rows: 65 rows are two passes of the sums' wave and walk
  // groups that straddle waves (1M x 1000 raw codes, 65 / 64 rows a block: 334 / 287
  // us; 300k x 400, 105 / 64 rows: 90 / 86; 300k x 200, 191 / 128 rows: 64 / 61),
  // unless only the larger blocks cover the rows with one on each CU (60k x
  // 250, 40 trees of depth 5, 8 classes, 244 / 192 rows: 25 / 30)
  const int64_t whole = RB - RB % 64;
  if (RB > 64 && !(n <= 256 * RB && n > 256 * whole)) RB = whole;
  if (RB < 8) return 0;
  *RB_out = (int32_t)RB;
  *lds_out = (size_t)(4 * T * H + RB * Sp + 8 * RB * (T + 1));
  return 1;
}

// block shape of predict_rows_kernel: 0 when the trees or rows do not fit
// (then predict_heap_kernel is used)
static int predict_rows_plan(int64_t S, int32_t K, int32_t H, int32_t n_rounds, int32_t* RB_out,
                      int32_t* TC_out, size_t* lds_out) {
  constexpr int64_t kBudget = 64 * 1024;
  // complete tables: (H - 1) / 2 node words and (H + 1) / 2 values per tree
  if (S % 16 != 0 || S > (1 << 16) || (int64_t)4 * H * K > 32 * 1024) return 0;
  const int64_t T = (int64_t)n_rounds * K;
  int64_t m = std::max<int64_t>(1, (16 * 1024) / ((int64_t)4 * H * K));
  int64_t TC = std::min<int64_t>(m * K, std::max<int64_t>(K, (T + K - 1) / K * K));
  const int64_t Sp = S + 4;
  int64_t RB = (kBudget - 4 * TC * H) / (Sp + 4 * (TC + 1));
  RB = std::min<int64_t>(RB, 256);
  RB = std::min<int64_t>(RB, (int64_t)kPredMaxAcc * kPredThreads / K);
  if (RB < 16) return 0;
  *RB_out = (int32_t)RB;
  *TC_out = (int32_t)TC;
  *lds_out = (size_t)(RB * Sp + 4 * TC * H + 4 * RB * (TC + 1));
  return 1;
}

// ---------------------------------------------------------------------------
// Column-block inference (same results as predict_rows_kernel): a workgroup
// holds 256 rows in LDS transposed, word (f, lane) = the code bytes of rows
// lane, lane + 64, lane + 128, lane + 192 at feature f, so a lane reads only
// its own bank whatever features its rows are at, and one word serves four
// rows.  A wave walks one tree for all 256 rows:
//   * the first kColsTop levels are evaluated for every node (the node words
//     are wave-uniform scalar loads): a code byte c goes right at bin b iff c
//     + (127 - b) has bit 7 set, four rows in one add, and each level's bits
//     select among the next level's (bit select) -- 15 word reads and no
//     node reads for 4 rows x 4 levels, where walking takes 32 byte and node
//     reads;
//   * the levels below, and the leaf, are walked row by row: a level's node
//     words are at most 64 consecutive words at the usual depths, so lanes at
//     different nodes read different banks.
// A leaf above the last level, or a tree shallower than kColsTop, continues as
// always-left nodes (complete tables).  Each class's trees are added in tree
// order: with VT = false wave w keeps the sums of classes w, w + waves, ... in
// registers; with VT = true (few classes) the waves share the chunk's trees,
// write each tree's values to LDS and one thread per (row, class) adds them.
// The row-at-a-time walkers take 12 reads a row and tree at depth 6, 39% of the
// LDS's cycles in conflicts of the row bytes; here it is 35 reads and 111 VALU
// instructions for 256 rows, which bound it about equally (2000 trees of depth
// 6 on 1M rows of 100 features: 3.60 -> 1.91 ms).
//   LDS: columns [S + 1][64] words (the last is zero: the always-left node's
//   column), the chunk's tables [TC][GW], values [TC][256] (VT).
// ---------------------------------------------------------------------------
constexpr uint32_t kBit7 = 0x80808080u;

// Per tree: kColsUni words, two top-level nodes each (column << 7 | 127 - bin;
// an always-left node names the zero column S with addend 0), then GW =
// 2^(D' + 1) - 2^kColsTop words, D' = max(D, kColsTop): the nodes below
// (column << 8 | bin; always left: bin 255) by heap index (1-based), and the
// 2^D' leaf values times lr (rounded to float32).
__global__ void cols_tables_kernel(const int32_t* __restrict__ feat,
                                   const int32_t* __restrict__ bin,
                                   const float* __restrict__ leaf, int64_t T, int32_t D,
                                   int32_t DX, int64_t S, float lr, uint32_t* __restrict__ uni,
                                   uint32_t* __restrict__ tab) {
  const int H = (2 << D) - 1;
  const int GW = (2 << DX) - (1 << kColsTop);
  const int per = kColsUni + GW;
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= T * per) return;
  const int64_t t = gid / per;
  const int j = (int)(gid - t * per);
  const int32_t* ft = feat + t * H;
  const bool top = j < kColsUni;
  // node word of heap index g: column and bin (always left: the zero column S
  // and 255)
  auto node = [&](int g, uint32_t& f, uint32_t& b) {
    const int d = 31 - __builtin_clz((unsigned)g);
    bool split = d < D;
    for (int k = 0; k <= d && split; ++k) split = ft[(g >> (d - k)) - 1] >= 0;
    f = (uint32_t)S;
    b = 255u;
    if (split) {
      f = (uint32_t)(ft[g - 1] < S ? ft[g - 1] : S - 1);
      b = (uint32_t)bin[t * H + g - 1] & 0xffu;
    }
  };
  uint32_t f = 0, b = 0;
  if (top) {
    uint32_t w = 0;
    for (int h = 0; h < 2; ++h) {
      const int gt = 2 * j + h + 1;
      if (gt >= (1 << kColsTop)) break;  // padding
      node(gt, f, b);
      // code bytes are at most 128: no byte goes right of a bin above 127
      const uint32_t x = b <= 127u ? f << 7 | (127u - b) : (uint32_t)S << 7;
      w |= x << (16 * h);
    }
    uni[t * kColsUni + j] = w;
    return;
  }
  const int g = j - kColsUni + (1 << kColsTop);
  if (g < (1 << DX)) {
    node(g, f, b);
    tab[t * GW + j - kColsUni] = f << 8 | b;
    return;
  }
  // leaf slot: the first node that is not a split on the path to its ancestor
  // at depth D
  const int h = (g >> (DX - D)) - 1;
  int a = h;
  for (int k = 0; k < D; ++k) {
    const int ak = ((h + 1) >> (D - k)) - 1;
    if (ft[ak] < 0) {
      a = ak;
      break;
    }
  }
  tab[t * GW + j - kColsUni] = __float_as_uint(lr * leaf[t * H + a]);
}

__device__ __forceinline__ uint32_t bit_select(uint32_t m, uint32_t a, uint32_t b) {
  return (m & a) | (~m & b);  // v_bfi_b32
}

template <bool VT>
__global__ __launch_bounds__(1024) void predict_cols_kernel(
    const int8_t* __restrict__ codes, int64_t n, int64_t S, int32_t num_bins,
    const uint32_t* __restrict__ uni, const uint32_t* __restrict__ tab, int32_t T, int32_t K,
    int32_t DX, int32_t TC, float* __restrict__ out, const int32_t* __restrict__ skip) {
  if (skip && *skip) return;  // uniform: the caller's fallback runs instead
  extern __shared__ uint32_t psm[];
  const int GW = (2 << DX) - (1 << kColsTop);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nw = blockDim.x >> 6;
  uint32_t* cols = psm;                        // [S + 1][64]
  uint32_t* tabs = psm + (S + 1) * 64;         // [TC][GW]
  float* vals = reinterpret_cast<float*>(tabs + TC * GW);  // [TC][256] (VT)
  const int64_t row0 = (int64_t)blockIdx.x * kColsRows;
  const uint32_t bb = (uint32_t)num_bins * 0x01010101u;
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  // stage: thread (lane, 16-column group) transposes 4 rows x 16 bytes
  for (int q = wave; q < (int)(S / 16); q += nw) {
    u4 x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t r = row0 + lane + 64 * j;
      x[j] = *(reinterpret_cast<const u4*>(codes + (r < n ? r : n - 1) * S) + q);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      uint32_t y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = walk_bytes(x[j][c], bb);
      const uint32_t l01 = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u);
      const uint32_t h01 = __builtin_amdgcn_perm(y[1], y[0], 0x07030602u);
      const uint32_t l23 = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u);
      const uint32_t h23 = __builtin_amdgcn_perm(y[3], y[2], 0x07030602u);
      uint32_t* d = cols + (16 * q + 4 * c) * 64 + lane;
      d[0] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
      d[64] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
      d[128] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
      d[192] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
    }
  }
  if (tid < 64) cols[S * 64 + tid] = 0u;
  // sums: VT: pair p = m * threads + tid = (row p % 256, class p / 256);
  // else wave's class slot m, rows lane + 64 j at [4 m + j]
  float acc[kColsMaxAcc];
#pragma unroll
  for (int m = 0; m < kColsMaxAcc; ++m) {
    const int p = m * (int)blockDim.x + tid;
    const int64_t r = VT ? row0 + (p & 255) : row0 + lane + 64 * (m & 3);
    const int k = VT ? p >> 8 : wave + (m >> 2) * nw;
    acc[m] = (k < K && r < n) ? out[r * K + k] : 0.0f;
  }
  const uint8_t* cols8 = reinterpret_cast<const uint8_t*>(cols);
  const uint32_t lane4 = (uint32_t)lane * 4u;
  // the values of tree t (table at LDS words tb) for the lane's four rows
  auto walk = [&](int t, const uint32_t* tb, float (&v)[4]) {
    const uint32_t* __restrict__ u = uni + (int64_t)t * kColsUni;
    uint32_t s[15];
#pragma unroll
    for (int i = 0; i < 15; ++i) {
      const uint32_t w = (u[i >> 1] >> (16 * (i & 1))) & 0xffffu;
      const uint32_t c = *reinterpret_cast<const uint32_t*>(cols8 + (((w >> 7) << 8) + lane4));
      s[i] = c + (w & 0x7fu) * 0x01010101u;
    }
    // bit 7 of each byte: the way at level 0, 1, 2, 3 of that row's path
    const uint32_t s0 = s[0];
    const uint32_t s1 = bit_select(s0, s[2], s[1]);
    const uint32_t s2 = bit_select(s0, bit_select(s1, s[6], s[5]), bit_select(s1, s[4], s[3]));
    const uint32_t s3 = bit_select(
        s0,
        bit_select(s1, bit_select(s2, s[14], s[13]), bit_select(s2, s[12], s[11])),
        bit_select(s1, bit_select(s2, s[10], s[9]), bit_select(s2, s[8], s[7])));
    // heap index 16 + path of each row, one byte each
    const uint32_t g4 = 0x10101010u | ((s0 & kBit7) >> 4) | ((s1 & kBit7) >> 5) |
                        ((s2 & kBit7) >> 6) | ((s3 & kBit7) >> 7);
    uint32_t g[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) g[j] = (g4 >> (8 * j)) & 0xffu;
    for (int d = kColsTop; d < DX; ++d) {
      uint32_t w[4], c[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = tb[(int)g[j] - (1 << kColsTop)];
#pragma unroll
      for (int j = 0; j < 4; ++j) c[j] = cols8[(w[j] & 0xffffff00u) | (lane4 + (uint32_t)j)];
#pragma unroll
      for (int j = 0; j < 4; ++j) g[j] = 2u * g[j] + (c[j] > (w[j] & 0xffu) ? 1u : 0u);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(tb[(int)g[j] - (1 << kColsTop)]);
  };
  for (int t0 = 0; t0 < T; t0 += TC) {
    const int tc = T - t0 < TC ? T - t0 : TC;
    __syncthreads();  // columns staged / the previous chunk's tables done with
    {
      const u4* src = reinterpret_cast<const u4*>(tab + (int64_t)t0 * GW);  // GW % 4 == 0
      u4* dst = reinterpret_cast<u4*>(tabs);
      for (int i = tid; i < tc * GW / 4; i += blockDim.x) dst[i] = src[i];
    }
    __syncthreads();
    if constexpr (VT) {
      for (int j = wave; j < tc; j += nw) {
        float v[4];
        walk(t0 + j, tabs + j * GW, v);
#pragma unroll
        for (int i = 0; i < 4; ++i) vals[j * kColsRows + lane + 64 * i] = v[i];
      }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < kColsMaxAcc; ++m) {
        const int p = m * (int)blockDim.x + tid;
        const int k = p >> 8;
        if (k < K) {  // (t0 is a multiple of K)
          float a = acc[m];
          for (int j = k; j < tc; j += K) a = a + vals[j * kColsRows + (p & 255)];
          acc[m] = a;
        }
      }
    } else {
#pragma unroll
      for (int m = 0; m < kColsMaxAcc / 4; ++m) {
        for (int j = wave + m * nw; j < tc && wave + m * nw < K; j += K) {
          float v[4];
          walk(t0 + j, tabs + j * GW, v);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[4 * m + i] = acc[4 * m + i] + v[i];
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < kColsMaxAcc; ++m) {
    const int p = m * (int)blockDim.x + tid;
    const int64_t r = VT ? row0 + (p & 255) : row0 + lane + 64 * (m & 3);
    const int k = VT ? p >> 8 : wave + (m >> 2) * nw;
    if (k < K && r < n) out[r * K + k] = acc[m];
  }
}
template __global__ void predict_cols_kernel<false>(const int8_t*, int64_t, int64_t, int32_t,
                                                    const uint32_t*, const uint32_t*, int32_t,
                                                    int32_t, int32_t, int32_t, float*,
                                                    const int32_t*);
template __global__ void predict_cols_kernel<true>(const int8_t*, int64_t, int64_t, int32_t,
                                                   const uint32_t*, const uint32_t*, int32_t,
                                                   int32_t, int32_t, int32_t, float*,
                                                   const int32_t*);

// block shape of predict_cols_kernel: waves, trees per chunk, whether values go
// through LDS; 0 when a chunk of one round does not fit
static int predict_cols_plan(int64_t S, int32_t K, int32_t D, int32_t n_rounds, int32_t* DX_out,
                      int32_t* waves_out, int32_t* TC_out, bool* vt_out, size_t* lds_out) {
  const int32_t DX = std::max(D, kColsTop);
  if (S % 16 != 0 || DX > 8 || S > 511) return 0;
  const int64_t GW = (int64_t(2) << DX) - (1 << kColsTop);
  const bool vt = K < 8;
  if (K > 16 * (kColsMaxAcc / 4)) return 0;
  const int64_t colb = (S + 1) * 256, per = 4 * GW + (vt ? 4 * kColsRows : 0);
  // tables of about 24 KB (48 KB with values) a chunk, in whole rounds
  int64_t rounds = std::max<int64_t>(1, (vt ? 48 : 24) * 1024 / (per * K));
  rounds = std::min<int64_t>(rounds, n_rounds);
  while (rounds > 1 && colb + rounds * K * per > 156 * 1024) --rounds;
  const int64_t lds = colb + rounds * K * per;
  if (lds > 156 * 1024) return 0;
  // waves: a class each, or 16 sharing the trees
  int32_t waves = 16;
  if (!vt) {
    const int32_t per_wave = (K + 15) / 16;
    waves = (K + per_wave - 1) / per_wave;
  }
  *DX_out = DX;
  *waves_out = waves;
  *TC_out = (int32_t)(rounds * K);
  *vt_out = vt;
  *lds_out = (size_t)lds;
  return 1;
}

// ---------------------------------------------------------------------------
// Which kernel a call of wgbm_predict_heap takes.
// ---------------------------------------------------------------------------
// More rows than one block of the column-block predictor on every CU, and two of
// its workgroups on a CU: it is taken.  1M x 100, 32 bins, us with the row
// walkers / with it: 2000 trees of depth 6, 10 classes 3600 / 1910; 100 trees, one
// class: depth 6 239 / 169, depth 5 213 / 136, depth 3 161 / 128; 200k x 300, 3
// classes, 300 trees of depth 8 430 / 243.
//
// Otherwise its time is that of one block, whatever the row count (or of as many
// as a CU gets): a class's trees one after the other, or a sixteenth of all
// trees.  The other kernels cut their row blocks smaller the more trees there are
// and fill the CUs (500 rows, 1700 trees of depth 1, 17 classes: 14 us against
// 118; 912 rows, 47 trees of depth 1: 14 / 11; 200k x 300, 100 trees of depth 5:
// 64 / 81), but lose to it where trees are few for the rows or deep (4000 rows,
// 120 trees of depth 8, 3 classes: 61 / 36).  So the times of both are estimated
// and the smaller is taken.  The estimates (us) were fitted to 7920 measured
// shapes (300 .. 300k rows, rows of 32 .. 384 bytes, 1 .. 32 classes, depths 0 ..
// 8, 2 .. 200 rounds): half of them within 5%, nine of ten within 16%; the
// kernel taken is on average 0.3% slower than the better of the two, less than
// 10% in 99 of 100 shapes.  Always taking it lost 5% or more in a quarter of them.
struct PredictSizes {
  int64_t n, S, K, R, T, H;
  int D;
  int64_t RB, TC;
};
static double ceil_div(int64_t a, int64_t b) { return (double)((a + b - 1) / b); }
// blocks of rows that a CU gets, one after the other
static double blocks_per_cu(int64_t n, int64_t rows) {
  return ceil_div((n + rows - 1) / rows, 256);
}
// rows of a wave that start on one LDS bank, but for the first
static double lds_conflicts(int64_t stride) {
  int64_t g = 64;
  while (stride % g) g /= 2;
  return (double)(g - 1);
}

static double est_cols(const PredictSizes& p, const PredictPlan& c) {
  const double below = c.DX - kColsTop;  // levels walked row by row
  const int64_t GW = (int64_t(2) << c.DX) - (1 << kColsTop);
  const double chunks = ceil_div(p.T, c.TC), blocks = blocks_per_cu(p.n, kColsRows);
  if (c.vt)
    return 5.1 + blocks * (ceil_div(p.T, 16) * (0.55 + 0.283 * below) +
                           0.030 * p.R * ceil_div(p.K, 4) + 1.18 * chunks + 0.0101 * p.S);
  return 7.0 + blocks * (p.R * ceil_div(p.K, c.waves) * (0.317 + 0.155 * below + 0.0281 * c.waves) +
                         chunks * (0.316 + 0.12 * (c.TC * GW / 1024.0)) + 0.0109 * p.S);
}

static double est_resident(const PredictSizes& p) {
  const int64_t G = 960 / p.RB;  // as the kernel's walkers
  const double conf = lds_conflicts(p.T + 1);
  const double walk = ceil_div((p.T + G - 1) / G, 2) * (0.378 + 0.068 * p.D + 0.0218 * conf);
  const double sums = ceil_div(p.RB * p.K, 64) * (0.28 + p.R * (0.0145 + 0.00068 * conf));
  return 6.1 + 0.586 * (p.T * p.H / 1024.0) + 0.069 * sums +
         blocks_per_cu(p.n, p.RB) * (std::max(walk, sums) + 0.39 * (p.RB * p.S / 16384.0));
}

static double est_rows(const PredictSizes& p) {
  const int64_t G = std::max<int64_t>(1, 1024 / p.RB);
  const double conf = 0.00435 * lds_conflicts(p.TC + 1);
  const double chunk = 0.687 + ceil_div((p.TC + G - 1) / G, 2) * (0.213 + 0.088 * p.D + 2 * conf) +
                       ceil_div(p.RB * p.K, 1024) * p.TC / p.K * conf +
                       0.254 * (p.TC * p.H / 1024.0);
  return 7.0 + 0.216 * (p.RB * p.S / 16384.0) +
         ceil_div(p.T, p.TC) * chunk * (1.0 + 0.52 * (blocks_per_cu(p.n, p.RB) - 1.0));
}

// a thread per (row, class), a dependent load a level: from the L2 while the
// tables fit it, and past ~2^17 threads bound by their number
static double est_heap(const PredictSizes& p) {
  const double mb = (double)p.T * p.H * 12 / (1 << 20);
  const double step = 0.24 + 0.33 * std::min(std::max((mb - 4.5) / 3.0, 0.0), 1.0);
  return 5.0 + p.R * (p.D + 1) *
                   std::max(step, (0.8 + 0.24 * p.D) * 1e-6 * (double)p.n * (double)p.K);
}

PredictPlan predict_plan(int64_t n, int64_t S, bool aligned16, int32_t K, int32_t D,
                         int32_t n_rounds) {
  PredictPlan o;
  const int32_t H = (int32_t)((int64_t(2) << D) - 1);
  if (predict_resident_plan(n, S, K, H, n_rounds, &o.RB, &o.lds))
    o.kind = kPredictResident;
  else if (predict_rows_plan(S, K, H, n_rounds, &o.RB, &o.TC, &o.lds))
    o.kind = kPredictRows;
  PredictPlan c;
  c.kind = kPredictCols;
  if (!aligned16 || !predict_cols_plan(S, K, D, n_rounds, &c.DX, &c.waves, &c.TC, &c.vt, &c.lds))
    return o;
  if (n > 255 * kColsRows && c.lds <= 80 * 1024) return c;
  const PredictSizes p{n, S, K, n_rounds, (int64_t)n_rounds * K, H, D, o.RB, o.TC};
  const double other = o.kind == kPredictResident ? est_resident(p)
                       : o.kind == kPredictRows   ? est_rows(p)
                                                  : est_heap(p);
  // over several blocks a CU the estimates lean to the row blocks by 10% and
  // to the column blocks by 5% where the trees are resident
  const double lean = n <= 255 * kColsRows ? 1.0 : o.kind == kPredictResident ? 0.95 : 1.1;
  return est_cols(p, c) < lean * other ? c : o;
}

// in-place row softmax over K logits: exp(x - max) / sum, sequential in k
// (up to kSoftmaxLds classes: a workgroup's 256 rows are one contiguous run,
// moved through LDS with coalesced loads and stores; a thread per row straight
// from memory touches 64 lines per load and read each row three times: 83 ->
// 26 us for 1M rows of 10 classes)
__global__ __launch_bounds__(256) void softmax_rows_kernel(float* __restrict__ x, int64_t n,
                                                           int32_t K) {
  extern __shared__ float xs[];  // [256][K | 1], staged rows
  const int64_t i0 = (int64_t)blockIdx.x * 256;
  const int64_t i = i0 + threadIdx.x;
  const bool staged = K <= kSoftmaxLds;
  const int ks = K | 1;  // odd: the rows of a wave start in different banks
  const int64_t left = n - i0;
  const int words = (int)(left < 256 ? left : 256) * K;
  if (staged) {
    for (int w = threadIdx.x; w < words; w += 256) xs[w / K * ks + w % K] = x[i0 * K + w];
    __syncthreads();
  }
  if (i < n) {
    float* r = staged ? xs + threadIdx.x * ks : x + i * K;
    float m = r[0];
    for (int k = 1; k < K; ++k) m = r[k] > m ? r[k] : m;
    float s = 0.0f;
    for (int k = 0; k < K; ++k) {
      const float e = wgbm_expf(r[k] - m);
      r[k] = e;
      s = s + e;
    }
    for (int k = 0; k < K; ++k) r[k] = r[k] / s;
  }
  if (staged) {
    __syncthreads();
    for (int w = threadIdx.x; w < words; w += 256) x[i0 * K + w] = xs[w / K * ks + w % K];
  }
}

// ---------------------------------------------------------------------------
// per-era split-gain importance (warpgbm/core.py:624-627): every internal node
// adds its per-era gains to acc[e][feature] with one float32 add per era, the
// nodes in the order the reference visits them.  node / fstart: the gain rows
// of the nodes grouped by feature (group f = node[fstart[f] .. fstart[f+1]),
// in visiting order), so each (feature, era) word is one thread's sequential
// sum and no two threads touch the same word.
// ---------------------------------------------------------------------------
__global__ void importance_add_kernel(float* __restrict__ acc, int32_t F, int32_t E,
                                      const float* __restrict__ gain,
                                      const int64_t* __restrict__ node,
                                      const int64_t* __restrict__ fstart) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (int64_t)F * E) return;
  const int f = (int)(gid / E), e = (int)(gid - (int64_t)f * E);
  float* w = acc + (int64_t)e * F + f;
  float s = *w;
  const int64_t i1 = fstart[f + 1];
  int64_t i = fstart[f];
  // batches of 16 gathers in flight ahead of their (sequential) adds, the
  // node indices of the next batch loaded with this batch's gains (one
  // memory round trip per batch; a feature can hold thousands of nodes)
  constexpr int U = 16;
  int64_t nx[U];
  if (i + U <= i1) {
#pragma unroll
    for (int u = 0; u < U; ++u) nx[u] = node[i + u];
  }
  for (; i + U <= i1; i += U) {
    float g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) g[u] = gain[nx[u] * E + e];
    if (i + 2 * U <= i1) {
#pragma unroll
      for (int u = 0; u < U; ++u) nx[u] = node[i + U + u];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) s = s + g[u];
  }
  for (; i < i1; ++i) s = s + gain[node[i] * E + e];
  *w = s;
}

}  // namespace wgbm
