// Ensemble prediction (est:863-884) with the rows' codes and the trees in
// LDS: every row walks every tree of its class, and lr * value of the leaves
// is added tree by tree from 0.0.
//
// What bounds it.  A step of a walk is a code byte and a node word from LDS
// and a few vector instructions, each step waiting for the one before it.
// The chip is full when a SIMD holds enough independent walks to hide that
// chain, and then the step's own instructions are the bound:
//   - a node is one 32-bit word (below) whose fields are LDS offsets, so that
//     a step is four vector instructions and two LDS reads;
//   - trees are renumbered breadth first (k_walk_pack), the children of a
//     node side by side: a level's nodes are neighbours, and the 64 lanes of
//     a wave read distinct LDS banks on levels of up to 64 nodes;
//   - leaves point to themselves with a threshold that no code exceeds, so
//     all walks of a tree take the same number of steps and no lane is masked
//     (deep trees: until all walks of a wave are at leaves, kDeepSteps);
//   - the root and its children come from one broadcast read, which takes
//     the first two levels' node reads off the chain;
//   - a lane walks kRpl rows through kTpl trees at once.  With four
//     neighbouring rows per lane (kRpl = 4) every lane's codes lie in its own
//     bank: no conflicts, and one 32-bit read gives the root codes of all four.
//     Smaller inputs spread one row per lane over more waves (kRpl = 1) and
//     take eight trees at a time instead.
// LDS reads then set the rate, about four clocks each per CU: 7 clocks per
// wave and step at 28 columns.  Measured (125-node trees of depth 6): 1M rows
// x 28 columns x 100 trees 117 us, where lanes that stopped at their leaf and
// column-strided codes (23 clocks a step) took 357; 100,000 rows x 100 columns
// x 300 trees 68 us (k_walk_split), 673 with the walk in HBM.
//
// A tree's node slots are a power of two: the root in slot 0, its number of
// levels in slot 1's word (own slots: in the upper half the slot of the tree
// kTpl trees on), pairs of children from slot 2 on; trees never cross a window
// of 1 << kWin bytes.  Node word:
//   bits 2 .. kWin - 1  the left child's byte offset in the window (a
//                       multiple of 8, so the right child's is "or 4")
//   bits kWin .. 23     the column
//   bits 24 .. 31       threshold: a code above it goes right
#include "kernels.h"

#include <hip/hip_ext.h>

#include <algorithm>

namespace bsscl {

namespace {

constexpr int kGroupNodes = kWalkGroupSlots;
static_assert(kWalkMaxNodes == kGroupNodes - 1, "slot 1 of a tree holds no node");
constexpr int kValsAt = kGroupNodes * 4;  // LDS byte offsets
constexpr int kCodesAt = kValsAt + kGroupNodes * 8;

// Trees deeper than kDeepSteps are grown on one side, and most rows end far
// above their deepest leaf: waves look whether all their walks have ended,
// first after kFreeSteps and then every kCheckSteps (a look costs about half a
// step).  1M rows through 100 chains of 62 splits: 287 us, 979 without; 1,000
// rows through 20 chains of 511 29 and 714.  Ensembles of trees grown at
// random lose up to 4% by looking with 62 or 127 splits (16 and 20 levels) and
// win 10% at 1M rows with 255 (21).  The depth comes from k_walk_pack: in the
// host's checks it cost 10 us for 37,500 nodes.
constexpr int kDeepSteps = 20, kFreeSteps = 10, kCheckSteps = 4;

// Windows of 256 slots, and of 1024 for trees that need more.
constexpr int kWinSmall = 10, kWinLarge = 12;
static_assert(kGroupNodes * 4 == 1 << kWinLarge, "a group is at most one large window");

// LDS by byte offset (the kernel has dynamic LDS only, which starts at 0).
template <typename T>
__device__ __forceinline__ T lds_get(uint32_t at) {
  return *(const __attribute__((address_space(3))) T *)(size_t)at;
}
template <typename T>
__device__ __forceinline__ void lds_put(uint32_t at, T v) {
  *(__attribute__((address_space(3))) T *)(size_t)at = v;
}
using Quad = __attribute__((ext_vector_type(4))) uint32_t;

}  // namespace

// One wave per entry: tree s is nodes [first[s], first[s] + count[s]) of
// `nodes` (a child's index is relative to first[s]) and goes to slot dest[s].
// count 0 is padding: one leaf of value 0.0, which adds +0.0 to a sum that is
// never -0.0.  A tree that is a single leaf gets a root over two copies of it.
// The host has checked that the nodes form a tree, so no slot past count[s]
// is reached.
__global__ __launch_bounds__(64) void k_walk_pack(
    const TreeNodeDev *__restrict__ nodes, const int32_t *__restrict__ first,
    const int32_t *__restrict__ count, const int32_t *__restrict__ dest,
    const uint8_t *__restrict__ remap, double lr, int32_t win, int32_t link,
    uint32_t *__restrict__ words, double *__restrict__ vals, int32_t *__restrict__ depth) {
  __shared__ int32_t order[kGroupNodes];
  const int32_t s = (int32_t)blockIdx.x, lane = (int32_t)threadIdx.x;
  const TreeNodeDev *tree = nodes + first[s];
  const int32_t cnt = count[s], slot = cnt + 1, to = dest[s];
  uint32_t *w = words + to;
  double *v = vals + to;
  // The tree's byte offset in its window.
  const uint32_t base = ((uint32_t)to * 4u) & ((1u << win) - 1u);
  // (Read only when that tree lies in the same group.)
  const uint32_t on = link > 0 && s + link < (int32_t)gridDim.x
                          ? (uint32_t)(dest[s + link] & (kGroupNodes - 1)) << 16
                          : 0u;
  if (cnt <= 0 || tree[0].feature < 0) {
    if (lane < 4) {
      // The root and both leaves: always left, to the left leaf.
      w[lane] = lane == 1 ? on | 1u : (255u << 24) | (base + 8u);
      v[lane] = cnt > 0 ? __dmul_rn(lr, tree[0].value) : 0.0;
    }
    return;
  }
  if (lane == 0) order[0] = 0;
  int32_t lo = 0, hi = 1, next = 2, d = 0;
  __syncthreads();
  while (lo < hi) {
    const int32_t level_end = next;
    for (int32_t i0 = lo; i0 < hi; i0 += 64) {
      const int32_t i = i0 + lane;
      const bool in = i < hi;
      TreeNodeDev nd;
      nd.feature = -1;
      if (in) nd = tree[order[i]];
      const unsigned long long split = __ballot(in && nd.feature >= 0);
      const int32_t pair = next + 2 * __popcll(split & ((1ull << lane) - 1ull));
      next += 2 * __popcll(split);
      if (in) {
        uint32_t word = (255u << 24) | (base + 4u * (uint32_t)i);  // a leaf: to itself
        if (nd.feature >= 0 && pair + 1 < slot) {
          // Threshold -1 sends every row right: the children change places
          // and every row goes left.
          const bool none = nd.threshold < 0;
          order[pair] = none ? nd.right : nd.left;
          order[pair + 1] = none ? nd.left : nd.right;
          const uint32_t thr = none ? 255u : (uint32_t)min(nd.threshold, 255);
          const uint32_t col = (uint32_t)remap[nd.feature];
          word = (thr << 24) | (col << win) | (base + 4u * (uint32_t)pair);
        }
        w[i] = word;
        v[i] = __dmul_rn(lr, nd.value);
      }
    }
    next = min(next, slot);
    lo = max(hi, 2);
    hi = next;
    if (level_end < next) ++d;
    __syncthreads();
  }
  if (lane == 0) {
    w[1] = on | (uint32_t)d;
    if (d > kDeepSteps) atomicMax(depth, d);
  }
}

#pragma clang fp contract(off)
template <int kRpl, int kTpl, int kTileLog2, int kWin, bool kDeep, bool kProba>
__device__ __forceinline__ void walk_rows(const WalkArgs &a) {
  constexpr int kTile = 1 << kTileLog2, kThreads = kTile / kRpl;
  constexpr int kWordLoads = kGroupNodes / 4 / kThreads, kValLoads = kGroupNodes / 2 / kThreads;
  constexpr uint32_t kChildMask = (1u << kWin) - 4u;
  constexpr uint32_t kColMask = 0xFFFFFFu & ~((1u << kWin) - 1u);
  const int tid = (int)threadIdx.x;
  const int32_t cls = (int32_t)blockIdx.y;
  const int64_t row0 = (int64_t)blockIdx.x * kTile;
  // The tile's codes, column by column.  (16-row runs past ld, the last
  // column's padding, are never read: rows there are >= n.  Rows from n on
  // hold any code; their walks stay in their trees.)
  for (int k = tid; k < a.n_cols * (kTile / 16); k += kThreads) {
    const int c = k / (kTile / 16), ch = k % (kTile / 16);
    const int64_t r = row0 + 16 * ch;
    const int64_t col = a.cols[c];
    if (r < a.ld)
      lds_put(kCodesAt + (c << kTileLog2) + 16 * ch,
              *reinterpret_cast<const Quad *>(a.codes + col * a.ld + r));
  }
  // Trees too large for eight at a time lie in slots of their own size, so
  // that small ones beside them do not fill a group each (their groups are
  // numbered, g0; else g0 is a group's first entry).  With the largest tree's
  // slots for all: 1M rows through one tree of 511 splits and 2,000 stumps
  // 4.7 ms, 0.95 so; 1,000 rows through 10 of 511 and 290 of 7 159 us and 78;
  // trees of one size are level to 4% slower.
  constexpr bool kOwn = kRpl == 1 && kTpl < 8;
  const int32_t t_end = a.ranges[2 * cls + 1];
  int32_t g0 = a.ranges[2 * cls];
  const uint32_t lane_at = (uint32_t)(tid * kRpl);
  auto code_at = [&](uint32_t w) {
    return ((w & kColMask) >> (kWin - kTileLog2)) | lane_at;
  };
  // The next group's words and values wait in registers while a group is
  // walked.
  Quad pw[kWordLoads], pv[kValLoads];
  int32_t cnt = 0;  // own slots: the group's record
  auto prefetch = [&]() {
    cnt = kOwn ? a.groups[g0] : min(a.per_group, t_end - g0);
    const int nw = kOwn ? kGroupNodes / 4 : cnt * a.slot / 4, nv = 2 * nw;
    const int64_t from = kOwn ? (int64_t)g0 * kGroupNodes : (int64_t)g0 * a.slot;
    const Quad *sw = reinterpret_cast<const Quad *>(a.words + from);
    const Quad *sv = reinterpret_cast<const Quad *>(a.vals + from);
#pragma unroll
    for (int q = 0; q < kWordLoads; ++q)
      if (tid + q * kThreads < nw) pw[q] = sw[tid + q * kThreads];
#pragma unroll
    for (int q = 0; q < kValLoads; ++q)
      if (tid + q * kThreads < nv) pv[q] = sv[tid + q * kThreads];
  };
  double F[kRpl];
#pragma unroll
  for (int r = 0; r < kRpl; ++r) F[r] = 0.0;
  if (g0 < t_end) prefetch();
  while (g0 < t_end) {
    const int32_t here = kOwn ? cnt & 0xffff : cnt;
    uint32_t next_at[kTpl];  // own slots: where the next trees start
    next_at[0] = 0u;
    if constexpr (kTpl > 1) next_at[1] = here > 1 ? (uint32_t)cnt >> 16 : 0u;
    const int nw = kOwn ? kGroupNodes / 4 : here * a.slot / 4, nv = 2 * nw;
    __syncthreads();  // the previous group's walks are done
#pragma unroll
    for (int q = 0; q < kWordLoads; ++q)
      if (tid + q * kThreads < nw) lds_put(16 * (tid + q * kThreads), pw[q]);
#pragma unroll
    for (int q = 0; q < kValLoads; ++q)
      if (tid + q * kThreads < nv) lds_put(kValsAt + 16 * (tid + q * kThreads), pv[q]);
    __syncthreads();
    g0 += kOwn ? 1 : a.per_group;
    if (g0 < t_end) prefetch();
    for (int32_t t = 0; t < here; t += kTpl) {
      int32_t steps = 2;
      uint32_t w[kTpl][kRpl], p[kTpl][kRpl], win[kTpl];
#pragma unroll
      for (int j = 0; j < kTpl; ++j) {
        const uint32_t at = kOwn ? next_at[j] * 4u : (uint32_t)((t + j) * a.slot * 4);
        win[j] = at & ~((1u << kWin) - 1u);
        const Quad top = lds_get<Quad>(at);  // root, levels, left and right child
        const int32_t top_y = __builtin_amdgcn_readfirstlane((int)top.y);
        steps = max(steps, kOwn ? top_y & 0xffff : top_y);
        if constexpr (kOwn) {
          // (After the last tree: the first of this step's again; an odd
          // last one is walked beside another and added alone.)
          next_at[j] = t + kTpl + j < here ? (uint32_t)top_y >> 16 : next_at[0];
        }
        const uint32_t thr = top.x >> 24;
        uint32_t c4;
        if constexpr (kRpl == 4) c4 = lds_get<uint32_t>(kCodesAt + code_at(top.x));
        else c4 = lds_get<uint8_t>(kCodesAt + code_at(top.x));
#pragma unroll
        for (int r = 0; r < kRpl; ++r) {
          const uint32_t code = kRpl == 4 ? (c4 >> (8 * r)) & 255u : c4;
          w[j][r] = code > thr ? top.w : top.z;
        }
      }
      // (Trees of one level take a second step, which their leaves' words
      // turn back to themselves.)
      auto step = [&]() {
#pragma unroll
        for (int j = 0; j < kTpl; ++j)
#pragma unroll
          for (int r = 0; r < kRpl; ++r)
            p[j][r] = lds_get<uint8_t>(kCodesAt + code_at(w[j][r]) + r);
        // (Every walk's read is issued before the first is waited for; the
        // scheduler otherwise saves registers instead: 5-8% slower.)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kTpl; ++j)
#pragma unroll
          for (int r = 0; r < kRpl; ++r) {
            const uint32_t code = p[j][r];
            p[j][r] = (w[j][r] & kChildMask) | (code > (w[j][r] >> 24) ? win[j] + 4u : win[j]);
          }
      };
      int32_t d = 2, stop = kDeep ? min(steps, kFreeSteps) : steps;
      while (true) {
        for (; d < stop; ++d) {
          step();
#pragma unroll
          for (int j = 0; j < kTpl; ++j)
#pragma unroll
            for (int r = 0; r < kRpl; ++r) w[j][r] = lds_get<uint32_t>(p[j][r]);
        }
        if (!kDeep || d >= steps) break;
        // (A leaf's word leads to itself.)
        bool on = false;
#pragma unroll
        for (int j = 0; j < kTpl; ++j)
#pragma unroll
          for (int r = 0; r < kRpl; ++r) on = on || win[j] + (w[j][r] & kChildMask) != p[j][r];
        if (!__any(on)) break;
        stop = min(steps, stop + kCheckSteps);
      }
      step();
#pragma unroll
      for (int j = 0; j < kTpl; ++j)
#pragma unroll
        for (int r = 0; r < kRpl; ++r)
          if (!kOwn || j == 0 || t + j < here)
            F[r] = __dadd_rn(F[r], lds_get<double>(kValsAt + 2 * p[j][r]));
    }
  }
#pragma unroll
  for (int r = 0; r < kRpl; ++r) {
    const int64_t i = row0 + lane_at + r;
    if (i >= a.n) continue;
    if constexpr (kProba) a.proba[i] = binary_proba(F[r], a.base_score);
    else a.out[cls * a.out_stride + i] = F[r];
  }
}
#pragma clang fp contract(on)

template <int kRpl, int kTpl, int kTileLog2, int kWin, bool kProba>
__global__ __launch_bounds__((1 << kTileLog2) / kRpl) void k_walk(WalkArgs a) {
  if (*a.depth > kDeepSteps) walk_rows<kRpl, kTpl, kTileLog2, kWin, true, kProba>(a);
  else walk_rows<kRpl, kTpl, kTileLog2, kWin, false, kProba>(a);
}

// The walk of few rows: the kSplitWaves waves of a block take 64 rows through
// eight trees each at a time, so a request of some rows is not one wave's
// walk of every tree (28 columns, 100 trees: 11 us at 64 rows, 27 in k_walk's
// blocks; where rows and classes alone fill the chip: kWalkSplitRows).
// The leaves' values wait in LDS, in place of the words they were reached
// by, and the first wave adds them in tree order.
constexpr int kSplitWaves = 8, kSplitTrees = 8 * kSplitWaves;

#pragma clang fp contract(off)
template <bool kProba>
__global__ __launch_bounds__(64 * kSplitWaves) void k_walk_split(WalkArgs a) {
  constexpr int kWin = kWinSmall, kTpl = 8;
  constexpr uint32_t kChildMask = (1u << kWin) - 4u;
  constexpr uint32_t kColMask = 0xFFFFFFu & ~((1u << kWin) - 1u);
  constexpr int kWaveBytes = kGroupNodes * 4;  // words of eight trees; then [8][64] values
  constexpr int kCodes = kSplitWaves * kWaveBytes;
  static_assert(kTpl * 64 * 8 <= kWaveBytes, "the values fit in place of the words");
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const int32_t cls = (int32_t)blockIdx.y;
  const int64_t row0 = (int64_t)blockIdx.x * 64;
  for (int k = (int)threadIdx.x; k < a.n_cols * 4; k += 64 * kSplitWaves) {
    const int64_t col = a.cols[k >> 2];
    lds_put(kCodes + 16 * k,
            *reinterpret_cast<const Quad *>(a.codes + col * a.ld + row0 + 16 * (k & 3)));
  }
  const uint32_t mine = (uint32_t)(wave * kWaveBytes);
  auto code_at = [&](uint32_t w) {
    return kCodes + (((w & kColMask) >> (kWin - 6)) | (uint32_t)lane);
  };
  const int32_t t_end = a.ranges[2 * cls + 1];
  double F = 0.0;
  for (int32_t g = a.ranges[2 * cls]; g < t_end; g += kSplitTrees) {
    // This wave's trees: slots [t0, t0 + nt), nt a multiple of kTpl or 0.  A
    // tree's words are relative to its window, and a group of trees starts
    // at a window.
    const int32_t t0 = g + wave * kTpl;
    const bool any = t0 < t_end;
    uint32_t p[kTpl];
    if (any) {
      const Quad *src = reinterpret_cast<const Quad *>(a.words + (int64_t)t0 * a.slot);
      const int nq = kTpl * a.slot / 4;
      for (int q = lane; q < nq; q += 64) lds_put(mine + 16 * q, src[q]);
    }
    __syncthreads();
    if (any) {
      int32_t steps = 2;
      uint32_t w[kTpl], win[kTpl];
      // Where the wave's trees start in their first window.
      const uint32_t lead = ((uint32_t)(t0 % a.per_group) * (uint32_t)a.slot * 4u) &
                            ((1u << kWin) - 1u);
#pragma unroll
      for (int j = 0; j < kTpl; ++j) {
        const uint32_t at = (uint32_t)(j * a.slot * 4);
        win[j] = mine + ((lead + at) & ~((1u << kWin) - 1u)) - lead;
        const Quad top = lds_get<Quad>(mine + at);
        steps = max(steps, __builtin_amdgcn_readfirstlane((int)top.y));
        w[j] = lds_get<uint8_t>(code_at(top.x)) > (top.x >> 24) ? top.w : top.z;
      }
      for (int32_t d = 1; d < steps; ++d) {
#pragma unroll
        for (int j = 0; j < kTpl; ++j) p[j] = lds_get<uint8_t>(code_at(w[j]));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kTpl; ++j)
          p[j] = win[j] + ((w[j] & kChildMask) | (p[j] > (w[j] >> 24) ? 4u : 0u));
        if (d + 1 < steps) {
#pragma unroll
          for (int j = 0; j < kTpl; ++j) w[j] = lds_get<uint32_t>(p[j]);
        }
      }
      double v[kTpl];
#pragma unroll
      for (int j = 0; j < kTpl; ++j)
        v[j] = a.vals[(int64_t)t0 * a.slot + (p[j] - mine) / 4];
      // (The wave's own words are read no more.)
#pragma unroll
      for (int j = 0; j < kTpl; ++j) lds_put(mine + (uint32_t)(j * 64 + lane) * 8, v[j]);
    }
    __syncthreads();
    if (wave == 0) {
      const int32_t nt = min(t_end - g, kSplitTrees);
      for (int32_t t = 0; t < nt; t += kTpl) {
#pragma unroll
        for (int j = 0; j < kTpl; ++j)
          F = F + lds_get<double>((uint32_t)(t / kTpl * kWaveBytes + (j * 64 + lane) * 8));
      }
    }
    __syncthreads();
  }
  const int64_t i = row0 + lane;
  if (wave == 0 && i < a.n) {
    if constexpr (kProba) a.proba[i] = binary_proba(F, a.base_score);
    else a.out[cls * a.out_stride + i] = F;
  }
}
#pragma clang fp contract(on)

bool walk_plan(int64_t n, int32_t K, int32_t n_cols, int32_t max_nodes, WalkPlan *plan) {
  if (n_cols < 1 || n_cols > kWalkMaxCols || max_nodes > kWalkMaxNodes) return false;
  WalkPlan &p = *plan;
  p.slot = 4;
  while (p.slot <= max_nodes) p.slot *= 2;  // (slot 1 holds no node)
  p.n_cols = n_cols;
  p.split = false;
  p.win = p.slot * 4 <= 1 << kWinSmall ? kWinSmall : kWinLarge;
  // Four rows per lane conflict least but need a full chip of 1,024-row
  // tiles, two of them per CU (28 columns, 100 trees: 67 us at 100,000 rows
  // and 117 at 1M, against 34 and 177 with one row; level at 400,000); from
  // 53 columns on, their LDS leaves too few waves (100 columns, 1M rows: 342
  // us against 197).
  if (n >= kWalkRows4 && n_cols <= kWalkCols4 && p.win == kWinSmall) {
    p.rpl = 4;
    p.tpl = 2;
  } else {
    p.rpl = 1;
    p.tpl = p.slot <= kGroupNodes / 8 ? 8 : p.slot <= kGroupNodes / 2 ? 2 : 1;
    p.split = n * K <= kWalkSplitRows && p.tpl == 8;
  }
  p.per_group = kGroupNodes / p.slot;
  p.own = p.rpl == 1 && p.tpl < 8;
  return true;
}

hipError_t launch_walk_pack(hipStream_t st, const TreeNodeDev *nodes, const int32_t *first,
                            const int32_t *count, const int32_t *dest, int32_t n_entries,
                            const uint8_t *remap, double lr, const WalkPlan &p, uint32_t *words,
                            double *vals, int32_t *depth) {
  if (n_entries <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_walk_pack, dim3((unsigned)n_entries), dim3(64), 0, st, nodes, first, count,
                     dest, remap, lr, p.win, p.own ? p.tpl : 0, words, vals, depth);
  return hipGetLastError();
}

namespace {

template <int kRpl, int kTpl, int kTileLog2, int kWin>
hipError_t run_walk(hipStream_t st, const WalkArgs &a, int32_t K, hipEvent_t ev_start,
                    hipEvent_t ev_stop) {
  constexpr int kTile = 1 << kTileLog2;
  const dim3 grid((unsigned)((a.n + kTile - 1) / kTile), (unsigned)K), block(kTile / kRpl);
  const size_t lds = (size_t)kCodesAt + ((size_t)a.n_cols << kTileLog2);
  if (a.proba)
    hipExtLaunchKernelGGL((k_walk<kRpl, kTpl, kTileLog2, kWin, true>), grid, block, lds, st,
                          ev_start, ev_stop, 0, a);
  else
    hipExtLaunchKernelGGL((k_walk<kRpl, kTpl, kTileLog2, kWin, false>), grid, block, lds, st,
                          ev_start, ev_stop, 0, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_walk(hipStream_t st, const WalkPlan &p, const WalkArgs &a, int32_t K,
                       hipEvent_t ev_start, hipEvent_t ev_stop) {
  if (a.n <= 0) return hipSuccess;
  if (p.split) {
    const dim3 grid((unsigned)((a.n + 63) / 64), (unsigned)K), block(64 * kSplitWaves);
    const size_t lds = (size_t)kSplitWaves * kGroupNodes * 4 + ((size_t)a.n_cols << 6);
    if (a.proba)
      hipExtLaunchKernelGGL(k_walk_split<true>, grid, block, lds, st, ev_start, ev_stop, 0, a);
    else
      hipExtLaunchKernelGGL(k_walk_split<false>, grid, block, lds, st, ev_start, ev_stop, 0, a);
    return hipGetLastError();
  }
  if (p.rpl == 4) return run_walk<4, 2, 10, kWinSmall>(st, a, K, ev_start, ev_stop);
  if (p.tpl == 8) return run_walk<1, 8, 8, kWinSmall>(st, a, K, ev_start, ev_stop);
  if (p.win == kWinSmall) return run_walk<1, 2, 8, kWinSmall>(st, a, K, ev_start, ev_stop);
  if (p.tpl == 2) return run_walk<1, 2, 8, kWinLarge>(st, a, K, ev_start, ev_stop);
  return run_walk<1, 1, 8, kWinLarge>(st, a, K, ev_start, ev_stop);
}

}  // namespace bsscl
