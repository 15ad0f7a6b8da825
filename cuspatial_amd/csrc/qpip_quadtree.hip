// quadtree_on_points on gfx950.
//
// Reference: cpp/src/indexing/point_quadtree.cu:154-180 (column API),
// detail/point_quadtree.cuh:238-272 (clamps), detail/index/construction/
// phase_1.cuh and phase_2.cuh (construction).
//
// The reference builds the tree bottom-up: it sorts the Morton keys, reduces the
// bottom cells, reduces every level above them into Q*(d+1)-sized arrays, then
// prunes the children of small nodes and recovers leaf offsets with two more
// sorts. This implementation computes the same five columns top-down from the
// sorted keys and never materialises pruned nodes:
//
//   1. keygen (fused with the radix sort's first digit count);
//   2. stable LSD radix sort of (key, point index) over the 2d+2 (at most 32)
//      key bits that can be non-zero;
//   3. starts: the node of level l that begins at sorted position i has more than
//      max_size points iff keys i and i + max_size share its prefix, so the nodes that
//      begin at a position, and which of them are internal, follow from a handful of
//      keys near it, for every level at once (tree_count_kernel marks the positions
//      and counts their nodes per level and block);
//   4. a scan of the blocks' counts gives every level's and block's first node number;
//   5. emit: each marked position writes its nodes straight into the output columns,
//      level-major and in key order within a level - the order of
//      reverse_tree_levels. Internal nodes get (length, offset) = (child count, first
//      child position) and leaves (point count, first point position).
//
// Equivalences with the reference (for the 5 output columns):
//   * a level-l node is kept by remove_unqualified_quads iff its parent has more
//     than max_size points (phase_2.cuh:256-281); since point counts shrink
//     downwards, that is iff all its ancestors are internal - the nodes of steps 3
//     to 5;
//   * a leaf's offset is the exclusive scan of leaf point counts in Morton order
//     (phase_2.cuh:105-184); leaves tile the sorted points in Morton order, so it
//     is the leaf's first sorted point position;
//   * when the root level holds R > 1 nodes (possible only if a point's cell
//     coordinate reaches 2^d, i.e. with a clamped scale), the reference's
//     num_parent_nodes = end - Q - 1 (phase_1.cuh:177) counts R - 1 extra
//     "parents", which are the first R - 1 bottom-level nodes in key order. Those
//     that survive pruning are flagged internal when they hold more than
//     max_size points, with length 0 and offset = number of nodes, and their
//     points drop out of the leaf-offset scan. Step 5 reproduces exactly that.
#include <algorithm>
#include <vector>

#include "qpip_sort.hpp"
#include "qpip_tree.hpp"

namespace qpip {

namespace {

constexpr int kMaxLevels = 16;
constexpr int kMaxMarked = 16;

struct TreeMeta {
  uint32_t level_begin[kMaxLevels + 1];  // first node of each level; [levels]: all nodes
  uint32_t num_marked;                   // E = R - 1 (d >= 1)
  uint32_t marked_key[kMaxMarked];
  uint32_t marked_internal[kMaxMarked];
  uint32_t marked_start[kMaxMarked];
  uint32_t marked_count[kMaxMarked];
  uint64_t num_nodes;
};

// --- 1. keygen: compute_point_keys_and_sorted_indices (phase_1.cuh:62-95) -------
// One block per radix-sort tile (4096 points). The block also counts the sort's
// first digit (key bits 0-7) into per-wave LDS histograms, so that the sort skips
// its first counting pass. Full tiles of 16-byte aligned inputs are read with
// 16-byte loads and the keys written as uint4 (thread t owns points 4t..4t+3 of
// each quarter of the tile). Points are either two coordinate arrays (the column
// API) or interleaved x, y pairs (vec_2d, the header-only API's layout).
template <bool XY>
__global__ void __launch_bounds__(256)
  keygen_kernel(double const* __restrict__ xs,  // XY: interleaved x, y pairs
                double const* __restrict__ ys,  // XY: unused
                uint64_t n,
                double min_x,
                double min_y,
                double max_x,
                double max_y,
                double scale,
                uint32_t outside_key,
                bool vec,
                uint32_t* __restrict__ keys,
                uint32_t* __restrict__ counts)
{
  constexpr int NW = 256 / kWave;
  __shared__ uint32_t h[NW][kRadix];
  int const w = threadIdx.x / kWave;
#pragma unroll
  for (int ww = 0; ww < NW; ++ww) h[ww][threadIdx.x] = 0;
  __syncthreads();
  uint64_t const lo = static_cast<uint64_t>(blockIdx.x) * kSortTile;
  if (vec && lo + kSortTile <= n) {
    constexpr int Q = kSortItems / 4;
    double px[kSortItems], py[kSortItems];
    if (XY) {
      double2 const* p2 = reinterpret_cast<double2 const*>(xs) + lo;
#pragma unroll
      for (int j = 0; j < Q; ++j) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          double2 const v   = p2[(j * 256 + threadIdx.x) * 4 + c];
          px[4 * j + c]     = v.x;
          py[4 * j + c]     = v.y;
        }
      }
    } else {
      double2 const* x2 = reinterpret_cast<double2 const*>(xs + lo);
      double2 const* y2 = reinterpret_cast<double2 const*>(ys + lo);
#pragma unroll
      for (int j = 0; j < Q; ++j) {
        int const e = (j * 256 + threadIdx.x) * 2;  // double2 index of point 4 * (j * 256 + t)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          double2 const xv  = x2[e + c];
          double2 const yv  = y2[e + c];
          px[4 * j + 2 * c] = xv.x;
          px[4 * j + 2 * c + 1] = xv.y;
          py[4 * j + 2 * c] = yv.x;
          py[4 * j + 2 * c + 1] = yv.y;
        }
      }
    }
    uint4* k4 = reinterpret_cast<uint4*>(keys + lo);
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      uint32_t k[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        k[c] = point_key(px[4 * j + c], py[4 * j + c], min_x, min_y, max_x, max_y, scale,
                         outside_key);
        wave_count_digit(h[w], k[c] & 0xFFu);
      }
      k4[j * 256 + threadIdx.x] = make_uint4(k[0], k[1], k[2], k[3]);
    }
  } else {
    double x[kSortItems], y[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
      uint64_t const i = lo + static_cast<uint64_t>(j) * 256 + threadIdx.x;
      x[j]             = i < n ? (XY ? xs[2 * i] : xs[i]) : 0.0;
      y[j]             = i < n ? (XY ? xs[2 * i + 1] : ys[i]) : 0.0;
    }
#pragma unroll
    for (int j = 0; j < kSortItems; ++j) {
      uint64_t const i   = lo + static_cast<uint64_t>(j) * 256 + threadIdx.x;
      uint32_t const key = point_key(x[j], y[j], min_x, min_y, max_x, max_y, scale, outside_key);
      if (i < n) keys[i] = key;
      wave_count_digit(h[w], i < n ? (key & 0xFFu) : static_cast<uint32_t>(kRadix));
    }
  }
  __syncthreads();
  uint32_t s = 0;
#pragma unroll
  for (int ww = 0; ww < NW; ++ww) s += h[ww][threadIdx.x];
  counts[static_cast<uint64_t>(blockIdx.x) * kRadix + threadIdx.x] = s;
}

// --- 3. starts --------------------------------------------------------------------
// Levels run from 0 to last = max(d, 1) - 1; a level-l node is the run of keys equal
// above bit 2 (last - l).
struct TreeShape {
  uint32_t const* K;  // sorted keys
  uint32_t n;
  int last;           // deepest level
  uint32_t max_size;

  __device__ __forceinline__ bool share(uint32_t a, uint32_t b, int l) const
  {
    return ((a ^ b) >> (2 * (last - l))) == 0;
  }
  // The deepest level at which keys a and b are in one node, -1 if none.
  __device__ __forceinline__ int common(uint32_t a, uint32_t b) const
  {
    if (a == b) return last;
    int const l = last - 1 - ((31 - __builtin_clz(a ^ b)) >> 1);
    return l < 0 ? -1 : l;
  }
  // What may_start reads.
  struct Near {
    uint32_t k, before, low, high;  // keys i, i - 1, i - 1 - h, i + h, h = max_size / 2
  };
  __device__ __forceinline__ Near load_near(uint32_t i) const
  {
    uint32_t const h = max_size / 2;
    return Near{K[i], K[i > 0 ? i - 1 : 0], K[i > h ? i - 1 - h : 0], K[n - i > h ? i + h : n - 1]};
  }
  // False for most positions that begin no kept node (inside a leaf). The first node that
  // can begin at i > 0 is a child of the node of level c = common(K[i - 1], K[i]), which
  // holds both and is internal only if it holds more than max_size positions; such a
  // range reaches i - 1 - h or i + h.
  __device__ __forceinline__ bool may_start(uint32_t i, Near const& v) const
  {
    int const c = common(v.before, v.k);
    if (i == 0 || c < 0) return true;
    uint32_t const h = max_size / 2;
    return c < last &&
           ((i > h && share(v.low, v.k, c)) || (n - i > h && share(v.high, v.k, c)));
  }
  // The level of the first node that begins at position i if it is kept (its parent,
  // which then holds i - 1 too, is internal), else last + 1.
  __device__ __forceinline__ int first_level(uint32_t i, uint32_t k) const
  {
    if (i == 0) return 0;
    int const c = common(K[i - 1], k);  // the parent's level
    if (c < 0) return 0;
    if (c == last) return last + 1;
    uint32_t const ms = max_size;
    if (i >= ms && share(K[i - ms], k, c)) return c + 1;
    // the parent begins after i - max_size
    uint32_t lo = i >= ms ? i - ms + 1 : 0, hi = i - 1;
    while (lo < hi) {
      uint32_t const mid = lo + ((hi - lo) >> 1);
      if (share(K[mid], k, c))
        hi = mid;
      else
        lo = mid + 1;
    }
    return n - lo > ms && share(K[lo + ms], k, c) ? c + 1 : last + 1;
  }
  // The leaf level of the chain of nodes that begins at i with level f: each node with
  // more than max_size points has its first child at i too.
  __device__ __forceinline__ int leaf_level(uint32_t i, uint32_t k, int f) const
  {
    int const c = n - i > max_size ? common(k, K[i + max_size]) : -1;
    if (c < f) return f;
    return c + 1 < last ? c + 1 : last;
  }
};

// Per block: nodes per level [0, 16) and the first marked position [16] (all ones:
// none); after the scan, the nodes before the block per level and the first marked
// position after it.
constexpr int kTreeCols   = 17;
constexpr int kTreeBlocks = 1024;  // entries per column

// Marks the positions of block b's range [b * per, (b + 1) * per) at which kept nodes
// begin (per is a multiple of kTreeStep: the blocks share no word of `marks`) and counts
// their nodes. Per kTreeSpan positions: first the positions that may start a node
// (eight per thread in flight), compacted in LDS, then those one per thread, so that a
// wave does not wait for a binary search in nearly every word (1e8 keys took 1109 us
// that way, 275 us so). Bound by the latency of its loads: 0.4 GB of keys from HBM, the
// other three reads of each are in the caches. With the scan and the emit the tree
// of 1e8 keys at depth 15 (1.2M nodes) takes 0.37 ms in 4 launches, against 0.46 ms in
// 30 as two launches per level (a search for every node's child boundaries), and that
// of 1e6 keys at depth 7 24 us in 4 launches against 95 us in 15.
constexpr int kTreeItems = 8;
constexpr int kTreeStep  = 256 * kTreeItems;  // positions per block and round
constexpr int kTreeSpan  = 256 * kWave;       // positions per LDS list

__global__ void __launch_bounds__(256)
  tree_count_kernel(TreeShape t, uint32_t per, uint64_t* __restrict__ marks,
                    uint32_t* __restrict__ cols)
{
  __shared__ uint16_t s_at[kTreeSpan];
  __shared__ unsigned long long s_word[kTreeSpan / kWave];
  __shared__ uint32_t s_cols[kTreeCols];
  __shared__ uint32_t s_total;
  if (threadIdx.x < kTreeCols) s_cols[threadIdx.x] = threadIdx.x == 16 ? 0xffffffffu : 0u;
  uint64_t const lo = static_cast<uint64_t>(blockIdx.x) * per;
  uint64_t const hi = lo + per < t.n ? lo + per : t.n;
  int const lane    = lane_id();
  uint32_t cnt = 0, first = 0xffffffffu;  // lane l: level l's nodes
  for (uint64_t i0 = lo; i0 < hi; i0 += kTreeSpan) {
    uint64_t const i1 = i0 + kTreeSpan < hi ? i0 + kTreeSpan : hi;
    s_word[threadIdx.x] = 0;
    if (threadIdx.x == 0) s_total = 0;
    __syncthreads();
    for (uint64_t r = i0; r < i1; r += kTreeStep) {
      TreeShape::Near v[kTreeItems];
#pragma unroll
      for (int u = 0; u < kTreeItems; ++u) {
        uint64_t const i = r + u * 256 + threadIdx.x;
        v[u]             = t.load_near(static_cast<uint32_t>(i < i1 ? i : i1 - 1));
      }
#pragma unroll
      for (int u = 0; u < kTreeItems; ++u) {
        uint64_t const i = r + u * 256 + threadIdx.x;
        bool const may   = i < i1 && t.may_start(static_cast<uint32_t>(i), v[u]);
        uint64_t const b = ballot(may);
        if (b == 0) continue;
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&s_total, static_cast<uint32_t>(__popcll(b)));
        at = uniform(at) + static_cast<uint32_t>(__popcll(b & lanemask_lt()));
        if (may) s_at[at] = static_cast<uint16_t>(i - i0);
      }
    }
    __syncthreads();
    uint32_t const total = s_total;
    for (uint32_t q = threadIdx.x; q - lane < total; q += 256) {
      int f = t.last + 1, leaf = -1;
      if (q < total) {
        uint32_t const at = s_at[q];
        uint32_t const i  = static_cast<uint32_t>(i0) + at;
        uint32_t const k  = t.K[i];
        f                 = t.first_level(i, k);
        if (f <= t.last) {
          leaf  = t.leaf_level(i, k, f);
          first = i < first ? i : first;
          atomicOr(&s_word[at / kWave], 1ull << (at % kWave));
        }
      }
      for (int l = 0; l <= t.last; ++l) {
        uint64_t const b = ballot(f <= l && l <= leaf);
        if (lane == l) cnt += static_cast<uint32_t>(__popcll(b));
      }
    }
    __syncthreads();
    if (i0 + threadIdx.x * kWave < i1) marks[i0 / kWave + threadIdx.x] = s_word[threadIdx.x];
    __syncthreads();
  }
  if (lane < 16 && cnt) atomicAdd(&s_cols[lane], cnt);
  if (first != 0xffffffffu) atomicMin(&s_cols[16], first);
  __syncthreads();
  if (threadIdx.x < kTreeCols) cols[threadIdx.x * kTreeBlocks + blockIdx.x] = s_cols[threadIdx.x];
}

// --- 4. scan of the blocks' counts, level sizes and the root-level quirk -----------
__global__ void __launch_bounds__(1024)
  tree_scan_kernel(TreeShape t, int d, uint32_t blocks, uint32_t* __restrict__ cols,
                   TreeMeta* __restrict__ meta)
{
  __shared__ uint32_t s_total[kMaxLevels];
  int const w = static_cast<int>(uniform(threadIdx.x / kWave)), lane = lane_id();
  // Waves 0 .. last scan the levels' columns and wave 15 (last <= 14) the first marked
  // positions; the values of up to 1024 blocks are loaded before they are scanned.
  if (w <= t.last || w == 15) {
    int const col = w == 15 ? 16 : w;
    uint32_t v[kTreeBlocks / kWave];
#pragma unroll
    for (int c = 0; c < kTreeBlocks / kWave; ++c) {
      uint32_t const b = static_cast<uint32_t>(c * kWave + lane);
      v[c]             = b < blocks ? cols[col * kTreeBlocks + b] : w == 15 ? 0xffffffffu : 0u;
    }
    if (w == 15) {
      uint32_t next = 0xffffffffu;
#pragma unroll
      for (int c = kTreeBlocks / kWave - 1; c >= 0; --c) {
        if (static_cast<uint32_t>(c * kWave) >= blocks) continue;
        uint32_t m = v[c];  // smallest of this lane's and the higher lanes'
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
          uint32_t const x = __shfl_down(m, o, kWave);
          if (lane + o < kWave) m = x < m ? x : m;
        }
        uint32_t const above = __shfl_down(m, 1, kWave);
        uint32_t const b     = static_cast<uint32_t>(c * kWave + lane);
        if (b < blocks)
          cols[16 * kTreeBlocks + b] = lane + 1 < kWave && above < next ? above : next;
        uint32_t const all = __shfl(m, 0, kWave);
        next               = all < next ? all : next;
      }
    } else {
      uint32_t run = 0;
#pragma unroll
      for (int c = 0; c < kTreeBlocks / kWave; ++c) {
        if (static_cast<uint32_t>(c * kWave) >= blocks) break;
        uint32_t const b    = static_cast<uint32_t>(c * kWave + lane);
        uint32_t const incl = wave_incl_scan(v[c]);
        if (b < blocks) cols[w * kTreeBlocks + b] = run + incl - v[c];
        run += __shfl(incl, kWave - 1, kWave);
      }
      if (lane == 0) s_total[w] = run;
    }
  }
  __syncthreads();
  if (w != 0) return;
  // Root level: distinct key >> 2d (d >= 1); at most 16 values.
  bool root_present = false;
  bool const many   = d >= 1 && (t.K[0] >> (2 * d)) != (t.K[t.n - 1] >> (2 * d));
  if (many && lane < 16) {
    uint32_t const lo = lower_bound_u32(t.K, 0, t.n, static_cast<uint64_t>(lane) << (2 * d));
    uint32_t const hi = lower_bound_u32(t.K, lo, t.n, static_cast<uint64_t>(lane + 1) << (2 * d));
    root_present      = hi > lo;
  }
  uint64_t const rm = ballot(root_present);
  if (lane != 0) return;
  uint32_t total = 0;
  for (int l = 0; l <= kMaxLevels; ++l) {
    meta->level_begin[l] = total;
    if (l <= t.last) total += s_total[l];
  }
  meta->num_nodes = total;
  int const R      = __popcll(rm);
  uint32_t const E = R > 1 ? static_cast<uint32_t>(R - 1) : 0u;
  meta->num_marked = E;
  // The first E distinct bottom-level keys (the extra "parents").
  uint32_t pos = 0;
  for (uint32_t e = 0; e < E; ++e) {
    meta->marked_internal[e] = meta->marked_start[e] = meta->marked_count[e] = 0;
    uint32_t const k    = pos < t.n ? t.K[pos] : 0xffffffffu;
    meta->marked_key[e] = k;
    if (pos < t.n) pos = lower_bound_u32(t.K, pos, t.n, static_cast<uint64_t>(k) + 1);
  }
}

// --- 5. emit ------------------------------------------------------------------------
struct TreeOut {
  uint32_t* key;
  uint8_t* level;
  uint8_t* internal;
  uint32_t* length;  // zeroed: an internal node's is counted by its children
  uint32_t* offset;
};

// Block b writes the nodes that begin in its range (tree_count_kernel's), 256 marked
// positions at a time: one per thread, ranked per level by ballots. A position's first
// node is a child of the last node of the level above that began before it.
__global__ void __launch_bounds__(256)
  tree_emit_kernel(TreeShape t, uint32_t per, uint64_t const* __restrict__ marks,
                   uint32_t const* __restrict__ cols, TreeMeta const* __restrict__ meta, TreeOut o)
{
  constexpr int NW = 256 / kWave;
  __shared__ uint16_t s_at[256 * kWave];  // marked positions of 256 words, relative
  __shared__ uint32_t s_scan[NW + 1];
  __shared__ uint32_t s_run[kMaxLevels];  // per level: the next node's number
  __shared__ uint32_t s_cnt[NW][kMaxLevels];
  __shared__ uint32_t s_open[2];  // the last leaf written, whose end is not known yet
  int const w = threadIdx.x / kWave, lane = lane_id();
  uint64_t const lo = static_cast<uint64_t>(blockIdx.x) * per;
  uint64_t const hi = lo + per < t.n ? lo + per : t.n;
  if (threadIdx.x < kMaxLevels)
    s_run[threadIdx.x] = meta->level_begin[threadIdx.x] + cols[threadIdx.x * kTreeBlocks + blockIdx.x];
  bool open = false;
  for (uint64_t i0 = lo; i0 < hi; i0 += 256 * kWave) {
    uint64_t const at = i0 + threadIdx.x * kWave;
    uint64_t word     = at < hi ? marks[at / kWave] : 0ull;
    uint32_t total;
    uint32_t slot = block_excl_scan<256>(static_cast<uint32_t>(__popcll(word)), s_scan, &total);
    while (word) {
      s_at[slot++] = static_cast<uint16_t>(threadIdx.x * kWave + __builtin_ctzll(word));
      word &= word - 1;
    }
    __syncthreads();
    if (total == 0) continue;
    if (open && threadIdx.x == 0)
      o.length[s_open[0]] = static_cast<uint32_t>(i0) + s_at[0] - s_open[1];
    open = true;
    for (uint32_t s0 = 0; s0 < total; s0 += 256) {
      uint32_t const s = s0 + threadIdx.x;
      bool const live  = s < total;
      uint32_t i = 0, k = 0;
      int f = t.last + 1, leaf = -1;
      if (live) {
        i    = static_cast<uint32_t>(i0) + s_at[s];
        k    = t.K[i];
        f    = i == 0 ? 0 : t.common(t.K[i - 1], k) + 1;
        leaf = t.leaf_level(i, k, f);
      }
      for (int l = 0; l <= t.last; ++l) {
        uint64_t const b = ballot(f <= l && l <= leaf);
        if (lane == 0) s_cnt[w][l] = static_cast<uint32_t>(__popcll(b));
      }
      __syncthreads();
      uint32_t above = 0;  // the node one level up (this position's, or its parent)
      for (int l = 0; l <= t.last; ++l) {
        uint64_t const b = ballot(f <= l && l <= leaf);
        uint32_t node    = s_run[l] + static_cast<uint32_t>(__popcll(b & lanemask_lt()));
        for (int q = 0; q < w; ++q) node += s_cnt[q][l];
        if (live && l == f - 1) above = node - 1;
        if (!(f <= l && l <= leaf)) continue;
        if (l > 0) {
          atomicAdd(&o.length[above], 1u);
          if (l > f) o.offset[above] = node;  // its first child
        }
        o.key[node]      = k >> (2 * (t.last - l));
        o.level[node]    = static_cast<uint8_t>(l);
        o.internal[node] = l < leaf ? 1 : 0;
        if (l == leaf) {
          o.offset[node] = i;
          if (s + 1 < total) {
            o.length[node] = static_cast<uint32_t>(i0) + s_at[s + 1] - i;
          } else {
            s_open[0] = node;
            s_open[1] = i;
          }
        }
        above = node;
      }
      __syncthreads();
      if (threadIdx.x <= static_cast<unsigned>(t.last)) {
        uint32_t add = 0;
        for (int q = 0; q < NW; ++q) add += s_cnt[q][threadIdx.x];
        s_run[threadIdx.x] += add;
      }
      __syncthreads();
    }
  }
  if (open && threadIdx.x == 0) {
    uint32_t const next = cols[16 * kTreeBlocks + blockIdx.x];
    o.length[s_open[0]] = (next == 0xffffffffu ? t.n : next) - s_open[1];
  }
}

// The extra "parents" among the bottom-level nodes: those that hold more than
// max_size points.
__global__ void __launch_bounds__(64)
  mark_extra_kernel(uint32_t const* __restrict__ key, uint32_t const* __restrict__ length,
                    uint32_t const* __restrict__ offset, int last, uint32_t max_size,
                    TreeMeta* __restrict__ meta)
{
  if (threadIdx.x != 0) return;
  uint32_t const lo0 = meta->level_begin[last];
  uint32_t const hi0 = static_cast<uint32_t>(meta->num_nodes);
  for (uint32_t e = 0; e < meta->num_marked; ++e) {
    uint32_t const mk = meta->marked_key[e];
    uint32_t const at = lower_bound_u32(key, lo0, hi0, mk);
    if (at < hi0 && key[at] == mk && length[at] > max_size) {
      meta->marked_internal[e] = 1;
      meta->marked_start[e]    = offset[at];
      meta->marked_count[e]    = length[at];
    }
  }
}

// Flags them internal and drops their points from the leaves' offsets.
__global__ void __launch_bounds__(256)
  apply_extra_kernel(TreeMeta const* __restrict__ meta, int last, uint64_t m, TreeOut o)
{
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < m;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    if (o.internal[i]) continue;
    uint32_t const key = o.key[i], start = o.offset[i];
    bool marked        = false;
    uint32_t skipped   = 0;
    for (uint32_t e = 0; e < meta->num_marked; ++e) {
      if (!meta->marked_internal[e]) continue;
      if (o.level[i] == last && meta->marked_key[e] == key) marked = true;
      if (meta->marked_start[e] < start) skipped += meta->marked_count[e];
    }
    if (marked) {
      o.internal[i] = 1;
      o.length[i]   = 0;
      o.offset[i]   = static_cast<uint32_t>(m);
    } else {
      o.offset[i] = start - skipped;
    }
  }
}

}  // namespace

// Host orchestration. Returns the number of nodes; outputs via `oa`.
static int64_t quadtree_on_points_impl(double const* x,
                                       double const* y,
                                       bool interleaved,  // x holds x, y pairs; y unused
                                       int64_t n,
                                       double x_min,
                                       double x_max,
                                       double y_min,
                                       double y_max,
                                       double scale,
                                       int8_t max_depth,
                                       int32_t max_size,
                                       OutputAllocator& oa,
                                       hipStream_t stream,
                                       uint32_t** point_indices,
                                       uint32_t** key,
                                       uint8_t** level,
                                       uint8_t** is_internal,
                                       uint32_t** length,
                                       uint32_t** offset)
{
  QPIP_EXPECTS(n < (int64_t{1} << 32), "number of points must be less than 2^32");
  // detail/point_quadtree.cuh:259-268
  double const min_x = std::min(x_min, x_max), max_x = std::max(x_min, x_max);
  double const min_y = std::min(y_min, y_max), max_y = std::max(y_min, y_max);
  max_size           = std::max(1, max_size);
  max_depth          = std::max(int8_t{0}, std::min(int8_t{15}, max_depth));
  int const d        = max_depth;
  scale = std::max(scale, std::max(max_x - min_x, max_y - min_y) / ((1 << d) + 2));

  // Cell coordinates are below 2^d + 3, so keys have at most 2*bits(2^d + 2) bits.
  int cbits = 0;
  while ((uint64_t{1} << cbits) <= (uint64_t{1} << d) + 2) ++cbits;
  int const key_bits = std::min(32, 2 * cbits);
  uint32_t const outside_key = static_cast<uint32_t>((1u << (2 * d)) - 1u);

  uint64_t const un = static_cast<uint64_t>(n);
  uint64_t const tiles = sort_tiles(un);
  // point_indices is written by the sort's last pass straight into the output
  uint32_t* pi = oa.make<uint32_t>(un);
  dbuf<uint32_t> keys_a(un), keys_b(un), vals_tmp(un);
  dbuf<uint32_t> counts0(static_cast<size_t>(tiles) * kRadix);
  {
    KernelTimer kt("keygen", stream);
    bool const vec = reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                     (interleaved || reinterpret_cast<uintptr_t>(y) % 16 == 0) &&
                     reinterpret_cast<uintptr_t>(keys_a.get()) % 16 == 0;
    if (interleaved)
      keygen_kernel<true><<<static_cast<unsigned>(tiles), 256, 0, stream>>>(
        x, nullptr, un, min_x, min_y, max_x, max_y, scale, outside_key, vec, keys_a.get(),
        counts0.get());
    else
      keygen_kernel<false><<<static_cast<unsigned>(tiles), 256, 0, stream>>>(
        x, y, un, min_x, min_y, max_x, max_y, scale, outside_key, vec, keys_a.get(),
        counts0.get());
    QPIP_LAUNCH_CHECK();
  }
  SortResult sorted = radix_sort_pairs(keys_a.get(), keys_b.get(), nullptr, pi, vals_tmp.get(),
                                       un, key_bits, stream, counts0.get(), "point_sort");
  vals_tmp.release();

  TreeShape const shape{sorted.keys, static_cast<uint32_t>(un), std::max(d, 1) - 1,
                        static_cast<uint32_t>(max_size)};
  // blocks of whole rounds, at most kTreeBlocks of them
  uint64_t per = (un + kTreeBlocks - 1) / kTreeBlocks;
  per          = std::max<uint64_t>(1, (per + kTreeStep - 1) / kTreeStep) * kTreeStep;
  uint32_t const blocks = static_cast<uint32_t>((un + per - 1) / per);
  dbuf<uint64_t> marks((un + kWave - 1) / kWave + 256 / kWave);
  dbuf<uint32_t> cols(kTreeBlocks * kTreeCols);
  dbuf<TreeMeta> meta(1);
  {
    KernelTimer kt("tree_count", stream);
    tree_count_kernel<<<blocks, 256, 0, stream>>>(shape, static_cast<uint32_t>(per), marks.get(),
                                                  cols.get());
    QPIP_LAUNCH_CHECK();
    tree_scan_kernel<<<1, 1024, 0, stream>>>(shape, d, blocks, cols.get(), meta.get());
    QPIP_LAUNCH_CHECK();
  }

  TreeMeta h_meta;
  read_back({{&h_meta, meta.get(), sizeof(TreeMeta)}}, stream);
  uint64_t const m = h_meta.num_nodes;

  uint32_t* o_key      = oa.make<uint32_t>(m);
  uint8_t* o_level     = oa.make<uint8_t>(m);
  uint8_t* o_internal  = oa.make<uint8_t>(m);
  uint32_t* o_length   = oa.make<uint32_t>(m);
  uint32_t* o_offset   = oa.make<uint32_t>(m);
  {
    KernelTimer kt("tree_emit", stream);
    TreeOut const out{o_key, o_level, o_internal, o_length, o_offset};
    fill_u32(o_length, m, 0u, stream);
    tree_emit_kernel<<<blocks, 256, 0, stream>>>(shape, static_cast<uint32_t>(per), marks.get(),
                                                 cols.get(), meta.get(), out);
    QPIP_LAUNCH_CHECK();
    if (h_meta.num_marked > 0) {
      mark_extra_kernel<<<1, 64, 0, stream>>>(o_key, o_length, o_offset, shape.last,
                                              shape.max_size, meta.get());
      QPIP_LAUNCH_CHECK();
      apply_extra_kernel<<<grid_for(m, 256), 256, 0, stream>>>(meta.get(), shape.last, m, out);
      QPIP_LAUNCH_CHECK();
    }
  }
  // no wait here: the outputs are ready for work queued on `stream` after this call
  *point_indices = pi;
  *key           = o_key;
  *level         = o_level;
  *is_internal   = o_internal;
  *length        = o_length;
  *offset        = o_offset;
  return static_cast<int64_t>(m);
}

}  // namespace qpip

namespace {

int quadtree_on_points_entry(const double* x,
                             const double* y,
                             bool interleaved,
                             int64_t num_points,
                             int64_t num_y,
                             double x_min,
                             double x_max,
                             double y_min,
                             double y_max,
                             double scale,
                             int8_t max_depth,
                             int32_t max_size,
                             const qpip_resource* mr,
                             void* stream,
                             uint32_t** point_indices,
                             uint32_t** key,
                             uint8_t** level,
                             uint8_t** is_internal_node,
                             uint32_t** length,
                             uint32_t** offset,
                             int64_t* num_nodes)
{
  using namespace qpip;
  try {
    QPIP_EXPECTS(point_indices && key && level && is_internal_node && length && offset && num_nodes,
                 "output pointers must not be null");
    *point_indices = nullptr;
    *key = nullptr, *level = nullptr, *is_internal_node = nullptr, *length = nullptr,
    *offset = nullptr, *num_nodes = 0;
    // cpp/src/indexing/point_quadtree.cu:166
    QPIP_EXPECTS(num_points == num_y, "x and y columns must have the same length");
    if (num_points <= 0) return QPIP_SUCCESS;
    QPIP_EXPECTS(x && (interleaved || y), "x and y must not be null");
    StreamScope scope(static_cast<hipStream_t>(stream));
    OutputAllocator oa(mr, static_cast<hipStream_t>(stream));
    *num_nodes = quadtree_on_points_impl(x, y, interleaved, num_points, x_min, x_max, y_min,
                                         y_max, scale, max_depth, max_size, oa,
                                         static_cast<hipStream_t>(stream), point_indices, key,
                                         level, is_internal_node, length, offset);
    oa.keep();
    return QPIP_SUCCESS;
  } catch (...) {
    return qpip::error_status();
  }
}

}  // namespace

extern "C" int qpip_quadtree_on_points(const double* x,
                                       const double* y,
                                       int64_t num_x,
                                       int64_t num_y,
                                       double x_min,
                                       double x_max,
                                       double y_min,
                                       double y_max,
                                       double scale,
                                       int8_t max_depth,
                                       int32_t max_size,
                                       const qpip_resource* mr,
                                       void* stream,
                                       uint32_t** point_indices,
                                       uint32_t** key,
                                       uint8_t** level,
                                       uint8_t** is_internal_node,
                                       uint32_t** length,
                                       uint32_t** offset,
                                       int64_t* num_nodes)
{
  return quadtree_on_points_entry(x, y, false, num_x, num_y, x_min, x_max, y_min, y_max, scale,
                                  max_depth, max_size, mr, stream, point_indices, key, level,
                                  is_internal_node, length, offset, num_nodes);
}

extern "C" int qpip_quadtree_on_points_xy(const double* points_xy,
                                          int64_t num_points,
                                          double x_min,
                                          double x_max,
                                          double y_min,
                                          double y_max,
                                          double scale,
                                          int8_t max_depth,
                                          int32_t max_size,
                                          const qpip_resource* mr,
                                          void* stream,
                                          uint32_t** point_indices,
                                          uint32_t** key,
                                          uint8_t** level,
                                          uint8_t** is_internal_node,
                                          uint32_t** length,
                                          uint32_t** offset,
                                          int64_t* num_nodes)
{
  return quadtree_on_points_entry(points_xy, nullptr, true, num_points, num_points, x_min, x_max, y_min,
                                  y_max, scale, max_depth, max_size, mr, stream, point_indices,
                                  key, level, is_internal_node, length, offset, num_nodes);
}
