// Device code of the quadrant / bounding-box join shared by the single-tree path
// and the batched (many trees) path: node-box classification and the descent of
// one breadth-first level.
#pragma once

#include "qpip_scan.hpp"

namespace qpip {

constexpr int kMaxJoinLevels = 16;

struct SplitTotal {
  uint64_t leaf;
  uint64_t quad;
};

struct JoinMeta {
  SplitTotal level[kMaxJoinLevels];  // per level: leaf pairs emitted, next frontier size
  uint64_t top_pairs;                // T * B
  uint32_t num_top;                  // T = count(level == 0)
  uint32_t max_leaf_offset;
  uint32_t overflow;
  uint32_t bad_index;
  uint32_t tickets;  // blocks of the setup that are done
};

// z_order.cuh:80-94
__device__ __forceinline__ uint32_t undilate_2(uint32_t x)
{
  x &= 0x55555555u;
  x = (x | (x >> 1)) & 0x33333333u;
  x = (x | (x >> 2)) & 0x0F0F0F0Fu;
  x = (x | (x >> 4)) & 0x00FF00FFu;
  x = (x | (x >> 8)) & 0x0000FFFFu;
  return x;
}

struct TreeView {
  uint32_t const* key;
  uint8_t const* level;
  uint8_t const* internal;
  uint32_t const* length;
  uint32_t const* offset;
  uint64_t m;
};

struct BoxView {
  double const* minx;
  double const* miny;
  double const* maxx;
  double const* maxy;
  uint64_t b;
};

// Geometry of the (single) quadtree: every node shares v_min, scale and depth.
struct Params {
  double vmin_x, vmin_y, scale;
  int max_depth;
  __device__ __forceinline__ void get(uint32_t, double& vx, double& vy, double& sc, int& d) const
  {
    vx = vmin_x;
    vy = vmin_y;
    sc = scale;
    d  = max_depth;
  }
};

// One box and the geometry of the quadtree it meets: the same for every node that a
// frontier element descends to.
struct BoxProbe {
  double minx, miny, maxx, maxy;
  double vmin_x, vmin_y, scale;
  int max_depth;
};

template <class Geom>
__device__ __forceinline__ BoxProbe make_probe(BoxView const& bx, Geom const& g, uint32_t node,
                                               uint32_t bbox)
{
  BoxProbe p{bx.minx[bbox], bx.miny[bbox], bx.maxx[bbox], bx.maxy[bbox], 0.0, 0.0, 0.0, 0};
  g.get(node, p.vmin_x, p.vmin_y, p.scale, p.max_depth);
  return p;
}

// intersection.cuh:99-128: 0 leaf, 1 quad, 2 none. The node extent is
// v_min + key * level_scale, which nvcc contracts to an FMA (default --fmad=true).
__device__ __forceinline__ int classify(BoxProbe const& p, uint32_t key, int level, bool internal)
{
  double const key_x = static_cast<double>(undilate_2(key));
  double const key_y = static_cast<double>(undilate_2(key >> 1));
  int const shift    = p.max_depth - 1 - level;
  double const ls    = p.scale * static_cast<double>(1 << (shift < 0 ? 0 : shift));
  double const nx0   = fma(key_x + 0, ls, p.vmin_x);
  double const ny0   = fma(key_y + 0, ls, p.vmin_y);
  double const nx1   = fma(key_x + 1, ls, p.vmin_x);
  double const ny1   = fma(key_y + 1, ls, p.vmin_y);
  if ((nx0 > p.maxx) || (nx1 < p.minx) || (ny0 > p.maxy) || (ny1 < p.miny)) return 2;
  return internal ? 1 : 0;
}

__device__ __forceinline__ uint64_t level_out_base(JoinMeta const* meta, int lvl)
{
  uint64_t b = 0;
  for (int l = 0; l < lvl; ++l) b += meta->level[l].leaf;
  return b;
}

// The traversal (quadtree_bbox_filtering.cuh:53-166, traversal.cuh:63-145) is breadth
// first: each (quad node, box) element of a frontier is replaced by its children that
// meet the box, leaves go to the output and quads to the next frontier, both in element
// order. A step here takes up to kJoinStep levels at once: an element's thread descends
// its subtree that far, counting its leaves per level and the quads below; after one
// scan of the four counts each level's leaves and the next frontier are written in the
// same order as level by level (within a level, path order is element order). Two
// launches per step instead of per level, for quads that one thread expands in turn (at
// most 21 per element at three levels, 5 at two); join_shape says how many levels.
constexpr int kJoinStep = 3;

// Counts of one element: leaves of the step's levels 0 and 1, of level 2 and quads.
struct StepCount {
  uint64_t a, b;  // leaf[0] | leaf[1] << 32, leaf[2] | quad << 32
};

struct JoinSink {
  JoinMeta* meta;
  uint32_t* out_node;
  uint32_t* out_bbox;
  uint32_t* out_key;  // null, or the leaves' offsets (the sort's keys)
  uint32_t* fr_node;
  uint32_t* fr_bbox;
  // cap_fr entries: the elements' counts of the counting pass (elements past them are
  // counted again: a descent costs more than 16 bytes)
  StepCount* counts;
  uint64_t cap_out, cap_fr;
  int lvl, levels;  // first level of the step, levels it takes
};

// Visits the nodes [first, first + n) of the step's level k and below, in path order:
// leaf(k, node) and, at the step's last level, quad(node). Nodes are looked at four at a
// time, so that their loads are in flight together.
template <int K, class Leaf, class Quad>
__device__ __forceinline__ void walk_nodes(TreeView const& t, BoxProbe const& p, JoinSink const& s,
                                           uint32_t first, uint32_t n, Leaf const& leaf,
                                           Quad const& quad)
{
  if (static_cast<uint64_t>(first) + n > t.m) {
    atomicOr(&s.meta->bad_index, 1u);
    return;
  }
  for (uint32_t j0 = 0; j0 < n; j0 += 4) {
    uint32_t key[4];
    int level[4];
    bool internal[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      uint32_t const node = first + (j0 + j < n ? j0 + j : n - 1);
      key[j]              = t.key[node];
      level[j]            = t.level[node];
      internal[j]         = t.internal[node] != 0;
    }
    uint32_t leaves = 0, quads = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      int const c = j0 + j < n ? classify(p, key[j], level[j], internal[j]) : 2;
      leaves |= (c == 0 ? 1u : 0u) << j;
      quads |= (c == 1 ? 1u : 0u) << j;
    }
    for (uint32_t both = leaves | quads; both; both &= both - 1) {
      uint32_t const j    = static_cast<uint32_t>(__builtin_ctz(both));
      uint32_t const node = first + j0 + j;
      if ((leaves >> j) & 1u) {
        leaf(K, node);
      } else if (K + 1 == kJoinStep || K + 1 == s.levels) {
        quad(node);
      } else if constexpr (K + 1 < kJoinStep) {
        walk_nodes<K + 1>(t, p, s, t.offset[node], t.length[node], leaf, quad);
      }
    }
  }
}

// Source: size() elements; root(i, node, bbox, first, n) gives an element's box, a node of
// its tree and the nodes its descent starts from, false where there is none.
template <class Source, class Geom>
__device__ __forceinline__ StepCount count_element(Source const& src, TreeView const& t,
                                                   BoxView const& bx, Geom const& g,
                                                   JoinSink const& s, uint64_t i)
{
  StepCount c{0, 0};
  uint32_t node, bbox, first, n;
  if (!src.root(t, i, node, bbox, first, n)) return c;
  BoxProbe const p = make_probe(bx, g, node, bbox);
  walk_nodes<0>(
    t, p, s, first, n,
    [&](int k, uint32_t) {
      c.a += k == 0 ? 1ull : k == 1 ? 1ull << 32 : 0ull;
      c.b += k == 2 ? 1ull : 0ull;
    },
    [&](uint32_t) { c.b += 1ull << 32; });
  return c;
}

template <class Source, class Geom>
__global__ void __launch_bounds__(kScanThreads)
  join_count_kernel(Source src, TreeView t, BoxView bx, Geom g, JoinSink s,
                    StepCount* __restrict__ partials)
{
  __shared__ uint64_t lds[2][kScanThreads / kWave];
  uint64_t lo, hi;
  chunk_range(src.size(), blockIdx.x, gridDim.x, lo, hi);
  StepCount acc{0, 0};
  for (uint64_t i = lo + threadIdx.x; i < hi; i += kScanThreads) {
    StepCount const c = count_element(src, t, bx, g, s, i);
    if (i < s.cap_fr) s.counts[i] = c;
    acc.a += c.a;
    acc.b += c.b;
  }
  acc.a = wave_sum(acc.a);
  acc.b = wave_sum(acc.b);
  if (lane_id() == 0) {
    lds[0][threadIdx.x / kWave] = acc.a;
    lds[1][threadIdx.x / kWave] = acc.b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    StepCount r{0, 0};
    for (int w = 0; w < kScanThreads / kWave; ++w) {
      r.a += lds[0][w];
      r.b += lds[1][w];
    }
    partials[blockIdx.x] = r;
  }
}

template <class Source, class Geom>
__global__ void __launch_bounds__(kScanThreads)
  join_emit_kernel(Source src, TreeView t, BoxView bx, Geom g, JoinSink s,
                   StepCount const* __restrict__ partials)
{
  __shared__ uint64_t lds[kScanThreads / kWave + 1];
  uint64_t lo, hi;
  chunk_range(src.size(), blockIdx.x, gridDim.x, lo, hi);
  StepCount before{0, 0}, all{0, 0};
  for (unsigned b = threadIdx.x; b < gridDim.x; b += kScanThreads) {
    StepCount const c = partials[b];
    all.a += c.a;
    all.b += c.b;
    if (b < blockIdx.x) {
      before.a += c.a;
      before.b += c.b;
    }
  }
  uint64_t base_a, base_b, total_a, total_b;
  block_excl_scan<kScanThreads>(before.a, lds, &base_a);
  block_excl_scan<kScanThreads>(before.b, lds, &base_b);
  block_excl_scan<kScanThreads>(all.a, lds, &total_a);
  block_excl_scan<kScanThreads>(all.b, lds, &total_b);
  constexpr uint64_t kLow = 0xFFFFFFFFull;
  uint64_t const total[kJoinStep] = {total_a & kLow, total_a >> 32, total_b & kLow};
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int k = 0; k < s.levels; ++k)
      s.meta->level[s.lvl + k] =
        SplitTotal{total[k], k + 1 == s.levels ? total_b >> 32 : uint64_t{0}};
  }
  uint64_t out[kJoinStep];  // first output row of each of the step's levels
  out[0] = level_out_base(s.meta, s.lvl);
  out[1] = out[0] + total[0];
  out[2] = out[1] + total[1];
  for (uint64_t t0 = lo; t0 < hi; t0 += kScanThreads) {
    uint64_t const i  = t0 + threadIdx.x;
    StepCount c{0, 0};
    if (i < hi) c = i < s.cap_fr ? s.counts[i] : count_element(src, t, bx, g, s, i);
    uint64_t tile_a, tile_b;
    uint64_t const ea = base_a + block_excl_scan<kScanThreads>(c.a, lds, &tile_a);
    uint64_t const eb = base_b + block_excl_scan<kScanThreads>(c.b, lds, &tile_b);
    base_a += tile_a;
    base_b += tile_b;
    if ((c.a | c.b) == 0) continue;
    uint64_t o0 = out[0] + (ea & kLow), o1 = out[1] + (ea >> 32), o2 = out[2] + (eb & kLow);
    uint64_t f  = eb >> 32;
    uint32_t node, bbox, first, n;
    src.root(t, i, node, bbox, first, n);
    BoxProbe const p = make_probe(bx, g, node, bbox);
    walk_nodes<0>(
      t, p, s, first, n,
      [&](int k, uint32_t leaf) {
        uint64_t const o = k == 0 ? o0++ : k == 1 ? o1++ : o2++;
        if (o < s.cap_out) {
          s.out_node[o] = leaf;
          s.out_bbox[o] = bbox;
          if (s.out_key) s.out_key[o] = t.offset[leaf];
        } else {
          atomicOr(&s.meta->overflow, 1u);
        }
      },
      [&](uint32_t q) {
        if (f < s.cap_fr) {
          s.fr_node[f] = q;
          s.fr_bbox[f] = bbox;
        } else {
          atomicOr(&s.meta->overflow, 1u);
        }
        ++f;
      });
  }
}

// The elements of a frontier written by an earlier step, whose length is *count. After
// a frontier overflow the recorded length exceeds what was stored (cap): the step is
// rerun with larger buffers, so the excess is skipped.
struct FrontierSource {
  uint64_t const* count;
  uint32_t const* in_node;
  uint32_t const* in_bbox;
  uint64_t cap;
  __device__ __forceinline__ uint64_t size() const { return *count; }
  __device__ __forceinline__ bool root(TreeView const& t, uint64_t i, uint32_t& node,
                                       uint32_t& bbox, uint32_t& first, uint32_t& n) const
  {
    if (i >= cap) return false;
    node  = in_node[i];
    bbox  = in_bbox[i];
    first = t.offset[node];
    n     = t.length[node];
    return true;
  }
};

// Levels per step and blocks of the grid, by the tree's nodes and the boxes. Measured
// with 3, 2 and 1 levels per step (us of all steps' kernels):
//   * no more nodes than boxes, so few of a step's nodes meet a box and the launches
//     count: one request of 20,000 points and 50,000 boxes 621 / 644 / 711 (whole call);
//   * more nodes, where a thread's quads in turn cost more than launches: 84 nodes and
//     200 boxes 27 / 25 / 43, 21,844 and 1,000 85 / 77 / 89, 1.22 million and 50,000 (of
//     36 edges) 260 / 216 / 246, and with boxes that cover the domain 5,456 nodes and 10
//     boxes 109 / 66 / 72, 113,432 and 20,000 257 / 186 / 214, 639,000 and 5,000
//     312 / 228 / 236;
//   * from 2^20 nodes and 64 per box the frontiers fill the GPU at every level: 1.21
//     million and 100 boxes 868 / 583 / 551, 1.4 million and 20,000 719 / 764 / 687, 2.18
//     million and 20,000 1959 / 1188 / 954 (1002 with the children classified twice).
// Two levels past the depth of a full tree of that many nodes few are left, and steps
// take three: a join of 89,916 nodes of 15 levels and 5,000 boxes 852 -> 845 us.
// The grid has a block per 64 boxes or 512 nodes, at most kScanBlocks and 64 at least: a
// box meets a few nodes of a level, or it covers many and their number is the nodes'.
// 1.21 million nodes and 100 boxes at three levels per step: 1367 us with 65 blocks (the
// boxes alone), 874 with this many or 1024; 84 nodes and 200 boxes 27 against 31.
struct JoinShape {
  int levels, deep;  // levels per step, and the level past which they are kJoinStep
  unsigned blocks;
};

inline JoinShape join_shape(uint64_t nodes, uint64_t boxes)
{
  uint64_t const want   = 64 + (boxes + nodes / 8) / 64;
  unsigned const blocks = static_cast<unsigned>(want < kScanBlocks ? want : kScanBlocks);
  int deep = 2;  // log4(nodes) + 2
  while (deep < kMaxJoinLevels && (uint64_t{1} << (2 * (deep - 1))) <= nodes) ++deep;
  if (nodes <= boxes) return {kJoinStep, deep, blocks};
  return {nodes >= (uint64_t{1} << 20) && nodes / 64 >= boxes ? 1 : 2, deep, blocks};
}

// The whole traversal of `depth` levels from the top elements; fr[2] are the frontiers'
// node and box arrays, used in turn.
template <class Top, class Geom>
void launch_join(Top const& top, TreeView const& t, BoxView const& bx, Geom const& g, JoinSink s,
                 uint32_t* const (&fr_node)[2], uint32_t* const (&fr_bbox)[2], int depth,
                 JoinShape shape, StepCount* partials, hipStream_t stream, char const* timer)
{
  unsigned const blocks = shape.blocks;
  for (int lvl = 0, step = 0; lvl < depth; lvl += s.levels, ++step) {
    KernelTimer kt(timer, stream);
    int const take = lvl > shape.deep ? kJoinStep : shape.levels;
    s.lvl          = lvl;
    s.levels       = depth - lvl < take ? depth - lvl : take;
    s.fr_node = fr_node[step % 2];
    s.fr_bbox = fr_bbox[step % 2];
    if (lvl == 0) {
      join_count_kernel<Top, Geom><<<blocks, kScanThreads, 0, stream>>>(top, t, bx, g, s, partials);
      QPIP_LAUNCH_CHECK();
      join_emit_kernel<Top, Geom><<<blocks, kScanThreads, 0, stream>>>(top, t, bx, g, s, partials);
    } else {
      FrontierSource const src{&s.meta->level[lvl - 1].quad, fr_node[(step + 1) % 2],
                               fr_bbox[(step + 1) % 2], s.cap_fr};
      join_count_kernel<FrontierSource, Geom>
        <<<blocks, kScanThreads, 0, stream>>>(src, t, bx, g, s, partials);
      QPIP_LAUNCH_CHECK();
      join_emit_kernel<FrontierSource, Geom>
        <<<blocks, kScanThreads, 0, stream>>>(src, t, bx, g, s, partials);
    }
    QPIP_LAUNCH_CHECK();
  }
}

}  // namespace qpip
