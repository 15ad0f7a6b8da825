// join_quadtree_and_bounding_boxes on gfx950.
//
// Reference: cpp/src/join/quadtree_bbox_filtering.cu:90-126 (column API, checks)
// and detail/join/quadtree_bbox_filtering.cuh:37-188 with intersection.cuh:79-136
// and traversal.cuh:63-145: a breadth-first traversal that starts from every
// (level-0 node, bbox) pair (node = i % T, bbox = i / T), classifies each pair
// as leaf / quad / none, emits leaf pairs in order, expands quad pairs to their
// children in order, and finally stable-sorts the leaf pairs by the leaf's first
// point position.
//
// Here the same traversal runs entirely on the device, one count/scan/emit per step
// of one to three levels (qpip_join.hpp) with the frontier length kept in device memory (the
// reference syncs the host on every level for sizes, traversal.cuh:222). The stable
// sort is the library's LSD radix sort over the bits of the largest leaf offset.
// Frontier/output capacities are preallocated; on overflow the traversal is
// rerun with the sizes the device recorded.
#include <algorithm>

#include "qpip_join.hpp"

namespace qpip {

namespace {

// Level 0: the virtual frontier i -> (i % T, i / T).
struct TopSource {
  JoinMeta const* meta;
  __device__ __forceinline__ uint64_t size() const { return meta->top_pairs; }
  __device__ __forceinline__ bool root(TreeView const&, uint64_t i, uint32_t& node, uint32_t& bbox,
                                       uint32_t& first, uint32_t& n) const
  {
    uint32_t const T = meta->num_top;
    node             = static_cast<uint32_t>(i % T);
    bbox             = static_cast<uint32_t>(i / T);
    first            = node;
    n                = 1;
    return true;
  }
};

// T = count(level == 0) (quadtree_bbox_filtering.cuh:53-56), T * B and the largest leaf
// offset (for the sort's bit count), into a zeroed *meta. One atomic per block and
// value; the last block to finish writes the product. (One atomic per wave on the
// largest offset took 50 us for 1.2M nodes, next to four launches for the rest.)
__global__ void __launch_bounds__(256)
  join_setup_kernel(uint8_t const* __restrict__ level, uint8_t const* __restrict__ internal,
                    uint32_t const* __restrict__ offset, uint64_t m, uint64_t boxes,
                    JoinMeta* __restrict__ meta)
{
  __shared__ uint32_t s_top[256 / kWave], s_max[256 / kWave];
  uint32_t top = 0, mx = 0;
#pragma unroll 4
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < m;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    uint32_t const o = offset[i];
    top += level[i] == 0 ? 1u : 0u;
    if (!internal[i]) mx = max(mx, o);
  }
  top = wave_sum(top);
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1)
    mx = max(mx, static_cast<uint32_t>(__shfl_xor(mx, o, kWave)));
  if (lane_id() == 0) {
    s_top[threadIdx.x / kWave] = top;
    s_max[threadIdx.x / kWave] = mx;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < 256 / kWave; ++w) {
    top += s_top[w];
    mx = max(mx, s_max[w]);
  }
  if (top) atomicAdd(&meta->num_top, top);
  if (mx) atomicMax(&meta->max_leaf_offset, mx);
  __threadfence();
  if (atomicAdd(&meta->tickets, 1u) + 1 == gridDim.x) {
    __threadfence();
    meta->top_pairs = static_cast<uint64_t>(atomicAdd(&meta->num_top, 0u)) * boxes;
  }
}

__global__ void __launch_bounds__(256)
  permute_pairs_kernel(uint32_t const* __restrict__ perm, uint32_t const* __restrict__ out_node,
                       uint32_t const* __restrict__ out_bbox, uint64_t k,
                       uint32_t* __restrict__ bbox_offset, uint32_t* __restrict__ quad_offset)
{
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < k;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    uint32_t const j = perm[i];
    bbox_offset[i]   = out_bbox[j];
    quad_offset[i]   = out_node[j];
  }
}

}  // namespace

}  // namespace qpip

extern "C" int qpip_join_quadtree_and_bounding_boxes(const uint32_t* key,
                                                     const uint8_t* level,
                                                     const uint8_t* is_internal_node,
                                                     const uint32_t* length,
                                                     const uint32_t* offset,
                                                     int64_t num_nodes,
                                                     const double* bbox_minx,
                                                     const double* bbox_miny,
                                                     const double* bbox_maxx,
                                                     const double* bbox_maxy,
                                                     int64_t num_bboxes,
                                                     double x_min,
                                                     double x_max,
                                                     double y_min,
                                                     double y_max,
                                                     double scale,
                                                     int8_t max_depth,
                                                     const qpip_resource* mr,
                                                     void* stream_,
                                                     uint32_t** bbox_offset,
                                                     uint32_t** quad_offset,
                                                     int64_t* num_pairs)
{
  using namespace qpip;
  try {
    QPIP_EXPECTS(bbox_offset && quad_offset && num_pairs, "output pointers must not be null");
    *bbox_offset = *quad_offset = nullptr;
    *num_pairs                  = 0;
    hipStream_t stream          = static_cast<hipStream_t>(stream_);
    // quadtree_bbox_filtering.cu:100-114
    QPIP_EXPECTS(scale > 0, "scale must be positive");
    QPIP_EXPECTS(x_min < x_max && y_min < y_max, "invalid bounding box (x_min, x_max, y_min, y_max)");
    QPIP_EXPECTS(max_depth > 0 && max_depth < 16, "maximum depth must be positive and less than 16");
    if (num_nodes <= 0 || num_bboxes <= 0) return QPIP_SUCCESS;
    QPIP_EXPECTS(num_nodes < (int64_t{1} << 32) && num_bboxes < (int64_t{1} << 32),
                 "quadtree and bounding box tables must have fewer than 2^32 rows");

    StreamScope scope(stream);
    TreeView tv{key, level, is_internal_node, length, offset, static_cast<uint64_t>(num_nodes)};
    BoxView bv{bbox_minx, bbox_miny, bbox_maxx, bbox_maxy, static_cast<uint64_t>(num_bboxes)};
    Params prm{x_min, y_min, scale, static_cast<int>(max_depth)};
    uint64_t const M = static_cast<uint64_t>(num_nodes);
    uint64_t const B = static_cast<uint64_t>(num_bboxes);

    dbuf<JoinMeta> meta(1);
    dbuf<StepCount> partials(kScanBlocks), counts;

    uint64_t cap_out = std::max<uint64_t>(uint64_t{1} << 20, 8 * B);
    uint64_t cap_fr  = std::max<uint64_t>(uint64_t{1} << 20, 8 * B);
    JoinMeta h_meta{};
    dbuf<uint32_t> out_node, out_bbox, ka, fa_node, fa_bbox, fb_node, fb_bbox;
    for (int attempt = 0;; ++attempt) {
      out_node.reset(cap_out);
      out_bbox.reset(cap_out);
      ka.reset(cap_out);
      counts.reset(cap_fr);
      fa_node.reset(cap_fr);
      fa_bbox.reset(cap_fr);
      fb_node.reset(cap_fr);
      fb_bbox.reset(cap_fr);
      QPIP_HIP(hipMemsetAsync(meta.get(), 0, sizeof(JoinMeta), stream));
      JoinMeta* dm = meta.get();
      {
        KernelTimer kt("join_setup", stream);
        join_setup_kernel<<<grid_for(M, 4 * 256, 256), 256, 0, stream>>>(level, is_internal_node,
                                                                         offset, M, B, dm);
        QPIP_LAUNCH_CHECK();
      }
      // quadtree_bbox_filtering.cuh:116-163: levels 0 .. max_depth - 1
      JoinSink const sink{dm, out_node.get(), out_bbox.get(), ka.get(), nullptr, nullptr,
                          counts.get(), cap_out, cap_fr, 0, 0};
      launch_join(TopSource{dm}, tv, bv, prm, sink, {fa_node.get(), fb_node.get()},
                  {fa_bbox.get(), fb_bbox.get()}, max_depth, join_shape(M, B), partials.get(), stream,
                  "join_level");
      read_back({{&h_meta, dm, sizeof(JoinMeta)}}, stream);
      if (h_meta.bad_index)
        throw logic_error("cuSpatial failure: quadtree child range exceeds the number of nodes");
      if (!h_meta.overflow) break;
      // grow to what the device saw (plus headroom) and rerun
      uint64_t tot_out = 0, max_fr = h_meta.top_pairs;
      for (int l = 0; l < max_depth; ++l) {
        tot_out += h_meta.level[l].leaf;
        max_fr = std::max<uint64_t>(max_fr, h_meta.level[l].quad);
      }
      cap_out = std::max<uint64_t>(cap_out * 2, tot_out + tot_out / 4 + 1024);
      cap_fr  = std::max<uint64_t>(cap_fr * 2, max_fr + max_fr / 4 + 1024);
      if (attempt > 8) throw device_error("join capacity growth did not converge");
    }
    uint64_t K = 0;
    for (int l = 0; l < max_depth; ++l) K += h_meta.level[l].leaf;
    if (K == 0) return QPIP_SUCCESS;
    QPIP_EXPECTS(K < (uint64_t{1} << 32), "join produced more than 2^32 pairs");

    // stable_sort_by_key(offset[leaf], (bbox, leaf)) (quadtree_bbox_filtering.cuh:152-166)
    dbuf<uint32_t> kb(K), va(K), vb(K);
    int bits = 1;
    while (bits < 32 && (h_meta.max_leaf_offset >> bits) != 0) ++bits;
    SortResult s = radix_sort_pairs(ka.get(), kb.get(), nullptr, va.get(), vb.get(), K, bits,
                                    stream, nullptr, "join_sort");
    OutputAllocator oa(mr, stream);
    uint32_t* o_bbox = oa.make<uint32_t>(K);
    uint32_t* o_quad = oa.make<uint32_t>(K);
    permute_pairs_kernel<<<grid_for(K, 256), 256, 0, stream>>>(s.values, out_node.get(),
                                                               out_bbox.get(), K, o_bbox, o_quad);
    QPIP_LAUNCH_CHECK();
    oa.keep();
    *bbox_offset = o_bbox;
    *quad_offset = o_quad;
    *num_pairs   = static_cast<int64_t>(K);
    return QPIP_SUCCESS;
  } catch (...) {
    return qpip::error_status();
  }
}
