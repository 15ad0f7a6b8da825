// quadtree_point_to_nearest_linestring and linestring_bounding_boxes.
//
// Nearest linestring (detail/join/quadtree_point_to_nearest_linestring.cuh:143-314,
// cpp/src/join/quadtree_point_to_nearest_linestring.cu:128-189): for every point of a
// leaf that the (linestring, quadrant) join paired with linestrings, the distance
// to each of those linestrings (detail/algorithm/point_linestring_distance.cuh:33-51)
// and the one kept by the reference's reduce_by_key operator: the smallest nonzero
// distance, ties to the lower linestring id; a zero distance yields to any other
// (:279-294). That operator is associative (zero distances are identities unless
// every distance is zero, when the last pair of the run wins), so a left fold over
// the run's pairs in pair order gives the reference's result.
//
// Output has one row per entry of point_indices (the reference sizes its outputs
// by the point count, :257-264): row p is (p, nearest linestring, distance) for a
// point in a paired leaf. The reference leaves the two index columns of the other
// rows uninitialized (distance 0); here they are (p, 0xffffffff, 0).
//
// The join sorts pairs by leaf offset, so the pairs on one leaf form a run. One wave
// per 64-point chunk of a run's leaf (nearest_chunk_kernel) finds each point's nearest
// linestring with a float32 distance in coordinates local to the chunk, and computes
// the reference's double arithmetic for that linestring alone; points whose float32
// distances do not decide fold over every linestring. Pairs that are not sorted, or
// that put two quadrants on one offset, take nearest_kernel, which finds the run of
// every pair as the reference does (lower and upper bound of its leaf's offset).
#include <algorithm>
#include <cmath>

#include "qpip_scan.hpp"

namespace qpip {

namespace {

struct NearestArgs {
  uint32_t const* pair_ls;
  uint32_t const* pair_quad;
  uint64_t num_pairs;
  uint32_t const* length;
  uint32_t const* offset;
  uint64_t num_nodes;
  uint32_t const* point_indices;
  uint64_t num_points;
  double const* x;
  double const* y;
  uint32_t const* ls_offsets;
  uint64_t num_ls;
  double const* lx;
  double const* ly;
  uint64_t num_vertices;
  uint32_t* out_point;
  uint32_t* out_ls;
  double* out_dist;
  uint32_t* bad;
};

// *bad: bit 1 an index out of range, bit 2 pairs that do not form runs of one leaf in
// offset order (or more chunks than the work list holds): nearest_kernel runs then.
constexpr uint32_t kBadIndex = 1u, kIrregular = 2u;

template <class T>
__device__ __forceinline__ T uniform_load(T const* p)
{
  return __builtin_amdgcn_readfirstlane(*p);
}

__device__ __forceinline__ double uniform_d(double const* p)
{
  uint64_t const b = static_cast<uint64_t>(__double_as_longlong(*p));
  uint32_t const lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b));
  uint32_t const hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b >> 32));
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

// dot(a, b) = a.x * b.x + a.y * b.y as fma(a.x, b.x, a.y * b.y): the form that
// reproduces the reference's expected distances bit for bit
// (quadtree_point_to_nearest_linestring_test_small.cu:173-192).
__device__ __forceinline__ double dot2(double ax, double ay, double bx, double by)
{
  return fma(ax, bx, ay * by);
}

// point_linestring_distance (detail/algorithm/point_linestring_distance.cuh:33-51):
// min over the segments (v[i], v[i+1]) of the squared distance, then the square
// root.
// One segment's squared distance, folded into dsq.
__device__ __forceinline__ double fold_segment(double dsq, double ax, double ay, double bx,
                                               double by, double px, double py)
{
  double const v1x = px - ax, v1y = py - ay;
  double const v2x = px - bx, v2y = py - by;
  double const ex = bx - ax, ey = by - ay;
  double const d0 = dot2(v1x, v1y, v1x, v1y);
  double const d1 = dot2(v2x, v2y, v2x, v2y);
  double const d2 = dot2(ex, ey, ex, ey);
  double const d3 = dot2(v1x, v1y, ex, ey);
  double const r  = d3 * d3 / d2;
  double const d  = (d3 <= 0.0 || r >= d2) ? fmin(d0, d1) : d0 - r;
  return fmin(dsq, d);
}

constexpr double kNoDistance = 1.7976931348623157e308;  // numeric_limits<double>::max()

// The linestring is the same in every lane (its vertices are loaded once per wave).
__device__ __forceinline__ double point_linestring_distance(NearestArgs const& a, uint32_t ls,
                                                            double px, double py)
{
  uint64_t v0 = uniform_load(a.ls_offsets + ls);
  uint64_t v1 = uniform_load(a.ls_offsets + ls + 1);
  if (v1 > a.num_vertices) v1 = a.num_vertices;
  double dsq = kNoDistance;
  for (uint64_t i = v0; i + 1 < v1; ++i)
    dsq = fold_segment(dsq, uniform_d(a.lx + i), uniform_d(a.ly + i), uniform_d(a.lx + i + 1),
                       uniform_d(a.ly + i + 1), px, py);
  return sqrt(dsq);
}

// Each lane has its own linestring.
__device__ __forceinline__ double own_linestring_distance(NearestArgs const& a, uint32_t ls,
                                                          double px, double py)
{
  uint64_t v0 = a.ls_offsets[ls], v1 = a.ls_offsets[ls + 1];
  if (v1 > a.num_vertices) v1 = a.num_vertices;
  double dsq = kNoDistance;
  if (v0 + 1 < v1) {
    double ax = a.lx[v0], ay = a.ly[v0];
    for (uint64_t i = v0 + 1; i < v1; ++i) {
      double const bx = a.lx[i], by = a.ly[i];
      dsq = fold_segment(dsq, ax, ay, bx, by, px, py);
      ax  = bx;
      ay  = by;
    }
  }
  return sqrt(dsq);
}

// The reference's choice between the kept (linestring, distance) and the next pair's
// (quadtree_point_to_nearest_linestring.cuh:279-294, lhs = kept, rhs = next).
__device__ __forceinline__ bool take_next(double best_d, uint32_t best_ls, double d, uint32_t ls)
{
  if (best_d == 0.0) return true;
  if (d == 0.0) return false;
  if (best_d == d) return !(best_ls < ls);
  return !(best_d < d);
}

// The fold over a run's pairs [rs, re), for every active lane.
__device__ __forceinline__ void fold_run(NearestArgs const& a, uint64_t rs, uint64_t re, double px,
                                         double py, uint32_t& best_ls, double& best_d, bool& err)
{
  best_ls = 0;
  best_d  = 0.0;
  for (uint64_t k = rs; k < re; ++k) {
    uint32_t const ls = uniform_load(a.pair_ls + k);
    if (ls >= a.num_ls) {
      err = true;
      continue;
    }
    double const d = point_linestring_distance(a, ls, px, py);
    if (k == rs || take_next(best_d, best_ls, d, ls)) {
      best_ls = ls;
      best_d  = d;
    }
  }
}

__device__ __forceinline__ double lane_value(double v, uint32_t lane)
{
  uint64_t const b = static_cast<uint64_t>(__double_as_longlong(v));
  auto half        = [&](uint64_t w) {
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w), lane));
  };
  return __longlong_as_double(
    static_cast<long long>((static_cast<uint64_t>(half(b >> 32)) << 32) | half(b)));
}

// The same fold for one point, (px, py) in every lane of a full wave: 64 pairs at a time,
// a linestring per lane. Where all distances are positive the fold is the smallest
// (distance, linestring), whatever the order; with a zero or a NaN among them it goes pair
// by pair.
__device__ __forceinline__ void fold_point(NearestArgs const& a, uint64_t rs, uint64_t re,
                                           double px, double py, uint32_t& best_ls,
                                           double& best_d, bool& err)
{
  best_ls = 0;
  best_d  = 0.0;
  for (uint64_t kb = rs; kb < re; kb += kWave) {
    bool const in = kb + lane_id() < re;
    uint32_t ls   = in ? a.pair_ls[kb + lane_id()] : 0u;
    bool const ok = in && ls < a.num_ls;
    if (in && !ok) err = true;
    double d = ok ? own_linestring_distance(a, ls, px, py) : INFINITY;
    if (ballot(ok && !(d > 0.0)) == 0) {
      if (!ok) ls = 0xffffffffu;
#pragma unroll
      for (int o = kWave / 2; o > 0; o >>= 1) {
        double const od   = __shfl_xor(d, o, kWave);
        uint32_t const ol = __shfl_xor(ls, o, kWave);
        if (od < d || (od == d && ol < ls)) {
          d  = od;
          ls = ol;
        }
      }
      if (ls < a.num_ls && take_next(best_d, best_ls, d, ls)) {
        best_ls = ls;
        best_d  = d;
      }
    } else {
      for (uint64_t m = ballot(ok); m; m &= m - 1) {
        uint32_t const j  = static_cast<uint32_t>(__builtin_ctzll(m));
        double const dj   = lane_value(d, j);
        uint32_t const lj = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ls), j));
        if (take_next(best_d, best_ls, dj, lj)) {
          best_ls = lj;
          best_d  = dj;
        }
      }
    }
  }
}

__global__ void __launch_bounds__(256) nearest_fill_kernel(NearestArgs a)
{
  uint64_t const p = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= a.num_points) return;
  a.out_point[p] = static_cast<uint32_t>(p);
  a.out_ls[p]    = 0xffffffffu;
  a.out_dist[p]  = 0.0;
}

// Pairs [base, base + waves of the grid): the host launches slices of 2^22 pairs so
// that a grid stays within 2^28 work-items.
__global__ void __launch_bounds__(256) nearest_kernel(NearestArgs a, uint64_t base)
{
  uint64_t const k0 = base + __builtin_amdgcn_readfirstlane(
    static_cast<uint32_t>(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave));
  if (k0 >= a.num_pairs) return;
  uint32_t const quad = uniform_load(a.pair_quad + k0);
  if (quad >= a.num_nodes) {
    if (lane_id() == 0) atomicOr(a.bad, kBadIndex);
    return;
  }
  uint32_t const len   = uniform_load(a.length + quad);
  uint32_t const first = uniform_load(a.offset + quad);
  // The run of pairs on this leaf, found as the reference finds it
  // (quadtree_point_to_nearest_linestring.cuh:44-61): lower and upper bound of the
  // leaf's offset among the pairs' quadrant offsets (the join orders pairs by them).
  auto off_at = [&](uint64_t k) -> uint32_t {
    uint32_t const q = uniform_load(a.pair_quad + k);
    return q < a.num_nodes ? uniform_load(a.offset + q) : 0xffffffffu;
  };
  uint64_t lo = 0, hi = k0;
  while (lo < hi) {
    uint64_t const mid = (lo + hi) / 2;
    if (off_at(mid) < first) lo = mid + 1;
    else hi = mid;
  }
  uint64_t const rs = lo;
  lo = k0 + 1;
  hi = a.num_pairs;
  while (lo < hi) {
    uint64_t const mid = (lo + hi) / 2;
    if (off_at(mid) <= first) lo = mid + 1;
    else hi = mid;
  }
  uint64_t const re     = lo;
  uint64_t const R      = re - rs;
  uint64_t const mine   = k0 - rs;
  uint64_t const chunks = (static_cast<uint64_t>(len) + kWave - 1) / kWave;
  int const lane        = lane_id();
  bool err              = false;
  for (uint64_t c = mine; c < chunks; c += R) {
    uint64_t const local = c * kWave + lane;
    if (local >= len) continue;
    uint64_t const pos = static_cast<uint64_t>(first) + local;
    if (pos >= a.num_points) {
      err = true;
      continue;
    }
    uint32_t const idx = a.point_indices[pos];
    if (idx >= a.num_points) {
      err = true;
      continue;
    }
    double const px = a.x[idx], py = a.y[idx];
    uint32_t best_ls;
    double best_d;
    fold_run(a, rs, re, px, py, best_ls, best_d, err);
    a.out_point[pos] = static_cast<uint32_t>(pos);
    a.out_ls[pos]    = best_ls;
    a.out_dist[pos]  = best_d;
  }
  if (err) atomicOr(a.bad, kBadIndex);
}

// Work list: the 64-point chunks of every run's leaf, as (first pair, chunk).
struct RunChunkOp {
  NearestArgs a;
  uint2* items;
  uint64_t cap;
  __device__ __forceinline__ uint32_t off(uint64_t k, uint32_t& q) const
  {
    q = a.pair_quad[k];
    return q < a.num_nodes ? a.offset[q] : 0xffffffffu;
  }
  __device__ uint64_t count(uint64_t k) const
  {
    uint32_t q, p = 0xffffffffu;
    uint32_t const o = off(k, q);
    if (q >= a.num_nodes) {
      atomicOr(a.bad, kBadIndex);
      return 0;
    }
    if (k > 0) {
      uint32_t const before = off(k - 1, p);
      if (before > o || (before == o && p != q)) atomicOr(a.bad, kIrregular);
    }
    return p == q ? 0ull : (static_cast<uint64_t>(a.length[q]) + kWave - 1) / kWave;
  }
  __device__ void emit(uint64_t k, uint64_t prefix) const
  {
    uint64_t const n = count(k);
    if (n == 0) return;
    if (prefix + n > cap) {
      atomicOr(a.bad, kIrregular);
      return;
    }
    for (uint64_t c = 0; c < n; ++c)
      items[prefix + c] = make_uint2(static_cast<uint32_t>(k), static_cast<uint32_t>(c));
  }
};

// One wave per work item. Each lane holds one point; a chunk of at most 32 points is
// held in 64 / 2^ceil(log2 points) copies that take different segments. The run's
// linestrings pass through the wave's LDS slot 63 segments at a time, in float32
// coordinates relative to the chunk's first point (start, direction and 1 / length^2
// per segment: 11 float32 instructions per point and segment instead of about 45
// double ones with a division), the vertices of the next batch in flight meanwhile.
//
// With M the largest float32 coordinate met (points and vertices), every float32
// distance is within 2^-19 M of the exact one (rounded ends, direction, projection and
// difference: at most 31 roundings of 2^-24 M), and so is the reference's double result
// (within 2^-23 M: the cancellation of d0 - r) except where
//  * the point lies on a segment: d0 - r may round below zero, and the distance is NaN;
//  * a segment's length^2 and its d3^2 underflow to 0: r = 0 / 0, and fmin drops the
//    segment, so the distance comes out larger.
// E = 2^-17 M + 1e-14 bounds both kinds of rounding. Where one float32 distance is more
// than 2 E below every other, no other linestring comes out as near, as zero or as NaN
// (the first exception needs a distance below 2^-23 M, the second only adds to one). If
// the reference's distance to that linestring is then within E of the float32 one it is
// the answer. Otherwise (an exception above, two linestrings that near, a zero distance,
// a linestring without segments, coordinates that are not finite or above 1e15) the point
// folds over the run's pairs, as the reference does: a few such points one after the
// other with a linestring per lane (fold_point), many at once with the linestrings in
// turn (fold_run), and so does every point of a run of one pair, which leaves no choice.
// One such point had held its wave for the whole fold: 1,000 points, 20,000 linestrings
// (1,355 per leaf) took 5.8 ms, 2.3 so and 4.5 with a wave per pair.
//
// Bound by the float32 instructions. 1e6 points, 20,000 linestrings of 2 to 32
// vertices (about 15 per leaf of 61 points): one wave per pair, each segment a chain of
// scalar loads and a double division, took 1232 us; this takes 253 us (359 with every point
// not decided in float32 folding with the linestrings in turn).
constexpr int kNearWaves = 4;
struct NearSegments {
  float4 s[kWave];  // start, direction
  float inv[kWave];
};

__global__ void __launch_bounds__(kNearWaves * kWave)
  nearest_chunk_kernel(NearestArgs a, uint2 const* __restrict__ items,
                       uint64_t const* __restrict__ total, uint64_t cap)
{
  __shared__ NearSegments s_seg[kNearWaves];
  NearSegments& S   = s_seg[threadIdx.x / kWave];
  uint64_t const w  = static_cast<uint64_t>(blockIdx.x) * kNearWaves + threadIdx.x / kWave;
  uint64_t const T  = *total;
  if (w >= T || T > cap) return;
  int const lane    = lane_id();
  uint2 const item  = items[w];
  uint64_t const rs = uniform(item.x);
  uint32_t const c  = uniform(item.y);
  uint32_t const quad  = uniform_load(a.pair_quad + rs);
  uint32_t const len   = uniform_load(a.length + quad);
  uint32_t const first = uniform_load(a.offset + quad);
  // the run's end: its pairs name the same quadrant
  uint64_t R = 0;
  while (true) {
    uint64_t const k = rs + R + lane;
    uint64_t const b = ballot(k < a.num_pairs && a.pair_quad[k] == quad);
    R += b == ~0ull ? 64 : __builtin_ctzll(~b);
    if (b != ~0ull) break;
  }
  uint32_t const q  = len - c * kWave < kWave ? len - c * kWave : kWave;
  uint32_t const lq = q > 1 ? 32u - static_cast<uint32_t>(__builtin_clz(q - 1)) : 0u;
  uint32_t const Q = 1u << lq, G = kWave >> lq;  // lanes per copy, copies
  uint32_t const at = static_cast<uint32_t>(lane) & (Q - 1), g = static_cast<uint32_t>(lane) >> lq;
  bool err       = false;
  bool valid     = at < q;
  uint64_t const pos = static_cast<uint64_t>(first) + c * static_cast<uint64_t>(kWave) + at;
  double px = 0.0, py = 0.0;
  if (valid) {
    uint32_t const idx = pos < a.num_points ? a.point_indices[pos] : 0xffffffffu;
    if (idx >= a.num_points) {
      err   = true;
      valid = false;
    } else {
      px = a.x[idx];
      py = a.y[idx];
    }
  }
  // readfirstlane of the first copy's first point (0 where that is not finite)
  auto first_lane = [](double v) {
    uint64_t const b = static_cast<uint64_t>(__double_as_longlong(v));
    return __longlong_as_double(static_cast<long long>(
      (static_cast<uint64_t>(uniform(static_cast<uint32_t>(b >> 32))) << 32) |
      uniform(static_cast<uint32_t>(b))));
  };
  double const ox = first_lane(isfinite(px) ? px : 0.0), oy = first_lane(isfinite(py) ? py : 0.0);
  float const fx = static_cast<float>(px - ox), fy = static_cast<float>(py - oy);
  constexpr float kTop = 1e15f;  // squares and their sums stay finite
  auto small = [](float x, float y) { return fabsf(x) <= kTop && fabsf(y) <= kTop; };  // not NaN
  bool decided = valid && small(fx, fy);
  float M      = decided ? fmaxf(fabsf(fx), fabsf(fy)) : 0.f;
  float m1 = INFINITY, m2 = INFINITY;
  uint64_t l1 = rs;
  bool odd    = false;  // a vertex or linestring index the float32 pass cannot take
  auto fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  for (uint64_t kb = 0; R > 1 && kb < R; kb += kWave) {
    // the next 64 pairs' vertex ranges, one per lane
    uint32_t const nj = R - kb < kWave ? static_cast<uint32_t>(R - kb) : kWave;
    uint32_t v_lo = 0, v_n = 0;  // first vertex, segments
    if (static_cast<uint32_t>(lane) < nj) {
      uint32_t const ls = a.pair_ls[rs + kb + lane];
      if (ls >= a.num_ls) {
        err = true;
      } else {
        uint64_t const b = a.ls_offsets[ls];
        uint64_t e       = a.ls_offsets[ls + 1];
        if (e > a.num_vertices) e = a.num_vertices;
        if (b + 1 < e) {
          v_lo = static_cast<uint32_t>(b);
          v_n  = static_cast<uint32_t>(e - b - 1);
        }
      }
    }
    // batches (pair j, segment s): 63 segments are 64 vertices, one per lane
    auto next_pair = [&](uint32_t j) {  // the first pair from j on with a segment
      uint64_t const m = ballot(v_n > 0) & (j < kWave ? ~0ull << j : 0ull);
      return m ? static_cast<uint32_t>(__builtin_ctzll(m)) : static_cast<uint32_t>(kWave);
    };
    auto rl = [](uint32_t v, uint32_t j) {
      return static_cast<uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(j)));
    };
    uint32_t j = next_pair(0), sb = 0;
    double vx = 0.0, vy = 0.0;
    auto load = [&](uint32_t jj, uint32_t ss) {
      uint32_t const n = rl(v_n, jj) - ss < 63u ? rl(v_n, jj) - ss : 63u;
      if (static_cast<uint32_t>(lane) <= n) {
        uint64_t const v = static_cast<uint64_t>(rl(v_lo, jj)) + ss + lane;
        vx               = a.lx[v];
        vy               = a.ly[v];
      }
    };
    if (j < kWave) load(j, 0);
    float m = INFINITY;
    while (j < kWave) {
      uint32_t const left = rl(v_n, j) - sb;
      uint32_t const n    = left < 63u ? left : 63u;
      float const sx = static_cast<float>(vx - ox), sy = static_cast<float>(vy - oy);
      if (static_cast<uint32_t>(lane) <= n) {
        if (small(sx, sy))
          M = fmaxf(M, fmaxf(fabsf(sx), fabsf(sy)));
        else
          odd = true;
      }
      float const ex = __shfl_down(sx, 1, kWave) - sx, ey = __shfl_down(sy, 1, kWave) - sy;
      float const l2 = ex * ex + ey * ey;
      fence();
      if (static_cast<uint32_t>(lane) < n) {
        S.s[lane]   = make_float4(sx, sy, ex, ey);
        S.inv[lane] = l2 > 1e-30f ? 1.f / l2 : 0.f;
      }
      fence();
      // the next batch's vertices
      bool const last   = left <= 63u;
      uint32_t const jn = last ? next_pair(j + 1) : j, sn = last ? 0u : sb + 63u;
      if (jn < kWave) load(jn, sn);
#pragma unroll 4
      for (uint32_t s = g; s < n; s += G) {
        float4 const e = S.s[s];
        float const wx = fx - e.x, wy = fy - e.y;
        float const t =
          __builtin_amdgcn_fmed3f(fmaf(wx, e.z, wy * e.w) * S.inv[s], 0.f, 1.f);
        float const dx = fmaf(-t, e.z, wx), dy = fmaf(-t, e.w, wy);
        m = fminf(m, fmaf(dx, dx, dy * dy));
      }
      if (last) {
        for (uint32_t o = Q; o < kWave; o <<= 1) m = fminf(m, __shfl_xor(m, o, kWave));
        if (m < m1) {
          m2 = m1;
          m1 = m;
          l1 = rs + kb + j;
        } else {
          m2 = fminf(m2, m);
        }
        m = INFINITY;
      }
      j  = jn;
      sb = sn;
    }
  }
  if (ballot(odd || err)) decided = false;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, kWave));
  float const E = fmaf(M, 0x1p-17f, 1e-14f);
  decided       = decided && m1 < INFINITY && sqrtf(m1) + E < sqrtf(m2) - E;
  bool const own = valid && g == 0;
  uint32_t best_ls = 0;
  double best_d    = 0.0;
  if (own && decided) {
    best_ls = a.pair_ls[l1];
    if (ballot(best_ls != uniform(best_ls)) == 0)  // one for all: its vertices loaded once
      best_d = point_linestring_distance(a, uniform(best_ls), px, py);
    else
      best_d = own_linestring_distance(a, best_ls, px, py);
    decided = best_d > 0.0 && fabs(best_d - static_cast<double>(sqrtf(m1))) <= E;  // not NaN
  }
  uint64_t const todo = ballot(own && !decided);
  if (3 * static_cast<uint64_t>(__popcll(todo)) * ((R + kWave - 1) / kWave) < R) {
    for (uint64_t m = todo; m; m &= m - 1) {
      uint32_t const j = static_cast<uint32_t>(__builtin_ctzll(m));
      uint32_t ls;
      double d;
      fold_point(a, rs, rs + R, lane_value(px, j), lane_value(py, j), ls, d, err);
      if (static_cast<uint32_t>(lane) == j) {
        best_ls = ls;
        best_d  = d;
      }
    }
  } else if (own && !decided) {
    fold_run(a, rs, rs + R, px, py, best_ls, best_d, err);
  }
  if (own) {
    a.out_point[pos] = static_cast<uint32_t>(pos);
    a.out_ls[pos]    = best_ls;
    a.out_dist[pos]  = best_d;
  }
  if (err) atomicOr(a.bad, kBadIndex);
}

__global__ void iota_i32_kernel(int32_t* __restrict__ p, int64_t n)
{
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = static_cast<int32_t>(i);
}

}  // namespace

}  // namespace qpip

using namespace qpip;

extern "C" int qpip_quadtree_point_to_nearest_linestring(const uint32_t* linestring_index,
                                                         const uint32_t* quad_index,
                                                         int64_t num_pairs,
                                                         const uint32_t* key,
                                                         const uint8_t* level,
                                                         const uint8_t* is_internal_node,
                                                         const uint32_t* length,
                                                         const uint32_t* offset,
                                                         int64_t num_nodes,
                                                         const uint32_t* point_indices,
                                                         int64_t num_point_indices,
                                                         const double* x,
                                                         const double* y,
                                                         int64_t num_x,
                                                         int64_t num_y,
                                                         const uint32_t* linestring_offsets,
                                                         int64_t num_linestring_offsets,
                                                         const double* linestring_x,
                                                         const double* linestring_y,
                                                         int64_t num_linestring_x,
                                                         int64_t num_linestring_y,
                                                         const qpip_resource* mr,
                                                         void* stream_,
                                                         uint32_t** point_index,
                                                         uint32_t** nearest_linestring_index,
                                                         double** distance,
                                                         int64_t* num_rows)
{
  (void)key;
  (void)level;
  (void)is_internal_node;
  try {
    QPIP_EXPECTS(point_index && nearest_linestring_index && distance && num_rows,
                 "output pointers must not be null");
    *point_index = *nearest_linestring_index = nullptr;
    *distance                                = nullptr;
    *num_rows                                = 0;
    auto stream = static_cast<hipStream_t>(stream_);
    // quadtree_point_to_nearest_linestring.cu:153-166 (column counts and dtypes are the
    // binding's: 2 + 5 columns, uint32 indices, f64 coordinates)
    QPIP_EXPECTS(num_point_indices == num_x && num_x == num_y,
                 "number of points must be the same for both x and y columns");
    QPIP_EXPECTS(num_linestring_x == num_linestring_y,
                 "numbers of vertices must be the same for both x and y columns");
    // :168-176: empty inputs give empty columns
    if (num_pairs == 0 || num_nodes == 0 || num_point_indices == 0 ||
        num_linestring_offsets == 0)
      return QPIP_SUCCESS;
    int64_t const n = num_point_indices;
    StreamScope scope(stream);
    OutputAllocator oa(mr, stream);
    uint32_t* o_point = oa.make<uint32_t>(n);
    uint32_t* o_ls    = oa.make<uint32_t>(n);
    double* o_dist    = oa.make<double>(n);
    dbuf<uint32_t> bad(1);
    fill_u32(bad.get(), 1, 0u, stream);
    NearestArgs a{linestring_index, quad_index, static_cast<uint64_t>(num_pairs), length, offset,
                  static_cast<uint64_t>(num_nodes), point_indices, static_cast<uint64_t>(n), x, y,
                  linestring_offsets, static_cast<uint64_t>(num_linestring_offsets - 1),
                  linestring_x, linestring_y, static_cast<uint64_t>(num_linestring_x), o_point,
                  o_ls, o_dist, bad.get()};
    uint64_t const K = static_cast<uint64_t>(num_pairs);
    auto fill = [&] {
      KernelTimer kt("nearest_fill", stream);
      nearest_fill_kernel<<<grid_for(static_cast<uint64_t>(n), 256, 1u << 30), 256, 0, stream>>>(a);
      QPIP_LAUNCH_CHECK();
    };
    uint32_t h_bad = 0;
    auto status = [&] { read_back({{&h_bad, bad.get(), sizeof(uint32_t)}}, stream); };
    fill();
    // chunks of the paired leaves: a tree's leaves hold each point once
    uint64_t const cap = static_cast<uint64_t>(n) / kWave +
                         std::min<uint64_t>(K, static_cast<uint64_t>(num_nodes));
    if (K < (uint64_t{1} << 32) && cap < (uint64_t{1} << 31)) {
      dbuf<uint2> items(cap);
      dbuf<uint64_t> partials(kScanBlocks), total(1);
      count_scan_emit<RunChunkOp, uint64_t, uint64_t>(RunChunkOp{a, items.get(), cap}, nullptr, K,
                                                      partials.get(), total.get(), stream,
                                                      scan_blocks_for(K), "nearest_chunks");
      {
        KernelTimer kt("nearest_linestring", stream);
        nearest_chunk_kernel<<<static_cast<unsigned>((cap + kNearWaves - 1) / kNearWaves),
                               kNearWaves * kWave, 0, stream>>>(a, items.get(), total.get(), cap);
        QPIP_LAUNCH_CHECK();
      }
      status();
    } else {
      h_bad = kIrregular;
    }
    if (h_bad & kIrregular) {
      fill_u32(bad.get(), 1, 0u, stream);
      fill();
      KernelTimer kt("nearest_linestring", stream);
      for (uint64_t b = 0; b < K; b += uint64_t{1} << 22) {
        uint64_t const m = std::min<uint64_t>(K - b, uint64_t{1} << 22);
        nearest_kernel<<<static_cast<unsigned>((m + 3) / 4), 256, 0, stream>>>(a, b);
        QPIP_LAUNCH_CHECK();
      }
      status();
    }
    if (h_bad)  // the outputs are released by `oa`
      throw logic_error(
        "cuSpatial failure: a quadrant, point or linestring index is out of range");
    oa.keep();
    *point_index              = o_point;
    *nearest_linestring_index = o_ls;
    *distance                 = o_dist;
    *num_rows                 = n;
    return QPIP_SUCCESS;
  } catch (...) {
    return qpip::error_status();
  }
}

extern "C" int qpip_linestring_bounding_boxes(const int32_t* linestring_offsets,
                                              int64_t num_linestring_offsets,
                                              const double* x,
                                              const double* y,
                                              int64_t num_x,
                                              int64_t num_y,
                                              double expansion_radius,
                                              const qpip_resource* mr,
                                              void* stream_,
                                              double** minx,
                                              double** miny,
                                              double** maxx,
                                              double** maxy,
                                              int64_t* num_boxes)
{
  try {
    QPIP_EXPECTS(minx && miny && maxx && maxy && num_boxes, "output pointers must not be null");
    *minx = *miny = *maxx = *maxy = nullptr;
    *num_boxes                    = 0;
    auto stream                   = static_cast<hipStream_t>(stream_);
    // linestring_bounding_boxes.cu:133-141
    int64_t const num_ls = num_linestring_offsets > 0 ? num_linestring_offsets - 1 : 0;
    QPIP_EXPECTS(num_x == num_y, "x and y must be the same size");
    QPIP_EXPECTS(expansion_radius >= 0, "expansion radius must be greater or equal than 0");
    QPIP_EXPECTS(num_x >= 2 * num_ls, "all linestrings must have at least 2 vertices");
    if (num_ls == 0 || num_x == 0) return QPIP_SUCCESS;
    // a linestring is a polygon with one ring: the same per-geometry reduction
    // (detail/bounding_boxes.cuh:97-131 and :139-184 both reduce by geometry id)
    StreamScope scope(stream);
    dbuf<int32_t> parts(num_ls + 1);
    iota_i32_kernel<<<grid_for(static_cast<uint64_t>(num_ls + 1), 256, 1u << 30), 256, 0,
                      stream>>>(parts.get(), num_ls + 1);
    QPIP_LAUNCH_CHECK();
    int const rc = qpip_polygon_bounding_boxes(parts.get(), num_ls + 1, linestring_offsets,
                                               num_linestring_offsets, x, y, num_x, num_y,
                                               expansion_radius, mr, stream_, minx, miny, maxx,
                                               maxy, num_boxes);
    return rc;
  } catch (...) {
    return qpip::error_status();
  }
}
