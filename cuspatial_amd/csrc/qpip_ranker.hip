// Learned candidate ranking for point location over a partition (no counterpart
// in the reference; an addition on top of the quadtree join).
//
// A coarse grid (dim x dim cells over the polygons' domain) lists, per cell, up to
// 16 candidate polygons: every polygon whose bounding box reaches the cell, so the
// list of a point's cell holds every polygon that can contain the point. A small
// MLP scores the candidates of a point's cell from the cell's learned embedding
// (64 values) and 32 Fourier features of the point's position inside the cell:
//
//     x[96] = [E[cell][0..63], sin/cos(pi k u), sin/cos(pi k v), k = 1..8]
//     h1 = relu(W1 x + b1)  (128)    h2 = relu(W2 h1 + b2)  (128)
//     logits = W3 h2 + b3   (16, one per candidate slot)
//
// bf16 operands, fp32 accumulation, on MFMA (v_mfma_f32_16x16x32_bf16, and
// v_mfma_f32_16x16x16_bf16 where the contraction is over the 16 slots). The
// locator tests the candidates in the order of their logits with the exact FP64
// point-in-polygon test of the quadtree path (same edge table, same arithmetic; for
// short rings a single-precision form first, whose outcome counts where it is certain)
// and stops at the first polygon that contains the point away from its edges.
// Points whose only hit is close to an edge, or whose cell lists more than 16
// candidates, or that have no hit after max_tests tests, are marked for the
// exact quadtree path; everything else is final.
//
// Training runs the forward pass, the masked softmax cross-entropy and the backward
// pass in one kernel per batch (mlp_kernel, which also gives the logits alone), a
// reduction of the workgroups' weight gradients, and Adam.
#include <algorithm>
#include <cmath>

#include "qpip_edges.hpp"

namespace qpip {

namespace {

constexpr int kCand   = 16;  // candidate slots per grid cell
constexpr int kEmb    = 64;  // cell embedding width
constexpr int kIn     = 96;  // kEmb + 32 Fourier features
constexpr int kHid    = 128; // hidden width
constexpr int kFreqs  = 8;   // frequencies per axis (2 axes x 8 x sin/cos = 32 features)

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Round to nearest even (v_cvt_pk_bf16_f32); NaN stays NaN.
__device__ __forceinline__ uint16_t to_bf16(float f)
{
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}
__device__ __forceinline__ float from_bf16(uint16_t h)
{
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

// D = A B + C on one 16x16x16 bf16 tile. Lane l supplies A[l % 16][4 (l / 16) + j]
// and B[4 (l / 16) + j][l % 16] (j = 0..3) and holds D[4 (l / 16) + j][l % 16].
__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Flat parameter layout (floats; the bf16 copy uses the same element offsets).
struct Layout {
  int64_t e, w1, b1, w2, b2, w3, b3, total;
  __host__ __device__ Layout() : Layout(0) {}
  __host__ __device__ explicit Layout(int64_t cells)
  {
    e     = 0;
    w1    = cells * kEmb;
    b1    = w1 + int64_t{kHid} * kIn;
    w2    = b1 + kHid;
    b2    = w2 + int64_t{kHid} * kHid;
    w3    = b2 + kHid;
    b3    = w3 + int64_t{kCand} * kHid;
    total = b3 + kCand;
  }
};

struct GridView {
  double x0, y0, cell, inv_cell;
  uint32_t dim;
  int32_t const* cand;
  uint8_t const* count;
};

// Cell coordinate floor((v - v0) * inv_cell) with inv_cell = 1 / cell, clamped to
// [0, dim - 1] (NaN -> 0). The function is monotone in v, so a polygon whose box
// spans [lo, hi] is listed in every cell from coord(lo) to coord(hi), which
// includes the cell of each point it contains.
__device__ __forceinline__ uint32_t grid_coord(double v, double v0, double inv_cell, uint32_t dim)
{
  double const t = floor((v - v0) * inv_cell);
  return static_cast<uint32_t>(fmin(fmax(t, 0.0), static_cast<double>(dim - 1)));  // NaN: 0
}

struct Loc {
  uint32_t cell;
  float u, v;
};

__device__ __forceinline__ Loc locate_cell(GridView const& g, double x, double y)
{
  uint32_t const ix = grid_coord(x, g.x0, g.inv_cell, g.dim);
  uint32_t const iy = grid_coord(y, g.y0, g.inv_cell, g.dim);
  double const u    = (x - (g.x0 + static_cast<double>(ix) * g.cell)) * g.inv_cell;
  double const v    = (y - (g.y0 + static_cast<double>(iy) * g.cell)) * g.inv_cell;
  return Loc{iy * g.dim + ix, static_cast<float>(u), static_cast<float>(v)};
}

// Fourier features of frequency index k (0..7): sin, cos of pi (k+1) u, then of v,
// from the hardware sine and cosine (v_sin_f32 / v_cos_f32 take revolutions:
// sin(pi (k+1) u) = sin(2 pi r) with r = (k+1) u / 2). Training and location use
// this same function, so the model sees identical features in both.
__device__ __forceinline__ void fourier4(float u, float v, int k, float (&f)[4])
{
  float const h  = 0.5f * static_cast<float>(k + 1);
  float const ru = h * u, rv = h * v;
  f[0]           = __builtin_amdgcn_sinf(ru);
  f[1]           = __builtin_amdgcn_cosf(ru);
  f[2]           = __builtin_amdgcn_sinf(rv);
  f[3]           = __builtin_amdgcn_cosf(rv);
}

// ---------------------------------------------------------------------------------
// Training kernels
// ---------------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
  features_kernel(GridView g, uint16_t const* __restrict__ emb, double const* __restrict__ xy,
                  int64_t n, uint16_t* __restrict__ X, uint32_t* __restrict__ cells)
{
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint16_t* x = X + i * kIn;
  Loc const L = locate_cell(g, xy[2 * i], xy[2 * i + 1]);
  cells[i]    = L.cell;
  uint16_t const* e = emb + static_cast<int64_t>(L.cell) * kEmb;
  for (int d = 0; d < kEmb; ++d) x[d] = e[d];
  for (int k = 0; k < kFreqs; ++k) {
    float f[4];
    fourier4(L.u, L.v, k, f);
    for (int j = 0; j < 4; ++j) x[kEmb + 4 * k + j] = to_bf16(f[j]);
  }
}

// The step's other kernels: Adam, and the fill of the embedding gradient with the
// packing of the weights.
__global__ void __launch_bounds__(256)
  adam_kernel(float* __restrict__ p, uint16_t* __restrict__ pb, float const* __restrict__ grad,
              float* __restrict__ m, float* __restrict__ v, int64_t n, float lr, float b1, float b2,
              float eps, float c1, float c2)
{
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float const g  = grad[i];
  float const mi = b1 * m[i] + (1.f - b1) * g;
  float const vi = b2 * v[i] + (1.f - b2) * g * g;
  m[i]           = mi;
  v[i]           = vi;
  float const q  = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  p[i]           = q;
  pb[i]          = to_bf16(q);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16x8 bf16x8_any __attribute__((aligned(2)));  // of a caller's array
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

constexpr int kKT = 32;  // K per v_mfma_f32_16x16x32_bf16

// A wave's LDS writes before, its reads after (and the other way round).
__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// D = A B + C on one 16x16x32 bf16 tile (gfx950). Lane l supplies
// A[l % 16][8 (l / 16) + j] and B[8 (l / 16) + j][l % 16] (j = 0..7) and holds
// D[4 (l / 16) + j][l % 16] (j = 0..3).
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Input column of k-slot j of K tile c for lane group g of a layer fed by the
// previous layer's output tiles: the B operand of that tile is output tiles 2c
// (slots 0..3: rows 4g + j) and 2c + 1 (slots 4..7: rows 16 + 4g + j - 4), so the
// weights of slot j sit in that column. The first layer's input is in natural
// order (32c + 8g + j).
__host__ __device__ __forceinline__ int chained_col(int c, int g, int j)
{
  return 32 * c + (j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4));
}

__device__ __forceinline__ __bf16 bf(float f) { return static_cast<__bf16>(f); }

// The weights in the order the MLP kernel's A operands take them, one fragment of
// 64 lanes x 8 (mfma32) or x 4 (mfma16) bf16 after another: a wave then reads a
// fragment with one coalesced 16- or 8-byte load per lane. The backward layers need
// the transposed weights, whose 8 values per lane lie a row apart in the parameters.
constexpr int kF1    = 0;                        // W1 forward: 8 M tiles x 3 K tiles
constexpr int kF2    = kF1 + 24 * 512;           // W2 forward: 8 x 4, chained columns
constexpr int kF3    = kF2 + 32 * 512;           // W3 forward: 1 x 4, chained columns
constexpr int kB2    = kF3 + 4 * 512;            // W2 transposed: 8 x 4, chained rows
constexpr int kB1    = kB2 + 32 * 512;           // W1 transposed, embedding inputs: 4 x 4
constexpr int kB3    = kB1 + 16 * 512;           // W3 transposed: 8 x 1, mfma16
constexpr int kPack  = kB3 + 8 * 256;            // elements
constexpr int kForward  = kB2;                   // the forward layers' share
constexpr int kBackward = kPack - kB2;
static_assert(kForward % 512 == 0 && kBackward % 512 == 0 && kBackward <= kForward,
              "staged 1 KB at a time into one slot");
constexpr int kPackThreads = kB3 / 8 + 8 * 64;   // one lane of one fragment each

__device__ __forceinline__ void pack_lane(uint16_t const* __restrict__ pb, Layout const& lay, int t,
                                          uint16_t* __restrict__ out)
{
  if (t >= kB3 / 8) {  // W3^T: A[m][4g + j] = W3[4g + j][16 mt + m]
    int const u = t - kB3 / 8, mt = u / kWave, l = u % kWave, g = l >> 4, r = l & 15;
    for (int j = 0; j < 4; ++j)
      out[kB3 + 4 * u + j] = pb[lay.w3 + static_cast<int64_t>(4 * g + j) * kHid + 16 * mt + r];
    return;
  }
  int const f = t / kWave, l = t % kWave, g = l >> 4, r = l & 15;
  for (int j = 0; j < 8; ++j) {
    int64_t at;
    if (f < 24) {
      at = lay.w1 + static_cast<int64_t>(16 * (f / 3) + r) * kIn + kKT * (f % 3) + 8 * g + j;
    } else if (f < 56) {
      int const q = f - 24;
      at = lay.w2 + static_cast<int64_t>(16 * (q / 4) + r) * kHid + chained_col(q % 4, g, j);
    } else if (f < 60) {
      at = lay.w3 + static_cast<int64_t>(r) * kHid + chained_col(f - 56, g, j);
    } else if (f < 92) {
      int const q = f - 60;
      at = lay.w2 + static_cast<int64_t>(chained_col(q % 4, g, j)) * kHid + 16 * (q / 4) + r;
    } else {
      int const q = f - 92;
      at = lay.w1 + static_cast<int64_t>(chained_col(q % 4, g, j)) * kIn + 16 * (q / 4) + r;
    }
    out[8 * t + j] = pb[at];
  }
}

// Packs the weights (the first blocks) and zeroes gE (the others, 16 bytes per
// store where gE is aligned).
constexpr int kPackBlocks = (kPackThreads + 255) / 256;
__global__ void __launch_bounds__(256)
  mlp_prepare_kernel(uint16_t const* __restrict__ pb, Layout lay, uint16_t* __restrict__ packed,
                     float* __restrict__ gE, int64_t n, bool vec)
{
  if (blockIdx.x < kPackBlocks) {
    int const t = static_cast<int>(blockIdx.x) * 256 + threadIdx.x;
    if (t < kPackThreads) pack_lane(pb, lay, t, packed);
    return;
  }
  int64_t const i0     = static_cast<int64_t>(blockIdx.x - kPackBlocks) * 256 + threadIdx.x;
  int64_t const stride = static_cast<int64_t>(gridDim.x - kPackBlocks) * 256;
  if (vec) {
    float4* v = reinterpret_cast<float4*>(gE);
    for (int64_t i = i0; i < n / 4; i += stride) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int64_t i = n / 4 * 4 + i0; i < n; i += stride) gE[i] = 0.f;
  } else {
    for (int64_t i = i0; i < n; i += stride) gE[i] = 0.f;
  }
}

// The ranker's whole network over one batch: logits (TRAIN = false), or the masked
// softmax cross-entropy, the backward pass, the embedding gradient (atomics on gE) and
// each workgroup's share of the weight gradients (partials, reduced by
// mlp_reduce_kernel in a fixed order).
//
// A workgroup of 4 waves takes tiles of 128 points, 32 per wave (two 16-point column
// tiles, so that a weight fragment serves two MFMAs). The layers chain in registers
// (chained_col), forward and backward. The weight gradients contract over the points,
// which lie across lanes, so each layer's activations and deltas pass through LDS as
// [feature][point] rows (272 bytes apart: the 16 rows a fragment reads start 4 banks
// apart), one layer at a time in the same two slots; wave w owns M tiles 2w and
// 2w + 1, whose accumulators stay in registers over all the workgroup's tiles. A bias
// gradient is one more column tile, against ones.
//
// The packed weights pass through LDS once per tile (global_load_lds, the backward
// ones during the loss): read as fragments straight from L2 by every wave they took
// the kernel 63 us instead of 27. Bound by latency: at the default batch of 16,384
// points each of 128 workgroups runs one tile, about 350 MFMAs per wave between its
// copies and barriers. Whole step (with Adam, 20 us at 6.4 TB/s) at that batch and
// 65,536 cells: 377 us as nine 16x16-tile GEMMs with 2-byte loads and their helper
// kernels, 63 us now.
constexpr int kMlpWaves = 4;
constexpr int kMlpCols  = 2;                            // 16-point tiles per wave
constexpr int kMlpTile  = kMlpWaves * kMlpCols * 16;    // points per workgroup tile
constexpr int kTPitch   = kMlpTile + 8;                 // bf16 per transposed row
constexpr int kTail     = kHid * kIn + kHid + kHid * kHid + kHid + kCand * kHid + kCand;
constexpr int kDxPitch  = kEmb + 4;                     // floats per point's embedding delta
static_assert(kMlpTile * kDxPitch * 4 <= 2 * kHid * kTPitch * 2, "the deltas fit the row slots");
static_assert(kTail % 4 == 0, "the reduction reads 16 bytes per lane");

struct MlpArgs {
  GridView g;
  uint16_t const* emb;     // bf16 embeddings
  uint16_t const* packed;  // kPack bf16
  float const* p;          // fp32 parameters (biases)
  Layout lay;
  double const* xy;
  int64_t n, tiles;
  float* Z;  // TRAIN = false: logits, n x 16
  int32_t const* labels;
  float scale;  // 1 / n
  float* gE;
  float* partials;  // gridDim.x x kTail
  float* stats;
};

template <bool TRAIN>
__global__ void __launch_bounds__(kMlpWaves * kWave, 1) mlp_kernel(MlpArgs a)
{
  __shared__ __attribute__((aligned(16))) uint16_t T[TRAIN ? 2 : 1][TRAIN ? kHid * kTPitch : 8];
  __shared__ __attribute__((aligned(16))) uint16_t W[kForward];  // forward, then backward
  __shared__ __attribute__((aligned(16))) float s_bias[2 * kHid + kCand];
  __shared__ float s_stats[3];
  int const wave = static_cast<int>(uniform(threadIdx.x / kWave));
  int const l = lane_id(), g = l >> 4, r = l & 15;
  for (int t = threadIdx.x; t < 2 * kHid + kCand; t += blockDim.x)
    s_bias[t] = a.p[t < kHid ? a.lay.b1 + t
                             : (t < 2 * kHid ? a.lay.b2 + t - kHid : a.lay.b3 + t - 2 * kHid)];
  f32x4 const zero = {0.f, 0.f, 0.f, 0.f};
  if (TRAIN && threadIdx.x < 3) s_stats[threadIdx.x] = 0.f;
  float loss = 0.f, correct = 0.f, labelled = 0.f;
  f32x4 dw1[2][kIn / 16], dw2[2][kHid / 16], dw3[2], db1[2], db2[2], db3 = zero;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    dw3[m] = db1[m] = db2[m] = zero;
#pragma unroll
    for (int t = 0; t < kIn / 16; ++t) dw1[m][t] = zero;
#pragma unroll
    for (int t = 0; t < kHid / 16; ++t) dw2[m][t] = zero;
  }
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = bf(1.f);

  // copies packed weights [at, at + 512 n) to the start of W, a KB per instruction
  auto stage = [&](int at, int n) {
    for (int f = wave; f < n; f += kMlpWaves)
      __builtin_amdgcn_global_load_lds(
        (__attribute__((address_space(1))) void const*)(a.packed + at + f * 512 + l * 8),
        (__attribute__((address_space(3))) void*)(W + f * 512), 16, 0, 0);
  };
  auto staged = [] {  // every wave's copies have landed
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  auto frag = [&](int at, int f) {  // of the staged range: fragment f from `at`
    return *reinterpret_cast<bf16x8 const*>(W + at + (f * kWave + l) * 8);
  };
  auto bias4 = [&](int at) {  // the bias of rows 4g .. 4g + 3 of a tile
    return *reinterpret_cast<f32x4 const*>(s_bias + at + 4 * g);
  };
  auto put = [&](f32x4 h, bf16x8& out, int half) {  // four rows into one half of a B operand
#pragma unroll
    for (int j = 0; j < 4; ++j) out[4 * half + j] = bf(h[j]);
  };
  auto relu = [](f32x4 h) {
    return f32x4{fmaxf(h[0], 0.f), fmaxf(h[1], 0.f), fmaxf(h[2], 0.f), fmaxf(h[3], 0.f)};
  };
  // rows [0, 16 x tiles of v) of a slot from chained operands, this wave's columns
  auto store_rows = [&](int slot, int t, int c, bf16x8 v) {
    uint16_t* row = T[slot] + (32 * c + 4 * g) * kTPitch + (wave * kMlpCols + t) * 16 + r;
    u16x8 const w = __builtin_bit_cast(u16x8, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) row[(j < 4 ? j : 16 + j - 4) * kTPitch] = w[j];
  };
  auto rows = [&](int slot, int tile, int ks) {
    return *reinterpret_cast<bf16x8 const*>(T[slot] + (16 * tile + r) * kTPitch + 32 * ks + 8 * g);
  };

  for (int64_t tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
    stage(0, kForward / 512);
    int64_t const base = tile * kMlpTile + wave * (kMlpCols * 16);
    uint32_t cell[kMlpCols];
    bf16x8 X[kMlpCols][kIn / kKT], H1[kMlpCols][kHid / kKT], H2[kMlpCols][kHid / kKT];
#pragma unroll
    for (int t = 0; t < kMlpCols; ++t) {
      int64_t const p = base + 16 * t + r;
      bool const in   = p < a.n;
      Loc const L     = locate_cell(a.g, in ? a.xy[2 * p] : 0.0, in ? a.xy[2 * p + 1] : 0.0);
      cell[t]         = L.cell;
      uint16_t const* e = a.emb + static_cast<int64_t>(L.cell) * kEmb;
#pragma unroll
      for (int c = 0; c < kEmb / kKT; ++c)
        X[t][c] = *reinterpret_cast<bf16x8_any const*>(e + kKT * c + 8 * g);
      // features 64 + 8g + j: frequencies 2g (j < 4) and 2g + 1 (j >= 4)
      float f0[4], f1[4];
      fourier4(L.u, L.v, 2 * g, f0);
      fourier4(L.u, L.v, 2 * g + 1, f1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        X[t][kEmb / kKT][j]     = bf(f0[j]);
        X[t][kEmb / kKT][j + 4] = bf(f1[j]);
      }
      if (!in)  // padding rows: zero features
        for (int c = 0; c < kIn / kKT; ++c) X[t][c] = bf16x8{};
    }
    staged();
#pragma unroll
    for (int mt = 0; mt < kHid / 16; ++mt) {
      f32x4 h[kMlpCols];
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) h[t] = bias4(16 * mt);
#pragma unroll
      for (int c = 0; c < kIn / kKT; ++c) {
        bf16x8 const w = frag(kF1, mt * (kIn / kKT) + c);
#pragma unroll
        for (int t = 0; t < kMlpCols; ++t) h[t] = mfma32(w, X[t][c], h[t]);
      }
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) put(relu(h[t]), H1[t][mt / 2], mt % 2);
    }
#pragma unroll
    for (int mt = 0; mt < kHid / 16; ++mt) {
      f32x4 h[kMlpCols];
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) h[t] = bias4(kHid + 16 * mt);
#pragma unroll
      for (int c = 0; c < kHid / kKT; ++c) {
        bf16x8 const w = frag(kF2, mt * (kHid / kKT) + c);
#pragma unroll
        for (int t = 0; t < kMlpCols; ++t) h[t] = mfma32(w, H1[t][c], h[t]);
      }
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) put(relu(h[t]), H2[t][mt / 2], mt % 2);
    }
    // logits: slots 4g + j of point r
    f32x4 z[kMlpCols];
#pragma unroll
    for (int t = 0; t < kMlpCols; ++t) z[t] = bias4(2 * kHid);
#pragma unroll
    for (int c = 0; c < kHid / kKT; ++c) {
      bf16x8 const w = frag(kF3, c);
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) z[t] = mfma32(w, H2[t][c], z[t]);
    }
    if constexpr (!TRAIN) {
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) {
        int64_t const p = base + 16 * t + r;
        if (p < a.n)
          for (int j = 0; j < 4; ++j) a.Z[p * kCand + 4 * g + j] = z[t][j];
      }
      __syncthreads();  // the next tile's weights overwrite W
    } else {
      __syncthreads();
      stage(kB2, kBackward / 512);  // lands during the loss
      // Masked softmax cross-entropy over the first count[cell] slots; the four lanes
      // of a point (g = 0..3) hold four slots each. A row whose label is negative or
      // outside the mask contributes nothing. dZ = (p - onehot) * scale.
      bf16x4 dz[kMlpCols];
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) {
        int64_t const p = base + 16 * t + r;
        int const cnt   = p < a.n ? (a.g.count[cell[t]] < kCand ? a.g.count[cell[t]] : kCand) : 0;
        int const y     = p < a.n ? a.labels[p] : -1;
        bool const use  = y >= 0 && y < cnt;
        float mx = -INFINITY;
        int best = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (4 * g + j < cnt && z[t][j] > mx) {
            mx   = z[t][j];
            best = 4 * g + j;
          }
#pragma unroll
        for (int o = 16; o < kWave; o <<= 1) {
          float const om = __shfl_xor(mx, o, kWave);
          int const ob   = __shfl_xor(best, o, kWave);
          if (om > mx || (om == mx && ob < best)) {
            mx   = om;
            best = ob;
          }
        }
        float e[4], sum = 0.f, zy = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          e[j] = 4 * g + j < cnt ? expf(z[t][j] - mx) : 0.f;
          sum += e[j];
          if (4 * g + j == y) zy = z[t][j];
        }
#pragma unroll
        for (int o = 16; o < kWave; o <<= 1) {
          sum += __shfl_xor(sum, o, kWave);
          zy += __shfl_xor(zy, o, kWave);  // the other lanes of the point hold 0
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float const q = 4 * g + j < cnt ? e[j] / sum : 0.f;
          dz[t][j] = use ? static_cast<short>(
                             to_bf16((q - (4 * g + j == y ? 1.f : 0.f)) * a.scale))
                         : short{0};
        }
        if (use && g == 0) {
          loss += logf(sum) - (zy - mx);
          correct += best == y ? 1.f : 0.f;
          labelled += 1.f;
        }
      }
      // slot 0: H2, slot 1: dZ
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) {
#pragma unroll
        for (int c = 0; c < kHid / kKT; ++c) store_rows(0, t, c, H2[t][c]);
        uint16_t* row = T[1] + 4 * g * kTPitch + (wave * kMlpCols + t) * 16 + r;
#pragma unroll
        for (int j = 0; j < 4; ++j) row[j * kTPitch] = static_cast<uint16_t>(dz[t][j]);
      }
      staged();
      // dH2 = (W3^T dZ) where H2 > 0
      auto gated = [](f32x4 d, bf16x8 h, int half) {
        f32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = static_cast<float>(h[4 * half + j]) > 0.f ? d[j] : 0.f;
        return o;
      };
      bf16x8 D2[kMlpCols][kHid / kKT];
#pragma unroll
      for (int mt = 0; mt < kHid / 16; ++mt) {
        bf16x4 const w =
          *reinterpret_cast<bf16x4 const*>(W + kB3 - kB2 + (mt * kWave + l) * 4);
#pragma unroll
        for (int t = 0; t < kMlpCols; ++t)
          put(gated(mfma16(w, dz[t], zero), H2[t][mt / 2], mt % 2), D2[t][mt / 2], mt % 2);
      }
#pragma unroll
      for (int ks = 0; ks < kMlpTile / 32; ++ks) {
        bf16x8 const d = rows(1, 0, ks);
#pragma unroll
        for (int m = 0; m < 2; ++m) dw3[m] = mfma32(d, rows(0, 2 * wave + m, ks), dw3[m]);
        if (wave == 0) db3 = mfma32(d, ones, db3);
      }
      __syncthreads();
      // slot 0: H1, slot 1: dH2
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t)
#pragma unroll
        for (int c = 0; c < kHid / kKT; ++c) {
          store_rows(0, t, c, H1[t][c]);
          store_rows(1, t, c, D2[t][c]);
        }
        // dH1 = (W2^T dH2) where H1 > 0
      bf16x8 D1[kMlpCols][kHid / kKT];
#pragma unroll
      for (int mt = 0; mt < kHid / 16; ++mt) {
        f32x4 d[kMlpCols];
#pragma unroll
        for (int t = 0; t < kMlpCols; ++t) d[t] = zero;
#pragma unroll
        for (int c = 0; c < kHid / kKT; ++c) {
          bf16x8 const w = frag(0, mt * (kHid / kKT) + c);
#pragma unroll
          for (int t = 0; t < kMlpCols; ++t) d[t] = mfma32(w, D2[t][c], d[t]);
        }
#pragma unroll
        for (int t = 0; t < kMlpCols; ++t)
          put(gated(d[t], H1[t][mt / 2], mt % 2), D1[t][mt / 2], mt % 2);
      }
      __syncthreads();
#pragma unroll
      for (int ks = 0; ks < kMlpTile / 32; ++ks) {
        bf16x8 d[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          d[m]   = rows(1, 2 * wave + m, ks);
          db2[m] = mfma32(d[m], ones, db2[m]);
        }
#pragma unroll
        for (int k = 0; k < kHid / 16; ++k) {
          bf16x8 const h = rows(0, k, ks);
#pragma unroll
          for (int m = 0; m < 2; ++m) dw2[m][k] = mfma32(d[m], h, dw2[m][k]);
        }
      }
      __syncthreads();
      // slot 0: X (natural order: features 32c + 8g + j), slot 1: dH1
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t) {
#pragma unroll
        for (int c = 0; c < kHid / kKT; ++c) store_rows(1, t, c, D1[t][c]);
#pragma unroll
        for (int c = 0; c < kIn / kKT; ++c) {
          uint16_t* row = T[0] + (32 * c + 8 * g) * kTPitch + (wave * kMlpCols + t) * 16 + r;
          u16x8 const w = __builtin_bit_cast(u16x8, X[t][c]);
#pragma unroll
          for (int j = 0; j < 8; ++j) row[j * kTPitch] = w[j];
        }
      }
        // embedding gradient: dX = W1^T dH1 (the embedding's inputs), rows 16 mt + 4g + j
      f32x4 dx[kMlpCols][kEmb / 16];
#pragma unroll
      for (int mt = 0; mt < kEmb / 16; ++mt) {
#pragma unroll
        for (int t = 0; t < kMlpCols; ++t) dx[t][mt] = zero;
#pragma unroll
        for (int c = 0; c < kHid / kKT; ++c) {
          bf16x8 const w = frag(kB1 - kB2, mt * (kHid / kKT) + c);
#pragma unroll
          for (int t = 0; t < kMlpCols; ++t) dx[t][mt] = mfma32(w, D1[t][c], dx[t][mt]);
        }
      }
      __syncthreads();
#pragma unroll
      for (int ks = 0; ks < kMlpTile / 32; ++ks) {
        bf16x8 d[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          d[m]   = rows(1, 2 * wave + m, ks);
          db1[m] = mfma32(d[m], ones, db1[m]);
        }
#pragma unroll
        for (int k = 0; k < kIn / 16; ++k) {
          bf16x8 const x = rows(0, k, ks);
#pragma unroll
          for (int m = 0; m < 2; ++m) dw1[m][k] = mfma32(d[m], x, dw1[m][k]);
        }
      }
      __syncthreads();
      // Through this wave's quarter of the slots, so that an atomic instruction adds one
      // point's 64 consecutive values (from the tile layout an instruction touched 16
      // points' lines for 16 bytes each, and the batch took 19 us more); after the last
      // barrier, which would wait for them.
      float* const row0 = reinterpret_cast<float*>(&T[0][0]) + wave * (kMlpCols * 16 * kDxPitch);
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t)
#pragma unroll
        for (int mt = 0; mt < kEmb / 16; ++mt)
          *reinterpret_cast<f32x4*>(row0 + (16 * t + r) * kDxPitch + 16 * mt + 4 * g) = dx[t][mt];
      wave_lds_sync();
#pragma unroll
      for (int t = 0; t < kMlpCols; ++t)
#pragma unroll 4
        for (int q = 0; q < 16; ++q) {
          if (base + 16 * t + q >= a.n) break;
          uint32_t const c = __builtin_amdgcn_readlane(cell[t], q);
          atomicAdd(a.gE + static_cast<int64_t>(c) * kEmb + l, row0[(16 * t + q) * kDxPitch + l]);
        }
      __syncthreads();  // the next tile's rows overwrite the slots
    }
  }
  if constexpr (TRAIN) {
    // this workgroup's share, in the parameters' order from w1 on
    float* o          = a.partials + static_cast<int64_t>(blockIdx.x) * kTail;
    float* const o_b1 = o + kHid * kIn;
    float* const o_w2 = o_b1 + kHid;
    float* const o_b2 = o_w2 + kHid * kHid;
    float* const o_w3 = o_b2 + kHid;
    float* const o_b3 = o_w3 + kCand * kHid;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int const row = 16 * (2 * wave + m) + 4 * g + j;
#pragma unroll
        for (int k = 0; k < kIn / 16; ++k) o[row * kIn + 16 * k + r] = dw1[m][k][j];
#pragma unroll
        for (int k = 0; k < kHid / 16; ++k) o_w2[row * kHid + 16 * k + r] = dw2[m][k][j];
        o_w3[(4 * g + j) * kHid + 16 * (2 * wave + m) + r] = dw3[m][j];
        if (r == 0) {
          o_b1[row] = db1[m][j];
          o_b2[row] = db2[m][j];
          if (wave == 0 && m == 0) o_b3[4 * g + j] = db3[j];
        }
      }
    loss     = wave_sum(loss);
    correct  = wave_sum(correct);
    labelled = wave_sum(labelled);
    if (l == 0) {
      atomicAdd(s_stats + 0, loss);
      atomicAdd(s_stats + 1, correct);
      atomicAdd(s_stats + 2, labelled);
    }
    __syncthreads();
    if (threadIdx.x < 3) atomicAdd(a.stats + threadIdx.x, s_stats[threadIdx.x]);
  }
}

// out[i] = sum over the workgroups' shares, in their order within each of four
// threads (16 bytes per load, eight loads in flight), then over the four.
__global__ void __launch_bounds__(256)
  mlp_reduce_kernel(float const* __restrict__ partials, int count, float* __restrict__ out)
{
  __shared__ float4 part[3][kWave];
  int const q = threadIdx.x / kWave, l = threadIdx.x % kWave;
  int const i = static_cast<int>(blockIdx.x) * kWave + l;  // float4 index
  float4 s    = make_float4(0.f, 0.f, 0.f, 0.f);
  if (i < kTail / 4) {
    float4 const* p = reinterpret_cast<float4 const*>(partials) + i;
#pragma unroll 8
    for (int b = q; b < count; b += 4) {
      float4 const v = p[static_cast<int64_t>(b) * (kTail / 4)];
      s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
    }
  }
  if (q > 0) part[q - 1][l] = s;
  __syncthreads();
  if (q == 0 && i < kTail / 4) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      float4 const v = part[k][l];
      s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
    }
    float const v[4] = {s.x, s.y, s.z, s.w};
    for (int j = 0; j < 4; ++j) out[4 * i + j] = v[j];
  }
}

// ---------------------------------------------------------------------------------
// Locator: MLP on MFMA + exact test in predicted order
// ---------------------------------------------------------------------------------
constexpr int kLocTiles   = 4;  // 16-point tiles per wave round: 64 points, one per lane
constexpr int kW1Frags    = (kHid / 16) * (kIn / kKT);    // 24
constexpr int kW2Frags    = (kHid / 16) * (kHid / kKT);   // 32
constexpr int kW3Frags    = (kCand / 16) * (kHid / kKT);  // 4
constexpr int kFrags      = kW1Frags + kW2Frags + kW3Frags;
constexpr int kFragElems  = 8;  // bf16 per lane per fragment
constexpr int kLogitPitch = kCand + 1;  // LDS row pitch of the logit transpose
constexpr int kLocWaves   = 4;

struct PolyView {
  uint32_t const* poly_offsets;
  int64_t num_polys;
  uint32_t const* ring_offsets;
  int64_t num_rings;
  Edge const* edges;
  EdgeB const* edges_b;
  uint32_t const* ring_edges;
  struct Record const* records;
  struct RingSlot const* slots;
};

// Per polygon with exactly one ring: its effective edges [e0, e0 + ne) and the y
// the ring's walk starts from (edges_b[e0].by), so a test needs one load before
// the edges. ne == kMultiRing marks a polygon tested through the ring tables.
constexpr uint32_t kMultiRing = 0xffffffffu;
struct alignas(16) Record {
  uint32_t e0, ne;
  double y0;
};

// A polygon of one short ring in single precision, in one 128-byte line: vertices
// relative to (cx, cy), the first the edges' first `b`, then each edge's `a`, and
// the largest magnitude among them. 20,000 cells of 6 edges: 2.6 MB, which one L2
// holds, against 4.5 MB of edges and 0.3 MB of records for the exact test.
// ne == kMultiRing: no slot (several rings, more than kSlotEdges edges, coordinates
// that are not finite, an extent outside [2^-60, 2^60]).
constexpr uint32_t kSlotEdges = 13;
struct alignas(128) RingSlot {
  float cx, cy, m;
  uint32_t ne;
  float2 v[kSlotEdges + 1];
};

__device__ __forceinline__ void fill_slot(PolyView const& P, Record const& rec, RingSlot& out)
{
  RingSlot s;
  s.cx = s.cy = s.m = 0.f;
  s.ne = kMultiRing;
#pragma unroll
  for (uint32_t i = 0; i <= kSlotEdges; ++i) s.v[i] = float2{0.f, 0.f};
  if (rec.ne <= kSlotEdges) {
    Edge const* E = P.edges + rec.e0;
    double2 w[kSlotEdges + 1];
    double mnx = __builtin_inf(), mxx = -mnx, mny = mnx, mxy = -mnx;
    uint32_t const nv = rec.ne ? rec.ne + 1 : 0u;
#pragma unroll
    for (uint32_t i = 0; i <= kSlotEdges; ++i)
      if (i < nv) {
        w[i] = i ? double2{E[i - 1].ax, E[i - 1].ay}
                 : double2{P.edges_b[rec.e0].bx, P.edges_b[rec.e0].by};
        mnx = fmin(mnx, w[i].x), mxx = fmax(mxx, w[i].x);
        mny = fmin(mny, w[i].y), mxy = fmax(mxy, w[i].y);
      }
    s.cx   = static_cast<float>(0.5 * mnx + 0.5 * mxx);
    s.cy   = static_cast<float>(0.5 * mny + 0.5 * mxy);
    bool ok = true;
#pragma unroll
    for (uint32_t i = 0; i <= kSlotEdges; ++i)
      if (i < nv) {
        s.v[i] = float2{static_cast<float>(w[i].x - static_cast<double>(s.cx)),
                        static_cast<float>(w[i].y - static_cast<double>(s.cy))};
        float const m = fmaxf(fabsf(s.v[i].x), fabsf(s.v[i].y));
        ok            = ok && fabsf(s.v[i].x) <= 0x1p60f && fabsf(s.v[i].y) <= 0x1p60f;
        s.m           = fmaxf(s.m, m);
      }
    s.m *= 1.f + 0x1p-20f;  // above every vertex's own magnitude, not its rounded one
    if (rec.ne == 0 || (ok && s.m >= 0x1p-60f)) s.ne = rec.ne;
  }
  out = s;
}

__global__ void __launch_bounds__(64)
  records_kernel(PolyView P, Record* __restrict__ out, RingSlot* __restrict__ slots)
{
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < P.num_polys;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    uint32_t const r0 = P.poly_offsets[i];
    uint32_t r1       = P.poly_offsets[i + 1];
    if (r1 > P.num_rings) r1 = static_cast<uint32_t>(P.num_rings);
    Record rec{0u, kMultiRing, 0.0};
    if (r1 == r0 + 1) {
      rec.e0 = P.ring_offsets[r0];
      rec.ne = P.ring_edges[r0];
      rec.y0 = rec.ne ? P.edges_b[rec.e0].by : 0.0;
    } else if (r1 <= r0) {
      rec.ne = 0;  // no rings: never contains a point
    }
    out[i] = rec;
    fill_slot(P, rec, slots[i]);
  }
}

struct LocateArgs {
  GridView g;
  uint16_t const* pb;  // bf16 parameters
  float const* p;      // fp32 parameters (biases)
  Layout lay;
  PolyView P;
  double const* xy;
  int64_t n;
  int max_tests;
  int32_t* out_poly;
  uint8_t* out_tests;
  uint8_t* out_flags;
  uint16_t* order;  // per point: the best 3 slots (4 bits each), then their number
};

// The exact test of the quadtree path for one point and one polygon, plus whether
// the point lies within the collinearity filter of any edge (then a neighbouring
// polygon's test could also hold, and the point goes to the quadtree path).
__device__ __forceinline__ void edge_step(Edge const& E, EdgeB const* eb, double px, double py,
                                          bool& y0, bool& inside, bool& on_edge, bool& near)
{
  double const lhs = (px - E.ax) * E.rise;  // run_to_point * rise
  double const rhs = E.run * (py - E.ay);   // run * rise_to_point
  double const gap = fma(fabs(rhs), -0x1p-48, fabs(rhs - lhs));
  if (!(gap > 0x1p-1020)) {
    near = true;
    if (float_equal(rhs, lhs)) {  // is_point_in_polygon.cuh:56-65
      double const bx   = eb->bx;
      double const minx = E.ax < bx ? E.ax : bx;
      double const maxx = E.ax < bx ? bx : E.ax;
      if (minx <= px && px <= maxx) on_edge = true;
    }
  }
  bool const y1 = E.ay > py;
  if (y1 != y0 && ((lhs < rhs) != y1)) inside = !inside;
  y0 = y1;
}

__device__ __forceinline__ void exact_test(PolyView const& P, uint32_t poly, double px, double py,
                                           bool& inside_out, bool& near_out)
{
  Record const rec = P.records[poly];
  if (rec.ne != kMultiRing) {
    bool inside = false, on_edge = false, near = false;
    bool y0 = rec.y0 > py;
    // four edges' loads in flight per wait (a lane's edges are its own, so each
    // load is a round trip to L2; vector loads complete in order)
    Edge const* E = P.edges + rec.e0;
    EdgeB const* B = P.edges_b + rec.e0;
    uint32_t e = 0;
    for (; e + 4 <= rec.ne; e += 4) {
      Edge const e0_ = E[e], e1_ = E[e + 1], e2_ = E[e + 2], e3_ = E[e + 3];
      edge_step(e0_, B + e, px, py, y0, inside, on_edge, near);
      edge_step(e1_, B + e + 1, px, py, y0, inside, on_edge, near);
      edge_step(e2_, B + e + 2, px, py, y0, inside, on_edge, near);
      edge_step(e3_, B + e + 3, px, py, y0, inside, on_edge, near);
    }
    for (; e < rec.ne; ++e) edge_step(E[e], B + e, px, py, y0, inside, on_edge, near);
    inside_out = inside && !on_edge;
    near_out   = near;
    return;
  }
  uint32_t const r0 = P.poly_offsets[poly];
  uint32_t r1       = P.poly_offsets[poly + 1];
  if (r1 > P.num_rings) r1 = static_cast<uint32_t>(P.num_rings);
  bool inside = false, on_edge = false, near = false;
  for (uint32_t r = r0; r < r1; ++r) {
    uint32_t const e0 = P.ring_offsets[r];
    uint32_t const ne = P.ring_edges[r];
    if (ne == 0) continue;
    bool y0 = P.edges_b[e0].by > py;
    for (uint32_t e = 0; e < ne; ++e)
      edge_step(P.edges[e0 + e], P.edges_b + e0 + e, px, py, y0, inside, on_edge, near);
  }
  inside_out = inside && !on_edge;
  near_out   = near;
}

// The test on a polygon's single-precision slot: false where it cannot vouch for the
// exact test's outcome. With s the point's and the vertices' largest magnitude about
// the slot's centre, a vertex relative to the point is known to within 2^-23 s (its
// rounding, the point's and the subtraction's, 2^-24 of at most s, s and 2 s, the
// first two never both at their largest), so an edge's lhs - rhs, two products of such,
// to within 2^-20 s^2 with their own rounding. Where every vertex's y is off the
// point's by more than 2^-21 s and every edge's |lhs - rhs| is above 2^-19 s^2, all signs
// are the exact test's, whose own error is 2^-48 of the same products, and no edge is
// within its collinearity filter (near). NaN and infinite points never pass.
__device__ __forceinline__ bool slot_test(RingSlot const& S, double px, double py, bool& inside)
{
  float4 const* q = reinterpret_cast<float4 const*>(&S);
  // the header and eight vertices (up to seven edges) in one round trip
  float4 const h = q[0];
  float4 a[4]    = {q[1], q[2], q[3], q[4]};
  uint32_t const ne = __float_as_uint(h.w);
  inside            = false;
  if (ne > kSlotEdges) return false;
  if (ne == 0) return true;
  float const dx = static_cast<float>(px - static_cast<double>(h.x));
  float const dy = static_cast<float>(py - static_cast<double>(h.y));
  float const s  = fabsf(dx) + fabsf(dy) + h.z;  // NaN if either is
  float bx = a[0].x - dx, by = a[0].y - dy;
  float my = fabsf(by), mt = INFINITY;
  uint32_t flip = 0;
  auto edge = [&](float vx, float vy) {
    float const ux = vx - dx, uy = vy - dy;
    float const t  = __builtin_fmaf(bx, uy, -(ux * by));
    my             = fminf(my, fabsf(uy));
    mt             = fminf(mt, fabsf(t));
    // toggles where the y signs differ and t's sign is the edge's end's
    flip ^= (__float_as_uint(uy) ^ __float_as_uint(by)) &
            ~(__float_as_uint(t) ^ __float_as_uint(uy));
    bx = ux, by = uy;
  };
  edge(a[0].z, a[0].w);
#pragma unroll
  for (uint32_t k = 1; k < 4; ++k) {
    if (2 * k <= ne) edge(a[k].x, a[k].y);
    if (2 * k + 1 <= ne) edge(a[k].z, a[k].w);
  }
  for (uint32_t k = 4; 2 * k <= ne; ++k) {
    float4 const w = q[1 + k];
    edge(w.x, w.y);
    if (2 * k + 1 <= ne) edge(w.z, w.w);
  }
  inside = (flip >> 31) != 0u;
  return my > 0x1p-21f * s && mt > 0x1p-19f * (s * s);
}

__device__ __forceinline__ bf16x8 load_frag(uint16_t const* lds, int frag, int lane)
{
  return *reinterpret_cast<bf16x8 const*>(lds +
                                          (static_cast<int64_t>(frag) * kWave + lane) * kFragElems);
}

// The next round's coordinates are loaded before layer 2 and its cells' embeddings and
// candidate counts before layer 3, into the registers that the layers in between have
// freed: the chain point -> cell -> embedding, two misses long, then runs under the MFMAs
// (20,000,000 points: 1337 -> 1105 us; the MFMAs alone are 490 us of it, the bf16
// conversions, features and the choice of the slots about as many VALU cycles).
// Two waves per SIMD (at most 256 registers, which also keeps the accumulators in
// VGPRs: no AGPR copies before the bf16 conversions), as many as two workgroups'
// LDS allows: one wave's feature and conversion work overlaps the other's MFMAs.
__global__ void __launch_bounds__(kLocWaves * kWave, 2) rank_kernel(LocateArgs a)
{
  __shared__ __attribute__((aligned(16))) uint16_t w_lds[kFrags * kWave * kFragElems];
  __shared__ float b_lds[kHid + kHid + kCand];
  __shared__ float logit_lds[kLocWaves][kWave * kLogitPitch];

  // Stage W1, W2, W3 in fragment order: fragment f (M tile mt, K tile c), lane l,
  // element j holds W[16 mt + l % 16][column of slot j of lane group l / 16].
  for (int t = threadIdx.x; t < kFrags * kWave; t += blockDim.x) {
    int const f = t / kWave, l = t % kWave, g = l >> 4;
    uint16_t const* W;
    int in, mt, c;
    bool chained;
    if (f < kW1Frags) {
      W = a.pb + a.lay.w1, in = kIn, mt = f / (kIn / kKT), c = f % (kIn / kKT), chained = false;
    } else if (f < kW1Frags + kW2Frags) {
      int const ff = f - kW1Frags;
      W = a.pb + a.lay.w2, in = kHid, mt = ff / (kHid / kKT), c = ff % (kHid / kKT), chained = true;
    } else {
      int const ff = f - kW1Frags - kW2Frags;
      W = a.pb + a.lay.w3, in = kHid, mt = ff / (kHid / kKT), c = ff % (kHid / kKT), chained = true;
    }
    uint16_t const* row = W + static_cast<int64_t>(16 * mt + (l & 15)) * in;
#pragma unroll
    for (int j = 0; j < kFragElems; ++j)
      w_lds[t * kFragElems + j] = row[chained ? chained_col(c, g, j) : kKT * c + 8 * g + j];
  }
  for (int t = threadIdx.x; t < kHid + kHid + kCand; t += blockDim.x)
    b_lds[t] = t < kHid ? a.p[a.lay.b1 + t]
                        : (t < 2 * kHid ? a.p[a.lay.b2 + t - kHid] : a.p[a.lay.b3 + t - 2 * kHid]);
  __syncthreads();

  int const wave = threadIdx.x / kWave;
  int const l = lane_id(), g = l >> 4, r = l & 15;
  float* lg   = logit_lds[wave];
  int64_t const waves = static_cast<int64_t>(gridDim.x) * kLocWaves;
  uint16_t const* W1s = w_lds;
  uint16_t const* W2s = w_lds + kW1Frags * kWave * kFragElems;
  uint16_t const* W3s = w_lds + (kW1Frags + kW2Frags) * kWave * kFragElems;

  int64_t base = (static_cast<int64_t>(blockIdx.x) * kLocWaves + wave) * kWave;
  if (base >= a.n) return;
  // the round's points, lane r of each group holding row r of every tile
  auto load_points = [&](int64_t from, double2 (&p)[kLocTiles]) {
#pragma unroll
    for (int t = 0; t < kLocTiles; ++t) {
      int64_t i = from + 16 * t + r;
      if (i >= a.n) i = a.n - 1;  // a row past the end: any point, its order is not written
      p[t] = double2{a.xy[2 * i], a.xy[2 * i + 1]};
    }
  };
  bf16x8 X[kLocTiles][kIn / kKT];
  float u[kLocTiles], v[kLocTiles];
  int count;  // candidates at this lane's own point (tile g, row r)
  // their cells; the embeddings and the count are on their way afterwards
  auto load_cells = [&](double2 const (&p)[kLocTiles]) {
    uint32_t own = 0;
#pragma unroll
    for (int t = 0; t < kLocTiles; ++t) {
      Loc const L = locate_cell(a.g, p[t].x, p[t].y);
      u[t] = L.u, v[t] = L.v;
      if (g == t) own = L.cell;
      uint16_t const* e = a.pb + a.lay.e + static_cast<int64_t>(L.cell) * kEmb;
#pragma unroll
      for (int c = 0; c < kEmb / kKT; ++c)
        X[t][c] = *reinterpret_cast<bf16x8 const*>(e + kKT * c + 8 * g);
    }
    count = a.g.count[own];
  };
  double2 pts[kLocTiles];
  load_points(base, pts);
  load_cells(pts);
  for (; base < a.n; base += waves * kWave) {
#pragma unroll
    for (int t = 0; t < kLocTiles; ++t) {
      // features 64 + 8g + j: frequencies 2g (j < 4) and 2g + 1 (j >= 4)
      float f0[4], f1[4];
      fourier4(u[t], v[t], 2 * g, f0);
      fourier4(u[t], v[t], 2 * g + 1, f1);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        X[t][kEmb / kKT][j]     = bf(f0[j]);
        X[t][kEmb / kKT][j + 4] = bf(f1[j]);
      }
    }
    int const cnt = count;
    // layer 1: output tile mt holds rows 16 mt + 4g + j; tiles 2c and 2c + 1 form
    // layer 2's K tile c (chained_col)
    f32x4 H[kLocTiles][kHid / 16];
#pragma unroll
    for (int mt = 0; mt < kHid / 16; ++mt) {
#pragma unroll
      for (int t = 0; t < kLocTiles; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) H[t][mt][j] = b_lds[16 * mt + 4 * g + j];
#pragma unroll
      for (int c = 0; c < kIn / kKT; ++c) {
        bf16x8 const w = load_frag(W1s, mt * (kIn / kKT) + c, l);
#pragma unroll
        for (int t = 0; t < kLocTiles; ++t) H[t][mt] = mfma32(w, X[t][c], H[t][mt]);
      }
    }
    // ReLU after the conversion: a bf16 value is negative exactly when its 16 bits
    // are as a signed integer, so a packed int16 max with 0 clamps two values per
    // instruction (bf16(max(x, 0)) and max(bf16(x), +0) agree for every non-NaN x)
    auto relu2 = [](float x, float y) {  // two values -> one word of bf16 pairs
      s16x2 v = __builtin_bit_cast(s16x2, __builtin_convertvector(f32x2{x, y}, bf16x2));
      return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(v, s16x2{0, 0}));
    };
    auto chain = [&](f32x4 const (&h)[kHid / 16], int c) {
      u32x4 const w{relu2(h[2 * c][0], h[2 * c][1]), relu2(h[2 * c][2], h[2 * c][3]),
                    relu2(h[2 * c + 1][0], h[2 * c + 1][1]),
                    relu2(h[2 * c + 1][2], h[2 * c + 1][3])};
      return __builtin_bit_cast(bf16x8, w);
    };
    load_points(base + waves * kWave, pts);  // the next round's (X is free from here)
    // layer 2
    f32x4 H2[kLocTiles][kHid / 16];
    {
      bf16x8 B1[kLocTiles][kHid / kKT];
#pragma unroll
      for (int t = 0; t < kLocTiles; ++t)
#pragma unroll
        for (int c = 0; c < kHid / kKT; ++c) B1[t][c] = chain(H[t], c);
#pragma unroll
      for (int mt = 0; mt < kHid / 16; ++mt) {
#pragma unroll
        for (int t = 0; t < kLocTiles; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j) H2[t][mt][j] = b_lds[kHid + 16 * mt + 4 * g + j];
#pragma unroll
        for (int c = 0; c < kHid / kKT; ++c) {
          bf16x8 const w = load_frag(W2s, mt * (kHid / kKT) + c, l);
#pragma unroll
          for (int t = 0; t < kLocTiles; ++t) H2[t][mt] = mfma32(w, B1[t][c], H2[t][mt]);
        }
      }
    }
    load_cells(pts);
    // layer 3: logits, then transpose through LDS (lane l -> point base + l)
    {
      f32x4 acc[kLocTiles];
#pragma unroll
      for (int t = 0; t < kLocTiles; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[t][j] = b_lds[2 * kHid + 4 * g + j];
#pragma unroll
      for (int c = 0; c < kHid / kKT; ++c) {
        bf16x8 const w = load_frag(W3s, c, l);
#pragma unroll
        for (int t = 0; t < kLocTiles; ++t) acc[t] = mfma32(w, chain(H2[t], c), acc[t]);
      }
#pragma unroll
      for (int t = 0; t < kLocTiles; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) lg[(16 * t + r) * kLogitPitch + 4 * g + j] = acc[t][j];
    }
    wave_lds_sync();
    float z[kCand];
#pragma unroll
    for (int s = 0; s < kCand; ++s) z[s] = lg[l * kLogitPitch + s];
    wave_lds_sync();

    // this lane's point is tile g, row r: base + 16 g + r = base + l
    int64_t const p = base + l;
    if (p >= a.n) continue;
    int const limit = cnt > kCand ? 0 : (cnt < a.max_tests ? cnt : a.max_tests);
    // The three best slots by decreasing logit (NaN lowest, near-ties to the lower
    // slot): each slot's key is the logit's order-preserving bits with the low 4
    // bits replaced by 15 - slot, so keys are distinct and three max passes find
    // them. The other slots are tested in list order after these; the order only
    // decides how many exact tests a point needs, never the answer.
    uint32_t key[kCand];
#pragma unroll
    for (int q = 0; q < kCand; ++q) {
      float const zq   = z[q] == z[q] ? z[q] : -INFINITY;
      uint32_t const b = __float_as_uint(zq);
      uint32_t const o = (b >> 31) ? ~b : (b | 0x80000000u);
      key[q]           = q < cnt ? ((o & 0xFFFFFFF0u) | static_cast<uint32_t>(15 - q)) : 0u;
    }
    uint32_t m0 = 0, m1 = 0, m2 = 0;
#pragma unroll
    for (int q = 0; q < kCand; ++q) m0 = max(m0, key[q]);
#pragma unroll
    for (int q = 0; q < kCand; ++q) m1 = max(m1, key[q] == m0 ? 0u : key[q]);
#pragma unroll
    for (int q = 0; q < kCand; ++q) m2 = max(m2, (key[q] == m0 || key[q] == m1) ? 0u : key[q]);
    uint32_t const ranked = static_cast<uint32_t>(limit < 3 ? limit : 3);
    a.order[p] = static_cast<uint16_t>((15u - (m0 & 15u)) | ((15u - (m1 & 15u)) << 4) |
                                       ((15u - (m2 & 15u)) << 8) | (ranked << 12));
  }
}

// Exact tests in predicted order, one lane per point. A wave takes `chunks` chunks of
// 64 points: each point's first candidate at once, the points it does not settle
// through a queue in LDS, so that second and later tests run in full waves too (the
// slowest of 64 points needs three or four). Bound by the scattered reads: a cell's
// count and candidate, and a polygon's line per test. 20,000,000 points, 20,000 cells
// of about 6 edges, 65,536 grid cells: 1658 us with a lane running its point's tests
// one after the other over 32-byte edges, 840 us so; 8 and 16 chunks: 850 and 890.
constexpr int kVerWaves     = 4;
constexpr uint32_t kVerMost = 4;  // chunks of a wave at most

struct Pending {  // a point in the queue
  uint32_t at;    // index in the wave's points | tests << 16 | count << 24
  uint32_t cell;
  uint32_t slots;  // order's three slots | the unranked slots as a mask << 16
};

__global__ void __launch_bounds__(kVerWaves * kWave, 7)
  verify_kernel(LocateArgs a, uint32_t chunks)
{
  __shared__ Pending s_queue[kVerWaves][2 * kWave];
  int const lane      = lane_id();
  Pending* const q    = s_queue[threadIdx.x / kWave];
  int64_t const first = (static_cast<int64_t>(blockIdx.x) * kVerWaves + threadIdx.x / kWave) *
                        static_cast<int64_t>(chunks) * kWave;
  uint32_t queued = 0;  // uniform

  // the point's outcome
  auto write = [&](int64_t p, int32_t result, uint32_t tests, uint32_t flags) {
    // the first prediction was not the answer (an overflowed cell makes none: 1, no test)
    if (!(result >= 0 && tests == 1) && !(tests == 0 && flags == 1u)) flags |= 2u;
    a.out_poly[p]  = (flags & 1u) ? -2 : result;
    a.out_tests[p] = static_cast<uint8_t>(tests);
    a.out_flags[p] = static_cast<uint8_t>(flags);
  };

  for (uint32_t k = 0;;) {
    // 64 queued points, or the next chunk, or the rest of the queue
    int64_t const next = first + static_cast<int64_t>(k) * kWave;
    bool const fresh   = queued < static_cast<uint32_t>(kWave) && k < chunks && next < a.n;
    if (!fresh && queued == 0) break;
    bool active;
    int64_t p = 0;
    double x = 0.0, y = 0.0;
    Pending e{};
    if (fresh) {
      p      = next + lane;
      active = p < a.n;
      if (active) {
        x = a.xy[2 * p], y = a.xy[2 * p + 1];
        uint32_t const order = a.order[p];  // issued with the point, before the cell lookup
        e.cell               = locate_cell(a.g, x, y).cell;
        uint32_t const cnt   = a.g.count[e.cell];
        if (cnt - 1u >= static_cast<uint32_t>(kCand)) {  // none, or overflowed: quadtree path
          write(p, -1, 0, cnt ? 1u : 0u);
          active = false;
        } else {
          uint32_t rest = (1u << cnt) - 1u;
          for (uint32_t i = 0; i < order >> 12; ++i) rest &= ~(1u << ((order >> (4 * i)) & 15u));
          e.at    = (k * kWave + static_cast<uint32_t>(lane)) | (cnt << 24);
          e.slots = order | (rest << 16);
        }
      }
      ++k;
    } else {
      uint32_t const take = queued < static_cast<uint32_t>(kWave) ? queued : kWave;
      queued -= take;
      active = static_cast<uint32_t>(lane) < take;
      wave_lds_sync();
      if (active) {
        e = q[queued + static_cast<uint32_t>(lane)];
        p = first + (e.at & 0xffffu);
        x = a.xy[2 * p], y = a.xy[2 * p + 1];
      }
      wave_lds_sync();
    }
    // one candidate of each point
    bool more = false;
    if (active) {
      uint32_t tests        = (e.at >> 16) & 0xffu;
      uint32_t const cnt    = e.at >> 24;
      uint32_t const ranked = (e.slots >> 12) & 15u;
      uint32_t slot;
      if (tests < ranked) {
        slot = (e.slots >> (4 * tests)) & 15u;
      } else {
        uint32_t const rest = e.slots >> 16;
        slot                = static_cast<uint32_t>(__ffs(static_cast<int>(rest))) - 1u;
        e.slots             = (e.slots & 0xffffu) | ((rest & (rest - 1u)) << 16);
      }
      ++tests;
      int32_t const poly = a.g.cand[static_cast<int64_t>(e.cell) * kCand + slot];
      if (poly < 0 || poly >= a.P.num_polys) {
        write(p, -1, tests, 1u);
      } else {
        bool inside, near = false;
        if (!slot_test(a.P.slots[poly], x, y, inside))
          exact_test(a.P, static_cast<uint32_t>(poly), x, y, inside, near);
        if (inside) {
          write(p, near ? -1 : poly, tests, near ? 1u : 0u);
        } else if (tests < cnt && tests < static_cast<uint32_t>(a.max_tests)) {
          more = true;
          e.at = (e.at & 0xff00ffffu) | (tests << 16);
        } else {
          write(p, -1, tests, tests < cnt ? 1u : 0u);  // stopped at max_tests, or no polygon
        }
      }
    }
    uint64_t const m = ballot(more);
    if (more) q[queued + static_cast<uint32_t>(__popcll(m & lanemask_lt()))] = e;
    queued += static_cast<uint32_t>(__popcll(m));
  }
}

// ---------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------
GridView grid_view(qpip_grid const* g)
{
  QPIP_EXPECTS(g != nullptr, "grid must not be null");
  QPIP_EXPECTS(g->dim > 0 && g->dim <= 65536, "grid dimension must be in [1, 65536]");
  QPIP_EXPECTS(g->cell > 0.0, "grid cell size must be positive");
  return GridView{g->x0, g->y0, g->cell, 1.0 / g->cell, static_cast<uint32_t>(g->dim),
                  g->candidates, g->counts};
}

void check_model(qpip_ranker const* m, qpip_grid const* g)
{
  QPIP_EXPECTS(m != nullptr && m->params != nullptr && m->params_bf16 != nullptr,
               "ranker parameters must not be null");
  QPIP_EXPECTS(m->num_cells == int64_t{g->dim} * g->dim,
               "ranker embedding count must equal the grid's cell count");
}

// Packed weights of one call, and with gE (cells x 64 floats) its zero fill.
void mlp_prepare(qpip_ranker const* m, Layout const& lay, uint16_t* packed, float* gE,
                 hipStream_t stream)
{
  int64_t const n    = gE ? lay.w1 : 0;
  unsigned const fill = gE ? grid_for(static_cast<uint64_t>(n), 256 * 4, 2048) : 0u;
  mlp_prepare_kernel<<<kPackBlocks + fill, 256, 0, stream>>>(
    m->params_bf16, lay, packed, gE, n, reinterpret_cast<uintptr_t>(gE) % 16 == 0);
  QPIP_LAUNCH_CHECK();
}

MlpArgs mlp_args(qpip_ranker const* m, GridView const& g, Layout const& lay,
                 uint16_t const* packed, double const* xy, int64_t n)
{
  MlpArgs a{};
  a.g = g, a.emb = m->params_bf16 + lay.e, a.packed = packed, a.p = m->params, a.lay = lay;
  a.xy = xy, a.n = n, a.tiles = (n + kMlpTile - 1) / kMlpTile;
  return a;
}

}  // namespace

}  // namespace qpip

using namespace qpip;

extern "C" int64_t qpip_ranker_num_params(int64_t num_cells)
{
  return num_cells < 0 ? -1 : Layout(num_cells).total;
}

extern "C" int qpip_ranker_features(const qpip_ranker* model,
                                    const qpip_grid* grid,
                                    const double* xy,
                                    int64_t num_points,
                                    uint16_t* features,
                                    uint32_t* cells,
                                    void* stream_)
{
  return guarded([&] {
    GridView const g = grid_view(grid);
    check_model(model, grid);
    QPIP_EXPECTS(num_points >= 0, "point count must not be negative");
    if (num_points == 0) return;
    auto stream = static_cast<hipStream_t>(stream_);
    StreamScope scope(stream);
    Layout const lay(model->num_cells);
    features_kernel<<<grid_for(static_cast<uint64_t>(num_points), 256, 1u << 30), 256, 0,
                      stream>>>(g, model->params_bf16 + lay.e, xy, num_points, features, cells);
    QPIP_LAUNCH_CHECK();
  });
}

extern "C" int qpip_ranker_logits(const qpip_ranker* model,
                                  const qpip_grid* grid,
                                  const double* xy,
                                  int64_t num_points,
                                  float* logits,
                                  void* stream_)
{
  return guarded([&] {
    GridView const g = grid_view(grid);
    check_model(model, grid);
    QPIP_EXPECTS(num_points >= 0, "point count must not be negative");
    if (num_points == 0) return;
    auto stream        = static_cast<hipStream_t>(stream_);
    StreamScope scope(stream);
    Layout const lay(model->num_cells);
    dbuf<uint16_t> packed(kPack);
    KernelTimer kt("ranker_forward", stream);
    mlp_prepare(model, lay, packed.get(), nullptr, stream);
    MlpArgs a = mlp_args(model, g, lay, packed.get(), xy, num_points);
    a.Z       = logits;
    mlp_kernel<false><<<grid_for(static_cast<uint64_t>(a.tiles), 1, 1u << 30),
                        kMlpWaves * kWave, 0, stream>>>(a);
    QPIP_LAUNCH_CHECK();
  });
}

extern "C" int qpip_ranker_gradients(const qpip_ranker* model,
                                     const qpip_grid* grid,
                                     const double* xy,
                                     const int32_t* labels,
                                     int64_t num_points,
                                     float* grad,
                                     float* stats,
                                     void* stream_)
{
  return guarded([&] {
    GridView const g = grid_view(grid);
    check_model(model, grid);
    QPIP_EXPECTS(num_points > 0, "a training batch needs at least one point");
    auto stream        = static_cast<hipStream_t>(stream_);
    StreamScope scope(stream);
    Layout const lay(model->num_cells);
    // One workgroup per CU at most: its weight gradients stay in registers over its
    // tiles, and fewer shares are left to reduce.
    int dev = 0, cus = 0;
    QPIP_HIP(hipGetDevice(&dev));
    QPIP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    dbuf<uint16_t> packed(kPack);
    MlpArgs a            = mlp_args(model, g, lay, packed.get(), xy, num_points);
    unsigned const wgs   = static_cast<unsigned>(std::min<int64_t>(a.tiles, cus));
    dbuf<float> partials(static_cast<size_t>(wgs) * kTail);
    a.labels   = labels;
    a.scale    = 1.f / static_cast<float>(num_points);
    a.gE       = grad + lay.e;
    a.partials = partials.get();
    a.stats    = stats;
    KernelTimer kt("ranker_gradients", stream);
    mlp_prepare(model, lay, packed.get(), a.gE, stream);
    mlp_kernel<true><<<wgs, kMlpWaves * kWave, 0, stream>>>(a);
    QPIP_LAUNCH_CHECK();
    mlp_reduce_kernel<<<(kTail / 4 + kWave - 1) / kWave, 256, 0, stream>>>(
      partials.get(), static_cast<int>(wgs), grad + lay.w1);
    QPIP_LAUNCH_CHECK();
  });
}

extern "C" int qpip_ranker_adam(float* params,
                                uint16_t* params_bf16,
                                const float* grad,
                                float* m,
                                float* v,
                                int64_t num_params,
                                float lr,
                                float beta1,
                                float beta2,
                                float eps,
                                int64_t step,
                                void* stream_)
{
  return guarded([&] {
    QPIP_EXPECTS(num_params >= 0, "parameter count must not be negative");
    QPIP_EXPECTS(step >= 1, "Adam step counts from 1");
    if (num_params == 0) return;
    auto stream    = static_cast<hipStream_t>(stream_);
    StreamScope scope(stream);
    float const c1 = 1.f / (1.f - std::pow(beta1, static_cast<float>(step)));
    float const c2 = 1.f / (1.f - std::pow(beta2, static_cast<float>(step)));
    KernelTimer kt("ranker_adam", stream);
    adam_kernel<<<grid_for(static_cast<uint64_t>(num_params), 256, 1u << 30), 256, 0, stream>>>(
      params, params_bf16, grad, m, v, num_params, lr, beta1, beta2, eps, c1, c2);
    QPIP_LAUNCH_CHECK();
  });
}

extern "C" int qpip_ranker_locate(const qpip_ranker* model,
                                  const qpip_grid* grid,
                                  const int32_t* poly_offsets,
                                  int64_t num_poly_offsets,
                                  const int32_t* ring_offsets,
                                  int64_t num_ring_offsets,
                                  const double* poly_x,
                                  const double* poly_y,
                                  int64_t num_vertices,
                                  const double* xy,
                                  int64_t num_points,
                                  int32_t max_tests,
                                  int32_t* out_polygon,
                                  uint8_t* out_tests,
                                  uint8_t* out_flags,
                                  void* stream_)
{
  return guarded([&] {
    GridView const g = grid_view(grid);
    check_model(model, grid);
    QPIP_EXPECTS(num_points >= 0, "point count must not be negative");
    QPIP_EXPECTS(max_tests >= 1, "max_tests must be at least 1");
    QPIP_EXPECTS(num_poly_offsets >= 1 && num_ring_offsets >= 1,
                 "offset columns need at least one entry");
    if (num_points == 0) return;
    auto stream           = static_cast<hipStream_t>(stream_);
    StreamScope scope(stream);
    int64_t const polys   = num_poly_offsets - 1;
    int64_t const rings   = num_ring_offsets - 1;
    dbuf<Edge> edges(std::max<int64_t>(num_vertices, 1));
    dbuf<EdgeB> edges_b(std::max<int64_t>(num_vertices, 1));
    dbuf<uint32_t> ring_edges(std::max<int64_t>(rings, 1));
    if (rings > 0) {
      KernelTimer kt("ranker_edges", stream);
      build_edges_kernel<<<grid_for(static_cast<uint64_t>(rings), 256 / kWave), 256, 0, stream>>>(
        reinterpret_cast<uint32_t const*>(ring_offsets), rings, poly_x, poly_y, num_vertices,
        edges.get(), edges_b.get(), ring_edges.get(), nullptr, nullptr, nullptr);
      QPIP_LAUNCH_CHECK();
    }
    LocateArgs a{};
    a.g   = g;
    a.pb  = model->params_bf16;
    a.p   = model->params;
    a.lay = Layout(model->num_cells);
    a.P   = PolyView{reinterpret_cast<uint32_t const*>(poly_offsets), polys,
                   reinterpret_cast<uint32_t const*>(ring_offsets), rings, edges.get(),
                   edges_b.get(), ring_edges.get()};
    a.xy        = xy;
    a.n         = num_points;
    a.max_tests = max_tests;
    a.out_poly  = out_polygon;
    a.out_tests = out_tests;
    a.out_flags = out_flags;
    dbuf<Record> records(std::max<int64_t>(polys, 1));
    dbuf<RingSlot> slots(std::max<int64_t>(polys, 1));
    a.P.records = records.get();
    a.P.slots   = slots.get();
    if (polys > 0) {
      records_kernel<<<grid_for(static_cast<uint64_t>(polys), 64), 64, 0, stream>>>(
        a.P, records.get(), slots.get());
      QPIP_LAUNCH_CHECK();
    }
    dbuf<uint16_t> order(num_points);
    a.order = order.get();
    int dev = 0, cus = 0;
    QPIP_HIP(hipGetDevice(&dev));
    QPIP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    uint64_t const groups = (static_cast<uint64_t>(num_points) + kWave - 1) / kWave;
    uint64_t const want   = (groups + kLocWaves - 1) / kLocWaves;
    unsigned const blocks = static_cast<unsigned>(std::min<uint64_t>(want, uint64_t(2) * cus));
    {
      KernelTimer kt("ranker_rank", stream);
      rank_kernel<<<blocks, kLocWaves * kWave, 0, stream>>>(a);
      QPIP_LAUNCH_CHECK();
    }
    {
      KernelTimer kt("ranker_verify", stream);
      // more chunks per wave only where every wave slot of the GPU (32 per CU) has one:
      // 10,000 points are one chunk for each of 157 waves, and a second chunk would
      // only lengthen their chain of loads
      uint64_t const chunks =
        std::clamp<uint64_t>(groups / (uint64_t(32) * cus), 1, kVerMost);
      verify_kernel<<<grid_for(groups, kVerWaves * chunks, 1u << 30), kVerWaves * kWave, 0,
                      stream>>>(a, static_cast<uint32_t>(chunks));
      QPIP_LAUNCH_CHECK();
    }
  });
}
