// Per-operation MLP inference on gfx950, one launch per layer.
//
// Network (analyzer/habitat/analysis/mlp/mlp.py:17-109): fc1 (F -> W), ReLU,
// `hidden` x [Linear(W, W), ReLU], fc2 (W -> 1), with W = 1024.  Input rows are
// standardised as RuntimePredictor.predict does (mlp.py:258-264): (x - mu) /
// sigma in fp64, then cast to fp32.
//
// Above kSplitAboveRows rows hbt_mlp_forward's hidden layers run on the 16-bit matrix
// cores: with every fp32 number in three bf16 pieces (mlp_split.h) or, from 1025 rows
// on, as a pair of fp16 numbers (mlp_pairs.h).  Up to there, in
// hbt_mlp_forward_fp32 and for networks whose weights are not for that (check_kernel),
// they run on the fp32 ones (below), with
// v_mfma_f32_32x32x2_f32: the A operand is a 32(n) x 2(k) weight fragment, the B
// operand a 2(k) x 32(m) activation fragment.  For these the weights are repacked
// once, at hbt_mlp_create, so that a fragment for 8 consecutive k is one fully
// coalesced 1 KiB load (16 B per lane) straight into the registers the MFMA reads: index
// [n-tile / 8][layer][k/8][n-tile % 8][lane][4] holds
// W_layer[32 * n-tile + lane%32][8*(k/8) + 4*(lane/32) + e].
//
// FLOPs per row: 2 * (F*1024 + hidden*1024^2 + 1024).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "../../include/habitat_mi.h"
#include "mlp_chain.h"
#include "mlp_pairs.h"
#include "mlp_split.h"
#include "wave_scale.h"

namespace hbt {

namespace {

using u32x4 = unsigned int __attribute__((ext_vector_type(4)));
using f32x2 = float __attribute__((ext_vector_type(2)));
using f32x4 = float __attribute__((ext_vector_type(4)));
using f32x16 = float __attribute__((ext_vector_type(16)));

// ReLU that hands a NaN on, as torch's does (a feature that is NaN or infinite,
// or a zero sigma, must give a NaN prediction as in the reference); the
// hardware's max would return the other operand, 0.
__device__ __forceinline__ float relu(float v) { return v < 0.f ? 0.f : v; }

constexpr int kWidth = 1024;      // hidden width the kernel is built for
constexpr int kRows = 32;         // rows per workgroup (one MFMA tile of m)
constexpr int kStride = kWidth + 4;  // LDS row stride in floats (mlp_fused_kernel)
constexpr int kMaxInPadded = 64;  // in_features padded to a multiple of 32, at most this

// ---------------------------------------------------------------------------
// Whole rounds of 32 rows per compute unit on the fp32 matrix cores
// (hbt_mlp_forward_fp32): one workgroup takes 32 rows through the whole
// network, with the activations in LDS.  Bound by the fp32 matrix cores: a
// round of 8192 rows takes 0.94 ms, 146 TFLOP/s of 157.
//
// FINISH: after the layers of mlp_pairs.h, the sum of a row's shares of the final dot
// product, and for the rows that are marked what this kernel makes of them.  A workgroup
// without a marked row is one trip to memory and two rows of 32 threads.
struct MlpArgs {
  const double* raw;     // [n][in_features]
  float* out;            // [n]
  int64_t n;
  int32_t in_features;
  int32_t in_padded;     // multiple of 32
  int32_t hidden;
  const double* mu;      // [in_features]
  const double* sigma;   // [in_features]
  const float* w_stream; // packed weights [waves][groups of all layers][tpw][64][4]
  const float* bias;     // [(hidden + 1)][kWidth]: fc1 bias, then hidden biases
  const float* w_last;   // fc2.weight [kWidth]
  float b_last;
  const float* part;     // FINISH: split::FinishArgs'
  int32_t rows_pad;
  const int32_t* redo;   // FINISH: [rows_pad] rows to be taken through the network here
};

// Fragments travel through a ring of four register slots.  Weight fragments are
// indexed by the wave's global k-group number (all layers, one stream) and are
// loaded three groups ahead, also across a layer boundary; activation
// fragments are loaded from LDS three groups ahead within the layer.
template <int TPW>
struct Ring {
  f32x4 w[4][TPW];
  f32x4 x[4];
};

// The wave's weight stream as a buffer resource: a load then takes the stream's
// base from scalar registers, the k-group's offset as a scalar and the lane's
// 16 bytes as one 32-bit register, with no 64-bit address arithmetic.
struct WeightStream {
  __amdgpu_buffer_rsrc_t rsrc;
  int lane_bytes;  // 16 * lane
};

__device__ __forceinline__ WeightStream weight_stream(const f32x4* stream, int64_t bytes,
                                                      int lane) {
  WeightStream w;
  w.rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<f32x4*>(stream), 0, (int)bytes, 0x00020000);
  w.lane_bytes = 16 * lane;
  return w;
}

template <int TPW, int SLOT>
__device__ __forceinline__ void ring_load_w(Ring<TPW>& r, const WeightStream& stream, int group,
                                            int lane) {
  const int group_bytes = group * (TPW * 64 * 16);
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(stream.rsrc, stream.lane_bytes + t * 1024,
                                                          group_bytes, 0);
    r.w[SLOT][t] = __builtin_bit_cast(f32x4, v);
  }
}

template <int TPW, int SLOT>
__device__ __forceinline__ void ring_load_x(Ring<TPW>& r, const float* act_lane, int g) {
  r.x[SLOT] = *reinterpret_cast<const f32x4*>(act_lane + 8 * g);
}

template <int TPW, int SLOT>
__device__ __forceinline__ void ring_mfma(const Ring<TPW>& r, f32x16 (&acc)[TPW]) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int t = 0; t < TPW; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(r.w[SLOT][t][e], r.x[SLOT][e], acc[t], 0, 0, 0);
}

// One layer's K loop: kg groups of 8 k (a multiple of 4) starting at global
// group `g0` of the wave's stream; `g_end` is the stream's last valid group.
// On entry ring slots 0..2 hold the weights of groups g0..g0+2.
template <int TPW>
__device__ __forceinline__ void layer_k_loop(Ring<TPW>& r, const WeightStream& stream,
                                             int g0, int kg, int g_end, const float* act_lane,
                                             f32x16 (&acc)[TPW]) {
  const int lane = threadIdx.x & 63;
  const int last = kg - 1;
  ring_load_x<TPW, 0>(r, act_lane, 0);
  ring_load_x<TPW, 1>(r, act_lane, min(1, last));
  ring_load_x<TPW, 2>(r, act_lane, min(2, last));
  for (int j = 0; j < kg; j += 4) {
    // The scheduling barriers keep the compiler from sinking a prefetch below
    // the MFMA block it is meant to overlap with.  Weight groups past the end
    // of the stream, and activation groups past the end of the layer, reload
    // the last valid one (unused values).
    ring_load_w<TPW, 3>(r, stream, min(g0 + j + 3, g_end), lane);
    ring_load_x<TPW, 3>(r, act_lane, min(j + 3, last));
    __builtin_amdgcn_sched_barrier(0);
    ring_mfma<TPW, 0>(r, acc);
    __builtin_amdgcn_sched_barrier(0);
    ring_load_w<TPW, 0>(r, stream, min(g0 + j + 4, g_end), lane);
    ring_load_x<TPW, 0>(r, act_lane, min(j + 4, last));
    __builtin_amdgcn_sched_barrier(0);
    ring_mfma<TPW, 1>(r, acc);
    __builtin_amdgcn_sched_barrier(0);
    ring_load_w<TPW, 1>(r, stream, min(g0 + j + 5, g_end), lane);
    ring_load_x<TPW, 1>(r, act_lane, min(j + 5, last));
    __builtin_amdgcn_sched_barrier(0);
    ring_mfma<TPW, 2>(r, acc);
    __builtin_amdgcn_sched_barrier(0);
    ring_load_w<TPW, 2>(r, stream, min(g0 + j + 6, g_end), lane);
    ring_load_x<TPW, 2>(r, act_lane, min(j + 6, last));
    __builtin_amdgcn_sched_barrier(0);
    ring_mfma<TPW, 3>(r, acc);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int WAVES, bool FINISH>
__global__ __launch_bounds__(WAVES * 64, 1) void mlp_fused_kernel(const MlpArgs a) {
  constexpr int TPW = (kWidth / 32) / WAVES;  // n-tiles per wave
  constexpr int THREADS = WAVES * 64;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* act = lds;                           // [kRows][kStride]
  float* red = lds + kRows * kStride;         // [THREADS / 32][32]
  float* bias_lds = red + (THREADS / 32) * 32;  // [kWidth]
  static_assert(THREADS * 4 == kWidth, "one float4 of bias per thread");

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int m = lane & 31, h = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * kRows;

  bool again = true;   // this thread's row of the tile, of the first 32 threads
  if (FINISH) {
    again = false;
    if (tid < kRows && row0 + tid < a.n) {
      again = a.redo[row0 + tid] != 0;
      a.out[row0 + tid] = split::sum_of_shares(a.part, a.rows_pad, row0 + tid, a.b_last);
    }
    if (wave == 0) {
      const bool any = __any(again);
      if (lane == 0) red[0] = any ? 1.f : 0.f;
    }
    __syncthreads();
    if (red[0] == 0.f) return;
  }

  // ---- stage standardised inputs: act[r][k], zero beyond in_features / n ----
  for (int idx = tid; idx < kRows * a.in_padded; idx += THREADS) {
    const int r = idx / a.in_padded, k = idx - r * a.in_padded;
    float v = 0.f;
    if (k < a.in_features && row0 + r < a.n) {
      const double x = a.raw[(row0 + r) * a.in_features + k];
      v = (float)((x - a.mu[k]) / a.sigma[k]);
    }
    act[r * kStride + k] = v;
  }
  // fc1's bias, where the accumulators will pick it up
  *reinterpret_cast<f32x4*>(bias_lds + 4 * tid) = *reinterpret_cast<const f32x4*>(a.bias + 4 * tid);
  __syncthreads();

  const float* act_lane = act + m * kStride + 4 * h;
  const int tile0 = wave * TPW;  // first n-tile of this wave

  // This wave's weight stream: fc1's groups, then 128 groups per hidden layer.
  const int kg_first = a.in_padded / 8;
  const int groups = kg_first + a.hidden * (kWidth / 8);
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int64_t stream_bytes = (int64_t)groups * TPW * 64 * 16;
  const WeightStream stream = weight_stream(
      reinterpret_cast<const f32x4*>(a.w_stream) + (size_t)wave_u * groups * TPW * 64, stream_bytes,
      lane);
  const int g_end = groups - 1;

  Ring<TPW> ring;
  ring_load_w<TPW, 0>(ring, stream, 0, lane);
  ring_load_w<TPW, 1>(ring, stream, min(1, g_end), lane);
  ring_load_w<TPW, 2>(ring, stream, min(2, g_end), lane);

  f32x16 acc[TPW];
  int g0 = 0;
  for (int layer = 0; layer <= a.hidden; ++layer) {
    // The accumulators start at this layer's bias, which the layer before
    // parked in LDS; every thread fetches four values of the next layer's now
    // and parks them after the K loop.  (Adding the bias here instead of in the
    // write-back leaves room there for a ReLU that hands NaNs on, at no more
    // instructions than add and max.)
    const int next_layer = layer < a.hidden ? layer + 1 : layer;
    const f32x4 bias_part =
        *reinterpret_cast<const f32x4*>(a.bias + (size_t)next_layer * kWidth + 4 * tid);
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 b =
            *reinterpret_cast<const f32x4*>(bias_lds + (tile0 + t) * 32 + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][4 * g + e] = b[e];
      }

    const int kg = (layer == 0) ? kg_first : kWidth / 8;
    layer_k_loop<TPW>(ring, stream, g0, kg, g_end, act_lane, acc);
    g0 += kg;

    __syncthreads();  // every wave has finished reading this layer's input and bias
    *reinterpret_cast<f32x4*>(bias_lds + 4 * tid) = bias_part;
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = (tile0 + t) * 32 + 8 * g + 4 * h;
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = relu(acc[t][4 * g + e]);
        *reinterpret_cast<f32x4*>(act + m * kStride + n) = o;
      }
    __syncthreads();
  }

  // ---- fc2: out[r] = sum_n act[r][n] * w_last[n] + b_last ----
  {
    constexpr int PARTS = THREADS / 32;
    constexpr int NPP = kWidth / PARTS;
    const int r = tid & 31, part = tid >> 5;
    const float* ap = act + r * kStride + part * NPP;
    const float* wl = a.w_last + part * NPP;
    float s = 0.f;
#pragma unroll 8
    for (int k = 0; k < NPP; k += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(ap + k);
      const f32x4 w = *reinterpret_cast<const f32x4*>(wl + k);
      s = fmaf(x[0], w[0], s);
      s = fmaf(x[1], w[1], s);
      s = fmaf(x[2], w[2], s);
      s = fmaf(x[3], w[3], s);
    }
    red[part * 32 + r] = s;
    __syncthreads();
    if (tid < 32 && row0 + tid < a.n && again) {
      float total = a.b_last;
#pragma unroll
      for (int p = 0; p < PARTS; ++p) total += red[p * 32 + tid];
      a.out[row0 + tid] = total;
    }
  }
}

// ---------------------------------------------------------------------------
// Up to kLayerMaxRows rows (one prediction, the operations of one trace, a trace
// for some devices): one launch per layer.
//
// A layer is spread over the chip in one of three shapes:
//
//   For a few rows (up to kSplitMaxRows) mlp_layer_kernel with four waves: a
//   workgroup takes one n-tile x one m-tile and an eighth of K (kSplit: 256
//   workgroups per layer), its waves split that eighth, each multiplies its
//   k-groups straight from global memory (no loop, no LDS staging), the waves
//   add their 32 x 32 accumulators through LDS, and the K-partials are written
//   as they are, [split][row][n]; they are summed, biased and rectified by
//   whoever reads them: the next layer's activation load, or the final dot
//   product.
//   Up to kHalfKMaxTiles m-tiles (128 rows) the same kernel with eight waves
//   and K over two workgroups, whose K-partials are stored by k-group (see
//   km_index), like all activations from here on.
//   Above that mlp_layer_tile_kernel: a wave per output tile, see there.
//
// The order of every sum is fixed, so results are reproducible.  Same packed
// weights, same MFMA instruction, same fragment layout as above.
constexpr int kSplit = 8;            // K-partials per hidden layer, up to kSplitMaxRows rows
// Rows up to which K is split over workgroups (the partials' traffic grows with
// the rows; beyond this the whole-K shapes are faster).
constexpr int kSplitMaxRows = 20;
// Rows that go through all layers in one launch (mlp_chain.h).
constexpr int kChainMaxRows = chain::kMaxRows;
constexpr size_t kChainHeader = 32;  // words before a handle's activations: the tickets
// Largest batch that takes this path: 224 m-tiles, 7 steps of the tile kernel on
// 256 compute units, just under what one round of the fused kernel costs
// whatever it holds.  Tuned on 256 compute units.
constexpr int kLayerMaxRows = 7168;
// m-tiles up to which the eight-wave shape splits K over two workgroups (128
// workgroups or fewer per layer would leave half the compute units idle).
constexpr int kHalfKMaxTiles = 4;
// Largest batch of hbt_mlp_forward that takes this path (256 rows: 7.6 us a layer
// here, 6.8 in the split path; 700 rows: 15.3 and 11.8).
constexpr int kSplitAboveRows = kHalfKMaxTiles * kRows;
// Input features up to which fc1 of a batch stored by k-group is computed with
// plain FMAs (mlp_first_fma_kernel); the reference's networks have 8 to 12.
constexpr int kFirstFmaMaxIn = 16;
constexpr int kFirstFmaSlices = 8;     // workgroups per m-tile (gridDim.y)
constexpr int kFirstFmaMinTiles = 64;  // m-tiles from which that kernel is used (2048 rows)
// Rows per compute unit that the split path takes at a time: one round of
// 256 x 256 workgroups per layer, with activations that stay in the 256 MB
// last-level cache: 1 M rows 72.9 ms, with two rounds 74.3 (and twice the scratch).
constexpr int64_t kSplitRowsPerUnit = 64;

struct LayerArgs {
  const float* w_stream;   // packed weights, see above
  int32_t groups_total;    // k-groups per wave stream (all layers)
  int32_t g0;              // first stream group of this layer
  int32_t kg;              // k-groups of this layer (K / 8)
  int32_t splits;          // K-partials this launch writes (gridDim.y)
  const float* p_in;       // m_pad x kWidth activations, or S_IN such blocks of K-partials
  const float* bias_in;    // [kWidth], bias of the previous layer (with partials)
  const float* bias_out;   // [kWidth], bias of this layer (FINAL)
  const double* raw;       // FIRST: [n][in_features], with mu and sigma
  const double* mu;
  const double* sigma;
  int32_t in_features;
  int64_t n;
  int32_t m_pad;           // rows rounded up to 32
  float* p_out;            // m_pad x kWidth activations (FINAL), else `splits` blocks of partials
  const float* w_first_t;  // fc1.weight transposed, [kFirstFmaMaxIn][kWidth] (mlp_first_fma_kernel)
};

// Outside the split-K shape activations are stored by k-group (KM below): element
// (row, n) at [row / 32][n / 8][row % 32][n % 8], so that the fragment a wave
// loads for one m-tile and k-group, 32 rows x 8 values, is 1 KiB of contiguous
// memory (8 cache lines used whole) where row-major storage spreads it over 32
// lines, 32 bytes of each.
__device__ __forceinline__ size_t km_index(int m_tile, int k_group, int m, int c) {
  return (((size_t)m_tile * (kWidth / 8) + k_group) * kRows + m) * 8 + c;
}

// G k-groups of a wave: the weight fragments of the n-tile and what the
// matching activation fragments are made from (the activations themselves, or
// S_IN K-partials and the bias that goes with them).
template <int G, int S_IN, int NT>
struct LayerFrag {
  f32x4 w[G][NT];
  f32x4 x[G][S_IN > 0 ? S_IN : 1];
  f32x4 bias[S_IN > 0 ? G : 1];
};

// One layer for one m-tile (blockIdx.z), NT n-tiles (blockIdx.x) and one
// K-partial (blockIdx.y of a.splits).  The WAVES waves split the partial's
// k-groups (at most G each); fc1 has fewer, so there each group is checked
// against the wave's count (wave-uniform).
//   FIRST: fc1, from the raw fp64 rows, standardised on the spot.
//   S_IN: 0 = the input holds activations; otherwise it holds that many
//     K-partials, to be summed, biased and rectified on the way in.
//   FINAL: the launch covers all of K (a.splits == 1), so the output is
//     biased and rectified here and the next layer reads activations.
//   PADDED_ROWS: rows past the end of the batch are read like the others (the
//     padded m-tile holds them) instead of being masked; masking saves most of
//     the traffic of a handful of rows, not masking keeps the loads of a full
//     tile free of branches.
//   NT: n-tiles per workgroup (blockIdx.x counts groups of NT); an activation
//     fragment then serves NT MFMAs.
//   DEPTH: k-groups whose loads are kept in flight ahead of the MFMAs; 0 leaves
//     the placement to the compiler (each group's loads next to its MFMAs, one
//     trip to memory after the other, which resident workgroups hide from each
//     other).
//   KM: activations (read, unless FIRST, and written) are stored by k-group.
//   S_OUT: K-partials this launch writes (a.splits; 1 with FINAL).
// The instantiations in use: fc1 (FIRST, FINAL, 4 waves) with row-major or
// k-group output; hidden layers with kSplit K-partials in and out (4 waves,
// rows masked); hidden layers with two K-partials in and out (8 waves, DEPTH 2,
// KM).
template <bool FIRST, int S_IN, bool FINAL, int WAVES, bool PADDED_ROWS, int DEPTH, int NT = 1,
          bool KM = false, int S_OUT = (FINAL ? 1 : kSplit)>
__global__ __launch_bounds__(WAVES * 64) void mlp_layer_kernel(const LayerArgs a) {
  static_assert((S_OUT == 1) == FINAL, "one K-partial is the whole sum");
  static_assert(8 % NT == 0, "a workgroup's n-tiles lie in one wave stream of the packed weights");
  static_assert(S_IN == 0 || !FINAL, "K-partials go in and come out together");
  static_assert(WAVES == 4 || WAVES == 8, "the reduction below is written for these");
  constexpr int G = FIRST ? kMaxInPadded / 8 / WAVES : kWidth / 8 / WAVES / S_OUT;
  __shared__ float red[WAVES][NT][16][64];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 31, h = lane >> 5;
  const int split = blockIdx.y;
  // rows past the end of the batch: computed (from zeros, or from what the
  // padded m-tile holds) and stored within the padded m-tile, never read out
  const int64_t row = (int64_t)blockIdx.z * kRows + m;
  const bool row_ok = PADDED_ROWS || row < a.n;

  // this wave's k-groups: [first, first + count) of the layer's kg
  const int per_split = a.kg / a.splits;
  const int per_wave = (per_split + WAVES - 1) / WAVES;
  const int first = split * per_split + wave * per_wave;
  int count = per_split - wave * per_wave;
  count = count < 0 ? 0 : (count > per_wave ? per_wave : count);

  // n-tile of the layer -> (weight stream, slot in its group)
  const int tile = blockIdx.x * NT;  // the first of the workgroup's NT
  const f32x4* w_lane = reinterpret_cast<const f32x4*>(a.w_stream) +
                        ((size_t)(tile >> 3) * a.groups_total + a.g0) * (8 * 64) +
                        (tile & 7) * 64 + lane;

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  LayerFrag<G, S_IN, NT> f;
  // Hidden layers fetch weights, activations (or K-partials) and bias through
  // buffer loads: bases in scalar registers, the k-group's offset a scalar, one
  // 32-bit register of lane offset each, no 64-bit address arithmetic.  A lane
  // whose row is past the end of the batch gets an offset beyond the buffer
  // instead of a branch around the load: such a load returns zeros.
  constexpr bool BUFFER = !FIRST;
  __amdgpu_buffer_rsrc_t w_rsrc, x_rsrc, b_rsrc;
  int w_lane_bytes = 0, x_lane_bytes = 0, w_base_bytes = 0;
  const int split_bytes = a.m_pad * (kWidth * 4);  // one K-partial, or the activations
  if (BUFFER) {
    w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.w_stream), 0,
                                               4 * a.groups_total * (8 * 64 * 16), 0x00020000);
    x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.p_in), 0,
                                               (S_IN > 0 ? S_IN : 1) * split_bytes, 0x00020000);
    b_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.bias_in), 0, kWidth * 4,
                                               0x00020000);
    w_lane_bytes = ((tile & 7) * 64 + lane) * 16;
    w_base_bytes = ((tile >> 3) * a.groups_total + a.g0) * (8 * 64 * 16);
    if (KM) x_lane_bytes = row_ok ? (int)km_index(blockIdx.z, 0, m, 4 * h) * 4 : 0x7fffff00;
    else x_lane_bytes = row_ok ? (int)row * (kWidth * 4) + 16 * h : 0x7fffff00;
  }
  auto load_group = [&](int j) {
    if (!FIRST || j < count) {
      const int gl = first + j;  // layer-local group
      if (BUFFER) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
          f.w[j][t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
              w_rsrc, w_lane_bytes + t * 1024, w_base_bytes + gl * (8 * 64 * 16), 0));
#pragma unroll
        for (int s = 0; s < (S_IN > 0 ? S_IN : 1); ++s)
          f.x[j][s] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
              x_rsrc, x_lane_bytes, s * split_bytes + gl * (KM ? kRows * 32 : 32), 0));
        if (S_IN > 0)
          f.bias[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
              b_rsrc, 16 * h, gl * 32, 0));
        return;
      }
      // fc1: a few groups, the raw fp64 features standardised on the spot
#pragma unroll
      for (int t = 0; t < NT; ++t) f.w[j][t] = w_lane[(size_t)gl * (8 * 64) + t * 64];
      const int k = 8 * gl + 4 * h;
      f32x4 v = zero;
      if (row_ok) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (k + e < a.in_features)
            v[e] = (float)((a.raw[row * a.in_features + k + e] - a.mu[k + e]) / a.sigma[k + e]);
      }
      f.x[j][0] = v;
    }
  };

  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  auto mfma_group = [&](int j) {
    if (!FIRST || j < count) {
      f32x4 v = f.x[j][0];
      if (S_IN > 0) {
        // the previous layer's K-partials, in their fixed order, then bias and ReLU
        v = f.bias[j];
#pragma unroll
        for (int s = 0; s < S_IN; ++s) v += f.x[j][s];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = relu(v[e]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.w[j][t][e], v[e], acc[t], 0, 0, 0);
    }
  };

  if (DEPTH == 0) {
    // the compiler places the loads: each group's next to its MFMAs, one trip
    // to memory after the other, which resident workgroups hide from each other
#pragma unroll
    for (int j = 0; j < G; ++j) load_group(j);
#pragma unroll
    for (int j = 0; j < G; ++j) mfma_group(j);
  } else {
    // DEPTH groups in flight ahead of the MFMAs
#pragma unroll
    for (int j = 0; j < (DEPTH < G ? DEPTH : G); ++j) load_group(j);
#pragma unroll
    for (int j = 0; j < G; ++j) {
      if (j + DEPTH < G) load_group(j + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
      mfma_group(j);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave][t][r][lane] = acc[t][r];
  __syncthreads();
  // thread (wave, lane) adds the waves' registers R*wave .. R*wave+R-1, in wave
  // order: accumulator register 4g + e of lane (m, h) is output n = 8g + 4h + e
  // of row m
  constexpr int R = 16 / WAVES;
  const int r0 = R * wave;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n0 = (tile + t) * 32 + 8 * (r0 >> 2) + 4 * h + (r0 & 3);
    float o[R];
#pragma unroll
    for (int e = 0; e < R; ++e) {
      float sum = red[0][t][r0 + e][lane];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) sum += red[w][t][r0 + e][lane];
      if (FINAL) sum = relu(sum + a.bias_out[n0 + e]);
      o[e] = sum;
    }
    float* dst = a.p_out + ((size_t)split * a.m_pad + (size_t)blockIdx.z * kRows + m) * kWidth + n0;
    if (KM)
      dst = a.p_out + (size_t)split * a.m_pad * kWidth + km_index(blockIdx.z, n0 >> 3, m, n0 & 7);
    if constexpr (R == 4) {
      *reinterpret_cast<f32x4*>(dst) = f32x4{o[0], o[1], o[2], o[3]};
    } else {
      *reinterpret_cast<f32x2*>(dst) = f32x2{o[0], o[1]};
    }
  }
}

// One hidden layer with a wave owning ONE output tile (32 rows x 32 outputs) for
// 1 / KS of K: no loop over tiles, accumulators in place for the wave's whole
// run of k-groups, fragments through a ring of SLOTS register slots (loads
// SLOTS - 1 k-groups ahead of their MFMAs, one 16-byte buffer load per lane and
// fragment, 1 KiB of contiguous memory per wave), no LDS staging.  A workgroup
// is four waves:
//   KS = 1   2 m-tiles x 2 n-tiles, no reduction, no barrier
//   KS = 2   1 m-tile x 2 n-tiles, two halves of K
//   KS = 4   1 m-tile x 1 n-tile, four quarters of K
// With KS > 1 the waves of a tile add their accumulators through LDS in wave
// order, each finishing 16 / KS of the tile's registers.  A tile for the whole
// of K is 13.7 us of one SIMD's matrix core, so a layer takes that times the
// tiles per SIMD, rounded up: KS trades a finer rounding (1024 / KS rows per
// step) against shorter runs per wave.  Activations in and out are stored by
// k-group (km_index); bias and ReLU are applied on the way out.
template <int KS, int SLOTS>
__global__ __launch_bounds__(256) void mlp_layer_tile_kernel(const LayerArgs a) {
  static_assert(KS == 1 || KS == 2 || KS == 4, "four waves per workgroup");
  constexpr int kGroups = kWidth / 8 / KS;  // per wave
  static_assert(kGroups % SLOTS == 0, "the ring turns a whole number of times");
  __shared__ float red[KS > 1 ? 4 : 1][16][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 31, h = lane >> 5;
  const int m_tiles = a.m_pad / kRows;
  // wave -> (part of K, n-tile, m-tile)
  const int k_part = wave % KS;
  const int n_tile = KS == 4 ? (int)blockIdx.x : (int)blockIdx.x * 2 + (KS == 2 ? wave >> 1 : wave & 1);
  const int m_tile = KS == 1 ? (int)blockIdx.y * 2 + (wave >> 1) : (int)blockIdx.y;
  if (m_tile >= m_tiles) return;  // KS = 1 only (no barrier there): an odd number of m-tiles

  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.w_stream), 0, 4 * a.groups_total * (8 * 64 * 16), 0x00020000);
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.p_in), 0, a.m_pad * (kWidth * 4), 0x00020000);
  const int first = k_part * kGroups;  // the wave's first k-group of the layer
  const int w_lane_bytes = ((n_tile & 7) * 64 + lane) * 16;
  const int w_base_bytes = ((n_tile >> 3) * a.groups_total + a.g0 + first) * (8 * 64 * 16);
  const int x_lane_bytes = m_tile * (kWidth * kRows * 4) + m * 32 + 16 * h;
  const int x_base_bytes = first * (kRows * 32);

  f32x4 w[SLOTS], x[SLOTS];
  auto load = [&](int slot, int group) {
    w[slot] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
        w_rsrc, w_lane_bytes, w_base_bytes + group * (8 * 64 * 16), 0));
    x[slot] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
        x_rsrc, x_lane_bytes, x_base_bytes + group * (kRows * 32), 0));
  };

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
  for (int s = 0; s < SLOTS - 1; ++s) load(s, s);
  for (int j = 0; j < kGroups; j += SLOTS) {
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      // past the wave's last group the last one is fetched again (unused)
      const int ahead = j + s + SLOTS - 1;
      load((s + SLOTS - 1) % SLOTS, ahead < kGroups ? ahead : kGroups - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(w[s][e], x[s][e], acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // accumulator register 4g + e of lane (m, h) is output n = 8g + 4h + e of row m
  auto finish = [&](int g, const f32x4 sum) {
    const int n0 = n_tile * 32 + 8 * g + 4 * h;
    const f32x4 bias = *reinterpret_cast<const f32x4*>(a.bias_out + n0);
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = relu(sum[e] + bias[e]);
    *reinterpret_cast<f32x4*>(a.p_out + km_index(m_tile, n0 >> 3, m, 4 * h)) = o;
  };
  if constexpr (KS == 1) {
#pragma unroll
    for (int g = 0; g < 4; ++g) finish(g, f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]});
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave][r][lane] = acc[r];
    __syncthreads();
    // the KS waves of a tile are wave0 .. wave0 + KS - 1; this one finishes the
    // register groups g0 .. g0 + 4 / KS - 1, adding the parts of K in wave order
    const int wave0 = wave - k_part;
#pragma unroll
    for (int i = 0; i < 4 / KS; ++i) {
      const int g = k_part * (4 / KS) + i;
      f32x4 sum;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = red[wave0][4 * g + e][lane];
#pragma unroll
        for (int p = 1; p < KS; ++p) v += red[wave0 + p][4 * g + e][lane];
        sum[e] = v;
      }
      finish(g, sum);
    }
  }
}

// fc1 for large batches stored by k-group, with at most kFirstFmaMaxIn input
// features: K is a dozen, so the layer is its 4 KiB-per-row write and little
// else, and plain FMAs from LDS do it without the matrix cores.  A workgroup
// takes one m-tile and an eighth of the outputs: it standardises the m-tile's
// raw fp64 rows (the 4-wave MFMA kernel does that once per n-tile, 32 times per
// row, this one 8 times), stages its slice of the transposed weights in LDS,
// and each lane (row m, half h) then produces four consecutive outputs per
// k-group of the next layer, 1 KiB of contiguous memory per wave and store.
// Sum order: bias, then k ascending.  Faster than the MFMA kernel from about
// 2048 rows (kFirstFmaMinTiles), slower below.
__global__ __launch_bounds__(256) void mlp_first_fma_kernel(const LayerArgs a) {
  __shared__ float xs[kRows][kFirstFmaMaxIn + 1];
  __shared__ __attribute__((aligned(16))) float wl[kFirstFmaMaxIn * (kWidth / kFirstFmaSlices)];  // [k][n of the slice]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int m = lane & 31, h = lane >> 5;
  const int m_tile = blockIdx.x;
  constexpr int slice_n = kWidth / kFirstFmaSlices;  // outputs of this workgroup
  const int n_base = (int)blockIdx.y * slice_n;
  for (int idx = tid; idx < kRows * kFirstFmaMaxIn; idx += 256) {
    const int r = idx / kFirstFmaMaxIn, k = idx - r * kFirstFmaMaxIn;
    const int64_t row = (int64_t)m_tile * kRows + r;
    float v = 0.f;
    if (k < a.in_features && row < a.n)
      v = (float)((a.raw[row * a.in_features + k] - a.mu[k]) / a.sigma[k]);
    xs[r][k] = v;
  }
  for (int idx = tid; idx < a.in_features * (slice_n / 4); idx += 256) {
    const int k = idx / (slice_n / 4), c = idx - k * (slice_n / 4);
    *reinterpret_cast<f32x4*>(wl + k * slice_n + 4 * c) =
        *reinterpret_cast<const f32x4*>(a.w_first_t + (size_t)k * kWidth + n_base + 4 * c);
  }
  __syncthreads();
  float x[kFirstFmaMaxIn];
#pragma unroll
  for (int k = 0; k < kFirstFmaMaxIn; ++k) x[k] = xs[m][k];
  for (int g = wave; g < slice_n / 8; g += 4) {
    const int local = 8 * g + 4 * h, n0 = n_base + local;
    f32x4 o = *reinterpret_cast<const f32x4*>(a.bias_out + n0);
#pragma unroll
    for (int k = 0; k < kFirstFmaMaxIn; ++k)
      if (k < a.in_features) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(wl + k * slice_n + local);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = fmaf(x[k], w[e], o[e]);
      }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = relu(o[e]);
    *reinterpret_cast<f32x4*>(a.p_out + km_index(m_tile, n0 >> 3, m, 4 * h)) = o;
  }
}

struct LastArgs {
  const float* p_in;     // m_pad x kWidth activations, or S_IN such blocks of K-partials
  const float* bias_in;  // [kWidth], bias of the last hidden layer (with partials)
  const float* w_last;   // [kWidth]
  float b_last;
  int64_t n;
  int32_t m_pad;
  float* out;            // [n]
  // hbt_mlp_predict_one: once out[0] is written, done_value is stored here
  // (host-visible memory) so that the caller need not wait for the stream
  uint32_t* done_flag;   // nullable
  uint32_t done_value;
};

// Publishes `value` to a waiting host thread after this thread's earlier stores.
__device__ __forceinline__ void publish_done(uint32_t* flag, uint32_t value) {
  __threadfence_system();
  __hip_atomic_store(flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// fc2 after the per-layer kernels: one wavefront per row.  S_IN as in mlp_layer_kernel.
template <int S_IN>
__global__ __launch_bounds__(256) void mlp_last_kernel(const LastArgs a) {
  constexpr int P = S_IN > 0 ? S_IN : 1;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.n) return;
  f32x4 part[kWidth / 256][P];
#pragma unroll
  for (int i = 0; i < kWidth / 256; ++i)
#pragma unroll
    for (int s = 0; s < P; ++s)
      part[i][s] = *reinterpret_cast<const f32x4*>(
          a.p_in + ((size_t)s * a.m_pad + row) * kWidth + 256 * i + 4 * lane);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kWidth / 256; ++i) {
    const int k = 256 * i + 4 * lane;
    f32x4 v = part[i][0];
    if (S_IN > 0) {
      v = *reinterpret_cast<const f32x4*>(a.bias_in + k);
#pragma unroll
      for (int s = 0; s < S_IN; ++s) v += part[i][s];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = relu(v[e]);
    }
    const f32x4 wl = *reinterpret_cast<const f32x4*>(a.w_last + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = fmaf(v[e], wl[e], sum);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off);
  if (lane == 0) {
    a.out[row] = sum + a.b_last;
    if (a.done_flag != nullptr && row == 0) publish_done(a.done_flag, a.done_value);
  }
}

// fc2 from activations stored by k-group: one workgroup per m-tile, its four
// waves take a quarter of K each; lane (m, h) reads 16 bytes of its row per
// k-group, so that a wave's load is the k-group's contiguous 1 KiB.
template <int S_IN>
__global__ __launch_bounds__(256) void mlp_last_km_kernel(const LastArgs a) {
  constexpr int kGroupsPerWave = kWidth / 8 / 4;
  __shared__ float part[4][kRows];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 31, h = lane >> 5;
  const f32x4* x = reinterpret_cast<const f32x4*>(
      a.p_in + km_index(blockIdx.x, wave * kGroupsPerWave, m, 4 * h));
  const f32x4* wl = reinterpret_cast<const f32x4*>(a.w_last + 8 * wave * kGroupsPerWave + 4 * h);
  constexpr int P = S_IN > 0 ? S_IN : 1;
  constexpr int kStep = 8;  // k-groups whose loads are issued together
  float sum = 0.f;
  for (int g0 = 0; g0 < kGroupsPerWave; g0 += kStep) {
    f32x4 v[kStep][P], w[kStep], bias[kStep];
#pragma unroll
    for (int j = 0; j < kStep; ++j) {
#pragma unroll
      for (int s = 0; s < P; ++s)
        v[j][s] = x[(size_t)(g0 + j) * (kRows * 2) + (size_t)s * a.m_pad * (kWidth / 4)];
      w[j] = wl[2 * (g0 + j)];
      if (S_IN > 0)
        bias[j] = *reinterpret_cast<const f32x4*>(
            a.bias_in + 8 * (wave * kGroupsPerWave + g0 + j) + 4 * h);
    }
    __builtin_amdgcn_sched_barrier(0);  // all of the step's loads before its arithmetic
#pragma unroll
    for (int j = 0; j < kStep; ++j) {
      f32x4 act = v[j][0];
      if (S_IN > 0) {
        // K-partials in their fixed order, then bias and ReLU
        act = bias[j];
#pragma unroll
        for (int s = 0; s < S_IN; ++s) act += v[j][s];
#pragma unroll
        for (int e = 0; e < 4; ++e) act[e] = relu(act[e]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = fmaf(act[e], w[j][e], sum);
    }
  }
  sum += __shfl_xor(sum, 32);
  if (h == 0) part[wave][m] = sum;
  __syncthreads();
  const int64_t row = (int64_t)blockIdx.x * kRows + threadIdx.x;
  if (threadIdx.x < kRows && row < a.n)
    a.out[row] = ((part[0][threadIdx.x] + part[1][threadIdx.x]) +
                  (part[2][threadIdx.x] + part[3][threadIdx.x])) + a.b_last;
}

constexpr size_t kOneOutOffset = 512;   // hbt_mlp_predict_one's result within its staging block
constexpr size_t kOneDoneOffset = 768;  // and the call number the last kernel publishes after it
constexpr size_t kOneOutsideOffset = 896;  // and what hbt_mlp_create's check_kernel leaves
constexpr size_t kOneOutsidePairsOffset = kOneOutsideOffset + 4;  // and its prepare kernels
constexpr size_t kOneBytes = 1024;
static_assert(kMaxInPadded * sizeof(double) <= kOneOutOffset, "a raw row fits below the result");

// Weight streams of 8 n-tiles each, and mlp_fused_kernel's waves: one per SIMD has
// fewer, longer MFMA runs between load bursts than two.
constexpr int kWaves = 4;
constexpr size_t kLdsBytes =
    (size_t)(kRows * kStride + (kWaves * 64 / 32) * 32 + kWidth) * sizeof(float);

}  // namespace

}  // namespace hbt

struct hbt_mlp {
  int32_t in_features, in_padded, width, hidden;
  int device;
  int compute_units;   // of that device
  void* blob;          // one device allocation holding everything below
  const double* mu;
  const double* sigma;
  const float* w_stream;
  const float* bias;
  const float* w_last;
  const float* w_first_t;  // fc1.weight transposed, [kFirstFmaMaxIn or kMaxInPadded][width]
  float b_last;
  const char* w_split; // the hidden layers' weights in bf16 pieces, kSplitLayerBytes each
  bool takes_pieces;   // whether they fit, and there are any
  // the same as fp16 pairs (mlp_pairs.h): weights, kPairsLayerBytes each, and the exponents
  // of the units' scales, F [hidden][kWidth] and G [hidden + 1][kWidth]
  const char* w_pairs;
  const int32_t* F;
  const int32_t* G;
  const int32_t* bias_most; // [hidden + 1]
  bool takes_pairs;
  int32_t* row_scales[2];   // of a layer's rows and of the next one's: [chunk_rows]
  int32_t* row_most[2];     // [kWidth / 32][chunk_rows]
  int32_t* redo;            // [chunk_rows] rows that the pairs do not hold
  int64_t chunk_rows;  // rows the split path takes at a time
  // the words of chain::Args of hbt_mlp_forward and hbt_mlp_predict_one, and of
  // hbt_mlp_forward_static; the counter of tickets comes first, in a block of its own
  uint64_t* chain[2];
  float* scratch[2];   // activations (or K-partials) of one layer and of the next
  float* part;         // split path: [kWidth / 32][chunk_rows] shares of the final dot product
  // hbt_mlp_predict_one: a pinned, device-visible block (one raw row in, one
  // prediction out at kOneOutOffset) and the lock that serialises its callers
  unsigned char* one_host;
  unsigned char* one_device;
  uint32_t one_calls;      // numbers the calls: the value the kernel publishes
  std::mutex one_lock;
};

namespace hbt {
namespace {

// Repack one layer, a row-major [kWidth][k_in] weight matrix (k_in <= k_padded),
// into the per-wave streams: wave w's copy goes to dst + w * wave_stride as
// [k_padded/8][tpw][64 lanes][4].
void pack_layer(const float* W, int k_in, int k_padded, int waves, float* dst, size_t wave_stride) {
  const int tpw = (kWidth / 32) / waves;
  const int kg = k_padded / 8;
  // (a tile's 32 rows at a time, each read through: 6.5 ms for eight hidden layers, 18 with
  // k outermost)
  for (int w = 0; w < waves; ++w)
    for (int t = 0; t < tpw; ++t)
      for (int j = 0; j < kg; ++j)
        for (int lane = 0; lane < 64; ++lane) {
          const int n = (w * tpw + t) * 32 + (lane & 31);
          const int k = 8 * j + 4 * (lane >> 5);
          float* out = dst + (size_t)w * wave_stride + (((size_t)j * tpw + t) * 64 + lane) * 4;
          const float* in = W + (size_t)n * k_in;
          if (k + 4 <= k_in) std::memcpy(out, in + k, 4 * sizeof(float));
          else
            for (int e = 0; e < 4; ++e) out[e] = k + e < k_in ? in[k + e] : 0.f;
        }
}

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

}  // namespace
}  // namespace hbt

// Scratch memory of hbt_mlp_forward_static: two buffers of activations (or
// K-partials) for up to HBT_MLP_STATIC_MAX_ROWS rows and the split path's shares
// of the final dot product, part of the code object (each GPU the library runs on
// holds its own copy until the process ends).  In host code this name is only a
// handle for hipGetSymbolAddress: kernels and copies get the per-device address
// kept in static_scratch_of().
constexpr int kStaticMaxRows = HBT_MLP_STATIC_MAX_ROWS;
constexpr size_t kStaticFloats =   // each of the two
    (size_t)(kStaticMaxRows / hbt::kRows) * hbt::split::kTileBytes / sizeof(float);
constexpr size_t kStaticShares = (size_t)(hbt::kWidth / 32) * kStaticMaxRows;
static_assert((size_t)hbt::kSplit * hbt::kRows * hbt::kWidth <= kStaticFloats &&
                  2 * (size_t)hbt::kHalfKMaxTiles * hbt::kRows * hbt::kWidth <= kStaticFloats &&
                  (size_t)kStaticMaxRows * hbt::kWidth <= kStaticFloats &&
                  kStaticMaxRows % hbt::kRows == 0 && kStaticMaxRows <= hbt::kLayerMaxRows,
              "the K-partials of the small shapes and the padded rows fit the static scratch");
static __device__ __align__(256) float scratch[2 * kStaticFloats + kStaticShares];

namespace {

// The device address of `scratch` on the current device, looked up once per
// device (nullptr and *rc set when the runtime refuses).
constexpr int kMaxDevices = 64;
float* static_scratch_of(int device, int* rc) {
  static std::mutex lock;
  static float* address[kMaxDevices] = {};
  *rc = HBT_OK;
  if (device < 0 || device >= kMaxDevices) {
    *rc = HBT_ESIZE;
    return nullptr;
  }
  std::lock_guard<std::mutex> guard(lock);
  if (address[device] == nullptr) {
    float* ptr = nullptr;
    if (hipGetSymbolAddress(reinterpret_cast<void**>(&ptr), HIP_SYMBOL(scratch)) != hipSuccess ||
        ptr == nullptr) {
      (void)hipGetLastError();
      *rc = HBT_EHIP;
      return nullptr;
    }
    address[device] = ptr;
  }
  return address[device];
}

// Into how many parts mlp_layer_tile_kernel splits K for a batch of m_tiles
// m-tiles.  A layer is 32 x m_tiles output tiles on 4 x compute_units SIMDs and
// takes ceil(32 m_tiles KS / SIMDs) steps of 1 / KS of a whole-K tile's time:
// the finest split is never worse by that count, but a wave's run gets shorter
// (a run of 32 k-groups is 3.4 us of MFMAs, next to about a microsecond until
// its first fragments arrive) and all workgroups should be resident at once (8
// per compute unit), so the coarsest split among the cheapest is taken: on 256
// compute units KS = 2 up to 4096 rows and KS = 4 up to 2048.
int tile_k_parts(int m_tiles, int compute_units) {
  const int simds = 4 * compute_units;  // 1024 on the GPU the thresholds were measured on
  // steps a layer takes with K in `ks` parts, in quarters of a whole-K step
  auto cost = [&](int ks) { return (32 * m_tiles * ks + simds - 1) / simds * (4 / ks); };
  int best = 1, best_cost = cost(1);
  if (m_tiles <= simds / 8 && cost(2) < best_cost) {
    best = 2;
    best_cost = cost(2);
  }
  if (m_tiles <= simds / 16 && cost(4) < best_cost) best = 4;
  return best;
}

// Up to kChainMaxRows rows through the whole network in one launch (mlp_chain.h).
int forward_chain(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out, uint64_t* chain,
                  hipStream_t stream, uint32_t* done_flag, uint32_t done_value) {
  hbt::chain::Args a{};
  a.w_stream = mlp->w_stream;
  a.first_groups = mlp->in_padded / 8;
  a.groups_total = a.first_groups + mlp->hidden * (hbt::kWidth / 8);
  a.hidden = mlp->hidden;
  a.w_first_t = mlp->w_first_t;
  a.bias = mlp->bias;
  a.w_last = mlp->w_last;
  a.b_last = mlp->b_last;
  a.raw = raw_features; a.mu = mlp->mu; a.sigma = mlp->sigma;
  a.in_features = mlp->in_features;
  a.n = (int32_t)n;
  a.out = out;
  a.done_flag = done_flag;
  a.done_value = done_value;
  a.tickets = chain;
  a.words = chain + hbt::kChainHeader;
  a.looks = hbt::chain::kMaxLooks;
  return hbt::chain::launch(a, stream) == hipSuccess ? HBT_OK : HBT_EHIP;
}

// One launch per layer for n <= kLayerMaxRows rows, through two buffers of
// activations or K-partials (each at least max(n rounded up to 32, kSplit * 32)
// x kWidth floats): the handle's, or the library's static ones.  The fewest rows
// take one launch for all layers.
int forward_layers(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                   float* const buffers[2], uint64_t* chain, hipStream_t stream,
                   uint32_t* done_flag = nullptr, uint32_t done_value = 0) {
  using namespace hbt;
  if (n <= kChainMaxRows && mlp->hidden > 0)
    return forward_chain(mlp, raw_features, n, out, chain, stream, done_flag, done_value);
  const int m_tiles = (int)((n + kRows - 1) / kRows);
  const bool split_k = n <= kSplitMaxRows;
  // with a few m-tiles the eight-wave shape splits K in two as well
  const int ks = (!split_k && m_tiles <= kHalfKMaxTiles) ? 2 : 1;
  LayerArgs l{};
  l.w_stream = mlp->w_stream;
  l.groups_total = mlp->in_padded / 8 + mlp->hidden * (kWidth / 8);
  l.raw = raw_features; l.mu = mlp->mu; l.sigma = mlp->sigma;
  l.in_features = mlp->in_features;
  l.n = n;
  l.m_pad = m_tiles * kRows;
  l.w_first_t = mlp->w_first_t;
  bool partials = false;
  const float* p_in = nullptr;
  const int tile_ks = tile_k_parts(m_tiles, mlp->compute_units);
  for (int layer = 0; layer <= mlp->hidden; ++layer) {
    l.g0 = (layer == 0) ? 0 : mlp->in_padded / 8 + (layer - 1) * (kWidth / 8);
    l.kg = (layer == 0) ? mlp->in_padded / 8 : kWidth / 8;
    l.splits = layer == 0 ? 1 : (split_k ? kSplit : ks);
    l.p_in = p_in;
    l.bias_in = (layer == 0) ? nullptr : mlp->bias + (size_t)(layer - 1) * kWidth;
    l.bias_out = mlp->bias + (size_t)layer * kWidth;
    l.p_out = buffers[layer & 1];
    const dim3 grid(kWidth / 32, (unsigned)l.splits, (unsigned)m_tiles);
    if (layer == 0 && split_k)
      hipLaunchKernelGGL((mlp_layer_kernel<true, 0, true, 4, false, 0>), grid, dim3(256), 0,
                         stream, l);
    else if (layer == 0 && mlp->in_features <= kFirstFmaMaxIn && m_tiles >= kFirstFmaMinTiles) {
      hipLaunchKernelGGL(mlp_first_fma_kernel, dim3((unsigned)m_tiles, kFirstFmaSlices), dim3(256), 0,
                         stream, l);
    } else if (layer == 0)
      hipLaunchKernelGGL((mlp_layer_kernel<true, 0, true, 4, false, 0, 1, true>), grid, dim3(256),
                         0, stream, l);
    else if (ks == 2 && !partials)
      hipLaunchKernelGGL((mlp_layer_kernel<false, 0, false, 8, true, 2, 1, true, 2>), grid,
                         dim3(512), 0, stream, l);
    else if (ks == 2)
      hipLaunchKernelGGL((mlp_layer_kernel<false, 2, false, 8, true, 2, 1, true, 2>), grid,
                         dim3(512), 0, stream, l);
    else if (!split_k && tile_ks == 1)
      hipLaunchKernelGGL((mlp_layer_tile_kernel<1, 4>),
                         dim3(kWidth / 64, (unsigned)((m_tiles + 1) / 2)), dim3(256), 0, stream, l);
    else if (!split_k && tile_ks == 2)
      hipLaunchKernelGGL((mlp_layer_tile_kernel<2, 4>), dim3(kWidth / 64, (unsigned)m_tiles),
                         dim3(256), 0, stream, l);
    else if (!split_k)
      hipLaunchKernelGGL((mlp_layer_tile_kernel<4, 4>), dim3(kWidth / 32, (unsigned)m_tiles),
                         dim3(256), 0, stream, l);
    else if (partials)
      hipLaunchKernelGGL((mlp_layer_kernel<false, kSplit, false, 4, false, 0>), grid, dim3(256),
                         0, stream, l);
    else
      hipLaunchKernelGGL((mlp_layer_kernel<false, 0, false, 4, false, 0>), grid, dim3(256), 0,
                         stream, l);
    p_in = l.p_out;
    partials = l.splits != 1;
  }
  LastArgs z{};
  z.p_in = p_in;
  z.bias_in = mlp->bias + (size_t)mlp->hidden * kWidth;
  z.w_last = mlp->w_last; z.b_last = mlp->b_last;
  z.n = n; z.m_pad = l.m_pad; z.out = out;
  z.done_flag = split_k ? done_flag : nullptr;  // (only the few-row shape publishes)
  z.done_value = done_value;
  const dim3 rows_grid((unsigned)((n + 3) / 4));
  if (partials && split_k)
    hipLaunchKernelGGL(mlp_last_kernel<kSplit>, rows_grid, dim3(256), 0, stream, z);
  else if (split_k) hipLaunchKernelGGL(mlp_last_kernel<0>, rows_grid, dim3(256), 0, stream, z);
  else if (partials && ks == 2)
    hipLaunchKernelGGL(mlp_last_km_kernel<2>, dim3((unsigned)m_tiles), dim3(256), 0, stream, z);
  else hipLaunchKernelGGL(mlp_last_km_kernel<0>, dim3((unsigned)m_tiles), dim3(256), 0, stream, z);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

// The fused kernel: one workgroup per 32 rows.
hbt::MlpArgs fused_args(const hbt_mlp* mlp, const double* raw_features, int64_t n, float* out) {
  hbt::MlpArgs a{};
  a.raw = raw_features;
  a.out = out;
  a.n = n;
  a.in_features = mlp->in_features;
  a.in_padded = mlp->in_padded;
  a.hidden = mlp->hidden;
  a.mu = mlp->mu;
  a.sigma = mlp->sigma;
  a.w_stream = mlp->w_stream;
  a.bias = mlp->bias;
  a.w_last = mlp->w_last;
  a.b_last = mlp->b_last;
  return a;
}

int forward_fused(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                  hipStream_t stream) {
  using namespace hbt;
  const MlpArgs a = fused_args(mlp, raw_features, n, out);
  hipLaunchKernelGGL((mlp_fused_kernel<kWaves, false>), dim3((unsigned)((n + kRows - 1) / kRows)),
                     dim3(kWaves * 64), kLdsBytes, stream, a);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

// The split path's hidden layers (mlp_split.h).
namespace split = hbt::split;
namespace pairs = hbt::pairs;
using hbt::kWidth;
constexpr size_t kSplitLayerBytes = (size_t)(kWidth / 32) * split::kTileBytes;

struct SplitLarge {
  using S = split::Large<4, 2, 2, 4, 24>;
  static constexpr auto kHidden = &split::large_kernel<4, 2, 2, 4, 24, false>;
  static constexpr auto kLast = &split::large_kernel<4, 2, 2, 4, 24, true>;
};
struct SplitMid192 {
  using S = split::Mid<1, 3, 4, 2, 2, 2>;
  static constexpr auto kHidden = &split::mid_kernel<1, 3, 4, 2, 2, 2, false>;
  static constexpr auto kLast = &split::mid_kernel<1, 3, 4, 2, 2, 2, true>;
};
template <int TN, int TM, int WAVES, int RING, int SETS>
struct SplitSmall {
  using S = split::Small<TN, TM, WAVES, RING, 4, SETS>;
  static constexpr auto kHidden = &split::small_kernel<TN, TM, WAVES, RING, 4, SETS, false>;
  static constexpr auto kLast = &split::small_kernel<TN, TM, WAVES, RING, 4, SETS, true>;
};
using SplitSmall1x1 = SplitSmall<1, 1, 8, 4, 2>;
using SplitSmall1x2 = SplitSmall<1, 2, 8, 3, 2>;
using SplitSmall2x2 = SplitSmall<2, 2, 8, 2, 2>;
using SplitSmall2x3 = SplitSmall<2, 3, 4, 2, 2>;
using SplitSmall2x4 = SplitSmall<2, 4, 4, 2, 2>;
using SplitSmall4x3 = SplitSmall<4, 3, 4, 2, 1>;
using SplitSmall4x4 = SplitSmall<4, 4, 4, 2, 1>;

template <class C>
bool split_ready_one() {
  const auto set = [](const void* f) {
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, C::S::LDS) ==
           hipSuccess;
  };
  return set(reinterpret_cast<const void*>(C::kHidden)) &&
         set(reinterpret_cast<const void*>(C::kLast));
}

template <class... C>
bool split_ready() {
  return (split_ready_one<C>() && ...);
}

template <class C>
void split_launch(const split::LayerArgs& a, bool last, hipStream_t stream) {
  const int m_blocks = (a.m_tiles + C::S::BM - 1) / C::S::BM;
  const dim3 grid((unsigned)((m_blocks + C::S::XM - 1) / C::S::XM * C::S::XM * C::S::NBLK));
  hipLaunchKernelGGL(last ? C::kLast : C::kHidden, grid, dim3(C::S::THREADS), C::S::LDS, stream,
                     a);
}

// The kernel for a layer of m_tiles m-tiles: each takes rounds of one workgroup
// per compute unit, whatever the last one holds, so the one whose rounds cost
// least.  Microseconds on 256 compute units, start + per round; what matters is
// their ratio where the choice changes (a full round of large_kernel takes 143, one
// of 12 289 rows 128).  Whole forwards of ten layers, us, in turn on one card:
//
//    rows   2x2   2x3   2x4   4x3   4x4   mid  large
//    1600   188   233   177   212   258   383    966   2x4 to 2048
//    4512   457   408   489   450   539   439    978   2x3 to 4608
//    4704   462   506   491   456   541   447    976   mid to 6144
//    5856   567   540   525   496   582   492    987
//    7936   746   765   693   707   645   869   1014   4x4 to 8192
//    9088   859   803   844   742   867   868   1019   4x3 to 9216
//   10240   932   918   876   923   900   905   1056   2x4 to 10 240
//   11392  1085  1025  1007   954   934   950   1081   mid to 12 288
//   12544  1143  1138  1154  1146  1169  1258   1078   large from 12 289
//   16384  1473  1418  1376  1396  1272  1351   1223
//
// Where mid_kernel and the 4 x 3 and 4 x 4 tiles are within 2 %, it is taken for its
// second set of sums (errors of 0.8 and 1.2 in 2^-24 of a layer's output).
using SplitLaunch = void (*)(const split::LayerArgs&, bool, hipStream_t);
SplitLaunch split_kernel_for(int m_tiles, int compute_units) {
  SplitLaunch best = nullptr;
  float best_us = 0.f;
  const auto consider = [&](auto kernel, float start, float round_us) {
    using C = decltype(kernel);
    const int per_round = C::S::BM * (compute_units / C::S::NBLK > 0 ? compute_units / C::S::NBLK : 1);
    const float us = start + round_us * (float)((m_tiles + per_round - 1) / per_round);
    if (best == nullptr || us < best_us) {
      best = split_launch<C>;
      best_us = us;
    }
  };
  consider(SplitSmall1x1(), 2.7f, 4.05f);   // rounds of 256 rows
  consider(SplitSmall1x2(), 2.f, 6.9f);     // 512
  consider(SplitSmall2x2(), 3.5f, 10.f);    // 1024
  consider(SplitSmall2x3(), 2.5f, 13.5f);   // 1536
  consider(SplitSmall2x4(), 4.f, 18.f);     // 2048
  consider(SplitSmall4x3(), 4.f, 24.5f);   // 3072
  consider(SplitSmall4x4(), 3.f, 32.f);    // 4096
  consider(SplitMid192(), 6.f, 44.f);      // 6144
  consider(SplitLarge(), 0.f, 122.f);      // 16 384
  return best;
}

// The split path for up to chunk_rows rows, through two buffers of activations in
// pieces (kTileBytes per m-tile) and one of the final dot product's shares
// ([kWidth / 32][m_tiles * 32]): the handle's, or the library's static ones.
int forward_split(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                  float* const scratch[2], float* part, hipStream_t stream) {
  using namespace hbt;
  const int m_tiles = (int)((n + kRows - 1) / kRows);
  char* const buffers[2] = {reinterpret_cast<char*>(scratch[0]),
                            reinterpret_cast<char*>(scratch[1])};
  split::FirstArgs f{};
  f.raw = raw_features; f.mu = mlp->mu; f.sigma = mlp->sigma;
  f.w_t = mlp->w_first_t; f.bias = mlp->bias;
  f.in_features = mlp->in_features; f.n = n;
  f.y = buffers[0];
  const dim3 first_grid((unsigned)m_tiles, split::kFirstSlices);
  if (mlp->in_features <= kFirstFmaMaxIn)
    hipLaunchKernelGGL(split::first_kernel<kFirstFmaMaxIn>, first_grid, dim3(256), 0, stream, f);
  else
    hipLaunchKernelGGL(split::first_kernel<kMaxInPadded>, first_grid, dim3(256), 0, stream, f);
  const SplitLaunch launch = split_kernel_for(m_tiles, mlp->compute_units);
  split::LayerArgs l{};
  l.w_last = mlp->w_last;
  l.part = part;
  l.m_tiles = m_tiles;
  for (int layer = 0; layer < mlp->hidden; ++layer) {
    l.w = mlp->w_split + (size_t)layer * kSplitLayerBytes;
    l.bias = mlp->bias + (size_t)(layer + 1) * kWidth;
    l.x = buffers[layer & 1];
    l.y = buffers[(layer + 1) & 1];
    const bool last = layer + 1 == mlp->hidden;
    launch(l, last, stream);
  }
  split::FinishArgs z{};
  z.part = part;
  z.rows_pad = m_tiles * kRows;
  z.b_last = mlp->b_last;
  z.n = n;
  z.out = out;
  hipLaunchKernelGGL(split::finish_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, z);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

// The pairs' hidden layers (mlp_pairs.h).
constexpr size_t kPairsLayerBytes = (size_t)(kWidth / 32) * pairs::kTileBytes;

template <class T, int TN, int TM, int KS, int NBUF, int RING, int FLUSH, int SPLIT>
struct PairsWide {
  using S = pairs::Wide<TN, TM, KS, NBUF, RING, FLUSH, SPLIT>;
  static constexpr auto kHidden = &pairs::wide_kernel<T, TN, TM, KS, NBUF, RING, FLUSH, SPLIT, false>;
  static constexpr auto kLast = &pairs::wide_kernel<T, TN, TM, KS, NBUF, RING, FLUSH, SPLIT, true>;
};
using PairsWide1x1 = PairsWide<double, 1, 1, 4, 3, 4, 4, 0>;
using PairsWide1x2 = PairsWide<float, 1, 2, 4, 3, 4, 8, 0>;
using PairsWide1x3 = PairsWide<float, 1, 3, 8, 2, 4, 8, 0>;
using PairsWide2x4 = PairsWide<float, 2, 4, 4, 3, 2, 64, 24>;

template <class C>
void pairs_launch(const pairs::LayerArgs& a, bool last, hipStream_t stream) {
  const int m_blocks = (a.m_tiles + C::S::BM - 1) / C::S::BM;
  const dim3 grid((unsigned)((m_blocks + C::S::XM - 1) / C::S::XM * C::S::XM * C::S::NBLK));
  hipLaunchKernelGGL(last ? C::kLast : C::kHidden, grid, dim3(C::S::THREADS), C::S::LDS, stream,
                     a);
}

// The kernel for a layer of m_tiles m-tiles, as split_kernel_for: in rounds of one
// workgroup per compute unit, the one whose rounds cost least, microseconds on 256 compute
// units.  Whole forwards of ten layers, us, in turn on one card:
//
//    rows   1x1   1x2   1x3   2x4   (three bf16 pieces)
//    1500   144                       155
//    2048   164   173                 196
//    4096         222   244   492     326
//    4500   370                       420
//    5911         362   293   499     482
//    8192         389   471   540     653
//   12288         630   579   567     962
//   16384         814   803   686    1196
//
// At 9217 to 12 288 rows 2 x 4 tiles are 2 % faster than 1 x 3; the sums of these are nearer.
//
// 1 x 1 tiles, with totals in double, have the nearest sums: errors of a prediction (eight
// networks, 2-norm, relative) 4.8e-8; 1 x 2 and 1 x 3 have 5.8e-8, 2 x 4 1.17e-7.  They are
// taken for a batch of up to one round, where they are the fastest too, and in two ranges in
// which the three bf16 pieces have their nearest sums, 4.8e-8 as well (in the others 6.5e-8,
// one set of sums 1.07e-7, large_kernel 1.41e-7), so that no batch is further from exact
// sums in pairs than in pieces: 2 to 2 1/4 rounds (4097 to 4608 rows; 4500: 370 us, 1 x 3 in
// one round of its own 293) and 4 1/2 to 5 (9217 to 10 240; 10 000: 631 and 570).
bool pairs_nearest(int m_tiles, int compute_units) {
  constexpr int kBlocks = PairsWide1x1::S::NBLK;
  const int round = compute_units / kBlocks > 0 ? compute_units / kBlocks : 1;   // of m-tiles
  return m_tiles <= round || (m_tiles > 2 * round && 4 * m_tiles <= 9 * round) ||
         (2 * m_tiles > 9 * round && m_tiles <= 5 * round);
}
struct PairsKernel {
  void (*launch)(const pairs::LayerArgs&, bool, hipStream_t);
  int parts;   // in which a layer leaves the rows' largest outputs
};
PairsKernel pairs_kernel_for(int m_tiles, int compute_units) {
  if (pairs_nearest(m_tiles, compute_units))
    return {pairs_launch<PairsWide1x1>, PairsWide1x1::S::PARTS};
  PairsKernel best{};
  float best_us = 0.f;
  const auto consider = [&](auto kernel, float start, float round_us) {
    using C = decltype(kernel);
    const int per_round = C::S::BM * (compute_units / C::S::NBLK > 0 ? compute_units / C::S::NBLK : 1);
    const float us = start + round_us * (float)((m_tiles + per_round - 1) / per_round);
    if (best.launch == nullptr || us < best_us) {
      best = {pairs_launch<C>, C::S::PARTS};
      best_us = us;
    }
  };
  consider(PairsWide1x2(), 1.5f, 22.5f);   // rounds of 4096 rows
  consider(PairsWide1x3(), 0.5f, 32.5f);   // 6144
  consider(PairsWide2x4(), 0.f, 81.f);     // 16 384
  return best;
}

// The same with pairs, through the handle's scratch.
int forward_pairs(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                  hipStream_t stream) {
  using namespace hbt;
  const int m_tiles = (int)((n + kRows - 1) / kRows);
  char* const buffers[2] = {reinterpret_cast<char*>(mlp->scratch[0]),
                            reinterpret_cast<char*>(mlp->scratch[1])};
  pairs::FirstArgs f{};
  f.raw = raw_features; f.mu = mlp->mu; f.sigma = mlp->sigma;
  f.w_t = mlp->w_first_t;
  f.units = {mlp->bias, nullptr, mlp->G, mlp->bias_most};
  f.in_features = mlp->in_features; f.n = n;
  f.y = buffers[0]; f.e_out = mlp->row_scales[0]; f.most_out = mlp->row_most[0];
  f.redo = mlp->redo;
  const dim3 first_grid((unsigned)m_tiles, split::kFirstSlices);
  if (mlp->in_features <= kFirstFmaMaxIn)
    hipLaunchKernelGGL(pairs::first_kernel<kFirstFmaMaxIn>, first_grid, dim3(256), 0, stream, f);
  else
    hipLaunchKernelGGL(pairs::first_kernel<kMaxInPadded>, first_grid, dim3(256), 0, stream, f);
  const PairsKernel kernel = pairs_kernel_for(m_tiles, mlp->compute_units);
  pairs::LayerArgs l{};
  l.w_last = mlp->w_last;
  l.part = mlp->part;
  l.m_tiles = m_tiles;
  l.most_count = pairs::kFirstParts;
  l.redo = mlp->redo;
  for (int layer = 0; layer < mlp->hidden; ++layer) {
    const int in = layer & 1, to = in ^ 1;
    l.w = mlp->w_pairs + (size_t)layer * kPairsLayerBytes;
    l.units = {mlp->bias + (size_t)(layer + 1) * kWidth, mlp->F + (size_t)layer * kWidth,
               mlp->G + (size_t)(layer + 1) * kWidth, mlp->bias_most + layer + 1};
    l.x = buffers[in]; l.e_in = mlp->row_scales[in]; l.most_in = mlp->row_most[in];
    l.y = buffers[to]; l.e_out = mlp->row_scales[to]; l.most_out = mlp->row_most[to];
    kernel.launch(l, layer + 1 == mlp->hidden, stream);
    l.most_count = kernel.parts;
  }
  MlpArgs z = fused_args(mlp, raw_features, n, out);
  z.part = mlp->part;
  z.rows_pad = m_tiles * kRows;
  z.redo = mlp->redo;
  hipLaunchKernelGGL((mlp_fused_kernel<kWaves, true>), dim3((unsigned)m_tiles), dim3(kWaves * 64),
                     kLdsBytes, stream, z);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

// Rows up to which the pieces stay: a layer there is a launch's start, loads' latency and
// the meeting of the sums, and pairs, with half the products and two thirds of the bytes,
// gain nothing (700 rows: 96 us in the form of split::small_kernel, 99 with pieces).
constexpr int kPairsAboveRows = 1024;

// Any number of rows on the fp32 matrix cores.  The fused kernel keeps every
// compute unit busy for whole rounds of 32 rows x compute units (about 0.94 ms
// each); what is left over after the last whole round would cost another one.
// Up to kLayerMaxRows leftover rows go through the per-layer path instead, which
// takes less for them.
int forward_fp32(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                 hipStream_t stream) {
  using namespace hbt;
  const int64_t round_rows = (int64_t)kRows * mlp->compute_units;
  const int64_t leftover = n % round_rows;
  if (leftover == 0 || leftover > kLayerMaxRows)
    return forward_fused(mlp, raw_features, n, out, stream);
  const int64_t done = n - leftover;
  if (done > 0) {
    const int rc = forward_fused(mlp, raw_features, done, out, stream);
    if (rc != HBT_OK) return rc;
  }
  return forward_layers(mlp, raw_features + done * mlp->in_features, leftover, out + done,
                        mlp->scratch, mlp->chain[0], stream);
}

// What hbt_mlp_forward and hbt_mlp_forward_fp32 refuse.
int check_forward(const hbt_mlp* mlp, const double* raw_features, int64_t n, const float* out) {
  if (mlp == nullptr || n < 0) return HBT_EINVAL;
  if (n == 0) return HBT_OK;
  if (raw_features == nullptr || out == nullptr) return HBT_EINVAL;
  if ((reinterpret_cast<uintptr_t>(raw_features) % 8) != 0 ||
      (reinterpret_cast<uintptr_t>(out) % 4) != 0)
    return HBT_EALIGN;
  if ((n + hbt::kRows - 1) / hbt::kRows > 0x7fffffff) return HBT_ESIZE;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    return HBT_EHIP;
  }
  return device != mlp->device ? HBT_EINVAL : HBT_OK;
}

}  // namespace

extern "C" {

hbt_mlp* hbt_mlp_create(int32_t in_features, int32_t width, int32_t hidden_layers,
                        const float* const* W, const float* const* b, const double* mu,
                        const double* sigma, int* err) {
  using namespace hbt;
  int dummy;
  if (err == nullptr) err = &dummy;
  *err = HBT_OK;
  if (W == nullptr || b == nullptr || mu == nullptr || sigma == nullptr || in_features <= 0 ||
      hidden_layers < 0) {
    *err = HBT_EINVAL;
    return nullptr;
  }
  for (int i = 0; i < hidden_layers + 2; ++i)
    if (W[i] == nullptr || b[i] == nullptr) { *err = HBT_EINVAL; return nullptr; }
  const int in_padded = (int)align_up((size_t)in_features, 32);
  if (width != kWidth || in_padded > kMaxInPadded || hidden_layers > 64) {
    *err = HBT_ESIZE;
    return nullptr;
  }
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    *err = HBT_EHIP;
    return nullptr;
  }

  int compute_units = 0;
  if (hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, device) !=
          hipSuccess ||
      compute_units <= 0) {
    (void)hipGetLastError();
    *err = HBT_EHIP;
    return nullptr;
  }

  // Host image of the device blob.
  // floats per wave: (fc1 groups + 128 per hidden layer) x tpw x 64 lanes x 4
  const int tpw = (kWidth / 32) / kWaves;
  const size_t group_floats = (size_t)tpw * 64 * 4;
  const size_t wave_stride = ((size_t)in_padded / 8 + (size_t)hidden_layers * (kWidth / 8)) * group_floats;
  const size_t n_stream = wave_stride * kWaves;
  const size_t n_bias = (size_t)(hidden_layers + 1) * kWidth;
  size_t off = 0;
  const size_t off_mu = off; off = align_up(off + sizeof(double) * in_features, 256);
  const size_t off_sigma = off; off = align_up(off + sizeof(double) * in_features, 256);
  const size_t off_stream = off; off = align_up(off + sizeof(float) * n_stream, 256);
  const size_t off_bias = off; off = align_up(off + sizeof(float) * n_bias, 256);
  const size_t off_last = off; off = align_up(off + sizeof(float) * kWidth, 256);
  const size_t first_t_rows = in_features <= kFirstFmaMaxIn ? kFirstFmaMaxIn : kMaxInPadded;
  const size_t off_first_t = off;
  off = align_up(off + sizeof(float) * first_t_rows * kWidth, 256);
  const size_t off_bias_most = off; off = align_up(off + sizeof(int32_t) * (hidden_layers + 1), 256);
  const size_t off_column_lost = off;
  off = align_up(off + sizeof(int32_t) * (size_t)hidden_layers * kWidth, 256);
  const size_t image = off;  // what is copied from the host; scratch follows
  const int64_t chunk_rows = kSplitRowsPerUnit * compute_units;
  size_t scratch_bytes = (size_t)(chunk_rows / kRows) * split::kTileBytes;
  const size_t layer_bytes = sizeof(float) * (size_t)kLayerMaxRows * kWidth;  // forward_layers
  if (scratch_bytes < layer_bytes) scratch_bytes = layer_bytes;
  const size_t off_split = off; off = align_up(off + (size_t)hidden_layers * kSplitLayerBytes, 256);
  const size_t off_pairs = off; off = align_up(off + (size_t)hidden_layers * kPairsLayerBytes, 256);
  const size_t unit_ints = (size_t)(hidden_layers + 1) * kWidth;
  const size_t off_F = off; off += sizeof(int32_t) * unit_ints;
  const size_t off_G = off; off += sizeof(int32_t) * unit_ints;
  const size_t off_sizes = off; off = align_up(off + sizeof(float) * unit_ints, 256);
  const size_t off_row_scales = off;
  off = align_up(off + sizeof(int32_t) * 2 * (1 + kWidth / 32) * (size_t)chunk_rows, 256);
  const size_t off_redo = off; off = align_up(off + sizeof(int32_t) * (size_t)chunk_rows, 256);
  const size_t off_scratch0 = off; off = align_up(off + scratch_bytes, 256);
  const size_t off_scratch1 = off; off = align_up(off + scratch_bytes, 256);
  const size_t off_part = off;
  off = align_up(off + sizeof(float) * (kWidth / 32) * (size_t)chunk_rows, 256);
  const size_t chain_bytes = align_up(sizeof(uint64_t) *
      (kChainHeader + (size_t)hidden_layers * chain::kMaxRows * kWidth), 256);
  const size_t off_chain = off; off += 2 * chain_bytes;
  const size_t total = off;

  std::vector<unsigned char> host;
  try {
    host.resize(image, 0);
  } catch (const std::bad_alloc&) {
    *err = HBT_ENOMEM;
    return nullptr;
  }
  std::memcpy(host.data() + off_mu, mu, sizeof(double) * in_features);
  std::memcpy(host.data() + off_sigma, sigma, sizeof(double) * in_features);
  float* stream = reinterpret_cast<float*>(host.data() + off_stream);
  pack_layer(W[0], in_features, in_padded, kWaves, stream, wave_stride);
  for (int l = 0; l < hidden_layers; ++l)
    pack_layer(W[1 + l], kWidth, kWidth, kWaves,
               stream + ((size_t)in_padded / 8 + (size_t)l * (kWidth / 8)) * group_floats, wave_stride);
  for (int l = 0; l <= hidden_layers; ++l)
    std::memcpy(host.data() + off_bias + sizeof(float) * (size_t)l * kWidth, b[l],
                sizeof(float) * kWidth);
  std::memcpy(host.data() + off_last, W[hidden_layers + 1], sizeof(float) * kWidth);
  float* first_t = reinterpret_cast<float*>(host.data() + off_first_t);  // zero beyond in_features
  for (int n = 0; n < kWidth; ++n)
    for (int k = 0; k < in_features; ++k)
      first_t[(size_t)k * kWidth + n] = W[0][(size_t)n * in_features + k];

  for (int l = 0; l <= hidden_layers; ++l)
    reinterpret_cast<int32_t*>(host.data() + off_bias_most)[l] = -pairs::kNotFinite;

  void* blob = nullptr;
  if (hipMalloc(&blob, total) != hipSuccess) {
    (void)hipGetLastError();
    *err = HBT_ENOMEM;
    return nullptr;
  }
  if (hipMemcpy(blob, host.data(), image, hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(blob);
    *err = HBT_EHIP;
    return nullptr;
  }
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_fused_kernel<kWaves, false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)kLdsBytes) != hipSuccess ||
      hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_fused_kernel<kWaves, true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)kLdsBytes) != hipSuccess ||
      !split_ready<SplitSmall1x1, SplitSmall1x2, SplitSmall2x2, SplitSmall2x3, SplitSmall2x4,
                   SplitSmall4x3, SplitSmall4x4, SplitMid192, SplitLarge, PairsWide1x1, PairsWide1x2,
                   PairsWide1x3, PairsWide2x4>()) {
    (void)hipGetLastError();
    (void)hipFree(blob);
    *err = HBT_EHIP;
    return nullptr;
  }
  if (hipMemset(static_cast<unsigned char*>(blob) + off_chain, 0, 2 * chain_bytes) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(blob);
    *err = HBT_EHIP;
    return nullptr;
  }
  void* one_host = nullptr;
  void* one_device = nullptr;
  if (hipHostMalloc(&one_host, kOneBytes, hipHostMallocDefault) != hipSuccess ||
      hipHostGetDevicePointer(&one_device, one_host, 0) != hipSuccess || one_device == nullptr) {
    (void)hipGetLastError();
    if (one_host != nullptr) (void)hipHostFree(one_host);
    (void)hipFree(blob);
    *err = HBT_ENOMEM;
    return nullptr;
  }
  std::memset(one_host, 0, kOneBytes);

  // the hidden layers' weights in bf16 pieces, from the packed fp32 ones
  for (int l = 0; l < hidden_layers; ++l) {
    split::PackArgs a{};
    a.w_stream = reinterpret_cast<const float*>(static_cast<unsigned char*>(blob) + off_stream);
    a.groups_total = in_padded / 8 + hidden_layers * (kWidth / 8);
    a.g0 = in_padded / 8 + l * (kWidth / 8);
    a.w = reinterpret_cast<char*>(blob) + off_split + (size_t)l * kSplitLayerBytes;
    hipLaunchKernelGGL(split::pack_kernel, dim3((kWidth / 32) * split::kSteps / 4), dim3(256), 0,
                       nullptr, a);
  }
  if (hidden_layers > 0) {
    split::CheckArgs a{};
    a.w_stream = reinterpret_cast<const float*>(static_cast<unsigned char*>(blob) + off_stream);
    a.groups_total = in_padded / 8 + hidden_layers * (kWidth / 8);
    a.g0 = in_padded / 8;
    // (through host memory: a copy back made the next call from an idle GPU 10 us slower)
    a.outside = reinterpret_cast<uint32_t*>(static_cast<unsigned char*>(one_device) +
                                            kOneOutsideOffset);
    hipLaunchKernelGGL(split::check_kernel, dim3(kWidth / 32, (unsigned)hidden_layers), dim3(64), 0,
                       nullptr, a);
    // and as fp16 pairs, after the sizes of the units, a layer after the other
    unsigned char* const base = static_cast<unsigned char*>(blob);
    pairs::PrepareArgs p{};
    p.w_stream = a.w_stream;
    p.groups_total = a.groups_total;
    p.w_first_t = reinterpret_cast<const float*>(base + off_first_t);
    p.in_features = in_features;
    p.bias = reinterpret_cast<const float*>(base + off_bias);
    p.G = reinterpret_cast<int32_t*>(base + off_G);
    p.bias_most = reinterpret_cast<int32_t*>(base + off_bias_most);
    p.size = reinterpret_cast<float*>(base + off_sizes);
    p.outside = reinterpret_cast<uint32_t*>(static_cast<unsigned char*>(one_device) +
                                            kOneOutsidePairsOffset);
    hipLaunchKernelGGL(pairs::prepare_first, dim3(kWidth / 256), dim3(256), 0, nullptr, p);
    for (int l = 0; l < hidden_layers; ++l) {
      p.g0 = in_padded / 8 + l * (kWidth / 8);
      p.G_in = p.G;
      p.size_in = p.size;
      p.F = reinterpret_cast<int32_t*>(base + off_F) + (size_t)l * kWidth;
      p.column_lost = reinterpret_cast<int32_t*>(base + off_column_lost) + (size_t)l * kWidth;
      p.G += kWidth;
      p.size += kWidth;
      p.bias += kWidth;
      ++p.bias_most;
      hipLaunchKernelGGL(pairs::prepare_layer, dim3(kWidth / 32), dim3(1024), 0, nullptr, p);
      pairs::PackArgs k{};
      k.w_stream = a.w_stream;
      k.groups_total = a.groups_total;
      k.g0 = p.g0;
      k.G_in = p.G_in;
      k.size_in = p.size_in;
      k.F = p.F;
      k.w = reinterpret_cast<char*>(base) + off_pairs + (size_t)l * kPairsLayerBytes;
      hipLaunchKernelGGL(pairs::pack_kernel, dim3((kWidth / 32) * split::kSteps / 4), dim3(256), 0,
                         nullptr, k);
    }
  }
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipHostFree(one_host);
    (void)hipFree(blob);
    *err = HBT_EHIP;
    return nullptr;
  }
  uint32_t outside[2] = {};
  std::memcpy(outside, static_cast<unsigned char*>(one_host) + kOneOutsideOffset, sizeof outside);

  hbt_mlp* m = new (std::nothrow) hbt_mlp();
  if (m == nullptr) {
    (void)hipHostFree(one_host);
    (void)hipFree(blob);
    *err = HBT_ENOMEM;
    return nullptr;
  }
  m->one_host = static_cast<unsigned char*>(one_host);
  m->one_device = static_cast<unsigned char*>(one_device);
  unsigned char* base = static_cast<unsigned char*>(blob);
  m->in_features = in_features;
  m->in_padded = in_padded;
  m->width = width;
  m->hidden = hidden_layers;
  m->device = device;
  m->compute_units = compute_units;
  m->blob = blob;
  m->mu = reinterpret_cast<const double*>(base + off_mu);
  m->sigma = reinterpret_cast<const double*>(base + off_sigma);
  m->w_stream = reinterpret_cast<const float*>(base + off_stream);
  m->bias = reinterpret_cast<const float*>(base + off_bias);
  m->w_last = reinterpret_cast<const float*>(base + off_last);
  m->w_first_t = reinterpret_cast<const float*>(base + off_first_t);
  m->w_split = reinterpret_cast<const char*>(base + off_split);
  m->takes_pieces = hidden_layers > 0 && outside[0] == 0;
  m->w_pairs = reinterpret_cast<const char*>(base + off_pairs);
  m->F = reinterpret_cast<const int32_t*>(base + off_F);
  m->G = reinterpret_cast<const int32_t*>(base + off_G);
  m->bias_most = reinterpret_cast<const int32_t*>(base + off_bias_most);
  m->takes_pairs = m->takes_pieces && outside[1] == 0;
  for (int i = 0; i < 2; ++i) {
    int32_t* const rows = reinterpret_cast<int32_t*>(base + off_row_scales) +
                          (size_t)i * (1 + kWidth / 32) * (size_t)chunk_rows;
    m->row_scales[i] = rows;
    m->row_most[i] = rows + chunk_rows;
  }
  m->redo = reinterpret_cast<int32_t*>(base + off_redo);
  m->chunk_rows = chunk_rows;
  for (int i = 0; i < 2; ++i)
    m->chain[i] = reinterpret_cast<uint64_t*>(base + off_chain + i * chain_bytes);
  m->part = reinterpret_cast<float*>(base + off_part);
  m->b_last = b[hidden_layers + 1][0];
  m->scratch[0] = reinterpret_cast<float*>(base + off_scratch0);
  m->scratch[1] = reinterpret_cast<float*>(base + off_scratch1);
  return m;
}

int hbt_mlp_forward(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                    void* hip_stream) {
  using namespace hbt;
  const int bad = check_forward(mlp, raw_features, n, out);
  if (bad != HBT_OK || n == 0) return bad;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  if (!mlp->takes_pieces) return forward_fp32(mlp, raw_features, n, out, stream);
  // Whole rounds of the 256 x 256 workgroups, then what is left over, with the
  // kernels that suit it.
  int64_t done = 0;
  while (done < n) {
    const int64_t rows = n - done < mlp->chunk_rows ? n - done : mlp->chunk_rows;
    const double* raw = raw_features + done * mlp->in_features;
    const int rc = rows <= kSplitAboveRows ? forward_fp32(mlp, raw, rows, out + done, stream)
                   : rows > kPairsAboveRows && mlp->takes_pairs
                       ? forward_pairs(mlp, raw, rows, out + done, stream)
                       : forward_split(mlp, raw, rows, out + done, mlp->scratch, mlp->part, stream);
    if (rc != HBT_OK) return rc;
    done += rows;
  }
  return HBT_OK;
}

int hbt_mlp_forward_fp32(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                         void* hip_stream) {
  const int bad = check_forward(mlp, raw_features, n, out);
  if (bad != HBT_OK || n == 0) return bad;
  return forward_fp32(mlp, raw_features, n, out, static_cast<hipStream_t>(hip_stream));
}

int hbt_mlp_forward_static(hbt_mlp* mlp, const double* raw_features, int64_t n, float* out,
                           void* hip_stream) {
  using namespace hbt;
  if (mlp == nullptr || n < 0) return HBT_EINVAL;
  if (n > kStaticMaxRows) return HBT_ESIZE;
  if (n == 0) return HBT_OK;
  if (raw_features == nullptr || out == nullptr) return HBT_EINVAL;
  if ((reinterpret_cast<uintptr_t>(raw_features) % 8) != 0 ||
      (reinterpret_cast<uintptr_t>(out) % 4) != 0)
    return HBT_EALIGN;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    return HBT_EHIP;
  }
  if (device != mlp->device) return HBT_EINVAL;
  int rc = HBT_OK;
  float* base = static_scratch_of(device, &rc);
  if (base == nullptr) return rc;
  // Every value a layer reads was written by the layer before it in this call
  // (rows past n within the last 32-row tile included), so nothing needs
  // clearing between calls.
  float* const buffers[2] = {base, base + kStaticFloats};
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  return n > kSplitAboveRows && mlp->takes_pieces
             ? forward_split(mlp, raw_features, n, out, buffers, base + 2 * kStaticFloats, stream)
             : forward_layers(mlp, raw_features, n, out, buffers, mlp->chain[1], stream);
}

int hbt_mlp_predict_one(hbt_mlp* mlp, const double* raw_row, float* out, void* hip_stream) {
  using namespace hbt;
  if (mlp == nullptr || raw_row == nullptr || out == nullptr) return HBT_EINVAL;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    return HBT_EHIP;
  }
  if (device != mlp->device) return HBT_EINVAL;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  // the call waits for its stream: a stream under graph capture cannot be used
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) != hipSuccess) {
    (void)hipGetLastError();
    return HBT_EHIP;
  }
  if (capture != hipStreamCaptureStatusNone) return HBT_EINVAL;

  std::lock_guard<std::mutex> guard(mlp->one_lock);
  std::memcpy(mlp->one_host, raw_row, sizeof(double) * (size_t)mlp->in_features);
  const uint32_t call = ++mlp->one_calls;
  const int rc = forward_layers(mlp, reinterpret_cast<const double*>(mlp->one_device), 1,
                                reinterpret_cast<float*>(mlp->one_device + kOneOutOffset),
                                mlp->scratch, mlp->chain[0], stream,
                                reinterpret_cast<uint32_t*>(mlp->one_device + kOneDoneOffset), call);
  if (rc != HBT_OK) return rc;
  // The last kernel publishes the call's number once the prediction is in the
  // block: watching for it takes microseconds less than waiting for the
  // stream's completion signal.  Should it not show up in time, the stream is
  // waited for, which is always right.
  if (!hbt::wait_published(reinterpret_cast<const uint32_t*>(mlp->one_host + kOneDoneOffset), call) &&
      hipStreamSynchronize(stream) != hipSuccess) {
    (void)hipGetLastError();
    return HBT_EHIP;
  }
  std::memcpy(out, mlp->one_host + kOneOutOffset, sizeof(float));
  return HBT_OK;
}

void hbt_mlp_destroy(hbt_mlp* mlp) {
  if (mlp == nullptr) return;
  if (mlp->one_host != nullptr) (void)hipHostFree(mlp->one_host);
  if (mlp->blob != nullptr) (void)hipFree(mlp->blob);
  delete mlp;
}

}  // extern "C"
