// A few rows through the whole network in one launch.
//
// Ten launches, one per layer, cost 3.6 to 4.8 us each whatever they hold: what
// bounds a handful of rows is that chain, not the 33.6 MB of weights (4 us).  Here
// a workgroup is one n-tile of one layer, and all of them, 32 per layer, start
// together: each fetches its 128 KiB of weights into registers at once, then waits
// for the activations of the layer before.  Those come as 8-byte words of a value
// and the number of the call, written and read with single atomic accesses, so a
// word that carries this call's number is the value itself: one trip through
// memory per layer, no fence, no counter, no clearing between calls.  Every
// kNumberAll-th call numbers the words of all kMaxRows rows, also those past its own:
// no word is older than that, and 32 bits of the number are enough for good.
//
// Order of workgroups: each takes the next ticket of the handle's counter when it
// starts, and the ticket says which tile of which layer it is.  So a workgroup
// waits only for ones that have started before it: nothing has to be resident
// together, and several such launches may share the GPU.  A workgroup that has
// waited too long computes its input by itself (alone()), in the same order of
// sums: a result never depends on how the waits went.
//
// The sums are those of mlp_layer_kernel and mlp_last_kernel for up to
// kSplitMaxRows rows, in the same order and as fused multiply-adds, which is how
// the fp32 matrix core rounds: the same results bit for bit.
//
// A layer takes about 1.9 us: the trip of the words, 0.2 us of multiply-adds per
// row, the sums through LDS.  Tried and not faster: half tiles, two workgroups to
// a compute unit (24 us for one row); waiting until the layer before the last one
// is done, longer pauses between looks; activations read from LDS by every lane
// instead of shared among 16 (21 us; the compiler's own sharing, 21.6).
//
// Included by mlp.hip, and by its test (tests/native/mlp_chain.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hbt {
namespace chain {

using f32x4 = float __attribute__((ext_vector_type(4)));

constexpr int kWidth = 1024;
constexpr int kTiles = kWidth / 32;
// Rows up to which this is the faster way: 19.2 / 23.9 / 27.6 / 29.9 us for 1 to 4
// (launches per layer 38.8 / 39.6 / 40.9 / 41.6); an earlier form took 39.5 and 46.0
// for 5 and 8 (42.0 and 44.2).  What a row adds is its share of the multiply-adds on
// a layer's 32 compute units, 0.2 us, and the reads of the next layer.
constexpr int kMaxRows = 4;
constexpr uint32_t kNumberAll = 1u << 16;  // calls
constexpr int kMaxIn = 64;
constexpr int kFewIn = 16;   // rows that w_first_t has at least, zero beyond the features
constexpr int kChains = 32;  // sums of 32 products that an output is added up from
// Looks at a word at full rate (about 200 us), and before a wait is given up (about
// 15 ms; a call in which every wait was given up at once took 0.4 ms).
constexpr int kBusyLooks = 256;
constexpr int kMaxLooks = 1 << 12;

struct Args {
  const float* w_stream;   // packed weights (mlp.hip)
  int32_t groups_total;    // k-groups per wave stream (all layers)
  int32_t first_groups;    // of them fc1's
  int32_t hidden;
  const float* w_first_t;  // fc1.weight transposed, [in_features][kWidth]
  const float* bias;       // [hidden + 1][kWidth]
  const float* w_last;     // [kWidth]
  float b_last;
  const double* raw;       // [n][in_features]
  const double* mu;
  const double* sigma;
  int32_t in_features;
  int32_t n;               // at most the instantiation's ROWS
  float* out;              // [n]
  uint32_t* done_flag;     // nullable, see LastArgs
  uint32_t done_value;
  uint64_t* tickets;       // counts all workgroups of all calls
  uint64_t* words;         // [hidden][kMaxRows][kWidth] activations and call numbers
  int32_t looks;           // at a word before a wait is given up (kMaxLooks)
};

// The i-th k that a sum takes: of each 8, the pairs (e, 4 + e) that the matrix core
// multiplies together.
__device__ __host__ constexpr int product(int i) {
  return (i & ~7) + 4 * (i & 1) + ((i >> 1) & 3);
}

// sum + the products of 16 weights, in the order of product(), with x, of which lane
// l of each 16 holds the l-th: 16 lanes share the values that they all want (read
// from LDS by every lane they took 0.4 us a row).  (The compiler makes two
// instructions of each step.  A value just written may not be shared at once,
// hence the wait states in front.)
template <int FIRST>
__device__ __forceinline__ float add_products(const f32x4 (&w)[4][2], float x, float sum) {
  constexpr int j = FIRST / 8;
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %1, %2 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %3 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %4 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %5 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %6 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %7 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %8 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %9 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %10 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %11 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %12 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %13 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %14 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %15 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %16 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, %1, %17 row_newbcast:15 row_mask:0xf bank_mask:0xf"
      : "+&v"(sum)
      : "v"(x), "v"(w[j][0][0]), "v"(w[j][1][0]), "v"(w[j][0][1]), "v"(w[j][1][1]),
        "v"(w[j][0][2]), "v"(w[j][1][2]), "v"(w[j][0][3]), "v"(w[j][1][3]),
        "v"(w[j + 1][0][0]), "v"(w[j + 1][1][0]), "v"(w[j + 1][0][1]), "v"(w[j + 1][1][1]),
        "v"(w[j + 1][0][2]), "v"(w[j + 1][1][2]), "v"(w[j + 1][0][3]), "v"(w[j + 1][1][3]));
  return sum;
}

__device__ __forceinline__ float relu(float v) { return v < 0.f ? 0.f : v; }

// Whether a word was written by this call.  Until then it holds the number of one of
// the 2 kNumberAll calls before, or the 0 of a new handle, whose first calls have
// other numbers.
__device__ __host__ constexpr bool carries(uint64_t word, uint32_t call) {
  return (uint32_t)(word >> 32) == call;
}

__device__ __forceinline__ void put(uint64_t* word, float value, uint32_t call) {
  __hip_atomic_store(word, (uint64_t)call << 32 | __builtin_bit_cast(uint32_t, value),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The values of ROWS words `stride` apart once all of the first n, for every lane of
// the wave, carry the number of this call (a loop for the wave: with one for each
// lane 2 to 4 rows took 1 us more).  While the first is not there only that one is
// asked for, and after kBusyLooks looks only now and then: all workgroups wait at
// a time, and where they asked for every row at full rate (twice as many, of half
// a tile, and eight rows: 33 MB a look) some waits did not end in a second, as if the
// reads had kept the write waited for from getting through (the cause was not
// found).  One row is 2 MB a look; 32 000 calls, half of them beside a kernel that
// takes all of the memory's bandwidth, then all took their usual time.  False, and
// no values, where the wait was given up after `looks`.
template <int ROWS>
__device__ __forceinline__ bool get(const uint64_t* words, int stride, int n, uint32_t call,
                                    int looks, float (&value)[ROWS]) {
  uint64_t v[ROWS] = {};
  const auto ask = [&](int r) {
    v[r] = __hip_atomic_load(words + (r < n ? r : 0) * stride, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
  };
  bool ready = false;
  for (int look = 0; !ready; ++look) {
    if (__builtin_expect(look == looks, 0)) break;
    if (look > 0) {
      if (look <= kBusyLooks) __builtin_amdgcn_s_sleep(1);
      else __builtin_amdgcn_s_sleep(127);
    }
    ask(0);
    ready = __all(carries(v[0], call));
    if (ROWS > 1 && ready) {
      bool all = true;
#pragma unroll
      for (int r = 1; r < ROWS; ++r) ask(r);
#pragma unroll
      for (int r = 1; r < ROWS; ++r) all = all && carries(v[r], call);
      ready = __all(all);
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) value[r] = __builtin_bit_cast(float, (uint32_t)v[r]);
  return ready;
}

// The packed weights of an output of a hidden layer, its k-groups 8 * 64 apart and
// the upper four k of a group 32 further.
__device__ __forceinline__ const f32x4* weights_of(const Args& a, int layer, int tile, int n) {
  return reinterpret_cast<const f32x4*>(a.w_stream) +
         ((size_t)(tile >> 3) * a.groups_total + a.first_groups + layer * (kWidth / 8)) * (8 * 64) +
         (tile & 7) * 64 + n;
}

// The rows standardised, zeros beyond them; thread = (row, feature).
template <int ROWS>
__device__ __forceinline__ void standardise(const Args& a, int tid, float (&xs)[ROWS][kMaxIn]) {
  if (tid < ROWS * kMaxIn) {
    const int r = tid / kMaxIn, k = tid % kMaxIn;
    float v = 0.f;
    if (r < a.n && k < a.in_features)
      v = (float)((a.raw[(size_t)r * a.in_features + k] - a.mu[k]) / a.sigma[k]);
    xs[r][k] = v;
  }
}

// One output of fc1: four sums, each of a quarter of the k-groups, as
// mlp_layer_kernel's waves.  wk: its weights, where in_features <= kFewIn.
template <int ROWS>
__device__ __forceinline__ void first_layer(const Args& a, int out, const float (&wk)[kFewIn],
                                            const float (&xs)[ROWS][kMaxIn], float (&v)[ROWS]) {
  float sum[ROWS];
  if (a.in_features <= kFewIn) {
    // two k-groups, each a sum of its own (the other two sums are zero)
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      float part[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < kFewIn; ++i) {
        const int k = product(i);
        part[k >> 3] = fmaf(wk[k], xs[r][k], part[k >> 3]);
      }
      sum[r] = part[0] + part[1];
    }
  } else {
    const int per_sum = (a.first_groups + 3) / 4;
    for (int s = 0; s < 4; ++s) {
      float part[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) part[r] = 0.f;
      for (int i = 8 * s * per_sum; i < 8 * (s + 1) * per_sum; ++i) {
        const int k = product(i);
        const float w1 = k < a.in_features ? a.w_first_t[(size_t)k * kWidth + out] : 0.f;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) part[r] = fmaf(w1, k < a.in_features ? xs[r][k] : 0.f, part[r]);
      }
#pragma unroll
      for (int r = 0; r < ROWS; ++r) sum[r] = s == 0 ? part[r] : sum[r] + part[r];
    }
  }
  const float b = a.bias[out];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) v[r] = relu(sum[r] + b);
}

// The input of layer `layer` into act, by this workgroup without any other: thread =
// output, its sums in the order of chain_kernel.  About 40 us a layer where all
// workgroups do it; it is there for waits that were given up and nothing else.
template <int ROWS>
__device__ __forceinline__ void alone(const Args& a, int layer, int tid, float (&xs)[ROWS][kMaxIn],
                                      float (&act)[ROWS][kWidth]) {
  float wk[kFewIn], v[ROWS];
  for (int k = 0; k < kFewIn; ++k) wk[k] = a.w_first_t[(size_t)k * kWidth + tid];
  standardise<ROWS>(a, tid, xs);
  __syncthreads();
  first_layer<ROWS>(a, tid, wk, xs, v);
#pragma unroll 1
  for (int l = 0; l < layer; ++l) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) act[r][tid] = v[r];
    __syncthreads();
    const f32x4* at = weights_of(a, l, tid >> 5, tid & 31);
    const float b = a.bias[(size_t)(l + 1) * kWidth + tid];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) v[r] = b;
#pragma unroll 1
    for (int p = 0; p < kChains; p += 4) {
      float part[ROWS];
#pragma unroll 1
      for (int c = p; c < p + 4; ++c) {
        float sum[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) sum[r] = 0.f;
#pragma unroll 1
        for (int j = 4 * c; j < 4 * c + 4; ++j) {
          const f32x4 lower = at[(size_t)j * (8 * 64)], upper = at[(size_t)j * (8 * 64) + 32];
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
              sum[r] = fmaf(lower[e], act[r][8 * j + e], sum[r]);
              sum[r] = fmaf(upper[e], act[r][8 * j + 4 + e], sum[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) part[r] = c == p ? sum[r] : part[r] + sum[r];
      }
#pragma unroll
      for (int r = 0; r < ROWS; ++r) v[r] += part[r];
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) v[r] = relu(v[r]);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) act[r][tid] = v[r];
  __syncthreads();
}

template <int ROWS>
__global__ __launch_bounds__(1024) void chain_kernel(const Args a) {
  __shared__ uint32_t taken[2];
  __shared__ uint32_t late;  // a thread's wait was given up
  __shared__ float xs[ROWS][kMaxIn];
  __shared__ __attribute__((aligned(16))) float act[ROWS][kWidth];
  __shared__ float red[ROWS][kChains][32];
  const int tid = threadIdx.x;
  const int blocks = a.hidden * kTiles + 1;
  if (tid == 0) {
    late = 0;
    const uint64_t t =
        __hip_atomic_fetch_add(a.tickets, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    taken[0] = (uint32_t)(t % (uint32_t)blocks);
    taken[1] = (uint32_t)(t / (uint32_t)blocks) + 1;
  }
  __syncthreads();
  const int block = __builtin_amdgcn_readfirstlane((int)taken[0]);
  const uint32_t call = __builtin_amdgcn_readfirstlane(taken[1]);
  const int layer = block / kTiles, tile = block % kTiles;  // layer == hidden: fc2

  // thread (n, c): output n of the tile, products 32 c .. 32 c + 31 of its sum,
  // k-groups 4 c .. 4 c + 3
  const int n = tid & 31, c = tid >> 5;
  f32x4 w[4][2];
  const auto load_weights = [&]() {
    const f32x4* at = weights_of(a, layer, tile, n) + 4 * c * (8 * 64);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) w[j][h] = at[j * (8 * 64) + 32 * h];
  };
  if (layer < a.hidden) load_weights();
  if (__builtin_expect(call % kNumberAll == 0, 0) && layer < a.hidden && c >= a.n && c < kMaxRows)
    put(a.words + ((size_t)layer * kMaxRows + c) * kWidth + tile * 32 + n, 0.f, call);

  if (layer == 0) {
    // fc1, by each of the first layer's workgroups for itself: thread = output
    float wk[kFewIn], v[ROWS];
#pragma unroll
    for (int k = 0; k < kFewIn; ++k) wk[k] = a.w_first_t[(size_t)k * kWidth + tid];
    standardise<ROWS>(a, tid, xs);
    __syncthreads();
    first_layer<ROWS>(a, tid, wk, xs, v);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) act[r][tid] = v[r];
  } else {
    float v[ROWS];
    if (!get<ROWS>(a.words + (size_t)(layer - 1) * kMaxRows * kWidth + tid, kWidth, a.n, call,
                   a.looks, v))
      late = 1;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) act[r][tid] = v[r];
  }
  __syncthreads();

  if (layer < a.hidden) {
    const auto finish_tile = [&](const uint32_t& given_up) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        if (r >= a.n) break;
        // (16 lanes share the values that they all want: read from LDS by every lane
        // they took 0.4 us a row)
        const float* x = &act[r][32 * c + product(tid & 15)];
        const float sum = add_products<0>(w, x[0], 0.f);
        red[r][c][n] = add_products<16>(w, x[16], sum);
      }
      __syncthreads();
      // a wave per row: four sums make a K-partial, the eight partials follow the
      // bias; lanes 0 to 31 add the first four, lanes 32 to 63 the others
      const int row = tid >> 6, upper = c & 1;
      if (row >= ROWS || row >= a.n) return;
      float p[kChains / 2];
#pragma unroll
      for (int i = 0; i < kChains / 2; ++i) p[i] = red[row][upper * (kChains / 2) + i][n];
      float v = a.bias[(size_t)(layer + 1) * kWidth + tile * 32 + n];
#pragma unroll
      for (int s = 0; s < kChains / 4 / 2; ++s)
        p[s] = ((p[4 * s] + p[4 * s + 1]) + p[4 * s + 2]) + p[4 * s + 3];
#pragma unroll
      for (int s = 0; s < kChains / 4 / 2; ++s) v += p[s];
      v = __shfl_up(v, 32);   // the lower half's sum, for the upper half
#pragma unroll
      for (int s = 0; s < kChains / 4 / 2; ++s) v += p[s];
      if (upper && given_up == 0)
        put(a.words + ((size_t)layer * kMaxRows + row) * kWidth + tile * 32 + n, relu(v), call);
    };
    finish_tile(late);
    if (__builtin_expect(late == 0, 1)) return;
    alone<ROWS>(a, layer, tid, xs, act);
    load_weights();
    finish_tile(0);
    return;
  }

  // fc2: a wave per row, summed as in mlp_last_kernel
  if (__builtin_expect(late != 0, 0)) alone<ROWS>(a, layer, tid, xs, act);
  const int lane = tid & 63, row = tid >> 6;
  if (row >= a.n) return;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kWidth / 256; ++i) {
    const int k = 256 * i + 4 * lane;
    const f32x4 v = *reinterpret_cast<const f32x4*>(&act[row][k]);
    const f32x4 wl = *reinterpret_cast<const f32x4*>(a.w_last + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = fmaf(v[e], wl[e], sum);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off);
  if (lane == 0) {
    a.out[row] = sum + a.b_last;
    if (a.done_flag != nullptr && row == 0) {
      __threadfence_system();
      __hip_atomic_store(a.done_flag, a.done_value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// The network for a.n rows, 1 to kMaxRows; hidden > 0.
inline hipError_t launch(const Args& a, hipStream_t stream) {
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.hidden * kTiles + 1)), dim3(1024), 0, stream, a);
  };
  if (a.n == 1) go(chain_kernel<1>);
  else if (a.n == 2) go(chain_kernel<2>);
  else go(chain_kernel<4>);
  return hipGetLastError();
}

}  // namespace chain
}  // namespace hbt
