// Hidden layers of the MLP on the fp16 matrix cores, at fp32 precision.
//
// An fp32 number of 24 bits is the sum of two fp16 numbers but for half of its last
// bit: x = x0 + x1, x0 = fp16(x), x1 = fp16(x - x0), 11 + 11 bits and the sign of x1.
// Three of the four products of two such pairs,
//     w x = w0 x0 + (w0 x1 + w1 x0) + ...,
// are the fp32 product to 2^-22, with either sign; their rms error, 1.2 x 2^-24 of a
// sum's own rms, is less than that sum's roundings cost (7 x 2^-24 on the fp32 matrix
// cores).  Products of fp16 are exact in the matrix core, sums are fp32, and gfx950's
// matrix cores run fp16 at the rate of bf16: half the products of the three bf16
// pieces of mlp_split.h, and two thirds of their bytes.
//
// What fp16 has not is fp32's range, so everything is scaled by powers of two, which
// costs no bit:
//   unit n of a layer by 2^G[n], chosen when the network is loaded (prepare_layer), so
//     that the units of a layer are of one size whatever their weights are;
//   row m of a batch by 2^e[m], chosen by the kernel that computes a layer, from the
//     largest of the row's (scaled) inputs and a bound on what the layer makes of it;
//   row n of a layer's weights by 2^-F[n], its largest weight to [2^14, 2^15).
// A scaled number below kHeldFrom is held to 2^-25: a weight to 2^-40 of its row's largest,
// an activation to 2^-40 of the bound on its row's, some 2^-32 of the row's usual ones.
// Where sums may hang on such numbers they are not made here: a network with many such
// weights in a row or column (kMostLostWeights), or with a unit that hangs on few of its
// inputs (kLeastShare), keeps the bf16 pieces; a row of a batch with many such activations,
// as where a few units are 2^10 times the others, or with hardly any above them
// (rows_lost), is marked while the layers run and goes through the
// network again on the fp32 matrix cores (mlp_fused_kernel).  An
// infinite activation is the second number of its pair, so that it meets nothing but
// the other operand's first number, whose sign is the weight's; a NaN stays one.
//
// Included by mlp.hip only.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "mlp_split.h"

namespace hbt {
namespace pairs {

using half2 = _Float16 __attribute__((ext_vector_type(2)));
using i32x4 = int32_t __attribute__((ext_vector_type(4)));
using half8 = _Float16 __attribute__((ext_vector_type(8)));
using split::f32x2;
using split::f32x4;
using split::f32x16;
using split::block_of;
using split::kRows;
using split::kSteps;
using split::kWidth;
using split::lds_void;
using split::relu_nan;
using split::wait_fetches;

// Layout as in mlp_split.h: [32-row tile][k-step][0 or 1][lane][8].
constexpr int kFragBytes = split::kFragBytes;
constexpr int kStepBytes = 2 * kFragBytes;
constexpr int kTileBytes = kSteps * kStepBytes;
constexpr int kTop = 15;  // scaled numbers are below 2^kTop
// From here on a scaled number is held to 2^-22 of itself, below to 2^-25.
constexpr float kHeldFrom = 0x1p-3f;
// Activations of a row below that.  Of 1024 that are of one size 0 to 20 are (networks of
// eight layers, any gain), and with one unit 2^4, 2^8, 2^10 and 2^12 times the others 1-21,
// 46-262, 185-527 and 472-551 (all that are not 0): errors of 5e-7, 4e-7, 6e-7 and 2e-6 where
// fp32 sums have 1e-6.
constexpr int kMostLost = 128;
// Weights of a row or column below that: of 1024 of one spread 0 to 2.
constexpr int kMostLostWeights = 16;

__device__ __forceinline__ size_t tile_offset(int tile, int step) {
  return (size_t)tile * kTileBytes + (size_t)step * kStepBytes;
}

// Weights and activations as buffers: a load takes its base from scalar registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tiles_rsrc(const char* tiles, int count) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(tiles), 0, count * kTileBytes, 0x00020000);
}

// One fragment into LDS (in a function of its own: the host's pass over a kernel does not
// know this builtin).
__device__ __forceinline__ void fetch_fragment(const char* tiles, int count, char* lds, int lane,
                                               int offset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(tiles_rsrc(tiles, count), (lds_void*)lds, 16, lane * 16,
                                           offset, 0, 0);
}

// Stores a lane's 8 scaled values of a fragment as pairs; `most` is the largest.  rest:
// what the values have beyond fp32 (nullable).
__device__ __forceinline__ void store_pairs(char* out, const float (&v)[8], const float* rest,
                                            float most) {
  using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
  u32x4 first, second;
  const auto put = [&](const float (&a)[8], const float* r) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const half2 p = __builtin_convertvector((f32x2){a[2 * j], a[2 * j + 1]}, half2);
      f32x2 q = {v[2 * j] - (float)p[0], v[2 * j + 1] - (float)p[1]};
      if (r != nullptr) q += (f32x2){r[2 * j], r[2 * j + 1]};
      first[j] = __builtin_bit_cast(uint32_t, p);
      second[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(q, half2));
    }
  };
  put(v, rest);
  if (__builtin_expect(!(most < 65504.f), 0)) {  // an infinity or a NaN
    float a[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = __builtin_isinf(v[j]) ? 0.f : v[j];
    put(a, nullptr);
  }
  *reinterpret_cast<u32x4*>(out) = first;
  *reinterpret_cast<u32x4*>(out + kFragBytes) = second;
}

// The power of two for a row of a layer's outputs, from the largest of its inputs and of
// the layer's biases (all scaled by unit), as the e of |v| < 2^e, which may be beyond
// fp32's.  With unit sizes u (put_size) a scaled output is at most
//     sum |w'| x' + b' <= 32 x 2 x largest + bias:
// u^2 is the sum of (w u)^2 over 1024 inputs, and u 2^G is in [1, 2).
constexpr int kNotFinite = 400;
constexpr int kInputsExponent = 6;       // 64 (and 8 x 2 for fc1's 64 features at most)
__device__ __forceinline__ int exponent_of(float v, int scale) {
  if (v == 0.f) return -kNotFinite;
  return v < __builtin_inff() ? __builtin_amdgcn_frexp_expf(v) - scale : kNotFinite;
}
__device__ __forceinline__ int row_exponent(int largest, int bias) {
  const int e = (largest + kInputsExponent > bias ? largest + kInputsExponent : bias) + 1;
  return kTop - (e > -kNotFinite ? e : -kNotFinite);
}

// What is known of the units of a layer.
struct Units {
  const float* bias;     // [kWidth]
  const int32_t* F;      // [kWidth] exponent of the scale of the unit's weights, and of what they make
  const int32_t* G;      // [kWidth] exponent of the scale of the unit itself
  const int32_t* bias_most;  // exponent_of the largest scaled bias
};

struct LayerArgs {
  const char* w;          // this layer's weights, [32 n-tiles] tiles
  const char* x;          // activations in, [m_tiles] tiles
  Units units;
  const int32_t* e_in;    // [m_tiles * 32] exponents of the rows' scales
  const int32_t* most_in; // [most_count][m_tiles * 32] part_of a row's inputs
  int32_t most_count;
  int32_t* redo;          // [m_tiles * 32] set where the inputs are not held
  char* y;                // not LAST: activations out, and what goes with them
  int32_t* e_out;
  int32_t* most_out;
  const float* w_last;    // LAST: fc2.weight [kWidth]
  float* part;            // LAST: [kWidth / 32][m_tiles * 32] shares of the final dot product
  int32_t m_tiles;
};

// A part of a row's outputs: exponent_of the largest, and how many are below kHeldFrom.
__device__ __forceinline__ int32_t part_of(int exponent, int lost) { return exponent * 256 + lost; }
__device__ __forceinline__ int part_exponent(int32_t part) { return part >> 8; }
__device__ __forceinline__ int part_lost(int32_t part) { return part & 255; }
__device__ __forceinline__ int32_t both_parts(int32_t a, int32_t b) {
  return (a > b ? a & -256 : b & -256) + part_lost(a) + part_lost(b);
}
// Whether a sum may hang on what a row has lost: there is much of it, or nothing is larger
// than 1 (all but some of the row's units are 0, and the bound was far from the others).
// most: part_exponent of the row, e: of its scale.
__device__ __forceinline__ bool rows_lost(int lost, int most, int e) {
  return lost > kMostLost || (lost > 0 && (most <= -kNotFinite || most + e <= 0));
}
__device__ __forceinline__ int is_lost(bool positive, float scaled) { return positive && scaled < kHeldFrom; }

// v of 4, 8 or 16 lanes together (in registers: a step through LDS is 100 cycles, and these
// come before the first MFMA).
template <int LANES, class Op>
__device__ __forceinline__ int over_lanes(int v, Op op) {
  static_assert(LANES == 4 || LANES == 8 || LANES == 16, "a row of lanes or a part of it");
  v = op(v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true));                    // 1 0 3 2
  v = op(v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true));                    // 2 3 0 1
  if (LANES > 4) v = op(v, __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true));    // half mirror
  if (LANES > 8) v = op(v, __builtin_amdgcn_mov_dpp(v, 0x140, 0xf, 0xf, true));    // mirror
  return v;
}

// The exponents of a block's rows, in and out, into LDS.  Some lanes to a row, each with its
// share of the parts, all loads at once: this comes before the first MFMA.
template <int ROWS, int THREADS, bool LAST>
__device__ __forceinline__ void row_scales(const LayerArgs& a, int m_tile0, bool store_out,
                                           int (*scales)[2]) {
  constexpr int kLanes = ROWS <= THREADS / 16 ? 16 : ROWS <= THREADS / 8 ? 8 : 4;
  constexpr int kLoads = kWidth / 32 / kLanes;
  static_assert(ROWS * kLanes <= THREADS, "one pass");
  const int rows = a.m_tiles * kRows, bias_most = *a.units.bias_most;
  const int r = threadIdx.x / kLanes, part = threadIdx.x % kLanes;
  const int row = m_tile0 * kRows + r < rows ? m_tile0 * kRows + r : rows - 1;
  const int e_in = a.e_in[row];
  int32_t v[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int p = part + j * kLanes;
    v[j] = a.most_in[(size_t)(p < a.most_count ? p : 0) * rows + row];
  }
  int most = v[0], lost = 0;
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    most = v[j] > most ? v[j] : most;
    lost += part + j * kLanes < a.most_count ? part_lost(v[j]) : 0;
  }
  most = part_exponent(over_lanes<kLanes>(most, [](int x, int y) { return x > y ? x : y; }));
  lost = over_lanes<kLanes>(lost, [](int x, int y) { return x + y; });
  if (part != 0 || r >= ROWS) return;
  const int e = row_exponent(most, bias_most);
  scales[r][0] = e_in;
  scales[r][1] = e;
  if (!store_out || m_tile0 * kRows + r >= rows) return;
  if (!LAST) a.e_out[row] = e;
  if (rows_lost(lost, most, e_in)) a.redo[row] = 1;
}

// Part `part` of a row's outputs: the largest, and how many are not held.
__device__ __forceinline__ void put_part(const LayerArgs& a, int part, int m_tile, int lane,
                                         float most, int lost, int e_out) {
  int32_t v = part_of(exponent_of(most, e_out), lost);
  v = both_parts(v, __shfl_xor(v, 32));
  if (lane < 32) a.most_out[(size_t)part * (a.m_tiles * kRows) + m_tile * kRows + lane] = v;
}

// What goes with a lane's 16 units of an n-tile, loaded once for all m-tiles: between the
// stores of one m-tile and the next the compiler would load it again and wait (1 x 3 tiles
// 0.7 us a layer, which is what counting is_lost takes).  Loaded before the k-steps it costs
// 1 x 1 tiles their second workgroup on a compute unit (1500 rows 146 -> 150 us).
template <bool LAST>
struct LaneUnits {
  f32x4 bias[4], w_last[4];
  i32x4 F[4], G[4];
  __device__ __forceinline__ LaneUnits(const LayerArgs& a, int n_tile, int lane) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = n_tile * 32 + 8 * g + 4 * (lane >> 5);
      bias[g] = *reinterpret_cast<const f32x4*>(a.units.bias + n);
      F[g] = *reinterpret_cast<const i32x4*>(a.units.F + n);
      if (LAST) w_last[g] = *reinterpret_cast<const f32x4*>(a.w_last + n);
      else G[g] = *reinterpret_cast<const i32x4*>(a.units.G + n);
    }
  }
};

// A lane's 8 outputs of a k-step of the next layer, registers 8 kk .. 8 kk + 7 of a tile,
// from their sums.  most: the largest of a row's so far; lost: those not held; share (LAST):
// of the final dot product.  Sums in double leave the pair one rounding, not an fp32 number's
// and its own.
template <bool LAST, class T>
__device__ __forceinline__ void finish_half(const LayerArgs& a, const LaneUnits<LAST>& units,
                                            const T (&sums)[8], int n_tile, int kk, int m_tile,
                                            int lane, int e_in, int e_out, float& most, int& lost,
                                            float& share) {
  float v[8], rest[8], largest = 0.f;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const f32x4 b = units.bias[2 * kk + g];
    const i32x4 F = units.F[2 * kk + g], G = units.G[2 * kk + g];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (std::is_same_v<T, double>) {
        const double y = __builtin_ldexp(sums[4 * g + e], F[e] - e_in) + (double)b[e];
        const float whole = (float)y;
        if (LAST) {
          v[4 * g + e] = relu_nan(whole);
          continue;
        }
        const double scaled = __builtin_ldexp(y, G[e] + e_out);
        const bool positive = whole > 0.f;
        // (what is infinite in fp32 is so here)
        v[4 * g + e] = relu_nan(whole < __builtin_inff() ? (float)scaled : whole);
        rest[4 * g + e] = positive ? (float)(scaled - (double)v[4 * g + e]) : 0.f;
        lost += is_lost(positive, v[4 * g + e]);
      } else {
        const float y = relu_nan(__builtin_ldexpf(sums[4 * g + e], F[e] - e_in) + b[e]);
        v[4 * g + e] = LAST ? y : __builtin_ldexpf(y, G[e] + e_out);
        if (!LAST) lost += is_lost(y > 0.f, v[4 * g + e]);
      }
    }
    if (LAST) {
#pragma unroll
      for (int e = 0; e < 4; ++e) share = fmaf(v[4 * g + e], units.w_last[2 * kk + g][e], share);
    }
  }
  if (LAST) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) largest = __builtin_elementwise_maximum(largest, v[e]);
  store_pairs(a.y + tile_offset(m_tile, 2 * n_tile + kk) + lane * 16, v,
              std::is_same_v<T, double> ? rest : nullptr, largest);
  most = __builtin_elementwise_maximum(most, largest);
}

// Outputs of one tile from its sums.
template <bool LAST, class T>
__device__ __forceinline__ void finish_tile(const LayerArgs& a, const LaneUnits<LAST>& units,
                                            const T (&sums)[16], int n_tile, int m_tile, int lane,
                                            int e_in, int e_out, float& most, int& lost) {
  float share = 0.f;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    T half[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) half[e] = sums[8 * kk + e];
    finish_half<LAST, T>(a, units, half, n_tile, kk, m_tile, lane, e_in, e_out, most, lost, share);
  }
  if (LAST) {
    share += __shfl_xor(share, 32);
    if (lane < 32) a.part[(size_t)n_tile * (a.m_tiles * kRows) + m_tile * kRows + lane] = share;
  }
}

// A hidden layer.  Bound by the matrix cores at the clock the power allows (a loop of
// nothing but these MFMAs on such data: 1.84 PFLOP/s), by what L2 delivers, and, where all
// workgroups end together, by the write of the activations (64 MB for 16 384 rows, 13 us).
//
// A workgroup is eight waves, each with TN n-tiles of its own and all of the workgroup's TM
// m-tiles.  So no two waves want the same weights: those come straight from L2 into a ring
// of RING k-steps of registers; the activations, which all want, go through LDS by direct
// loads, KS k-steps at a time (a slab, one barrier), NBUF slabs.  With weights in LDS too,
// and four or two waves reading each fragment of both, LDS was busy 1280 of a step's 1536
// cycles of MFMAs (whole forwards, 128 x 192 per workgroup: 5911 rows 300 us, 286 this way;
// 256 x 256: 12 288 rows 594 us, 2 x 4 tiles this way 567).  The direct loads are buffer loads:
// among global ones the compiler waits for all of the ring at each slab (5911 rows 303 us).
//
// Order of the sum.  The matrix core adds eight products and rounds the running sum, and a
// rounding costs half an ulp of what the sum has grown to (errors in 2^-24 of the output's
// rms, from a model of it that agrees with the matrix core in 94 of 100 sums):
//   FLUSH < 64: three sets of sums, for TN x TM <= 3.  The small products have one of their
//     own, the leading ones another that is added to the third, the total, every FLUSH
//     k-steps.  With FLUSH = 8 the error is 2.0 (three bf16 pieces with two sets 2.3, fp32
//     matrix cores 6.8).  A total in double (T) and FLUSH = 4 leave little but the pairs'
//     own error, 1.2.
//   FLUSH = 64: one set, for 2 x 4 tiles.  The last SPLIT_STEPS k-steps come for their small
//     products first, while the sum is small, and for their leading ones at the end, two to a
//     unit of the loop.  With 24 the error is 4.8 (three bf16 pieces in this order 5.2), with
//     none 6.0 and 2.5 % less time, with all 3.7.
//
//   TN x TM  rows of a round  us a layer  PFLOP/s of fp16  three bf16 pieces
//   1 x 1 double  2048           16-18        0.74           19-24
//   1 x 2         4096           24            1.1            34
//   1 x 3         6144           32            1.2            52
//   2 x 4        16384           81            1.27          143
template <int TN, int TM, int KS, int NBUF, int RING, int FLUSH, int SPLIT_STEPS>
struct Wide {
  static constexpr int WAVES = 8, BN = WAVES * TN, BM = TM;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int FRAGS = TM * KS * 2;
  static constexpr int LPW = (FRAGS + WAVES - 1) / WAVES;
  static constexpr int SLAB = FRAGS * kFragBytes;
  static constexpr int LDS = SLAB * NBUF + BM * kRows * 2 * (int)sizeof(int);
  static constexpr int NBLK = (kWidth / 32) / BN, XM = 8;
  static constexpr int PARTS = NBLK * WAVES;
  static constexpr int kFull = kSteps - SPLIT_STEPS;
  static constexpr int kUnits = kSteps + SPLIT_STEPS / 2, SLABS = kUnits / KS;
  static_assert(FLUSH % KS == 0 && kSteps % FLUSH == 0, "whole slabs to a part of the sum");
  static_assert(SPLIT_STEPS % (2 * KS) == 0, "whole slabs");
  static_assert(TN * 32 < 256, "part_of holds the count of a part's numbers");
  static_assert(KS % RING == 0 && KS % 2 == 0, "the rings turn a whole number of times in a slab");
};

template <class T, int TN, int TM, int KS, int NBUF, int RING, int FLUSH, int SPLIT_STEPS, bool LAST>
__global__ __launch_bounds__(512, 2) void wide_kernel(const LayerArgs a) {
  using S = Wide<TN, TM, KS, NBUF, RING, FLUSH, SPLIT_STEPS>;
  constexpr bool PARTED = FLUSH < kSteps;   // three sets of sums
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  int(*const scales)[2] = reinterpret_cast<int(*)[2]>(lds + S::SLAB * NBUF);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int n_blk, m_blk;
  block_of<S::NBLK, 1>((int)blockIdx.x, n_blk, m_blk);
  if (m_blk * S::BM >= a.m_tiles) return;
  const int n_tile0 = n_blk * S::BN + wave * TN, m_tile0 = m_blk * S::BM;

  // The k-steps come in units: the last SPLIT_STEPS for their small products, the others
  // whole, then the last ones' leading products, two steps to a unit.
  const auto unit_at = [](int u) {
    return (u < SPLIT_STEPS ? S::kFull + u : u < kSteps ? u - SPLIT_STEPS : S::kFull + 2 * (u - kSteps)) *
           kStepBytes;
  };
  const auto stride_of = [](int u) { return u < kSteps ? kFragBytes : kStepBytes; };

  int src[S::LPW], q[S::LPW], dst[S::LPW];
#pragma unroll
  for (int i = 0; i < S::LPW; ++i) {
    int f = wave * S::LPW + i;
    if (S::FRAGS % S::WAVES != 0) f = f < S::FRAGS ? f : S::FRAGS - 1;
    const int m_t = m_tile0 + f / (KS * 2);
    q[i] = f % (KS * 2);
    src[i] = (m_t < a.m_tiles ? m_t : a.m_tiles - 1) * kTileBytes;
    dst[i] = f * kFragBytes;
  }
  auto fetch = [&](int slab, int buf) {
    const int u = (slab < S::SLABS ? slab : S::SLABS - 1) * KS;
#pragma unroll
    for (int i = 0; i < S::LPW; ++i)
      fetch_fragment(a.x, a.m_tiles, lds + buf * S::SLAB + dst[i], lane,
                     src[i] + unit_at(u) + q[i] * stride_of(u));
  };
  const __amdgpu_buffer_rsrc_t w_rsrc = tiles_rsrc(a.w, kWidth / 32);
  half8 w[RING][2][TN];
  auto load_w = [&](int slot, int unit) {
    const int u = unit < S::kUnits ? unit : S::kUnits - 1;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int i = 0; i < TN; ++i)
        w[slot][p][i] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(
            w_rsrc, lane * 16, (n_tile0 + i) * kTileBytes + unit_at(u) + p * stride_of(u), 0));
  };
#pragma unroll
  for (int s = 0; s < NBUF; ++s) fetch(s, s);
#pragma unroll
  for (int s = 0; s < RING - 1; ++s) load_w(s, s);
  row_scales<S::BM * kRows, S::THREADS, LAST>(a, m_tile0, n_blk == 0, scales);

  f32x16 sums[PARTED ? 2 : 1][TN][TM];   // leading products', small ones'
  T total[PARTED ? TN : 1][PARTED ? TM : 1][16] = {};   // PARTED: finished parts'
  f32x16(&leading)[TN][TM] = sums[0], (&small)[TN][TM] = sums[PARTED ? 1 : 0];
#pragma unroll
  for (int t = 0; t < (PARTED ? 2 : 1); ++t)
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) sums[t][i][j][r] = 0.f;

  half8 x[2][2][TM];
  auto load_x = [&](half8(&d)[2][TM], int buf, int k) {
    const char* at = lds + buf * S::SLAB + k * kStepBytes + lane * 16;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        d[p][j] = *reinterpret_cast<const half8*>(at + j * (KS * kStepBytes) + p * kFragBytes);
  };
  auto mm = [&](f32x16(&d)[TN][TM], const half8(&p)[TN], const half8(&q)[TM]) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        d[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(p[i], q[j], d[i][j], 0, 0, 0);
  };
  wait_fetches<0>();
  __builtin_amdgcn_s_barrier();
  load_x(x[0], 0, 0);
  int buf = 0;
  // phase 0: the small products, 1: all, 2: the leading ones of two steps
  auto slab_body = [&](auto phase, int s) {
    constexpr int P = decltype(phase)::value;
    const int next = buf + 1 == NBUF ? 0 : buf + 1;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      load_w((k + RING - 1) % RING, s * KS + k + RING - 1);
      if (k == KS - 1) {
        // (what may be on its way: the weights ahead, and later slabs)
        wait_fetches<2 * TN * (RING - 1) + 2>();
        __builtin_amdgcn_s_barrier();
        fetch(s + NBUF, buf);
        HBT_FENCE;
        load_x(x[(k + 1) % 2], next, 0);
      } else {
        load_x(x[(k + 1) % 2], buf, k + 1);
      }
      // (2 x 4 tiles 0.8 % slower without it, the others 1 to 2 % slower with it)
      if (!PARTED) HBT_FENCE;
      half8(&wk)[2][TN] = w[k % RING];
      half8(&xk)[2][TM] = x[k % 2];
      if (P != 0) mm(leading, wk[0], xk[0]);
      if (P == 2) mm(leading, wk[1], xk[1]);
      if (P != 2) mm(small, wk[0], xk[1]);
      if (P != 2) mm(small, wk[1], xk[0]);
      HBT_FENCE;
    }
    buf = next;
  };
  int s = 0;
  if constexpr (PARTED) {
#pragma unroll 1
    while (s < S::SLABS) {
#pragma unroll 1
      for (int end = s + FLUSH / KS; s < end; ++s) slab_body(std::integral_constant<int, 1>(), s);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            total[i][j][r] += (T)leading[i][j][r];
            leading[i][j][r] = 0.f;
          }
    }
  } else {
#pragma unroll 1
    for (; s < SPLIT_STEPS / KS; ++s) slab_body(std::integral_constant<int, 0>(), s);
#pragma unroll 1
    for (; s < kSteps / KS; ++s) slab_body(std::integral_constant<int, 1>(), s);
#pragma unroll 1
    for (; s < S::SLABS; ++s) slab_body(std::integral_constant<int, 2>(), s);
  }
  wait_fetches<0>();

  const int m = lane & 31;
  float most[TM] = {};
  int lost[TM] = {};
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const LaneUnits<LAST> units(a, n_tile0 + i, lane);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      if (m_tile0 + j >= a.m_tiles) continue;
      const int* const e = scales[j * kRows + m];
      T sum[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sum[r] = (T)small[i][j][r];
        if constexpr (PARTED) sum[r] += total[i][j][r];
      }
      finish_tile<LAST, T>(a, units, sum, n_tile0 + i, m_tile0 + j, lane, e[0],
                           LAST ? 0 : e[1], most[j], lost[j]);
    }
  }
  if (LAST) return;
#pragma unroll
  for (int j = 0; j < TM; ++j)
    if (m_tile0 + j < a.m_tiles)
      put_part(a, n_blk * S::WAVES + wave, m_tile0 + j, lane, most[j], lost[j], scales[j * kRows + m][1]);
}

// ---------------------------------------------------------------------------
// When a network is loaded.

// Least share that a unit's inputs have together in what it is made of: (sum of its
// weights times the inputs' sizes)^2 over the sum of their squares, 768 for 1024
// weights of one spread.  A pair's error does not average out over a sum of few
// products; and of 256 inputs at least half are held in any row that is not marked.
constexpr double kLeastShare = 256.;

// Units whose size is beyond 2^+-kUnitRange are not for pairs: their activations would leave
// fp32, where layers that make nearly nothing of their inputs follow each other, while
// their scaled ones do not.
constexpr int kUnitRange = 100;

struct PrepareArgs {
  const float* w_stream;   // packed fp32 weights (mlp.hip)
  int32_t groups_total;    // k-groups per wave stream
  int32_t g0;              // first k-group of the layer
  const float* w_first_t;  // fc1.weight transposed, [in_features][kWidth]
  int32_t in_features;
  const float* bias;       // [kWidth] of the layer
  const int32_t* G_in;     // [kWidth] of the units of the layer before, and their sizes
  const float* size_in;    //   times 2^G, in [1, 2) or 0
  int32_t* F;              // [kWidth]
  int32_t* G;
  float* size;
  int32_t* bias_most;      // of the layer; at the least there is before
  int32_t* column_lost;    // [kWidth] weights below kHeldFrom of an input; zeroes before
  uint32_t* outside;       // set where the layer is not for pairs
};

// Size of a unit: what it is for inputs of their sizes and either sign, and its bias.
__device__ __forceinline__ void put_size(const PrepareArgs& a, int n, double squares) {
  const double u = sqrt(squares) + fabs((double)a.bias[n]);
  if (u != 0. && !(u >= ldexp(1., -kUnitRange) && u < ldexp(1., kUnitRange))) *a.outside = 1;
  const int e = u > 0. ? __builtin_amdgcn_frexp_exp(u) - 1 : 0;
  a.G[n] = -e;
  a.size[n] = (float)ldexp(u, -e);
  const float b = a.bias[n];
  if (b > 0.f) atomicMax(a.bias_most, __builtin_amdgcn_frexp_expf(b) - e);
}

__global__ __launch_bounds__(256) void prepare_first(const PrepareArgs a) {
  const int n = (int)blockIdx.x * 256 + threadIdx.x;
  double squares = 0.;
  for (int k = 0; k < a.in_features; ++k) {
    const double w = a.w_first_t[(size_t)k * kWidth + n];
    squares += w * w;
  }
  put_size(a, n, squares);
}

// One workgroup per n-tile, K over its 16 waves.
__global__ __launch_bounds__(1024) void prepare_layer(const PrepareArgs a) {
  __shared__ double sums[2][16][32];
  __shared__ double largest[16][32];
  __shared__ int lost_of[16][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tile = blockIdx.x;
  const int m = lane & 31, h = lane >> 5;
  const f32x4* in = reinterpret_cast<const f32x4*>(a.w_stream) +
                    ((size_t)(tile >> 3) * a.groups_total + a.g0) * (8 * 64) + (tile & 7) * 64 + lane;
  double s[2] = {0., 0.};
  double most = 0.;   // (2^-149 of a weight times a unit's 2^-100 is no fp32 number)
#pragma unroll
  for (int i = 0; i < kWidth / 8 / 16; ++i) {
    const int g = wave * (kWidth / 8 / 16) + i, k = 8 * g + 4 * h;
    const f32x4 v = in[(size_t)g * (8 * 64)];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double w = ldexp((double)v[e], -a.G_in[k + e]);
      const double x = w * a.size_in[k + e];
      s[0] += fabs(x);
      s[1] += x * x;
      // (a unit of size 0 is always 0 or NaN: its weights take no part, and are packed as 0)
      if (a.size_in[k + e] > 0.f) most = fmax(most, fabs(w));
    }
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    s[t] += __shfl_xor(s[t], 32);
    sums[t][wave][m] = s[t];
  }
  largest[wave][m] = fmax(most, __shfl_xor(most, 32));
  __syncthreads();
  double total = 0., squares = 0.;
  for (int w = 0; w < 16; ++w) {
    total += sums[0][w][m];
    squares += sums[1][w][m];
    most = fmax(most, largest[w][m]);
  }
  const int F = most > 0. ? __builtin_amdgcn_frexp_exp(most) - kTop : 0;
  int lost = 0;
  for (int i = 0; i < kWidth / 8 / 16; ++i) {
    const int g = wave * (kWidth / 8 / 16) + i, k = 8 * g + 4 * h;
    const f32x4 v = in[(size_t)g * (8 * 64)];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (a.size_in[k + e] > 0.f && v[e] != 0.f &&
          ldexp(fabs((double)v[e]), -a.G_in[k + e] - F) < kHeldFrom) {
        ++lost;
        if (atomicAdd(a.column_lost + k + e, 1) >= kMostLostWeights) *a.outside = 1;
      }
  }
  lost += __shfl_xor(lost, 32);
  lost_of[wave][m] = lost;
  __syncthreads();
  if (threadIdx.x >= 32) return;
  lost = 0;
  for (int w = 0; w < 16; ++w) lost += lost_of[w][m];
  // (a weight that is not finite has been found by check_kernel)
  if (!(total * total >= kLeastShare * squares) || lost > kMostLostWeights) *a.outside = 1;
  const int n = tile * 32 + m;
  a.F[n] = F;
  put_size(a, n, squares);
}

// The packed fp32 weights of one layer as pairs.  One wavefront per (n-tile, k-step).
struct PackArgs {
  const float* w_stream;
  int32_t groups_total;
  int32_t g0;
  const int32_t* G_in;
  const float* size_in;
  const int32_t* F;
  char* w;
};
__global__ __launch_bounds__(256) void pack_kernel(const PackArgs a) {
  const int lane = threadIdx.x & 63;
  const int item = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int tile = item / kSteps, step = item % kSteps;
  const f32x4* in = reinterpret_cast<const f32x4*>(a.w_stream) +
                    ((size_t)(tile >> 3) * a.groups_total + a.g0 + 2 * step) * (8 * 64) +
                    (tile & 7) * 64 + lane;
  const int F = a.F[tile * 32 + (lane & 31)];
  half8 first, second;
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = 16 * step + 8 * g + 4 * (lane >> 5) + e;
      const float w = a.size_in[k] > 0.f ? in[g * (8 * 64)][e] : 0.f;
      const float v = ldexpf(w, -a.G_in[k] - F);
      _Float16 p = (_Float16)v, q = (_Float16)(v - (float)p);
      if (p == (_Float16)0.f && w != 0.f) {  // keeps its sign for an infinite activation
        p = (_Float16)(w > 0.f ? 0x1p-24f : -0x1p-24f);
        q = -p;
      }
      first[4 * g + e] = p;
      second[4 * g + e] = q;
    }
  char* out = a.w + tile_offset(tile, step) + lane * 16;
  *reinterpret_cast<half8*>(out) = first;
  *reinterpret_cast<half8*>(out + kFragBytes) = second;
}

struct FirstArgs {
  const double* raw;     // [n][in_features]
  const double* mu;
  const double* sigma;
  const float* w_t;      // fc1.weight transposed, [MAX_IN][kWidth]
  Units units;           // (F is not used)
  int32_t in_features;
  int64_t n;
  char* y;               // activations out, [m_tiles] tiles, and what goes with them
  int32_t* e_out;
  int32_t* most_out;     // [kFirstParts][m_tiles * 32]
  int32_t* redo;         // [m_tiles * 32] cleared
};
constexpr int kFirstParts = 4 * split::kFirstSlices;

// fc1, as split::first_kernel.
template <int MAX_IN>
__global__ __launch_bounds__(256) void first_kernel(const FirstArgs a) {
  constexpr int kSlice = kWidth / split::kFirstSlices;
  __shared__ float xs[kRows][MAX_IN + 1];
  __shared__ __attribute__((aligned(16))) float wl[MAX_IN * kSlice];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 31, h = lane >> 5;
  const int m_tile = blockIdx.x, n_base = (int)blockIdx.y * kSlice;
  for (int idx = tid; idx < kRows * MAX_IN; idx += 256) {
    const int r = idx / MAX_IN, k = idx - r * MAX_IN;
    const int64_t row = (int64_t)m_tile * kRows + r;
    float v = 0.f;
    if (k < a.in_features && row < a.n)
      v = (float)((a.raw[row * a.in_features + k] - a.mu[k]) / a.sigma[k]);
    xs[r][k] = v;
  }
  for (int idx = tid; idx < a.in_features * (kSlice / 4); idx += 256) {
    const int k = idx / (kSlice / 4), c = idx - k * (kSlice / 4);
    *reinterpret_cast<f32x4*>(wl + k * kSlice + 4 * c) =
        *reinterpret_cast<const f32x4*>(a.w_t + (size_t)k * kWidth + n_base + 4 * c);
  }
  __syncthreads();
  float most_in = 0.f;
  for (int k = 0; k < a.in_features; ++k)
    most_in = __builtin_elementwise_maximum(most_in, fabsf(xs[m][k]));
  const int e_out = row_exponent(exponent_of(most_in, 0), *a.units.bias_most);
  if (blockIdx.y == 0 && wave == 0 && h == 0) {
    a.e_out[m_tile * kRows + m] = e_out;
    a.redo[m_tile * kRows + m] = 0;
  }
  float most = 0.f;
  int lost = 0;
  for (int s = wave; s < kSlice / 16; s += 4) {
    float v[8];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(a.units.bias + n_base + 16 * s + 8 * g + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * g + e] = b[e];
    }
    for (int k = 0; k < a.in_features; ++k) {
      const float x = xs[m][k];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(wl + k * kSlice + 16 * s + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * g + e] = fmaf(x, w[e], v[4 * g + e]);
      }
    }
    float largest = 0.f;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const i32x4 G = *reinterpret_cast<const i32x4*>(a.units.G + n_base + 16 * s + 8 * g + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float y = relu_nan(v[4 * g + e]);
        v[4 * g + e] = __builtin_ldexpf(y, G[e] + e_out);
        lost += is_lost(y > 0.f, v[4 * g + e]);
        largest = __builtin_elementwise_maximum(largest, v[4 * g + e]);
      }
    }
    store_pairs(a.y + tile_offset(m_tile, n_base / 16 + s) + lane * 16, v, nullptr, largest);
    most = __builtin_elementwise_maximum(most, largest);
  }
  int32_t part = part_of(exponent_of(most, e_out), lost);
  part = both_parts(part, __shfl_xor(part, 32));
  if (h == 0)
    a.most_out[(size_t)((int)blockIdx.y * 4 + wave) * ((size_t)gridDim.x * kRows) + m_tile * kRows + m] =
        part;
}

}  // namespace pairs
}  // namespace hbt
