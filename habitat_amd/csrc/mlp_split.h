// Hidden layers of the MLP on the bf16 matrix cores, at fp32 precision.
//
// What bounds a batch of rows is the matrix cores, and gfx950's do 16 times as
// many multiply-adds per cycle on bf16 as on fp32.  An fp32 number is the exact
// sum of three bf16 numbers (8 + 8 + 8 bits of mantissa):
//     x = x0 + x1 + x2,  x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1
// so weights and activations are kept as three such pieces, and of the nine
// products of pieces the six that matter are multiplied:
//     w x = w0 x0 + (w0 x1 + w1 x0) + (w1 x1 + w0 x2 + w2 x0) + ...
// What is left out, w1 x2 + w2 x1 + w2 x2, is below 2^-23 of the product, with
// either sign: beside the roundings of a sum of 1024 products it does not show.
// Products of bf16 are exact in the matrix core and sums are fp32, so the layer
// is an fp32 layer at 16 / 6 of the fp32 rate.
//
// Where it is not: below 2^-110 the third piece falls under bf16's smallest number,
// 2^-133, and a weight or activation is held to 2^-134 and no longer to 24 bits (a
// single product with an activation of 2^-114: off by 1e-6, of 2^-122 by 2.4e-4;
// products and sums that small are kept otherwise, the matrix core does not flush
// them).  Beside a bias or another product of ordinary size that does not show: what
// is lost is 2^-134 of the other operand.  Weights whose products could overflow do
// not come here (fits_pieces).  And a product takes more
// roundings than on the fp32 matrix cores, so that with a few nonzero products to a
// sum the error is larger: for a single one up to 1.7 x 2^-24 with two sets of sums (small_kernel
// to 2 x 4 tiles, mid_kernel), 3.7 with one (the larger tiles, large_kernel), 1.0 in
// fp32.  Sparse weights therefore do not come here either (kLeastNonzero); a layer
// whose input has fewer than some 100 active units of 1024 can see it.
//
// The order of the sum decides its error: the matrix core adds eight products
// and rounds the running sum, and a rounding costs half an ulp of what the sum
// has grown to.  Over one layer of 1024 (errors in 2^-24 of the output's rms):
// fp32 matrix cores 6.7, the six products of each step in turn 7.9, the five
// small products of all steps before the leading ones 2.4.
//
// Batches of 1025 rows and more come here only where the network is not for fp16 pairs
// (mlp_pairs.h), which take half the products; the ranges named below are such networks'.
//
// Included by mlp.hip only.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace hbt {
namespace split {

using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));
using f32x4 = float __attribute__((ext_vector_type(4)));
using f32x16 = float __attribute__((ext_vector_type(16)));

using bf16x2 = __bf16 __attribute__((ext_vector_type(2)));
using f32x2 = float __attribute__((ext_vector_type(2)));

// Layout.  A layer is computed transposed, Out^T[n][m] = sum_k W[n][k] Act[m][k],
// with v_mfma_f32_32x32x16_bf16: 32 outputs x 32 rows x 16 k (a k-step).  Weights
// and activations are both stored as the register image of its operands:
//     [32-row tile][k-step][piece][lane][8],
// lane (r, h) = (lane % 32, lane / 32) holding row r of the tile and
//     k = 16 step + 8 (j / 4) + 4 h + j % 4,  j = 0..7.
// That order of k within a step is the accumulator's own: register 4 g + e of
// lane (m, h) is output n = 8 g + 4 h + e of row m, so a lane's registers 8 kk ..
// 8 kk + 7 are its part of the next layer's k-step 2 tile + kk as they are, and
// every load and store of a wave is 1 KiB of contiguous memory.
constexpr int kWidth = 1024;
constexpr int kRows = 32;                        // rows of a tile
constexpr int kSteps = kWidth / 16;
constexpr int kPieces = 3;
constexpr int kFragBytes = 64 * 16;              // one operand of one MFMA
constexpr int kStepBytes = kPieces * kFragBytes;
constexpr int kTileBytes = kSteps * kStepBytes;

// Two floats rounded to bf16 in one register (low half first), and back.
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}
__device__ __forceinline__ float low2(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float high2(uint32_t v) {
  return __builtin_bit_cast(float, v & 0xffff0000u);
}

// The pieces of N values, two to a register.
template <int N>
struct Split {
  uint32_t p[kPieces][N / 2];
};

// HUGE_VALUES: some of the values are kHuge or more in magnitude, where rounding
// to bf16 overflows.  A finite one then gets the largest bf16 as its first
// piece; an infinity becomes its LAST piece alone, which meets nothing but the
// other operand's first piece, so that inf * w is what it is in fp32 and no
// inf - inf or inf * 0 comes up that fp32 would not have.
constexpr float kHuge = 0x1.FFp+127f;
constexpr float kMaxBf16 = 0x1.FEp+127f;

template <bool HUGE_VALUES, int N>
__device__ __forceinline__ Split<N> split_values(const float (&values)[N]) {
  Split<N> s;
#pragma unroll
  for (int j = 0; j < N / 2; ++j) {
    float a = values[2 * j], b = values[2 * j + 1];
    const bool inf_a = HUGE_VALUES && __builtin_isinf(a), inf_b = HUGE_VALUES && __builtin_isinf(b);
    if (inf_a) a = 0.f;
    if (inf_b) b = 0.f;
    uint32_t hi;
    if (HUGE_VALUES) {  // (a NaN stays one: it is not beyond either bound)
      const float ca = a > kMaxBf16 ? kMaxBf16 : a < -kMaxBf16 ? -kMaxBf16 : a;
      const float cb = b > kMaxBf16 ? kMaxBf16 : b < -kMaxBf16 ? -kMaxBf16 : b;
      hi = pack2(ca, cb);
    } else {
      hi = pack2(a, b);
    }
    a -= low2(hi);
    b -= high2(hi);
    const uint32_t mid = pack2(a, b);
    a = inf_a ? values[2 * j] : a - low2(mid);
    b = inf_b ? values[2 * j + 1] : b - high2(mid);
    s.p[0][j] = hi;
    s.p[1][j] = mid;
    s.p[2][j] = pack2(a, b);
  }
  return s;
}

// Stores a lane's 8 (or first or last 4) values of a fragment in pieces; `out`
// is their place in the first one.
template <int N>
__device__ __forceinline__ void store_split(char* out, const float (&v)[N]) {
  using V = uint32_t __attribute__((ext_vector_type(N / 2)));
  float most = 0.f;
#pragma unroll
  for (int j = 0; j < N; ++j) most = fmaxf(most, fabsf(v[j]));
  Split<N> s = split_values<false, N>(v);
  if (__builtin_expect(most >= kHuge, 0)) s = split_values<true, N>(v);
#pragma unroll
  for (int p = 0; p < kPieces; ++p) {
    V packed;
#pragma unroll
    for (int j = 0; j < N / 2; ++j) packed[j] = s.p[p][j];
    *reinterpret_cast<V*>(out + p * kFragBytes) = packed;
  }
}

// Byte offset of k-step `step` of a tile (weights or activations).
__device__ __forceinline__ size_t tile_offset(int tile, int step) {
  return (size_t)tile * kTileBytes + (size_t)step * kStepBytes;
}

struct LayerArgs {
  const char* w;        // this layer's weights, [32 n-tiles] tiles
  const char* x;        // activations in, [m_tiles] tiles
  const float* bias;    // [kWidth]
  char* y;              // activations out (not LAST)
  const float* w_last;  // LAST: fc2.weight [kWidth]
  float* part;          // LAST: [kWidth / 32][m_tiles * 32] shares of the final dot product
  int32_t m_tiles;
};

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

// Keeps the compiler from moving a load below the MFMAs it is meant to overlap.
#define HBT_FENCE __builtin_amdgcn_sched_barrier(0)

// ReLU that hands a NaN on, as torch's does, in one instruction.
__device__ __forceinline__ float relu_nan(float v) { return __builtin_elementwise_maximum(v, 0.f); }

// Waits until at most N of this wave's fetches are still on their way, and for
// all of its reads from LDS.
template <int N>
__device__ __forceinline__ void wait_fetches() {
  static_assert(N >= 0 && N < 64, "the counter holds 63");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// Which n-block and m-block a workgroup takes.  Consecutive workgroups go
// round-robin over the 8 XCDs: XCD x of XN x XM takes every XM-th m-block and
// an XN-th of the n-blocks.
template <int NBLK, int XN>
__device__ __forceinline__ void block_of(int id, int& n_blk, int& m_blk) {
  constexpr int XM = 8 / XN, PER = NBLK / XN;
  static_assert(NBLK % XN == 0, "the XCDs share the n-blocks evenly");
  const int xcd = id & 7, i = id >> 3;
  n_blk = (xcd % XN) * PER + i % PER;
  m_blk = (i / PER) * XM + xcd / XN;
}

// Outputs of one tile: bias is in; ReLU, then stored in pieces, or (LAST) the
// tile's share of the final dot product.
template <bool LAST>
__device__ __forceinline__ void finish_tile(const LayerArgs& a, const f32x16& acc, int n_tile,
                                            int m_tile, int lane) {
  const int m = lane & 31, h = lane >> 5;
  if (LAST) {
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 wl = *reinterpret_cast<const f32x4*>(a.w_last + n_tile * 32 + 8 * g + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = fmaf(relu_nan(acc[4 * g + e]), wl[e], sum);
    }
    sum += __shfl_xor(sum, 32);
    if (h == 0) a.part[(size_t)n_tile * (a.m_tiles * kRows) + m_tile * kRows + m] = sum;
  } else {
    char* out = a.y + tile_offset(m_tile, 2 * n_tile) + lane * 16;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = relu_nan(acc[8 * kk + e]);
      store_split(out + kk * kStepBytes, v);
    }
  }
}

// A hidden layer for thousands of rows.  Bound by the matrix cores, at the clock
// that the card's power allows them (a loop of nothing but these MFMAs on such
// data: 1.7 to 1.9 PFLOP/s of the nominal 2.5), and beside them by LDS.
//
// A workgroup of WN x WM waves takes BN x BM tiles; the waves' fragments of a
// k-step (a slab: three fragments per tile) go through LDS, where they are
// shared, by direct loads (no registers, no instructions but the load's own).
// 4 x 2 tiles per wave and 2 x 4 waves, 256 outputs x 256 rows: per slab and
// compute unit 3072 cycles of MFMAs, 1152 of LDS reads and 768 of LDS fills.
// Two waves per SIMD, so that one's reads and barriers lie beside the other's
// MFMAs.  Three slabs of LDS: slab s + 3 is fetched when slab s has been read,
// two thirds of the way through its MFMAs.
//
// Order of the sum: for the last SPLIT_STEPS k-steps only the five small
// products at first, while the sum is still small; then the other steps whole;
// then the leading products of the last ones, three steps to a slab.  24 of 64
// steps give an error of 5.5 (see above) for 2.5 % more time than none; all of
// them 2.4 for 8 % more.
//
// 16 384 rows, one layer: 0.143-0.15 ms, 235 TFLOP/s of fp32 work = 1.41 PFLOP/s
// of bf16 (the fp32 matrix cores: 0.235 ms, 147 TFLOP/s).  From 12 289 rows on.  Tried and not faster:
// 128 x 256 and 128 x 128 per workgroup, two workgroups to a compute unit (1.39,
// 1.45 against 1.55 PFLOP/s without the write-back), four waves of 4 x 4 tiles
// (1.19), fragments stored by k-step first, fetching a slab earlier.
template <int TN, int TM, int WN, int WM, int SPLIT_STEPS>
struct Large {
  static constexpr int BN = TN * WN, BM = TM * WM, TILES = BN + BM, WAVES = WN * WM;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int FRAGS = TILES * kPieces;
  static constexpr int LPW = FRAGS / WAVES;  // fragments a wave fetches per slab
  static constexpr int SLAB = FRAGS * kFragBytes;
  static constexpr int NBUF = 3;
  static constexpr int LDS = SLAB * NBUF;
  static constexpr int NBLK = (kWidth / 32) / BN, XM = 8;
  static_assert(FRAGS % WAVES == 0, "every wave fetches as many fragments");
  static_assert(SPLIT_STEPS % 3 == 0, "three leading products to a slab");
};

template <int TN, int TM, int WN, int WM, int SPLIT_STEPS, bool LAST>
__global__ __launch_bounds__(WN * WM * 64, 2) void large_kernel(const LayerArgs a) {
  using S = Large<TN, TM, WN, WM, SPLIT_STEPS>;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5;
  const int wn = wave % WN, wm = wave / WN;
  int n_blk, m_blk;
  block_of<S::NBLK, 1>((int)blockIdx.x, n_blk, m_blk);
  if (m_blk * S::BM >= a.m_tiles) return;
  const int n_tile0 = n_blk * S::BN, m_tile0 = m_blk * S::BM;

  // this wave's fragments of a slab (an m-block past the end of the batch reads
  // its last tile again and stores nothing)
  const char* src[S::LPW];
  int q[S::LPW];
#pragma unroll
  for (int i = 0; i < S::LPW; ++i) {
    const int f = wave * S::LPW + i, tile = f / kPieces;
    q[i] = f % kPieces;
    const int m_t = m_tile0 + tile - S::BN;
    src[i] = tile < S::BN ? a.w + tile_offset(n_tile0 + tile, 0)
                          : a.x + tile_offset(m_t < a.m_tiles ? m_t : a.m_tiles - 1, 0);
  }
  constexpr int kFull = kSteps - SPLIT_STEPS, kSlabs = kSteps + SPLIT_STEPS / 3;
  const uint32_t lane16 = (uint32_t)lane * 16;
  auto fetch = [&](int slab, int buf) {
    int step, q_stride = kFragBytes;
    if (slab < SPLIT_STEPS) step = kFull + slab;
    else if (slab < kSteps) step = slab - SPLIT_STEPS;
    else { step = kFull + 3 * (slab - kSteps); q_stride = kStepBytes; }
    if (slab >= kSlabs) step = 0;  // (not used)
#pragma unroll
    for (int i = 0; i < S::LPW; ++i)
      __builtin_amdgcn_global_load_lds(
          (global_void*)(src[i] + (uint32_t)(step * kStepBytes + q[i] * q_stride) + lane16),
          (lds_void*)(lds + buf * S::SLAB + (wave * S::LPW + i) * kFragBytes), 16, 0, 0);
  };

  f32x16 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int w_off = wn * TN * kStepBytes + lane * 16;
  const int x_off = (S::BN + wm * TM) * kStepBytes + lane * 16;
  bf16x8 w[kPieces][TN], x[kPieces][TM], w_next[TN], x_next[TM];
  auto load_w = [&](bf16x8(&d)[TN], int buf, int p) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
      d[i] = *reinterpret_cast<const bf16x8*>(lds + buf * S::SLAB + w_off + i * kStepBytes +
                                              p * kFragBytes);
  };
  auto load_x = [&](bf16x8(&d)[TM], int buf, int p) {
#pragma unroll
    for (int j = 0; j < TM; ++j)
      d[j] = *reinterpret_cast<const bf16x8*>(lds + buf * S::SLAB + x_off + j * kStepBytes +
                                              p * kFragBytes);
  };
  auto mm = [&](const bf16x8(&p)[TN], const bf16x8(&q)[TM]) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p[i], q[j], acc[i][j], 0, 0, 0);
  };
  fetch(0, 0);
  fetch(1, 1);
  fetch(2, 2);
  wait_fetches<2 * S::LPW>();
  __builtin_amdgcn_s_barrier();
  load_w(w[0], 0, 0);
  load_x(x[0], 0, 0);
  int buf = 0, s = 0;
  // Everybody has read slab s, slab s + 1 is there for everybody, slab s + 2 on
  // its way: slab s + 3 may take the place of slab s.
  auto turn = [&]() {
    wait_fetches<S::LPW>();
    __builtin_amdgcn_s_barrier();
    fetch(s + 3, buf);
  };
  auto body = [&](auto leading) {
    const int next = buf == 2 ? 0 : buf + 1;
    load_x(x[1], buf, 1);
    load_w(w[1], buf, 1);
    HBT_FENCE;
    if (leading) mm(w[0], x[0]);
    HBT_FENCE;
    load_x(x[2], buf, 2);
    load_w(w[2], buf, 2);
    HBT_FENCE;
    mm(w[0], x[1]);
    mm(w[1], x[0]);
    HBT_FENCE;
    turn();
    HBT_FENCE;
    mm(w[1], x[1]);
    HBT_FENCE;
    load_w(w_next, next, 0);
    load_x(x_next, next, 0);
    HBT_FENCE;
    mm(w[0], x[2]);
    mm(w[2], x[0]);
    HBT_FENCE;
#pragma unroll
    for (int i = 0; i < TN; ++i) w[0][i] = w_next[i];
#pragma unroll
    for (int j = 0; j < TM; ++j) x[0][j] = x_next[j];
    buf = next;
  };
#pragma unroll 1
  for (; s < SPLIT_STEPS; ++s) body(std::false_type());
#pragma unroll 1
  for (; s < kSteps; ++s) body(std::true_type());
#pragma unroll 1
  for (; s < kSlabs; ++s) {
    const int next = buf == 2 ? 0 : buf + 1;
    load_x(x[1], buf, 1);
    load_w(w[1], buf, 1);
    HBT_FENCE;
    mm(w[0], x[0]);
    HBT_FENCE;
    load_x(x[2], buf, 2);
    load_w(w[2], buf, 2);
    turn();
    HBT_FENCE;
    mm(w[1], x[1]);
    HBT_FENCE;
    load_w(w_next, next, 0);
    load_x(x_next, next, 0);
    HBT_FENCE;
    mm(w[2], x[2]);
    HBT_FENCE;
#pragma unroll
    for (int i = 0; i < TN; ++i) w[0][i] = w_next[i];
#pragma unroll
    for (int j = 0; j < TM; ++j) x[0][j] = x_next[j];
    buf = next;
  }
  wait_fetches<0>();

#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int n_tile = n_tile0 + wn * TN + i;
    f32x4 b[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
      b[g] = *reinterpret_cast<const f32x4*>(a.bias + n_tile * 32 + 8 * g + 4 * h);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] += b[r >> 2][r & 3];
      const int m_tile = m_tile0 + wm * TM + j;
      if (m_tile < a.m_tiles) finish_tile<LAST>(a, acc[i][j], n_tile, m_tile, lane);
    }
  }
}

// A hidden layer for 4609 to 6144 and 10 241 to 12 288 rows, in rounds of one workgroup
// per compute unit: smaller blocks than large_kernel's, so that a batch fills the
// card, and for the same reason bound by LDS as much as by the matrix cores.
// 1 x 3 tiles per wave, 4 x 2 waves, 128 outputs x 192 rows: 6144 rows in 50-57
// us, 228-250 TFLOP/s of fp32 (the fp32 matrix cores: 90 us; small_kernel in two
// rounds: 54; whole forwards of 4700 to 6144 rows are within 4 % of those with its 4 x 3
// tiles, which have one set of sums).  Slabs of KS = 2 k-steps (one barrier for both: 37 us a layer at
// 4096 rows against 47 with one step), two slabs of LDS.  A wave holds all
// fragments of a step in registers and reads the next step's during its MFMAs, so
// a slab's place is free for the next but one at the barrier.  Registers allow
// two sets of sums, the leading products' and the small ones': the error is 2.4
// (see above).
template <int TN, int TM, int WN, int WM, int KS, int NBUF>
struct Mid {
  static constexpr int BN = TN * WN, BM = TM * WM, TILES = BN + BM, WAVES = WN * WM;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int FRAGS = TILES * KS * kPieces;
  static constexpr int LPW = (FRAGS + WAVES - 1) / WAVES;
  static constexpr int SLAB = FRAGS * kFragBytes;
  static constexpr int LDS = SLAB * NBUF;
  static constexpr int NBLK = (kWidth / 32) / BN, XM = 8;
  static constexpr int SLABS = kSteps / KS;
};

template <int TN, int TM, int WN, int WM, int KS, int NBUF, bool LAST>
__global__ __launch_bounds__(WN * WM * 64, 2) void mid_kernel(const LayerArgs a) {
  using S = Mid<TN, TM, WN, WM, KS, NBUF>;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5;
  const int wn = wave % WN, wm = wave / WN;
  int n_blk, m_blk;
  block_of<S::NBLK, 1>((int)blockIdx.x, n_blk, m_blk);
  if (m_blk * S::BM >= a.m_tiles) return;
  const int n_tile0 = n_blk * S::BN, m_tile0 = m_blk * S::BM;

  const char* src[S::LPW];
  int dst[S::LPW];
#pragma unroll
  for (int i = 0; i < S::LPW; ++i) {
    int f = wave * S::LPW + i;
    if (S::FRAGS % S::WAVES != 0) f = f < S::FRAGS ? f : S::FRAGS - 1;
    const int tile = f / (KS * kPieces), q = f % (KS * kPieces);
    const int m_t = m_tile0 + tile - S::BN;
    src[i] = (tile < S::BN ? a.w + tile_offset(n_tile0 + tile, 0)
                           : a.x + tile_offset(m_t < a.m_tiles ? m_t : a.m_tiles - 1, 0)) +
             q * kFragBytes;
    dst[i] = f * kFragBytes;
  }
  const uint32_t lane16 = (uint32_t)lane * 16;
  auto fetch = [&](int slab, int buf) {
#pragma unroll
    for (int i = 0; i < S::LPW; ++i)
      __builtin_amdgcn_global_load_lds(
          (global_void*)(src[i] + (uint32_t)slab * (uint32_t)(KS * kStepBytes) + lane16),
          (lds_void*)(lds + buf * S::SLAB + dst[i]), 16, 0, 0);
  };

  f32x16 leading[TN][TM], small[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) leading[i][j][r] = small[i][j][r] = 0.f;

  const int w_off = wn * TN * (KS * kStepBytes) + lane * 16;
  const int x_off = (S::BN + wm * TM) * (KS * kStepBytes) + lane * 16;
  bf16x8 w[kPieces][TN], x[kPieces][TM];
  auto load = [&](bf16x8(&wd)[kPieces][TN], bf16x8(&xd)[kPieces][TM], int buf, int k) {
    const char* at = lds + buf * S::SLAB + k * kStepBytes;
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
        wd[p][i] = *reinterpret_cast<const bf16x8*>(at + w_off + i * (KS * kStepBytes) + p * kFragBytes);
#pragma unroll
      for (int j = 0; j < TM; ++j)
        xd[p][j] = *reinterpret_cast<const bf16x8*>(at + x_off + j * (KS * kStepBytes) + p * kFragBytes);
    }
  };
  auto mm = [&](f32x16(&d)[TN][TM], const bf16x8(&p)[TN], const bf16x8(&q)[TM]) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        d[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p[i], q[j], d[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < NBUF; ++s) fetch(s, s);
  wait_fetches<(NBUF - 1) * S::LPW>();
  __builtin_amdgcn_s_barrier();
  load(w, x, 0, 0);
  int buf = 0;
#pragma unroll 1
  for (int s = 0; s < S::SLABS; ++s) {
    const int next = buf + 1 == NBUF ? 0 : buf + 1;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      bf16x8 wf[kPieces][TN], xf[kPieces][TM];
      if (k == KS - 1) {
        wait_fetches<(NBUF - 2) * S::LPW>();
        __builtin_amdgcn_s_barrier();
        const int ahead = s + NBUF;
        fetch(ahead < S::SLABS ? ahead : S::SLABS - 1, buf);
        HBT_FENCE;
        load(wf, xf, next, 0);
      } else {
        load(wf, xf, buf, k + 1);
      }
      HBT_FENCE;
      mm(leading, w[0], x[0]);
      mm(small, w[0], x[1]);
      mm(small, w[1], x[0]);
      mm(small, w[1], x[1]);
      mm(small, w[0], x[2]);
      mm(small, w[2], x[0]);
      HBT_FENCE;
#pragma unroll
      for (int p = 0; p < kPieces; ++p) {
#pragma unroll
        for (int i = 0; i < TN; ++i) w[p][i] = wf[p][i];
#pragma unroll
        for (int j = 0; j < TM; ++j) x[p][j] = xf[p][j];
      }
    }
    buf = next;
  }
  wait_fetches<0>();

#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int n_tile = n_tile0 + wn * TN + i;
    f32x4 b[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
      b[g] = *reinterpret_cast<const f32x4*>(a.bias + n_tile * 32 + 8 * g + 4 * h);
#pragma unroll
    for (int j = 0; j < TM; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) leading[i][j][r] = (leading[i][j][r] + small[i][j][r]) + b[r >> 2][r & 3];
      const int m_tile = m_tile0 + wm * TM + j;
      if (m_tile < a.m_tiles) finish_tile<LAST>(a, leading[i][j], n_tile, m_tile, lane);
    }
  }
}

// A hidden layer for 129 to 4608 and 6145 to 10 240 rows, in rounds of one workgroup
// per compute unit of TN x TM tiles, K split over its waves.  A wave multiplies all of the
// workgroup's tiles over its part of K, so no fragment is wanted by two waves:
// they come straight from L2 into a ring of RING k-steps of registers (no LDS,
// no barrier until the end), where the waves' sums then meet in wave order.
// What bounds it is the L2 of those loads, (TN + TM) x 192 KiB per workgroup,
// beside TN x TM x 1.3 us of MFMAs and some 3 us to start and to write back.
// Microseconds per layer at a full round, and on the fp32 matrix cores:
//
//   tiles  waves  rows    here  fp32        tiles  waves  rows    here  fp32
//   1 x 1    8     256     6.8   7.6        2 x 4    4    2048    19-24   33
//   1 x 2    8     512     8.9  12          4 x 3    4    3072    28      47
//   2 x 2    8    1024    12    18          4 x 4    4    4096    32-34   61
//   2 x 3    4    1536    15.5  26
//
// (mid_kernel with 128 x 128 blocks took 37-40 at 3072 and 4096 rows.)  Four
// waves have twice the registers each: room for more tiles, where one wave per
// SIMD and a ring of two k-steps keep the matrix cores fed.  With 12 and 16 tiles
// there is room for one set of sums only; K in four parts still keeps its error
// below the fp32 kernels' (1.0e-7 of an fp64 evaluation against 1.6e-7; with two
// sets 4.6e-8 against 0.9-1.2e-7).
// XN = 4: an XCD reads a quarter of the weights and half of the activations
// (1, 2 and 8 are within 5 %).  Tried and not faster: 16 waves (6.9 us at 160
// rows, 16.8 at 700), 2 x 4 tiles on eight waves (out of registers), four waves
// of 2 x 2 (12.4), 1 x 3 on eight (11.1 at 700 rows, 2 x 2 11.4), deeper rings.
template <int TN, int TM, int WAVES, int RING, int XN, int SETS = 2>
struct Small {
  static constexpr int BN = TN, BM = TM, TILES = TN * TM, XM = 8 / XN;
  static constexpr int THREADS = WAVES * 64;
  static constexpr int STEPS = kSteps / WAVES;     // per wave
  static constexpr int PHASES = WAVES * TILES > 40 ? 2 : 1;  // the sums meet in as many parts
  static constexpr int PART = TILES / PHASES;      // tiles of a part
  static constexpr int HALVES = 2 * PART;          // half tiles: a k-step of the next layer
  static constexpr int LDS = WAVES * PART * 16 * 64 * (int)sizeof(float);
  static constexpr int NBLK = (kWidth / 32) / BN;
  static_assert(kSteps % WAVES == 0 && RING <= STEPS, "every wave has as many steps");
  static_assert(TILES % PHASES == 0 && LDS <= 160 * 1024, "the sums of all waves fit the LDS");
};

template <int TN, int TM, int WAVES, int RING, int XN, int SETS, bool LAST>
__global__ __launch_bounds__(WAVES * 64, WAVES / 4) void small_kernel(const LayerArgs a) {
  using S = Small<TN, TM, WAVES, RING, XN, SETS>;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  float* const red = reinterpret_cast<float*>(lds);  // [wave][tile][register][lane]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 31, h = lane >> 5;
  int n_blk, m_blk;
  block_of<S::NBLK, XN>((int)blockIdx.x, n_blk, m_blk);
  if (m_blk * TM >= a.m_tiles) return;
  const int n_tile0 = n_blk * TN, m_tile0 = m_blk * TM;

  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(a.w), 0, (kWidth / 32) * kTileBytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(a.x), 0, a.m_tiles * kTileBytes, 0x00020000);
  const int step0 = wave * S::STEPS * kStepBytes;
  int x_base[TM];  // (a tile past the end of the batch: the last one again, nothing stored)
#pragma unroll
  for (int j = 0; j < TM; ++j)
    x_base[j] = (m_tile0 + j < a.m_tiles ? m_tile0 + j : a.m_tiles - 1) * kTileBytes + step0;
  const int w_base = n_tile0 * kTileBytes + step0;

  bf16x8 w[RING][kPieces][TN], x[RING][kPieces][TM];
  auto load = [&](int slot, int step) {
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
        w[slot][p][i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
            w_rsrc, lane * 16 + p * kFragBytes, w_base + i * kTileBytes + step * kStepBytes, 0));
#pragma unroll
      for (int j = 0; j < TM; ++j)
        x[slot][p][j] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
            x_rsrc, lane * 16 + p * kFragBytes, x_base[j] + step * kStepBytes, 0));
    }
  };
  f32x16 acc[SETS][TN][TM];  // with two: the leading products' and the small ones'
#pragma unroll
  for (int t = 0; t < SETS; ++t)
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][i][j][r] = 0.f;
  auto mm = [&](f32x16(&d)[TN][TM], const bf16x8(&p)[TN], const bf16x8(&q)[TM]) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        d[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p[i], q[j], d[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < RING - 1; ++s) load(s, s);
#pragma unroll
  for (int s = 0; s < S::STEPS; ++s) {
    const int c = s % RING;
    if (s + RING - 1 < S::STEPS) load((s + RING - 1) % RING, s + RING - 1);
    HBT_FENCE;
    mm(acc[0], w[c][0], x[c][0]);
    mm(acc[SETS - 1], w[c][0], x[c][1]);
    mm(acc[SETS - 1], w[c][1], x[c][0]);
    mm(acc[SETS - 1], w[c][1], x[c][1]);
    mm(acc[SETS - 1], w[c][0], x[c][2]);
    mm(acc[SETS - 1], w[c][2], x[c][0]);
    HBT_FENCE;
  }

#pragma unroll
  for (int phase = 0; phase < S::PHASES; ++phase) {
    if (phase > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < S::PART; ++t) {
      const int i = (phase * S::PART + t) / TM, j = (phase * S::PART + t) % TM;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        red[((wave * S::PART + t) * 16 + r) * 64 + lane] =
            SETS == 2 ? acc[0][i][j][r] + acc[SETS - 1][i][j][r] : acc[0][i][j][r];
    }
    __syncthreads();
    // half tiles go round the waves: accumulator registers 8 kk .. 8 kk + 7 of a tile
    constexpr int kPerWave = (S::HALVES + WAVES - 1) / WAVES;
    float share[kPerWave];
#pragma unroll
    for (int q = 0; q < kPerWave; ++q) {
      const int half = wave + q * WAVES;
      share[q] = 0.f;
      if (S::HALVES % WAVES != 0 && half >= S::HALVES) continue;
      const int t = half >> 1, kk = half & 1, tile = phase * S::PART + t;
      const int n_tile = n_tile0 + tile / TM, m_tile = m_tile0 + tile % TM;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float sum = red[(t * 16 + 8 * kk + e) * 64 + lane];
#pragma unroll
        for (int p = 1; p < WAVES; ++p) sum += red[((p * S::PART + t) * 16 + 8 * kk + e) * 64 + lane];
        v[e] = sum;
      }
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int n = n_tile * 32 + 16 * kk + 8 * g + 4 * h;
        const f32x4 b = *reinterpret_cast<const f32x4*>(a.bias + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * g + e] = relu_nan(v[4 * g + e] + b[e]);
        if (LAST) {
          const f32x4 wl = *reinterpret_cast<const f32x4*>(a.w_last + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) share[q] = fmaf(v[4 * g + e], wl[e], share[q]);
        }
      }
      if (LAST)
        share[q] += __shfl_xor(share[q], 32);
      else if (m_tile < a.m_tiles)
        store_split(a.y + tile_offset(m_tile, 2 * n_tile + kk) + lane * 16, v);
    }
    if (LAST) {
      // a tile's two half shares of the final dot product
      __syncthreads();
#pragma unroll
      for (int q = 0; q < kPerWave; ++q) {
        const int half = wave + q * WAVES;
        if (half < S::HALVES && h == 0) red[half * 32 + m] = share[q];
      }
      __syncthreads();
      for (int i = threadIdx.x; i < S::PART * 32; i += S::THREADS) {
        const int t = i >> 5, row = i & 31, tile = phase * S::PART + t;
        const int n_tile = n_tile0 + tile / TM, m_tile = m_tile0 + tile % TM;
        if (m_tile < a.m_tiles)
          a.part[(size_t)n_tile * (a.m_tiles * kRows) + m_tile * kRows + row] =
              red[(2 * t) * 32 + row] + red[(2 * t + 1) * 32 + row];
      }
    }
  }
}

// The packed fp32 weights of one layer (pack_layer in mlp.hip) in pieces; once,
// when the network is loaded.  One wavefront per (n-tile, k-step).
struct PackArgs {
  const float* w_stream;
  int32_t groups_total;  // k-groups per wave stream
  int32_t g0;            // first k-group of this layer
  char* w;
};
__global__ __launch_bounds__(256) void pack_kernel(const PackArgs a) {
  const int lane = threadIdx.x & 63;
  const int item = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int tile = item / kSteps, step = item % kSteps;
  const f32x4* in = reinterpret_cast<const f32x4*>(a.w_stream) +
                    ((size_t)(tile >> 3) * a.groups_total + a.g0 + 2 * step) * (8 * 64) +
                    (tile & 7) * 64 + lane;
  float v[8];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[4 * g + e] = in[g * (8 * 64)][e];
  store_split(a.w + tile_offset(tile, step) + lane * 16, v);
}

// Whether a layer may hold this weight and be an fp32 layer in pieces.  From
// kMostWeight on (an infinity too) the products of its smaller pieces with a large
// activation's can overflow with another sign than the leading product's: NaN where
// fp32 has an infinity.
constexpr float kMostWeight = 0x1p7f;
__device__ __host__ constexpr bool fits_pieces(float w) { return w < kMostWeight && w > -kMostWeight; }
// Nonzero weights that an output has at least, or none.  A nonzero product takes up
// to six roundings of the running sum here and one on the fp32 matrix cores; over a
// whole row those are more, because they add two products at a time and not eight.
// Errors in 2^-24 of the output's rms, here and there, for the kernels with one set
// of sums, weights of both signs: 0.95 / 1.13 and 0.85 / 0.82 with 32 and 64, 1.10 /
// 0.94 with 128, 0.88 / 0.99 with 192, 1.22 / 2.29 with all; large_kernel, all positive: 1.57 /
// 1.41 with 32, 1.97 / 1.97 with 64, 3.83 / 7.82 with all.
constexpr int kLeastNonzero = 192;

// Sets *outside where a layer's weights are not for pieces; once, when the network
// is loaded.  One wavefront per n-tile (blockIdx.x) and layer (blockIdx.y).
struct CheckArgs {
  const float* w_stream;
  int32_t groups_total;  // k-groups per wave stream
  int32_t g0;            // first k-group of the first layer
  uint32_t* outside;
};
__global__ __launch_bounds__(64) void check_kernel(const CheckArgs a) {
  const int lane = threadIdx.x, tile = blockIdx.x;
  const f32x4* in = reinterpret_cast<const f32x4*>(a.w_stream) +
                    ((size_t)(tile >> 3) * a.groups_total + a.g0 + blockIdx.y * (kWidth / 8)) * (8 * 64) +
                    (tile & 7) * 64 + lane;
  bool fits = true;
  int nonzero = 0;
#pragma unroll 8
  for (int g = 0; g < kWidth / 8; ++g) {
    const f32x4 v = in[(size_t)g * (8 * 64)];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      fits = fits && fits_pieces(v[e]);
      nonzero += v[e] != 0.f;
    }
  }
  nonzero += __shfl_xor(nonzero, 32);
  if (!fits || (nonzero > 0 && nonzero < kLeastNonzero)) *a.outside = 1;  // (all the same value)
}

struct FirstArgs {
  const double* raw;     // [n][in_features]
  const double* mu;
  const double* sigma;
  const float* w_t;      // fc1.weight transposed, [MAX_IN][kWidth]
  const float* bias;
  int32_t in_features;
  int64_t n;
  char* y;               // activations out, [m_tiles] tiles
};
constexpr int kFirstSlices = 8;

// fc1: K is a dozen, so the layer is its 6 KiB-per-row write and little else, and
// plain FMAs from LDS do it.  A workgroup takes one m-tile and a slice of the
// outputs (an eighth: 2 / 8 / 16 / 32 slices took 19.4 / 8.4 / 10.0 / 13.6 us at
// 4096 rows when the output was fp32).  Sum order: bias, then k ascending.
// 16 384 rows: 20.5 us, 4.9 TB/s (a large copy on this card: 4.8).
template <int MAX_IN>
__global__ __launch_bounds__(256) void first_kernel(const FirstArgs a) {
  constexpr int kSlice = kWidth / kFirstSlices;
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
  for (int s = wave; s < kSlice / 16; s += 4) {
    float v[8];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(a.bias + n_base + 16 * s + 8 * g + 4 * h);
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
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = relu_nan(v[j]);
    store_split(a.y + tile_offset(m_tile, n_base / 16 + s) + lane * 16, v);
  }
}

struct FinishArgs {
  const float* part;  // [kWidth / 32][rows_pad] shares of the final dot product
  int32_t rows_pad;
  float b_last;
  int64_t n;
  float* out;         // [n]
};

// fc2: the shares of the final dot product that the last hidden layer left, added in
// n-tile order, in double: in fp32 these 32 sums were half of a prediction's error.
__device__ __forceinline__ float sum_of_shares(const float* part, int32_t rows_pad, int64_t row,
                                               float b_last) {
  float v[kWidth / 32];
#pragma unroll
  for (int t = 0; t < kWidth / 32; ++t) v[t] = part[(size_t)t * rows_pad + row];
  double sum = b_last;
#pragma unroll
  for (int t = 0; t < kWidth / 32; ++t) sum += (double)v[t];
  return (float)sum;
}

__global__ __launch_bounds__(256) void finish_kernel(const FinishArgs a) {
  const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (row < a.n) a.out[row] = sum_of_shares(a.part, a.rows_pad, row, a.b_last);
}

}  // namespace split
}  // namespace hbt
