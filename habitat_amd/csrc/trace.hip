// Trace-level prediction for a sweep of destination devices: the sums the
// reference forms in Python after scaling each kernel, fused into the scaling.
//
//   hbt_wave_scale_sum   per destination d and segment s (one segment per
//                        forward/backward pass of an operation):
//                        sum over the segment's kernel records of the scaled
//                        time t'(d)  — the sum in RunTimePrediction.run_time_ms
//                        (analyzer/habitat/analysis/run_time.py:50-58) over the
//                        kernels Predictor._wave_scale predicted
//                        (analyzer/habitat/analysis/predictor.py:116-124).
//                        Scaled times never reach HBM: traffic is the record
//                        columns once per destination row of the grid (they stay
//                        in L2) plus 8 bytes per (destination, segment).  Sums of
//                        runs that span wavefronts meet in floating-point atomics.
//   hbt_wave_scale_sum_ordered
//                        the same sums for segments that are runs of consecutive
//                        records, added in the records' order as the reference
//                        adds them, without atomics: the scaled times pass
//                        through a caller's workspace and one thread per
//                        (segment, destination) adds them up.
//   hbt_wave_scale_sum_totals
//                        the same with each destination's total, for some rows of a
//                        sweep's destinations.
//   hbt_ratio_scale      per destination and MLP-predicted operation:
//                        run_time_ms * pred_dest / pred_origin, negative -> 0
//                        (predictor.py:132-148 and :182,218,238,283), the
//                        per-destination sum of those and the number replaced;
//   hbt_ratio_scale_kinds
//                        for all kinds of operation in one launch: all that a sweep
//                        does once its networks are done (five launches of 4 to 11 us
//                        each before, and the sums' seven).
//
// Destinations live in a device-resident table (hbt_device_table) so that one
// launch covers all of them: blockIdx.y is a group of destinations, and their
// constants come through scalar loads.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <new>
#include <vector>

#include "../../include/habitat_mi.h"
#include "occupancy.h"
#include "wave_scale.h"

#pragma clang fp contract(off)

#include "wave_scale_device.h"

struct hbt_device_table {
  int32_t n_dest;
  int32_t model;           // dev::kModel...: which occupancy models the kernel needs
  int device;
  hbt::OriginArgs origin;
  hbt::DestArgs* dests;    // device memory, [n_dest]
};

namespace hbt {
namespace {

using namespace dev;

constexpr int kBlock = 256;
// Destinations one thread of wave_scale_sum_kernel walks over (blockIdx.y counts
// groups of this many): the record is loaded and its origin part computed once
// per group, and the occupancy model runs once per run of destinations with
// equal occupancy constants within the group.
constexpr int kSumGroup = 8;

// Where destination d's results go: row d of the outputs, or the row that `rows` names;
// -1 where there is no such row.
struct OutputRows {
  const int32_t* rows;  // [n_dest], nullable
  int32_t count;        // of the outputs' rows
  __device__ int of(int d) const {
    const int row = rows != nullptr ? rows[d] : d;
    return row >= 0 && row < count ? row : -1;
  }
};

struct SumArgs {
  int64_t n;
  int32_t n_segments;
  int32_t n_dest;
  const int32_t* num_blocks;
  const int32_t* block_size;
  const int32_t* dynamic_smem;
  const int32_t* static_smem;
  const int32_t* regs;
  const int32_t* dest_regs;    // nullable
  const double* run_time_ns;
  const double* flop_sp_efficiency;
  const double* dram_read_bytes;
  const double* dram_write_bytes;
  const uint8_t* has_metrics;  // nullable
  const int32_t* segment;      // nullable: all records in segment 0
  double* out_sum;             // [n_dest][n_segments]
  int32_t* out_bad;            // [n_dest], nullable
  double* work;                // ORDERED: [n_dest][n]
  const DestArgs* dests;
  OriginArgs origin;
  OutputRows out;              // ORDERED: rows of out_bad
};

__global__ void fill_zero_kernel(double* sums, int64_t n_sums, int32_t* bad, int32_t n_bad) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_sums) sums[i] = 0.0;
  if (bad != nullptr && i < n_bad) bad[i] = 0;
}

__global__ void zero_rows_kernel(int32_t* bad, int32_t n_dest, OutputRows out) {
  const int d = (int)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n_dest) return;
  const int row = out.of(d);
  if (row >= 0) bad[row] = 0;
}

// One thread per record and group of kSumGroup destinations.  Within a
// wavefront, consecutive records of the same segment are summed with a
// segmented scan and the last lane of each run adds the run's total to the
// segment's sum, per destination.
// ORDERED: no sums here; each scaled time (+0 where the reference would raise)
// goes to a.work[destination][record] for segment_sum_ordered_kernel to add up
// in the records' order.
template <int MODEL, bool ORDERED>
__global__ __launch_bounds__(kBlock) void wave_scale_sum_kernel(const SumArgs a) {
  const int d0 = blockIdx.y * kSumGroup;
  const int d1 = d0 + kSumGroup < a.n_dest ? d0 + kSumGroup : a.n_dest;
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool in_range = i < a.n;
  const int64_t j = in_range ? i : 0;

  RecordIn r;
  r.nb = a.num_blocks[j];
  r.block = a.block_size[j];
  r.smem_total = smem_sum(a.static_smem[j], a.dynamic_smem[j]);
  r.regs = a.regs[j];
  r.dest_regs = a.dest_regs != nullptr ? a.dest_regs[j] : -1;
  r.metrics = a.has_metrics != nullptr ? a.has_metrics[j] != 0 : true;
  r.t = a.run_time_ns[j];
  r.eff = a.flop_sp_efficiency[j];
  r.rd = a.dram_read_bytes[j];
  r.wr = a.dram_write_bytes[j];
  // lanes past the end form a run of their own so that they never swallow a tail
  const int32_t seg = (in_range && !ORDERED) ? (a.segment != nullptr ? a.segment[j] : 0) : -1;

  RecordMid m = origin_part<MODEL>(a.origin, r);
  if (__builtin_expect(m.redo_gflops, 0))
    m.num_gflops = origin_gflops_exact(a.origin.peak_gflops, r.eff, r.t);
  finish_mid<false>(m, 0.0);

  // Runs of equal segment ids get increasing run numbers, so that equal run
  // numbers at any distance mean "same run" even if a segment id repeats later.
  const int32_t prev_seg = __shfl_up(seg, 1);
  const bool head = lane == 0 || prev_seg != seg;
  const unsigned long long heads = __ballot(head);
  const int32_t run = (int32_t)__popcll(heads & ((2ull << lane) - 1ull));
  const int32_t next_run = __shfl_down(run, 1);
  const bool tail = lane == 63 || next_run != run;
  const bool adds = tail && in_range && seg >= 0 && seg < a.n_segments;

  int32_t occ_d = 0;
  for (int d = d0; d < d1; ++d) {
    const DestArgs& p = a.dests[d];
    // the first destination of a group never carries the mark
    if (!(p.dev.flags & kSameOccAsPrev)) occ_d = dest_occupancy<MODEL>(p, r, m);
    const double gamma = roofline_gamma(p, m.num_gflops, m.total_gb, r.metrics);
    RecordOut o = dest_scale<MODEL, false>(p, r, m, occ_d, gamma, 0.0);
    if (__builtin_expect(o.in_order, 0))
      o.t = scaled_time_in_order(r.t, o.gamma, p.log2_bw, p.log2_clk, p.log2_clk_sm);

    const bool ok = in_range && o.status == HBT_ST_OK;
    double v = ok ? o.t : 0.0;
    if (a.out_bad != nullptr) {
      const unsigned long long bad = __ballot(in_range && o.status != HBT_ST_OK);
      const int row = ORDERED ? a.out.of(d) : d;
      if (lane == 0 && bad != 0 && row >= 0) atomicAdd(a.out_bad + row, (int32_t)__popcll(bad));
    }
    if (ORDERED) {
      if (in_range) a.work[(int64_t)d * a.n + i] = v;
      continue;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double other = __shfl_up(v, off);
      const int32_t other_run = __shfl_up(run, off);
      if (lane >= off && other_run == run) v += other;
    }
    if (adds) unsafeAtomicAdd(a.out_sum + (int64_t)d * a.n_segments + seg, v);
  }
}

struct OrderedSumArgs {
  int64_t n;
  int32_t n_segments;
  const double* work;            // [n_dest][n], from wave_scale_sum_kernel<., true>
  const int64_t* segment_start;  // [n_segments + 1]
  double* out_sum;               // [rows][n_segments]
  OutputRows out;
  // a sweep's totals: constant_ms + the segments' sums in milliseconds, NaN where a record
  // was bad
  double* out_total;             // [rows], nullable
  const int32_t* out_bad;        // [rows], with out_total
  double constant_ms;
  int32_t per_block;             // segments that a workgroup takes at a time, up to kBlock
  bool totals_here;              // kBlock at a time, and all of a destination's
};

// Sum of `v` over the workgroup, in one order; for thread 0.
__device__ __forceinline__ double block_sum(double v, double (&part)[kBlock / 64]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  double total = 0.0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) total += part[w];
  return total;
}

__device__ __forceinline__ void put_total(const OrderedSumArgs& a, int row, double mine,
                                          double (&part)[kBlock / 64]) {
  const double total = block_sum(mine, part);
  if (threadIdx.x == 0)
    a.out_total[row] = a.out_bad[row] > 0 ? __builtin_nan("") : a.constant_ms + total / 1e6;
}

// A thread per segment, up to 256 of them and a destination (blockIdx.x) to a workgroup: a
// thread adds its segment's scaled times one after the other in the records' order, as the
// reference adds a pass's kernels (run_time.py:50-58).  No floating-point atomics: the sum is
// the same every time, and the same as a sequential sum of the per-record kernel's times.
// Bound by that chain of additions for the longest segment (an optimizer pass is several
// hundred kernels): the times come through LDS, kStage of them at a time, so that no addition
// waits for memory (256 destinations of a ResNet-50's records: 21 us with loads of their own,
// 8 us).  A workgroup takes segments for about one stage (per_block), since those of the next
// stages would wait for them, and the workgroups of a destination are spread over gridDim.y
// where the destinations alone do not fill the GPU: one destination, a million records in
// 100 000 segments 28 us with the scaling and in 1000 segments 32, by one workgroup
// 3660 and 5390.
constexpr int kStage = 2048;
constexpr int kFillGrid = 1024;   // workgroups that fill the GPU
__global__ __launch_bounds__(kBlock) void segment_sum_ordered_kernel(const OrderedSumArgs a) {
  __shared__ double staged[kStage];
  __shared__ double part[kBlock / 64];
  __shared__ long long range[2];
  const int d = blockIdx.x, row = a.out.of(d);
  if (row < 0) return;
  const double* v = a.work + (int64_t)d * a.n;
  double mine = 0.0;
  for (int64_t s0 = (int64_t)blockIdx.y * a.per_block; s0 < a.n_segments;
       s0 += (int64_t)gridDim.y * a.per_block) {
    const int64_t s = (int)threadIdx.x < a.per_block ? s0 + (int)threadIdx.x : a.n_segments;
    // (clamped to the columns: a wrong boundary must not become a stray read)
    int64_t begin = 0, end = 0;
    if (s < a.n_segments) {
      begin = a.segment_start[s];
      end = a.segment_start[s + 1];
      begin = begin < 0 ? 0 : begin;
      end = end > a.n ? a.n : end;
    }
    if (threadIdx.x == 0) {
      range[0] = a.n;
      range[1] = 0;
    }
    __syncthreads();
    if (begin < end) {
      atomicMin(&range[0], (long long)begin);
      atomicMax(&range[1], (long long)end);
    }
    __syncthreads();
    const int64_t first = range[0], last = range[1];
    double sum = 0.0;
    for (int64_t c = first; c < last; c += kStage) {
      const int count = (int)(last - c < kStage ? last - c : kStage);
      __syncthreads();
      for (int j = threadIdx.x; j < count; j += kBlock) staged[j] = v[c + j];
      __syncthreads();
      const int from = (int)(begin > c ? (begin - c < count ? begin - c : count) : 0);
      const int to = (int)(end > c ? (end - c < count ? end - c : count) : 0);
#pragma unroll 8
      for (int j = from; j < to; ++j) sum += staged[j];
    }
    if (s < a.n_segments) a.out_sum[(int64_t)row * a.n_segments + s] = sum;
    mine += sum;
    __syncthreads();   // range is read above and set again
  }
  if (!a.totals_here) return;
  put_total(a, row, mine, part);
}

// The totals of destinations whose segments were spread, in the order of a workgroup that
// has them 256 at a time.
__global__ __launch_bounds__(kBlock) void segment_totals_kernel(const OrderedSumArgs a) {
  __shared__ double part[kBlock / 64];
  const int row = a.out.of(blockIdx.x);
  if (row < 0) return;
  double mine = 0.0;
  for (int64_t s = threadIdx.x; s < a.n_segments; s += kBlock)
    mine += a.out_sum[(int64_t)row * a.n_segments + s];
  put_total(a, row, mine, part);
}

struct GammaArgs {
  int64_t n;
  const double* run_time_ns;
  const double* flop_sp_efficiency;
  const double* dram_read_bytes;
  const double* dram_write_bytes;
  double* out_gamma;
  double peak_gflops;   // origin
  DestArgs dest;
};

// gamma alone (roofline.py:68-104), one thread per record; NaN where the
// reference's assertion 0 <= gamma <= 1 fails.
__global__ __launch_bounds__(kBlock) void roofline_gamma_kernel(const GammaArgs a) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= a.n) return;
  const double t = a.run_time_ns[i], eff = a.flop_sp_efficiency[i];
  const double total_gb = (a.dram_read_bytes[i] + a.dram_write_bytes[i]) * 0x1p-30;
  const double scaled = div_const<C100>(eff) * a.peak_gflops * t;
  double num_gflops = div_const<C1e9>(scaled);
  if (!(div_const_safe(eff) && div_const_safe(scaled)))
    num_gflops = origin_gflops_exact(a.peak_gflops, eff, t);
  const double gamma = roofline_gamma(a.dest, num_gflops, total_gb, true);
  a.out_gamma[i] = (gamma >= 0 && gamma <= 1) ? gamma : __builtin_nan("");
}

struct RatioArgs {
  hbt_ratio_kind kinds[HBT_RATIO_MAX_KINDS];
  int32_t n_kinds, n_dest;
  double* out_total;          // [n_dest], nullable; added to
  int32_t* out_clamped;       // [n_dest], nullable
  bool add_clamped;           // added to, or written
};

// blockIdx.x = destination; the block's threads stride over the operations of one kind
// after the other.  Operations with equal features share one column of pred.
__global__ __launch_bounds__(kBlock) void ratio_scale_kernel(const RatioArgs a) {
  __shared__ double part[kBlock / 64];
  __shared__ int32_t count;
  const int d = blockIdx.x;
  if (threadIdx.x == 0) count = 0;
  __syncthreads();
  double total = a.out_total != nullptr ? a.out_total[d] : 0.0;
  for (int k = 0; k < a.n_kinds; ++k) {
    const hbt_ratio_kind& kind = a.kinds[k];
    const float* dest = kind.pred + (int64_t)d * kind.n_rows;
    const float* orig = kind.pred + (int64_t)a.n_dest * kind.n_rows;
    double acc = 0.0;
    int32_t clamped = 0;
    for (int o = threadIdx.x; o < kind.n_ops; o += kBlock) {
      const int32_t row = kind.op_row != nullptr ? kind.op_row[o] : o;
      double ms = __builtin_nan("");
      if (row >= 0 && row < kind.n_rows) {
        // predictor.py:182: operation.run_time_ms * pred_dest / pred_orig, in fp64
        ms = kind.run_time_ms[o] * (double)dest[row] / (double)orig[row];
        if (ms < 0) {   // predictor.py:135-141: warned about and replaced by 0
          ms = 0.;
          ++clamped;
        }
      }
      if (kind.out_ms != nullptr) kind.out_ms[(int64_t)d * kind.n_ops + o] = ms;
      acc += ms;
    }
    if (a.out_total != nullptr) total += block_sum(acc, part);
    if (clamped > 0) atomicAdd(&count, clamped);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (a.out_total != nullptr) a.out_total[d] = total;
  if (a.out_clamped != nullptr) a.out_clamped[d] = a.add_clamped ? a.out_clamped[d] + count : count;
}

}  // namespace
}  // namespace hbt

extern "C" {

hbt_device_table* hbt_device_table_create(const hbt_device_spec* origin,
                                          const hbt_device_spec* dests, int32_t n_dest,
                                          int* err) {
  using namespace hbt;
  int dummy;
  if (err == nullptr) err = &dummy;
  *err = HBT_OK;
  if (origin == nullptr || dests == nullptr || n_dest <= 0) {
    *err = HBT_EINVAL;
    return nullptr;
  }
  if (n_dest > 65535) {
    *err = HBT_ESIZE;
    return nullptr;
  }
  int rc = hbt_device_spec_check(origin);
  for (int32_t d = 0; d < n_dest && rc == HBT_OK; ++d) rc = hbt_device_spec_check(&dests[d]);
  if (rc != HBT_OK) {
    *err = rc;
    return nullptr;
  }
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    *err = HBT_EHIP;
    return nullptr;
  }
  hbt_device_table* t = new (std::nothrow) hbt_device_table();
  if (t == nullptr) {
    *err = HBT_ENOMEM;
    return nullptr;
  }
  t->n_dest = n_dest;
  t->device = device;
  t->origin = make_origin_args(*origin);
  std::vector<DestArgs> host((size_t)n_dest);
  for (int32_t d = 0; d < n_dest; ++d) {
    host[d] = make_dest_args(*origin, dests[d]);
    // within a group of kSumGroup destinations, one that has the occupancy
    // constants of the one before it shares that one's occupancies
    if (d % kSumGroup != 0 && same_occupancy_constants(host[d - 1].dev, host[d].dev))
      host[d].dev.flags |= kSameOccAsPrev;
  }
  t->model = dev::model_for(t->origin.dev, host.data(), n_dest);
  t->dests = nullptr;
  const size_t bytes = sizeof(DestArgs) * (size_t)n_dest;
  if (hipMalloc(reinterpret_cast<void**>(&t->dests), bytes) != hipSuccess) {
    (void)hipGetLastError();
    delete t;
    *err = HBT_ENOMEM;
    return nullptr;
  }
  if (hipMemcpy(t->dests, host.data(), bytes, hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(t->dests);
    delete t;
    *err = HBT_EHIP;
    return nullptr;
  }
  return t;
}

void hbt_device_table_destroy(hbt_device_table* table) {
  if (table == nullptr) return;
  if (table->dests != nullptr) (void)hipFree(table->dests);
  delete table;
}

int32_t hbt_device_table_size(const hbt_device_table* table) {
  return table != nullptr ? table->n_dest : 0;
}

int hbt_wave_scale_sum(const hbt_device_table* table, int64_t n, const int32_t* num_blocks,
                       const int32_t* block_size, const int32_t* dynamic_smem,
                       const int32_t* static_smem, const int32_t* regs, const int32_t* dest_regs,
                       const double* run_time_ns, const double* flop_sp_efficiency,
                       const double* dram_read_bytes, const double* dram_write_bytes,
                       const uint8_t* has_metrics, const int32_t* segment, int32_t n_segments,
                       double* out_sum, int32_t* out_bad, void* hip_stream) {
  using namespace hbt;
  if (table == nullptr || n < 0 || n_segments <= 0 || out_sum == nullptr) return HBT_EINVAL;
  if (n > 0 && (!num_blocks || !block_size || !dynamic_smem || !static_smem || !regs ||
                !run_time_ns || !flop_sp_efficiency || !dram_read_bytes || !dram_write_bytes))
    return HBT_EINVAL;
  const int64_t blocks = (n + kBlock - 1) / kBlock;
  // (the clearing launch covers n_dest * n_segments sums with 256 threads per block)
  if (blocks > 0x7fffffff || (int64_t)n_segments * table->n_dest > ((int64_t)1 << 38))
    return HBT_ESIZE;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    return HBT_EHIP;
  }
  if (device != table->device) return HBT_EINVAL;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);

  const int64_t n_sums = (int64_t)table->n_dest * n_segments;
  const int64_t fill = n_sums > table->n_dest ? n_sums : table->n_dest;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((fill + kBlock - 1) / kBlock)), dim3(kBlock),
                     0, stream, out_sum, n_sums, out_bad, table->n_dest);
  if (hipGetLastError() != hipSuccess) return HBT_EHIP;
  if (n == 0) return HBT_OK;

  SumArgs a{};
  a.n = n;
  a.n_segments = n_segments;
  a.n_dest = table->n_dest;
  a.num_blocks = num_blocks; a.block_size = block_size; a.dynamic_smem = dynamic_smem;
  a.static_smem = static_smem; a.regs = regs; a.dest_regs = dest_regs;
  a.run_time_ns = run_time_ns; a.flop_sp_efficiency = flop_sp_efficiency;
  a.dram_read_bytes = dram_read_bytes; a.dram_write_bytes = dram_write_bytes;
  a.has_metrics = has_metrics; a.segment = segment;
  a.out_sum = out_sum; a.out_bad = out_bad;
  a.dests = table->dests;
  a.origin = table->origin;
  const dim3 grid((unsigned)blocks, (unsigned)((table->n_dest + kSumGroup - 1) / kSumGroup));
  dev::with_model(table->model, [&](auto m) {
    hipLaunchKernelGGL((wave_scale_sum_kernel<decltype(m)::value, false>), grid, dim3(kBlock), 0,
                       stream, a);
  });
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

int hbt_wave_scale_sum_totals(const hbt_device_table* table, int64_t n, const int32_t* num_blocks,
                              const int32_t* block_size, const int32_t* dynamic_smem,
                              const int32_t* static_smem, const int32_t* regs,
                              const int32_t* dest_regs, const double* run_time_ns,
                              const double* flop_sp_efficiency, const double* dram_read_bytes,
                              const double* dram_write_bytes, const uint8_t* has_metrics,
                              const int64_t* segment_start, int32_t n_segments, double* workspace,
                              const int32_t* out_rows, int32_t n_rows, double constant_ms,
                              double* out_sum, int32_t* out_bad, double* out_total,
                              void* hip_stream) {
  using namespace hbt;
  if (table == nullptr || n < 0 || n_segments <= 0 || out_sum == nullptr ||
      segment_start == nullptr || n_rows < 0 || (out_total != nullptr && out_bad == nullptr) ||
      (out_rows == nullptr && n_rows != table->n_dest))
    return HBT_EINVAL;
  if (n > 0 && (!num_blocks || !block_size || !dynamic_smem || !static_smem || !regs ||
                !run_time_ns || !flop_sp_efficiency || !dram_read_bytes || !dram_write_bytes ||
                !workspace))
    return HBT_EINVAL;
  const int64_t blocks = (n + kBlock - 1) / kBlock;
  if (blocks > 0x7fffffff || (int64_t)n_segments * table->n_dest > ((int64_t)1 << 38))
    return HBT_ESIZE;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    return HBT_EHIP;
  }
  if (device != table->device) return HBT_EINVAL;
  hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  const OutputRows out{out_rows, n_rows};
  if (out_bad != nullptr) {
    hipLaunchKernelGGL(zero_rows_kernel, dim3((unsigned)((table->n_dest + kBlock - 1) / kBlock)),
                       dim3(kBlock), 0, stream, out_bad, table->n_dest, out);
    if (hipGetLastError() != hipSuccess) return HBT_EHIP;
  }
  if (n > 0) {
    SumArgs a{};
    a.n = n;
    a.n_segments = n_segments;
    a.n_dest = table->n_dest;
    a.num_blocks = num_blocks; a.block_size = block_size; a.dynamic_smem = dynamic_smem;
    a.static_smem = static_smem; a.regs = regs; a.dest_regs = dest_regs;
    a.run_time_ns = run_time_ns; a.flop_sp_efficiency = flop_sp_efficiency;
    a.dram_read_bytes = dram_read_bytes; a.dram_write_bytes = dram_write_bytes;
    a.has_metrics = has_metrics;
    a.out_bad = out_bad;
    a.out = out;
    a.work = workspace;
    a.dests = table->dests;
    a.origin = table->origin;
    const dim3 grid((unsigned)blocks, (unsigned)((table->n_dest + kSumGroup - 1) / kSumGroup));
    dev::with_model(table->model, [&](auto m) {
      hipLaunchKernelGGL((wave_scale_sum_kernel<decltype(m)::value, true>), grid, dim3(kBlock), 0,
                         stream, a);
    });
    if (hipGetLastError() != hipSuccess) return HBT_EHIP;
  }
  OrderedSumArgs b{};
  b.n = n;
  b.n_segments = n_segments;
  b.work = workspace;
  b.segment_start = segment_start;
  b.out_sum = out_sum;
  b.out = out;
  b.out_total = out_total;
  b.out_bad = out_bad;
  b.constant_ms = constant_ms;
  const int64_t stage = n > 0 ? (int64_t)kStage * n_segments / n : kBlock;
  b.per_block = (int32_t)(stage > kBlock || stage >= n_segments ? kBlock : stage > 0 ? stage : 1);
  const int64_t blocks_all = ((int64_t)n_segments + b.per_block - 1) / b.per_block;
  const int64_t fill = table->n_dest < kFillGrid ? kFillGrid / table->n_dest : 1;
  const dim3 sum_grid((unsigned)table->n_dest, (unsigned)(blocks_all < fill ? blocks_all : fill));
  b.totals_here = out_total != nullptr && b.per_block == kBlock && sum_grid.y == 1;
  hipLaunchKernelGGL(segment_sum_ordered_kernel, sum_grid, dim3(kBlock), 0, stream, b);
  if (out_total != nullptr && !b.totals_here)
    hipLaunchKernelGGL(segment_totals_kernel, dim3((unsigned)table->n_dest), dim3(kBlock), 0, stream,
                       b);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

int hbt_wave_scale_sum_ordered(const hbt_device_table* table, int64_t n, const int32_t* num_blocks,
                               const int32_t* block_size, const int32_t* dynamic_smem,
                               const int32_t* static_smem, const int32_t* regs,
                               const int32_t* dest_regs, const double* run_time_ns,
                               const double* flop_sp_efficiency, const double* dram_read_bytes,
                               const double* dram_write_bytes, const uint8_t* has_metrics,
                               const int64_t* segment_start, int32_t n_segments, double* workspace,
                               double* out_sum, int32_t* out_bad, void* hip_stream) {
  return hbt_wave_scale_sum_totals(table, n, num_blocks, block_size, dynamic_smem, static_smem, regs,
                                   dest_regs, run_time_ns, flop_sp_efficiency, dram_read_bytes,
                                   dram_write_bytes, has_metrics, segment_start, n_segments,
                                   workspace, nullptr, table != nullptr ? table->n_dest : 0, 0.0,
                                   out_sum, out_bad, nullptr, hip_stream);
}

int hbt_roofline_gamma(const hbt_device_spec* origin, const hbt_device_spec* dest, int64_t n,
                       const double* run_time_ns, const double* flop_sp_efficiency,
                       const double* dram_read_bytes, const double* dram_write_bytes,
                       double* out_gamma, void* hip_stream) {
  using namespace hbt;
  if (origin == nullptr || dest == nullptr || n < 0) return HBT_EINVAL;
  int rc = hbt_device_spec_check(origin);
  if (rc == HBT_OK) rc = hbt_device_spec_check(dest);
  if (rc != HBT_OK) return rc;
  if (n == 0) return HBT_OK;
  if (!run_time_ns || !flop_sp_efficiency || !dram_read_bytes || !dram_write_bytes || !out_gamma)
    return HBT_EINVAL;
  const void* cols[] = {run_time_ns, flop_sp_efficiency, dram_read_bytes, dram_write_bytes,
                        out_gamma};
  for (const void* p : cols)
    if (reinterpret_cast<uintptr_t>(p) % 8 != 0) return HBT_EALIGN;
  const int64_t blocks = (n + kBlock - 1) / kBlock;
  if (blocks > 0x7fffffff) return HBT_ESIZE;
  if (hbt_device_count() <= 0) return HBT_EHIP;
  GammaArgs a{};
  a.n = n;
  a.run_time_ns = run_time_ns; a.flop_sp_efficiency = flop_sp_efficiency;
  a.dram_read_bytes = dram_read_bytes; a.dram_write_bytes = dram_write_bytes;
  a.out_gamma = out_gamma;
  a.peak_gflops = origin->peak_gflops;
  a.dest = make_dest_args(*origin, *dest);
  hipLaunchKernelGGL(roofline_gamma_kernel, dim3((unsigned)blocks), dim3(kBlock), 0,
                     static_cast<hipStream_t>(hip_stream), a);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

int hbt_ratio_scale(const float* pred, int32_t n_dest, int32_t n_rows, const int32_t* op_row,
                    int32_t n_ops, const double* run_time_ms, double* out_ms, double* out_total,
                    int32_t* out_clamped, void* hip_stream) {
  using namespace hbt;
  if (n_dest < 0 || n_ops < 0 || n_rows < 0) return HBT_EINVAL;
  if (op_row == nullptr && n_rows != n_ops) return HBT_EINVAL;
  if (n_dest == 0 || n_ops == 0) return HBT_OK;
  if (pred == nullptr || run_time_ms == nullptr ||
      (out_ms == nullptr && out_total == nullptr && out_clamped == nullptr))
    return HBT_EINVAL;
  if (n_rows == 0) return HBT_EINVAL;
  RatioArgs a{};
  a.kinds[0] = {pred, op_row, run_time_ms, out_ms, n_rows, n_ops};
  a.n_kinds = 1;
  a.n_dest = n_dest;
  a.out_total = out_total;
  a.out_clamped = out_clamped;
  a.add_clamped = true;
  hipLaunchKernelGGL(ratio_scale_kernel, dim3((unsigned)n_dest), dim3(kBlock), 0,
                     static_cast<hipStream_t>(hip_stream), a);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

int hbt_ratio_scale_kinds(const hbt_ratio_kind* kinds, int32_t n_kinds, int32_t n_dest,
                          double* out_total, int32_t* out_clamped, void* hip_stream) {
  using namespace hbt;
  if (n_dest < 0 || n_kinds < 0 || n_kinds > HBT_RATIO_MAX_KINDS || (n_kinds > 0 && !kinds))
    return HBT_EINVAL;
  for (int k = 0; k < n_kinds; ++k) {
    const hbt_ratio_kind& kind = kinds[k];
    if (kind.n_ops < 0 || kind.n_rows < 0) return HBT_EINVAL;
    if (kind.n_ops > 0 && (kind.pred == nullptr || kind.run_time_ms == nullptr || kind.n_rows == 0 ||
                           (kind.op_row == nullptr && kind.n_rows != kind.n_ops)))
      return HBT_EINVAL;
  }
  if (n_dest == 0) return HBT_OK;
  RatioArgs a{};
  for (int k = 0; k < n_kinds; ++k) a.kinds[k] = kinds[k];
  a.n_kinds = n_kinds;
  a.n_dest = n_dest;
  a.out_total = out_total;
  a.out_clamped = out_clamped;
  hipLaunchKernelGGL(ratio_scale_kernel, dim3((unsigned)n_dest), dim3(kBlock), 0,
                     static_cast<hipStream_t>(hip_stream), a);
  return hipGetLastError() == hipSuccess ? HBT_OK : HBT_EHIP;
}

}  // extern "C"
