// The few-row MLP kernel (habitat_amd/csrc/mlp_chain.h) with its hand-over's memory
// in the caller's hands: tests/test_mlp_chain_gpu.py sets the counter of calls to
// where years of calls would have brought it.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../habitat_amd/csrc/mlp_chain.h"

extern "C" {

int chain_carries(uint64_t word, uint32_t call) { return hbt::chain::carries(word, call); }

int chain_max_rows() { return hbt::chain::kMaxRows; }
int chain_max_looks() { return hbt::chain::kMaxLooks; }

// Device pointers; the shapes are those of hbt::chain::Args.
int chain_forward(const float* w_stream, int32_t first_groups, int32_t hidden,
                  const float* w_first_t, const float* bias, const float* w_last, float b_last,
                  const double* raw, const double* mu, const double* sigma, int32_t in_features,
                  int32_t n, float* out, uint64_t* tickets, uint64_t* words, int32_t looks,
                  void* stream) {
  if (looks < 0 || looks > hbt::chain::kMaxLooks || n < 1 || n > hbt::chain::kMaxRows || hidden < 1 || in_features < 1 ||
      in_features > 8 * first_groups || 8 * first_groups > hbt::chain::kMaxIn)
    return -1;
  hbt::chain::Args a{};
  a.w_stream = w_stream;
  a.first_groups = first_groups;
  a.groups_total = first_groups + hidden * (hbt::chain::kWidth / 8);
  a.hidden = hidden;
  a.w_first_t = w_first_t;
  a.bias = bias;
  a.w_last = w_last;
  a.b_last = b_last;
  a.raw = raw; a.mu = mu; a.sigma = sigma;
  a.in_features = in_features;
  a.n = n;
  a.out = out;
  a.tickets = tickets;
  a.words = words;
  a.looks = looks;
  return hbt::chain::launch(a, static_cast<hipStream_t>(stream)) == hipSuccess ? 0 : -2;
}

}  // extern "C"
