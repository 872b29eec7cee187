// Signed gathers out of many small parameter tensors (CDNA4, gfx950).
//
// A layer's kernels read its parameters in assembled forms -- the heads'
// intertwiners as one block matrix, the readout heads as one mixing matrix per
// input frequency, the trunks stacked -- whose every entry is one parameter,
// possibly negated, or zero.  The reference assembles them with concatenations
// and stacks per head and block on every call (nn/attention.py:653-669,
// nn/kernels.py:506-546); here one launch writes every assembled form of a
// layer, and one launch in the backward writes every parameter's gradient:
//
//   out[e] = sum over u < uses of s(code[u][e]) src[t(code)][o(code)]
//
// with the terms added in order (deterministic).  Launch-bound: the forms of an
// eight-head layer of 160 reals take one launch of about 10 us in place of 46
// launches forward and 110 backward.
#include <hip/hip_runtime.h>

#include "common.hpp"

namespace gm {
namespace {

// Tensors a launch reads: their addresses travel in the kernel's arguments
// (2 KiB of the 4 KiB a launch may carry).
constexpr int kMaxSources = 256;

struct GatherArgs {
  const float* src[kMaxSources];
  const int64_t* codes;  // (uses, n): -1 (zero) or t << 40 | offset << 1 | negative
  float* out;
  int64_t n;
  int uses;
};

constexpr int kThreads = 256;

__global__ __launch_bounds__(kThreads) void signed_gather_kernel(GatherArgs a) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= a.n) return;
  float sum = 0.f;
  for (int u = 0; u < a.uses; ++u) {
    const int64_t code = a.codes[u * a.n + e];
    if (code < 0) continue;
    const float* p = a.src[code >> 40];
    if (p == nullptr) continue;  // an absent gradient
    const float x = p[(code >> 1) & ((int64_t(1) << 39) - 1)];
    const float s = (code & 1) ? -x : x;
    sum = u == 0 ? s : sum + s;
  }
  a.out[e] = sum;
}

}  // namespace
}  // namespace gm

extern "C" int gm_signed_gather_f32(const float* const* src, int64_t n_src, const int64_t* codes, int64_t uses,
                                    int64_t n, float* out, void* stream) {
  GM_REQUIRE(n_src >= 0 && n_src <= gm::kMaxSources, "at most 256 source tensors");
  GM_REQUIRE(n >= 0 && uses >= 1 && uses <= 64, "n must be non-negative and uses in [1, 64]");
  if (n == 0) return GM_OK;
  GM_REQUIRE((n_src == 0 || src) && codes && out, "src must be a host array, codes and out device pointers");
  gm::GatherArgs a;
  for (int64_t i = 0; i < gm::kMaxSources; ++i) a.src[i] = i < n_src ? src[i] : nullptr;
  a.codes = codes;
  a.out = out;
  a.n = n;
  a.uses = (int)uses;
  hipLaunchKernelGGL(gm::signed_gather_kernel, dim3((unsigned)((n + gm::kThreads - 1) / gm::kThreads)),
                     dim3(gm::kThreads), 0, (hipStream_t)stream, a);
  return gm::check_launch("signed_gather");
}
