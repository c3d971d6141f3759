// A short host list of integers to device memory through kernel arguments.
//
// A request's block table reaches the single-request calls as a host list. A
// copy from pageable memory makes the host wait for everything queued on the
// stream (two of them were 45 us of a 67 us single-request decode); as kernel
// arguments the values travel with the launch itself, and the call stays
// asynchronous. A kernel argument block holds 4 KB, so a launch carries 960
// 32-bit values (block ids are checked against the pool before). Measured: a single-request
// fp16 decode of 2,048 tokens, 32/8 heads of 128, 68.0 us per call with two
// copies, 33.8 us; a 500-query chunk after 16,000 keys 159 and 140 us.
#include "mlr_common.h"

namespace mlr {
namespace {

constexpr int kPerLaunch = 960;
constexpr int64_t kMost = 4 * kPerLaunch;  // a longer list is a copy's work

struct StageArgs {
  int32_t v[kPerLaunch];
  int64_t *dst;
  int n;
};

__global__ __launch_bounds__(kPerLaunch) void stage_kernel(StageArgs a) {
  // Read as memory: indexing the by-value array by thread would first copy it
  // to every thread's scratch.
  typedef __attribute__((address_space(4))) const int32_t const_i32;
  const const_i32 *v = (const const_i32 *)__builtin_amdgcn_kernarg_segment_ptr();
  const int i = threadIdx.x;
  if (i < a.n) a.dst[i] = v[i];
}

}  // namespace
}  // namespace mlr

using namespace mlr;

extern "C" int mlr_stage_i64(const int64_t *host_values, int64_t n, int64_t *dst, void *stream) {
  clear_error();
  MLR_REQUIRE(n >= 0 && n <= kMost, "mlr_stage_i64: n must be in [0, %lld]", (long long)kMost);
  if (n == 0) return MLR_OK;
  MLR_REQUIRE(host_values && dst, "mlr_stage_i64: null pointer argument");
  for (int64_t i = 0; i < n; ++i)
    MLR_REQUIRE(host_values[i] >= INT32_MIN && host_values[i] <= INT32_MAX,
                "mlr_stage_i64: value %lld does not fit 32 bits", (long long)host_values[i]);
  for (int64_t at = 0; at < n; at += kPerLaunch) {
    StageArgs a;
    a.n = static_cast<int>(n - at < kPerLaunch ? n - at : kPerLaunch);
    for (int i = 0; i < a.n; ++i) a.v[i] = static_cast<int32_t>(host_values[at + i]);
    a.dst = dst + at;
    const unsigned threads = static_cast<unsigned>(ceil_div(a.n, kWave) * kWave);
    stage_kernel<<<1, threads, 0, static_cast<hipStream_t>(stream)>>>(a);
    const int rc = check_launch("mlr_stage_i64");
    if (rc != MLR_OK) return rc;
  }
  return MLR_OK;
}
