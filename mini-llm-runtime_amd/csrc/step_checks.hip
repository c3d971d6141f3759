// The device-side checks of a step's metadata, in one launch.
//
// The host layer validates what a call was given before anything is written:
// context lengths against the block tables, block ids against the pool, each
// token's position and slot against its request's table, and no slot twice
// (reference: kernels/reference/paged_attention.py:224-238,
// model/qwen2.py:578-602, runtime/paged_kv_cache.py:235-239). As torch
// operations that is 12 to 30 launches of a few values each, which is what a
// small call then spends its time on: the checked decode of four short FP32
// requests took 105 us for a 7 us kernel.
//
// Workgroup j takes the table rows j, j + G, ... (one row at a time, its 256
// threads along the columns) and the tokens [64 j, 64 j + 64): it finds each
// token's request by binary search in query_start_loc, compares position and
// slot with what the table gives, and its slot with those of all earlier
// tokens, which pass through LDS as broadcast reads, a quarter per wave
// (6.4 us at 1,021 tokens, 9.5 at 2,048, where a sort takes 22 and 27). Every workgroup writes one word of
// flags of its own, so there is nothing to clear first and nothing to add
// up; the host reads the words in the one transfer that it waits for anyway.
#include <algorithm>

#include "mlr_common.h"

namespace mlr {
namespace {

constexpr int kThreads = 256;
constexpr int kTokens = 64;       // tokens per workgroup
constexpr int kTile = 1024;       // earlier tokens staged at a time
constexpr int kMaxGroups = 256;   // workgroups, unless the tokens need more
constexpr int64_t kMaxTokens = 8192;  // past this a sort finds a repeat sooner

// Flags; the values are in mlr_attn.h.
struct CheckParams {
  const int64_t *bt;
  int64_t bt_stride;
  int width;
  const int64_t *ctx;
  int reqs;
  const int64_t *qsl;  // null: token t is request t's only one
  const int64_t *positions;
  const int64_t *slots;
  int tokens;
  const uint8_t *decoding;  // [reqs] or null (every token in the prefill flags)
  int64_t block_size, num_blocks, max_query_len;
  int64_t *out;  // [groups] flags, then, with detail, qsl, ctx and bad rows
  int detail;
};

__global__ __launch_bounds__(kThreads) void check_step(CheckParams p) {
  __shared__ __align__(16) int64_t keys[kTile];
  __shared__ int64_t own[kTokens];
  __shared__ unsigned int wave_flags[kThreads / kWave];
  const int tid = threadIdx.x, groups = gridDim.x;
  const int64_t bs = p.block_size;
  unsigned int flags = 0;

  for (int r = blockIdx.x; r < p.reqs; r += groups) {
    const int64_t ctx = p.ctx[r];
    // Blocks the context needs; none when it is not positive.
    const int64_t need = ctx > 0 ? (ctx - 1) / bs + 1 : 0;
    bool bad = false;
    for (int c = tid; c < p.width && c < need; c += kThreads) {
      const int64_t blk = p.bt[r * p.bt_stride + c];
      bad |= blk < 0 || blk >= p.num_blocks;
    }
    const bool any = __syncthreads_or(bad);
    if (tid == 0) {
      if (ctx <= 0) flags |= MLR_CHECK_CONTEXT;
      if (need > p.width) flags |= MLR_CHECK_WIDTH;
      if (any) flags |= MLR_CHECK_BLOCK;
      if (p.qsl != nullptr) {
        const int64_t len = p.qsl[r + 1] - p.qsl[r];
        if (len <= 0) flags |= MLR_CHECK_QSL_ORDER;
        if (len > p.max_query_len) flags |= MLR_CHECK_QUERY_LEN;
        if (ctx < len) flags |= MLR_CHECK_COVER;
      }
      if (p.detail) {
        int64_t *d = p.out + groups;
        d[r] = p.qsl[r];
        if (r == p.reqs - 1) d[p.reqs] = p.qsl[p.reqs];
        d[p.reqs + 1 + r] = ctx;
        d[2 * p.reqs + 1 + r] = any;
      }
    }
  }
  if (blockIdx.x == 0 && tid == 0 && p.qsl != nullptr) {
    if (p.qsl[0] != 0) flags |= MLR_CHECK_QSL_START;
    if (p.qsl[p.reqs] != p.tokens) flags |= MLR_CHECK_QSL_END;
  }

  // Lane i of every wave holds token first + i; wave 0 checks it, and all four
  // look for its slot among a quarter of the earlier tokens each.
  const int first = blockIdx.x * kTokens, lane = tid % kWave, wave = tid / kWave;
  const int t = first + lane;
  if (first < p.tokens) {  // uniform
    // The request of token u: how many request ends lie at or before it.
    auto owner = [&](int u) -> int {
      if (p.qsl == nullptr) return u;
      int lo = 0, hi = p.reqs;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (p.qsl[mid + 1] <= u) lo = mid + 1;
        else hi = mid;
      }
      return min(lo, p.reqs - 1);
    };
    // Tokens of different phases may share a slot: the phase in the low bit.
    auto key_of = [&](int u) -> int64_t {
      const int64_t slot = p.slots[u];
      return p.decoding == nullptr ? slot : slot * 2 + (p.decoding[owner(u)] != 0);
    };
    int64_t mine = 0;
    unsigned int shift = 0;
    if (t < p.tokens) {
      mine = key_of(t);
      if (p.decoding != nullptr && p.decoding[owner(t)]) shift = MLR_CHECK_DECODE_SHIFT;
    }
    if (wave == 0 && t < p.tokens) {
      const int64_t slot = p.slots[t];
      if (slot < 0 || slot >= p.num_blocks * bs) flags |= MLR_CHECK_SLOT_RANGE;
      if (p.reqs > 0) {
        const int r = owner(t);
        const int64_t start = p.qsl != nullptr ? p.qsl[r] : t;
        const int64_t len = p.qsl != nullptr ? p.qsl[r + 1] - start : 1;
        const int64_t pos = p.positions[t];
        if (pos != p.ctx[r] - len + (t - start)) flags |= MLR_CHECK_POSITION << shift;
        int64_t col = pos >= 0 ? pos / bs : 0;
        col = col > p.width - 1 ? p.width - 1 : col;
        const int64_t in = pos - (pos >= 0 ? pos / bs : -((bs - 1 - pos) / bs)) * bs;
        if (p.width > 0 && slot != p.bt[r * p.bt_stride + col] * bs + in)
          flags |= MLR_CHECK_SLOT << shift;
      }
    }
    bool same = false;
    // Whole workgroups of earlier tokens: no bounds, two keys a read.
    for (int base = 0; base < first; base += kTile) {
      const int n = min(kTile, first - base);  // a multiple of kTokens
      __syncthreads();
      for (int i = tid; i < n; i += kThreads) keys[i] = key_of(base + i);
      __syncthreads();
      const longlong2 *part = reinterpret_cast<const longlong2 *>(keys + wave * (n / 4));
#pragma unroll 8
      for (int i = 0; i < n / 8; ++i) {
        const longlong2 k = part[i];
        same |= k.x == mine || k.y == mine;
      }
    }
    if (wave == 0) {  // its own earlier lanes, through LDS within the wave
      own[lane] = mine;
      __builtin_amdgcn_wave_barrier();
      for (int i = 0; i < kTokens; ++i) same |= i < lane && own[i] == mine;
    }
    if (same && t < p.tokens) flags |= MLR_CHECK_REPEAT << shift;
  }

#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) flags |= __shfl_xor(flags, o);
  if (tid % kWave == 0) wave_flags[tid / kWave] = flags;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kThreads / kWave; ++w) flags |= wave_flags[w];
    p.out[blockIdx.x] = flags;
  }
}

}  // namespace
}  // namespace mlr

using namespace mlr;

extern "C" int64_t mlr_check_step_groups(int64_t num_reqs, int64_t num_tokens) {
  if (num_reqs < 0 || num_tokens < 0 || num_tokens > kMaxTokens || num_reqs >= INT32_MAX) return 0;
  return std::max<int64_t>({1, std::min<int64_t>(num_reqs, kMaxGroups),
                            ceil_div(num_tokens, kTokens)});
}

extern "C" int mlr_check_step(const int64_t *block_tables, int64_t block_table_stride,
                              int64_t max_blocks, const int64_t *context_lens, int64_t num_reqs,
                              const int64_t *query_start_loc, const int64_t *positions,
                              const int64_t *slot_mapping, int64_t num_tokens,
                              const uint8_t *decoding, int64_t block_size, int64_t num_blocks,
                              int64_t max_query_len, int detail, int64_t *out, int64_t out_len,
                              void *stream) {
  clear_error();
  const int64_t groups = mlr_check_step_groups(num_reqs, num_tokens);
  MLR_REQUIRE(groups > 0, "mlr_check_step: more than %lld tokens", (long long)kMaxTokens);
  MLR_REQUIRE(block_size > 0 && num_blocks > 0 && num_blocks <= INT64_MAX / 2 / block_size,
              "mlr_check_step: bad block_size or num_blocks");
  MLR_REQUIRE(max_blocks >= 0 && max_blocks < INT32_MAX && block_table_stride >= max_blocks,
              "mlr_check_step: bad block table width/stride");
  MLR_REQUIRE(num_reqs == 0 || (context_lens && (block_tables || max_blocks == 0)),
              "mlr_check_step: null block_tables or context_lens");
  MLR_REQUIRE(num_tokens == 0 || (slot_mapping && (num_reqs == 0 || positions)),
              "mlr_check_step: null positions or slot_mapping");
  MLR_REQUIRE(query_start_loc || num_tokens == 0 || num_reqs == 0 || num_tokens == num_reqs,
              "mlr_check_step: without query_start_loc every request has one token");
  MLR_REQUIRE(!(decoding && num_reqs == 0) && !(query_start_loc && num_reqs == 0),
              "mlr_check_step: no requests");
  MLR_REQUIRE(!detail || query_start_loc, "mlr_check_step: detail needs query_start_loc");
  MLR_REQUIRE(out && out_len >= groups + (detail ? 3 * num_reqs + 1 : 0),
              "mlr_check_step: out is too small");
  CheckParams p{block_tables, block_table_stride, static_cast<int>(max_blocks), context_lens,
                static_cast<int>(num_reqs), query_start_loc, positions, slot_mapping,
                static_cast<int>(num_tokens), decoding, block_size, num_blocks, max_query_len,
                out, detail};
  check_step<<<static_cast<unsigned>(groups), kThreads, 0, static_cast<hipStream_t>(stream)>>>(p);
  return check_launch("mlr_check_step");
}

extern "C" int mlr_check_step_wait(const int64_t *block_tables, int64_t block_table_stride,
                                   int64_t max_blocks, const int64_t *context_lens,
                                   int64_t num_reqs, const int64_t *query_start_loc,
                                   const int64_t *positions, const int64_t *slot_mapping,
                                   int64_t num_tokens, const uint8_t *decoding,
                                   int64_t block_size, int64_t num_blocks,
                                   int64_t max_query_len, int detail, int64_t *out,
                                   int64_t out_len, void *stream) {
  clear_error();
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone)
    return set_error(MLR_ERR_INVALID, "mlr_check_step_wait: the stream is being captured");
  const int rc = mlr_check_step(block_tables, block_table_stride, max_blocks, context_lens,
                                num_reqs, query_start_loc, positions, slot_mapping, num_tokens,
                                decoding, block_size, num_blocks, max_query_len, detail, out,
                                out_len, stream);
  if (rc != MLR_OK) return rc;
  const hipError_t err = hipStreamSynchronize(s);
  if (err != hipSuccess)
    return set_error(MLR_ERR_HIP, "mlr_check_step_wait: %s", hipGetErrorString(err));
  return MLR_OK;
}
