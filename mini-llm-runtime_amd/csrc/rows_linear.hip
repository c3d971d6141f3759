// Linear layers over a few rows (a decode step's projections) on the matrix
// cores: out[r, n] = sum_k x[r, k] * w[n, k] (+ bias[n]), and the same for a
// stacked gate/up weight with silu(gate) * up in the epilogue.
//
// With at most 32 rows the product is a read of the weight: its floor is the
// weight's bytes, 2 to 17 MB at the layer sizes of a 0.5B model, a few us.
// What a call spends beyond that is latency: the round trip of its loads,
// the launch, and the chain of a long k loop in too few wavefronts. So every
// workgroup takes 16 output columns (a gate/up pair: the same 16 of both) and
// its waves deal the k blocks round-robin, each wave issuing the loads of
// kUnroll blocks before it computes any; there is no LDS staging, as no
// weight byte is used twice by one wave. A k block is 128 bytes of each row:
// lane l takes row l%16, bytes [64 j + 16 (l/16), +16), j < 2, so its four lanes
// cover one whole cache line. The lane's two 16-byte chunks are the A
// operands of two 16x16x32 MFMAs (bf16, fp16) or of eight 16x16x4 ones (FP32):
// the k order inside a block differs from memory order the same way for w
// and x, which a sum over k does not see. x goes through the same loads (it
// stays in L2: a few rows). The waves' FP32 sums are added in wave order
// through LDS, so a row's result does not depend on the other rows.
//
// Measured (graphs, weights from HBM, 16 rows, bf16; GEMM library before):
// 896 columns of k 896 4.0 us (5.4), of k 4864 7.7 us (17.1; 12.2 in one
// workgroup per tile, 14.1 before every load of a batch left first), gate/up
// 4864 of k 896 with silu 8.4 us (11.3 as GEMM and silu_mul), gate/up 8960 of
// k 1536 16.7 us (42), 3.3 TB/s. FP32: 5.6 (7.4), 10.3 (15.1), 13.5 (15.2).
//
// All loads go through buffer resources that end with the tile's rows; lanes
// past the last row or the last k ask for an offset beyond them and get zeros.
//
// Rounding: FP32 accumulation, bias added in FP32, one rounding to the
// element type, as the GEMM library's epilogue does; the gated form rounds
// gate and up to the element type first and then follows mlr_silu_mul.
#include <algorithm>

#include "mlr_common.h"
#include "silu.h"

namespace mlr {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kMaxSplits = 4;
constexpr int kTileN = 16;         // output columns per workgroup
constexpr int kBlockBytes = 128;   // bytes of a row per k block
constexpr uint32_t kOutside = 0x7fffffffu;  // an offset past every resource

struct RowsLinearParams {
  const void *x;
  int64_t x_stride;  // elements
  const void *w;     // [n or 2n, k] contiguous
  const void *bias;  // [n] or null
  void *out;
  int64_t out_stride;
  int rows, n, k;
  int splits;      // workgroups that share a tile's k blocks
  float *partial;  // [splits][rows][n] FP32 sums when splits > 1
};

// One lane's share of a k block: 32 bytes of w and of x.
template <typename T>
__device__ __forceinline__ f32x4_t mma_block(const uint4 (&w)[2], const uint4 (&x)[2], f32x4_t c);
template <>
__device__ __forceinline__ f32x4_t mma_block<bf16_t>(const uint4 (&w)[2], const uint4 (&x)[2],
                                                     f32x4_t c) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[j]),
                                                __builtin_bit_cast(bf16x8_t, x[j]), c, 0, 0, 0);
  return c;
}
template <>
__device__ __forceinline__ f32x4_t mma_block<f16_t>(const uint4 (&w)[2], const uint4 (&x)[2],
                                                    f32x4_t c) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, w[j]),
                                               __builtin_bit_cast(f16x8_t, x[j]), c, 0, 0, 0);
  return c;
}
template <>
__device__ __forceinline__ f32x4_t mma_block<float>(const uint4 (&w)[2], const uint4 (&x)[2],
                                                    f32x4_t c) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const f32x4_t a = __builtin_bit_cast(f32x4_t, w[j]), b = __builtin_bit_cast(f32x4_t, x[j]);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
  }
  return c;
}

__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// kRT row tiles of 16; kG weight tiles (2: gate and up).
template <typename T, int kRT, int kG, int kUnroll, int kMaxWaves>
__global__ __launch_bounds__(64 * kMaxWaves) void rows_linear_kernel(RowsLinearParams p) {
  using E = Elem<T>;
  constexpr int kSize = static_cast<int>(sizeof(T));
  constexpr int kAcc = kRT * kG;
  extern __shared__ __align__(16) f32x4_t red[];  // [waves][kAcc][64]
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * kTileN;
  const uint32_t row_bytes = static_cast<uint32_t>(p.k) * kSize;
  const uint32_t wrows = static_cast<uint32_t>(min(kTileN, p.n - n0));
  __amdgpu_buffer_rsrc_t wr[kG];
#pragma unroll
  for (int t = 0; t < kG; ++t)
    wr[t] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T *>(static_cast<const T *>(p.w) + (static_cast<int64_t>(t) * p.n + n0) * p.k),
        0, wrows * row_bytes, 0x00020000);
  const uint32_t xrow_bytes = static_cast<uint32_t>(p.x_stride) * kSize;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void *>(p.x), 0, static_cast<uint32_t>(p.rows - 1) * xrow_bytes + row_bytes,
      0x00020000);
  const uint32_t w_lane = m < static_cast<int>(wrows) ? m * row_bytes : kOutside;

  f32x4_t acc[kAcc];
#pragma unroll
  for (int a = 0; a < kAcc; ++a) acc[a] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int blocks = (row_bytes + kBlockBytes - 1) / kBlockBytes;
  // This workgroup's k blocks: [lo, hi).
  const int per = (blocks + p.splits - 1) / p.splits;
  const int lo = blockIdx.y * per, hi = min(blocks, lo + per);
  for (int kb0 = lo + wave; kb0 < hi; kb0 += waves * kUnroll) {
    uint4 wv[kUnroll][kG][2], xv[kUnroll][kRT][2];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int kb = kb0 + u * waves;
        const uint32_t at = static_cast<uint32_t>(kb) * kBlockBytes + 64u * j + 16u * g;
        const bool in = kb < hi && at < row_bytes;
#pragma unroll
        for (int t = 0; t < kG; ++t)
          wv[u][t][j] = load16(wr[t], in && w_lane != kOutside ? w_lane + at : kOutside);
#pragma unroll
        for (int t = 0; t < kRT; ++t) {
          const int row = 16 * t + m;
          xv[u][t][j] = load16(xr, in && row < p.rows ? row * xrow_bytes + at : kOutside);
        }
      }
    // Every load of the batch leaves before the first MFMA waits: left to
    // itself the compiler keeps five loads in flight to save registers.
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
#pragma unroll
      for (int t = 0; t < kG; ++t)
#pragma unroll
        for (int r = 0; r < kRT; ++r)
          acc[t * kRT + r] = mma_block<T>(wv[u][t], xv[u][r], acc[t * kRT + r]);
  }
  // Lane l of accumulator (t, r) holds columns n0 + 4g + i of row 16 r + m.
#pragma unroll
  for (int a = 0; a < kAcc; ++a) red[(wave * kAcc + a) * 64 + lane] = acc[a];
  __syncthreads();
  // Thread (r, c) of the tile: column c fastest, so a row's 16 outputs are
  // stored together.
  const float *flat = reinterpret_cast<const float *>(red);
  for (int e = threadIdx.x; e < kRT * 256; e += blockDim.x) {
    const int row = e >> 4, c = e & 15;
    if (row >= p.rows || n0 + c >= p.n) continue;
    const int r = row >> 4;
    const int at = ((c >> 2) * 16 + (row & 15)) * 4 + (c & 3);
    float v[kG];
#pragma unroll
    for (int t = 0; t < kG; ++t) {
      float s = 0.f;
      for (int w = 0; w < waves; ++w) s += flat[(w * kAcc + t * kRT + r) * 256 + at];
      v[t] = s;
    }
    if (kG == 1 && p.splits > 1) {  // uniform
      p.partial[(static_cast<int64_t>(blockIdx.y) * p.rows + row) * p.n + n0 + c] = v[0];
      continue;
    }
    T *dst = static_cast<T *>(p.out) + row * p.out_stride + n0 + c;
    if constexpr (kG == 2) {
      *dst = silu_mul_elem<T>(E::from_f32(v[0]), E::from_f32(v[1]));
    } else {
      if (p.bias != nullptr) v[0] += E::to_f32(static_cast<const T *>(p.bias)[n0 + c]);
      *dst = E::from_f32(v[0]);
    }
  }
}

// The splits' sums of one (row, column), added in split order.
template <typename T>
__global__ __launch_bounds__(256) void rows_linear_reduce(RowsLinearParams p) {
  using E = Elem<T>;
  const int c = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;
  if (c >= p.n) return;
  const float *src = p.partial + static_cast<int64_t>(row) * p.n + c;
  const int64_t step = static_cast<int64_t>(p.rows) * p.n;
  float v[kMaxSplits];
#pragma unroll
  for (int s = 0; s < kMaxSplits; ++s) v[s] = s < p.splits ? src[s * step] : 0.f;
  float sum = v[0];
#pragma unroll
  for (int s = 1; s < kMaxSplits; ++s)
    if (s < p.splits) sum += v[s];
  if (p.bias != nullptr) sum += E::to_f32(static_cast<const T *>(p.bias)[c]);
  static_cast<T *>(p.out)[row * p.out_stride + c] = E::from_f32(sum);
}

// Workgroups that share a tile's k blocks. A tile's k loop is one batch of
// loads while 16 waves of four blocks cover it; a longer one in few tiles
// leaves most CUs idle (896 columns are 56 workgroups), so its blocks are
// dealt to about one workgroup per CU and a second kernel adds the sums.
int splits_of(int64_t n, int64_t k, int64_t size, bool gated) {
  const int64_t blocks = ceil_div(k * size, kBlockBytes), tiles = ceil_div(n, kTileN);
  if (gated || blocks <= 64 || tiles >= 192) return 1;
  return static_cast<int>(std::min<int64_t>(kMaxSplits, ceil_div(256, tiles)));
}

template <typename T, int kRT, int kG, int kUnroll>
int launch_rows(const RowsLinearParams &p, hipStream_t stream) {
  // Waves: enough for each to issue all its k blocks at once, up to 16 (8
  // where 16 waves' accumulators would pass 64 KB of LDS).
  const int64_t blocks = ceil_div(static_cast<int64_t>(p.k) * sizeof(T), kBlockBytes);
  constexpr int kMax = kRT > 1 ? 8 : 16;
  const int waves = static_cast<int>(
      std::min<int64_t>(kMax, ceil_div(ceil_div(blocks, p.splits), kUnroll)));
  const size_t lds = static_cast<size_t>(waves) * kRT * kG * 64 * sizeof(f32x4_t);
  const dim3 grid(static_cast<unsigned>(ceil_div(p.n, kTileN)), p.splits);
  rows_linear_kernel<T, kRT, kG, kUnroll, kMax><<<grid, 64 * waves, lds, stream>>>(p);
  const int rc = check_launch("mlr_rows_linear");
  if (rc != MLR_OK || p.splits == 1) return rc;
  rows_linear_reduce<T><<<dim3(static_cast<unsigned>(ceil_div(p.n, 256)), p.rows), 256, 0,
                          stream>>>(p);
  return check_launch("mlr_rows_linear(reduce)");
}

template <typename T, int kG>
int launch_tiles(const RowsLinearParams &p, hipStream_t stream) {
  if (p.rows <= 16) return launch_rows<T, 1, kG, 4>(p, stream);
  return launch_rows<T, 2, kG, 3>(p, stream);
}

template <typename T>
int launch_type(const RowsLinearParams &p, bool gated, hipStream_t stream) {
  return gated ? launch_tiles<T, 2>(p, stream) : launch_tiles<T, 1>(p, stream);
}

}  // namespace
}  // namespace mlr

using namespace mlr;

extern "C" size_t mlr_rows_linear_workspace_size(int64_t rows, int64_t n, int64_t k, int gated,
                                                 int dtype) {
  const int64_t size = dtype_size(dtype);
  if (rows <= 0 || n <= 0 || k <= 0 || size == 0) return 0;
  const int splits = splits_of(n, k, size, gated != 0);
  return splits > 1 ? static_cast<size_t>(splits) * rows * n * sizeof(float) : 0;
}

extern "C" int mlr_rows_linear(const void *x, int64_t x_stride, const void *weight,
                               const void *bias, void *out, int64_t out_stride, int64_t rows,
                               int64_t n, int64_t k, int gated, int dtype, void *workspace,
                               size_t workspace_bytes, void *stream) {
  clear_error();
  MLR_REQUIRE(rows >= 0 && rows <= 32, "mlr_rows_linear: rows must be in [0, 32]");
  MLR_REQUIRE(n > 0 && k > 0, "mlr_rows_linear: n and k must be > 0");
  if (rows == 0) return MLR_OK;
  MLR_REQUIRE(x && weight && out, "mlr_rows_linear: null x, weight or out");
  MLR_REQUIRE(!(gated && bias), "mlr_rows_linear: the gated form takes no bias");
  MLR_REQUIRE(dtype == MLR_DTYPE_BF16 || dtype == MLR_DTYPE_F16 || dtype == MLR_DTYPE_F32,
              "mlr_rows_linear: dtype %d not supported (bf16, fp16, fp32)", dtype);
  MLR_REQUIRE(x_stride >= k && out_stride >= n, "mlr_rows_linear: a row stride is too small");
  const int64_t size = dtype_size(dtype);
  // 16-byte loads; a tile's rows and all rows of x under 32-bit offsets.
  MLR_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight)) & 15u) == 0 &&
                  k * size % 16 == 0 && x_stride * size % 16 == 0,
              "mlr_rows_linear: x and weight rows must be 16-byte aligned");
  MLR_REQUIRE(k < (int64_t(1) << 24) && n < (int64_t(1) << 30) &&
                  x_stride < (int64_t(1) << 22),
              "mlr_rows_linear: k, n or the row stride is too large");
  RowsLinearParams p{x, x_stride, weight, bias, out, out_stride, static_cast<int>(rows),
                     static_cast<int>(n), static_cast<int>(k),
                     splits_of(n, k, size, gated != 0), static_cast<float *>(workspace)};
  if (workspace_bytes < mlr_rows_linear_workspace_size(rows, n, k, gated, dtype))
    return set_error(MLR_ERR_WORKSPACE, "mlr_rows_linear: workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MLR_DTYPE_BF16) return launch_type<bf16_t>(p, gated != 0, s);
  if (dtype == MLR_DTYPE_F16) return launch_type<f16_t>(p, gated != 0, s);
  return launch_type<float>(p, gated != 0, s);
}
