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
#include <type_traits>

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
  // With the fused norm: x is the layer's delta, normalised after the residual
  // add; rows of at most 2 * 64 16-byte chunks.
  const void *residual;
  int64_t residual_stride;
  void *residual_out;  // [rows, k] contiguous
  const void *norm_weight;
  float norm_factor, norm_eps;
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

// Two values packed to a 16-bit type (round to nearest even) and back.
template <typename T> struct Pair;
template <> struct Pair<bf16_t> {
  __device__ static uint32_t pack(float lo, float hi) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
  }
  __device__ static float lo(uint32_t w) { return __uint_as_float(w << 16); }
  __device__ static float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};
template <> struct Pair<f16_t> {
  __device__ static uint32_t pack(float lo, float hi) {
    return static_cast<uint32_t>(float_to_f16_bits(lo)) |
           (static_cast<uint32_t>(float_to_f16_bits(hi)) << 16);
  }
  __device__ static float lo(uint32_t w) { return f16_bits_to_float(static_cast<uint16_t>(w)); }
  __device__ static float hi(uint32_t w) { return f16_bits_to_float(static_cast<uint16_t>(w >> 16)); }
};

// The gate/up product of a decoder layer's MLP with the residual add and
// RMSNorm before it, in one launch: out = silu(gate) * up of n(r), r =
// residual + x: r and n(r) as mlr_rms_norm gives them, bit for bit, the products
// up to the order of FP32 sums (the gated form deals k to waves by its length).
//
// A decode step of a 0.5B layer spent 4.7 us (and a launch's gap) on the norm
// of 16 rows of 896, which is latency. Here every workgroup normalises all rows
// (28 KB, from L2) into LDS while its weight loads, issued behind those of the
// rows, are on their way; workgroup 0 stores r. 4 kRT waves, four rows each.
// Measured in the 24-layer decode graph, 16 rows, 896 to 2 x 4864, bf16: 10.6 us
// against 4.7 + 8.8 for the two launches and the gap between them; with the
// norm behind the sums of the down projection 1,290 -> 1,203 us per step.
template <typename T, int kRT>
__global__ __launch_bounds__(256 * kRT) void norm_rows_linear_kernel(RowsLinearParams p) {
#pragma clang fp contract(off)
  using E = Elem<T>;
  constexpr int kN = 8, kK = 2, kRows = 4, kWaves = 4 * kRT, kUnroll = 4, kAcc = 2 * kRT;
  struct alignas(16) Chunk {
    T v[kN];
  };
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * kTileN;
  const uint32_t row_bytes = static_cast<uint32_t>(p.k) * 2;
  const uint32_t lds_row = row_bytes + 16;  // rows four banks apart
  const int chunks = p.k / kN;

  // The wave's rows and the norm's weight, requested first.
  Chunk x[kRows][kK], r[kRows][kK], w[kK];
#pragma unroll
  for (int u = 0; u < kRows; ++u) {
    const int row = min(wave * kRows + u, p.rows - 1);
    const T *xr = static_cast<const T *>(p.x) + row * p.x_stride;
    const T *rr = static_cast<const T *>(p.residual) + row * p.residual_stride;
#pragma unroll
    for (int k = 0; k < kK; ++k) {
      const int c = min(lane + kWave * k, chunks - 1);
      x[u][k] = reinterpret_cast<const Chunk *>(xr)[c];
      r[u][k] = reinterpret_cast<const Chunk *>(rr)[c];
    }
  }
#pragma unroll
  for (int k = 0; k < kK; ++k)
    w[k] = static_cast<const Chunk *>(p.norm_weight)[min(lane + kWave * k, chunks - 1)];

  const uint32_t wrows = static_cast<uint32_t>(min(kTileN, p.n - n0));
  __amdgpu_buffer_rsrc_t wr[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
    wr[t] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T *>(static_cast<const T *>(p.w) + (static_cast<int64_t>(t) * p.n + n0) * p.k),
        0, wrows * row_bytes, 0x00020000);
  const uint32_t w_lane = m < static_cast<int>(wrows) ? m * row_bytes : kOutside;
  const int blocks = (row_bytes + kBlockBytes - 1) / kBlockBytes;
  uint4 wv[kUnroll][2][2];
  auto load_w = [&](int kb0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t at =
            static_cast<uint32_t>(kb0 + u * kWaves) * kBlockBytes + 64u * j + 16u * g;
        const bool in = at < row_bytes && w_lane != kOutside;
#pragma unroll
        for (int t = 0; t < 2; ++t) wv[u][t][j] = load16(wr[t], in ? w_lane + at : kOutside);
      }
  };
  __builtin_amdgcn_sched_barrier(0);
  load_w(wave);
  __builtin_amdgcn_sched_barrier(0);

  // The four norms, in the order of mlr_rms_norm: a lane's chunks, then the
  // wave's butterfly. Roundings go two at a time through the packed hardware
  // conversion (12 instructions per element; with the bit-wise one 40, and
  // 13.9 us per call instead of 10.6), which gives a NaN other bits: only
  // the stored r needs the canonical ones.
  using P = Pair<T>;
#pragma unroll
  for (int u = 0; u < kRows; ++u) {
    const int row = wave * kRows + u;
    uint32_t rp[kK][4];
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < kK; ++k) {
      const uint4 xb = __builtin_bit_cast(uint4, x[u][k]), rb = __builtin_bit_cast(uint4, r[u][k]);
      const uint32_t xw[4] = {xb.x, xb.y, xb.z, xb.w}, rw[4] = {rb.x, rb.y, rb.z, rb.w};
      const bool in = lane + kWave * k < chunks;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        rp[k][e] = P::pack(P::lo(rw[e]) + P::lo(xw[e]), P::hi(rw[e]) + P::hi(xw[e]));
        const float f0 = P::lo(rp[k][e]), f1 = P::hi(rp[k][e]);
        if (in) {
          sum += f0 * f0;
          sum += f1 * f1;
        }
      }
    }
    sum = wave_sum(sum);
    const float inv = rsqrtf(sum * p.norm_factor + p.norm_eps);
#pragma unroll
    for (int k = 0; k < kK; ++k) {
      const int c = lane + kWave * k;
      if (c >= chunks) continue;
      const uint4 wb = __builtin_bit_cast(uint4, w[k]);
      const uint32_t ww[4] = {wb.x, wb.y, wb.z, wb.w};
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float f0 = P::lo(rp[k][e]) * inv, f1 = P::hi(rp[k][e]) * inv;
        // The FP32 rounding of the product stays, as in mlr_rms_norm.
        if constexpr (std::is_same<T, f16_t>::value) asm volatile("" : "+v"(f0), "+v"(f1));
        const uint32_t nv = P::pack(f0, f1);
        o[e] = P::pack(P::lo(ww[e]) * P::lo(nv), P::hi(ww[e]) * P::hi(nv));
      }
      *reinterpret_cast<uint4 *>(smem + row * lds_row + 16 * c) = make_uint4(o[0], o[1], o[2], o[3]);
      if (blockIdx.x == 0 && row < p.rows) {
        Chunk keep;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          keep.v[2 * e] = E::from_f32(P::lo(rp[k][e]));
          keep.v[2 * e + 1] = E::from_f32(P::hi(rp[k][e]));
        }
        reinterpret_cast<Chunk *>(static_cast<T *>(p.residual_out) +
                                  static_cast<int64_t>(row) * p.k)[c] = keep;
      }
    }
  }
  // lgkmcnt(0) and a barrier: the LDS rows are there, the weight loads may
  // still be in flight.
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();

  f32x4_t acc[kAcc];
#pragma unroll
  for (int a = 0; a < kAcc; ++a) acc[a] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int kb0 = wave; kb0 < blocks; kb0 += kWaves * kUnroll) {
    if (kb0 != wave) {
      load_w(kb0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) {
        uint4 xv[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          // A chunk past the row meets weights that are zero: chunk 0 stands in.
          const uint32_t at =
              static_cast<uint32_t>(kb0 + u * kWaves) * kBlockBytes + 64u * j + 16u * g;
          xv[j] = *reinterpret_cast<const uint4 *>(smem + (16 * rt + m) * lds_row +
                                                   (at < row_bytes ? at : 0u));
          if (at >= row_bytes) xv[j] = make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[t * kRT + rt] = mma_block<T>(wv[u][t], xv, acc[t * kRT + rt]);
      }
    }
  }
  __syncthreads();  // the rows' LDS becomes the waves' sums
  f32x4_t *red = reinterpret_cast<f32x4_t *>(smem);
#pragma unroll
  for (int a = 0; a < kAcc; ++a) red[(wave * kAcc + a) * 64 + lane] = acc[a];
  __syncthreads();
  const float *flat = reinterpret_cast<const float *>(red);
  for (int e = threadIdx.x; e < kRT * 256; e += 64 * kWaves) {
    const int row = e >> 4, c = e & 15;
    if (row >= p.rows || n0 + c >= p.n) continue;
    const int rt = row >> 4;
    const int at = ((c >> 2) * 16 + (row & 15)) * 4 + (c & 3);
    float v[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float s = 0.f;
#pragma unroll
      for (int ww = 0; ww < kWaves; ++ww) s += flat[(ww * kAcc + t * kRT + rt) * 256 + at];
      v[t] = s;
    }
    static_cast<T *>(p.out)[row * p.out_stride + n0 + c] =
        silu_mul_elem<T>(E::from_f32(v[0]), E::from_f32(v[1]));
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
  if (rc != MLR_OK || p.splits == 1 || p.out == nullptr) return rc;
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
  // Without `out` a split product stops at its workgroups' sums.
  const bool sums_only = out == nullptr && dtype_size(dtype) > 0 &&
                         mlr_rows_linear_workspace_size(rows, n, k, gated, dtype) > 0;
  MLR_REQUIRE(x && weight && (out || sums_only), "mlr_rows_linear: null x, weight or out");
  MLR_REQUIRE(!(sums_only && bias), "mlr_rows_linear: sums take no bias");
  MLR_REQUIRE(!(gated && bias), "mlr_rows_linear: the gated form takes no bias");
  MLR_REQUIRE(dtype == MLR_DTYPE_BF16 || dtype == MLR_DTYPE_F16 || dtype == MLR_DTYPE_F32,
              "mlr_rows_linear: dtype %d not supported (bf16, fp16, fp32)", dtype);
  MLR_REQUIRE(x_stride >= k && (sums_only || out_stride >= n), "mlr_rows_linear: a row stride is too small");
  const int64_t size = dtype_size(dtype);
  // 16-byte loads; a tile's rows and all rows of x under 32-bit offsets.
  MLR_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight)) & 15u) == 0 &&
                  k * size % 16 == 0 && x_stride * size % 16 == 0,
              "mlr_rows_linear: x and weight rows must be 16-byte aligned");
  MLR_REQUIRE(k < (int64_t(1) << 24) && n < (int64_t(1) << 30) &&
                  x_stride < (int64_t(1) << 22),
              "mlr_rows_linear: k, n or the row stride is too large");
  RowsLinearParams p{};
  p.x = x;
  p.x_stride = x_stride;
  p.w = weight;
  p.bias = bias;
  p.out = out;
  p.out_stride = out_stride;
  p.rows = static_cast<int>(rows);
  p.n = static_cast<int>(n);
  p.k = static_cast<int>(k);
  p.splits = splits_of(n, k, size, gated != 0);
  p.partial = static_cast<float *>(workspace);
  if (workspace_bytes < mlr_rows_linear_workspace_size(rows, n, k, gated, dtype))
    return set_error(MLR_ERR_WORKSPACE, "mlr_rows_linear: workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MLR_DTYPE_BF16) return launch_type<bf16_t>(p, gated != 0, s);
  if (dtype == MLR_DTYPE_F16) return launch_type<f16_t>(p, gated != 0, s);
  return launch_type<float>(p, gated != 0, s);
}

extern "C" int mlr_norm_rows_linear(const void *x, int64_t x_stride, const void *residual,
                                    int64_t residual_stride, void *residual_out,
                                    const void *norm_weight, double eps, const void *weight,
                                    void *out, int64_t out_stride, int64_t rows, int64_t n,
                                    int64_t k, int dtype, void *stream) {
  clear_error();
  MLR_REQUIRE(rows >= 0 && rows <= 32, "mlr_norm_rows_linear: rows must be in [0, 32]");
  MLR_REQUIRE(n > 0 && n < (int64_t(1) << 30), "mlr_norm_rows_linear: bad n");
  MLR_REQUIRE(k > 0 && k <= 1024 && k % 8 == 0,
              "mlr_norm_rows_linear: k must be a multiple of 8 up to 1024");
  MLR_REQUIRE(rows <= 16 || k <= 1008, "mlr_norm_rows_linear: the rows pass 64 KB of LDS");
  MLR_REQUIRE(dtype == MLR_DTYPE_BF16 || dtype == MLR_DTYPE_F16,
              "mlr_norm_rows_linear: bf16 or fp16 only");
  MLR_REQUIRE(eps > 0, "mlr_norm_rows_linear: eps must be > 0");
  if (rows == 0) return MLR_OK;
  MLR_REQUIRE(x && residual && residual_out && norm_weight && weight && out,
              "mlr_norm_rows_linear: null pointer argument");
  MLR_REQUIRE(residual_out != residual && residual_out != x,
              "mlr_norm_rows_linear: residual_out must be a buffer of its own");
  MLR_REQUIRE(x_stride >= k && residual_stride >= k && out_stride >= n && x_stride % 8 == 0 &&
                  residual_stride % 8 == 0,
              "mlr_norm_rows_linear: bad row stride");
  MLR_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(residual) |
                reinterpret_cast<uintptr_t>(residual_out) |
                reinterpret_cast<uintptr_t>(norm_weight) |
                reinterpret_cast<uintptr_t>(weight)) & 15u) == 0,
              "mlr_norm_rows_linear: operands must be 16-byte aligned");
  RowsLinearParams p{};
  p.x = x;
  p.x_stride = x_stride;
  p.w = weight;
  p.out = out;
  p.out_stride = out_stride;
  p.rows = static_cast<int>(rows);
  p.n = static_cast<int>(n);
  p.k = static_cast<int>(k);
  p.residual = residual;
  p.residual_stride = residual_stride;
  p.residual_out = residual_out;
  p.norm_weight = norm_weight;
  // The scale torch's mean applies, as mlr_rms_norm takes it.
  p.norm_factor = static_cast<float>(rows) / static_cast<float>(rows * k);
  p.norm_eps = static_cast<float>(eps);
  p.splits = 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned grid = static_cast<unsigned>(ceil_div(n, kTileN));
  auto run = [&](auto tag, auto rt) {
    using T = decltype(tag);
    constexpr int kRT = decltype(rt)::value;
    const size_t rows_lds = static_cast<size_t>(16 * kRT) * (k * 2 + 16);
    const size_t sums_lds = static_cast<size_t>(4 * kRT) * 2 * kRT * 64 * sizeof(f32x4_t);
    norm_rows_linear_kernel<T, kRT>
        <<<grid, 256 * kRT, std::max(rows_lds, sums_lds), s>>>(p);
    return check_launch("mlr_norm_rows_linear");
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if (dtype == MLR_DTYPE_BF16) return rows <= 16 ? run(bf16_t{}, One{}) : run(bf16_t{}, Two{});
  return rows <= 16 ? run(f16_t{}, One{}) : run(f16_t{}, Two{});
}
