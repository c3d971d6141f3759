// FP32 paged chunk prefill on gfx950 matrix cores (v_mfma_f32_32x32x2_f32).
//
// One workgroup = 32 queries of one query head; its waves deal the 32-key
// tiles of the context round-robin and merge their (m, l, O) through LDS at
// the end. Per wave and tile:
//   S^T[32 keys x 32 queries] = K[32 keys x D] . Q^T[D x 32 queries], D/2
//     MFMAs. Lane l holds K row l%32 and Q row l%32, floats 8j + 4(l/32) ..
//     +4 of 8-float block j (one 16-byte load each): MFMA e of block j takes
//     element e of both, so the k pairs of an MFMA lie 4 floats apart in K and
//     Q alike. Q is loaded once, at head sizes 64 and 128 pre-multiplied by
//     scale*log2(e) (see below for the others).
//   Lane l then holds the scores of query l%32 and keys 8(i/4) + 4(l/32) + i%4,
//     i < 16: the row max is 15 maxima and one swap with lane l^32; row sums
//     stay per lane until the end. Online softmax in FP32, base 2.
//   O^T[32 dims x 32 queries] += V^T[32 dims x 2 keys] . P^T[2 keys x 32
//     queries], 16 steps for each of D/32 accumulators: step i takes the two
//     keys whose probabilities lanes l and l^32 hold in register i. Dim m of
//     accumulator c is dim VC*m + c (VC = D/32), so lane l loads VC
//     consecutive floats of a V row.
//
// What bounds it: the FP32 matrix cores (152 TFLOP/s by a large product), if
// the loads arrive in time. K and V of a tile are 16 KB (D = 64) for 8192
// matrix-core cycles, so each wave reads them straight from L2 without LDS.
// There is one buffer of each: the next tile's K is requested once this
// tile's S^T has read K, and lands during the softmax and P.V; the next V
// once P.V has read V, and lands during S^T. Block ids come 32 tiles at a
// time, one per lane, so no load waits for a table lookup. The kernel before
// this one (16 queries a wave, one 16-key block in flight behind a block id
// load each) took 256 us for 4 sequences of 100..700 queries on prefixes up
// to 1,500, 14/2 heads of 64 (36 TFLOP/s); this one takes 117 us (78 TFLOP/s), and 8
// x 512 queries after 2,000 keys 454 and 334 us (99 TFLOP/s).
//
// K rows past the last key the workgroup needs are read as that key's row and
// masked, V rows past it as zeros. Of an out-of-range block, V rows are zeros and
// pool row 0 stands in for K, masked: it may hold anything, no score of it is
// used. Head sizes other than 64 and 128 (multiples of 4 up to 128) run in the
// kernel of 32, 64 or 128 dims that holds them, with the dims past the head as
// zeros, each score in four chains, and q unscaled (the score is scaled instead).
//
// A V row that is not finite reaches the queries that see its key and no other,
// though a masked key is in the MFMAs with probability 0: see the mask and the
// loop after the tiles. Looking for one costs a masked tile 16 D / 32 multiply-adds;
// no measurable time at 64 and 128 (4 x 300 tokens, 28/4 heads of 128, 52.1 and
// 52.7 us), 8-10% at padded sizes, whose registers are full (3 chunks, 10/2 heads of
// 80, 131 and 144 us).
//
// Numerics: FP32 products and sums throughout (the reference's FP32 path,
// kernels/reference/paged_attention.py:346-434); the scale is folded into q
// (one FP32 rounding) at the unpadded head sizes. The reference's tile_size only orders its FP32
// accumulation, as the tiles and waves here do.
//
// Work: items are (sequence, 32-query tile) pairs, each run once per query
// head. Workgroup b goes to XCD b mod 8 (the dispatcher deals workgroups to
// the XCDs in turn), and the query heads of one item get workgroups of one
// residue mod 8, so the K/V rows a GQA group re-reads come from one L2.
// Items start with the most keys first: ranked by every workgroup where there
// are at most 256 of several sequences, else last query tile first.
#include "paged_prefill.h"

namespace mlr {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr float kLog2eF32 = 1.4426950408889634f;
constexpr int kBMF = 32;   // queries per workgroup
constexpr int kBNF = 32;   // keys per tile
// Work items ranked by their keys: at most kRankMax of them, and only where
// contexts pass kRankKeys keys (the ranking takes 3 us: 25 us against 22 for
// 4 x 300 tokens, but 117 against 173 for 4 ragged chunks on ragged prefixes).
constexpr int kRankMax = 256;
constexpr int kRankKeys = 512;

template <int VC> struct VecOf { typedef float type __attribute__((ext_vector_type(VC))); };
template <> struct VecOf<1> { typedef float type; };

__device__ __forceinline__ float other_half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x),
                                                  false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// kWaves waves per workgroup.
template <int D, int kWaves, bool kPad>
__global__ __launch_bounds__(64 * kWaves) void prefill_f32_mfma(PrefillParams p) {
  constexpr int QK = D / 8;   // 8-float blocks of a row
  constexpr int VC = D / 32;  // dims per lane and V row; O^T accumulators
  typedef typename VecOf<VC>::type vec_t;
  const int nqt = p.n_qtiles;
  const int nitems = p.num_seqs * nqt;
  const int b = static_cast<int>(blockIdx.x);
  const int tb = b >> 3;
  const int h = tb % p.hq;
  const int rank = (tb / p.hq) * 8 + (b & 7);
  if (rank >= nitems) return;  // uniform: the grid is padded to whole groups of 8
  int seq = rank % p.num_seqs, qt = nqt - 1 - rank / p.num_seqs;
  if (kWaves >= 4 && p.num_seqs > 1 && nitems <= kRankMax &&
      p.max_blocks * p.block_size > kRankKeys) {  // uniform
    // The item with `rank` items of more keys (ties by index).
    __shared__ __align__(16) int keys_s[kRankMax];
    __shared__ int item_s;
    const int i = threadIdx.x;
    int mine = 0;
    if (i < kRankMax) {
      if (i < nitems) {
        const SeqRange r = seq_range(p, i / nqt);
        const int64_t lo = static_cast<int64_t>(i % nqt) * kBMF;
        mine = lo < r.qlen ? static_cast<int>(r.prefix + min<int64_t>(r.qlen, lo + kBMF)) : 0;
      }
      keys_s[i] = mine;
    }
    __syncthreads();
    if (i < nitems) {
      int above = 0;
      for (int j = 0; j < nitems; j += 4) {
        const int4 o = *reinterpret_cast<const int4 *>(keys_s + j);
        above += (o.x > mine || (o.x == mine && j < i)) + (o.y > mine || (o.y == mine && j + 1 < i)) +
                 (o.z > mine || (o.z == mine && j + 2 < i)) +
                 (o.w > mine || (o.w == mine && j + 3 < i));
      }
      if (above == rank) item_s = i;
    }
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(item_s);
    seq = item / nqt;
    qt = item % nqt;
  }
  const int q0 = qt * kBMF;
  const SeqRange rg = seq_range(p, seq);
  const int qlen = static_cast<int>(rg.qlen);
  if (q0 >= qlen) return;  // uniform
  const int prefix = static_cast<int>(rg.prefix);
  const int kvh = h / p.group;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 31, half = lane >> 5;
  const int d = kPad ? p.d : D;

  // Q^T fragments of query q0 + m (zeros past the chunk and past the head).
  const int qi = q0 + m;
  const bool q_ok = qi < qlen;
  // The score's factor, positive. With kPad it is kept in two floats and applied
  // to the score, so the exponent is rounded once and not by c2 and the product
  // too.
  const double c64 = p.scale * 1.4426950408889634;
  const float c2 = kPad ? static_cast<float>(c64) : static_cast<float>(p.scale) * kLog2eF32;
  const float c2_lo = kPad ? static_cast<float>(c64 - c2) : 0.f;
  f32x4_t qf[QK];
  {
    const float *qrow = static_cast<const float *>(p.q) +
                        (rg.q0 + (q_ok ? qi : q0)) * p.q_st + static_cast<int64_t>(h) * p.q_sh;
#pragma unroll
    for (int j = 0; j < QK; ++j) {
      const int e = 8 * j + 4 * half;
      const f32x4_t v = *reinterpret_cast<const f32x4_t *>(qrow + (kPad && e >= d ? 0 : e));
      qf[j] = q_ok && !(kPad && e >= d) ? (kPad ? v : v * c2) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }
  // Keys the workgroup needs: up to its last query's position.
  const int kv_end = prefix + min(qlen, q0 + kBMF);
  const int ntiles = (kv_end + kBNF - 1) / kBNF;
  const int qpos = prefix + qi;
  const int first_masked = prefix + q0;  // tiles ending at or before it see no mask
  const int bs_log2 = p.bs_log2;
  const int bs_mask = (1 << bs_log2) - 1;
  const int64_t row_elems = static_cast<int64_t>(p.hkv) * d;
  const uint32_t row_bytes = static_cast<uint32_t>(p.hkv) * d * 4;
  // Lane offsets inside a span: K row m%16 (with 64-bit bases: a tile's rows lie
  // in two spans), V row 4 half and the lane's dims.
  const uint32_t k_lane = 16u * half;
  const uint32_t v_lane = 4u * half * row_bytes + 4u * (kPad && VC * m >= d ? 0 : VC * m);
  const float *kc = static_cast<const float *>(p.kc) + static_cast<int64_t>(kvh) * d;
  const float *vc = static_cast<const float *>(p.vc) + static_cast<int64_t>(kvh) * d;
  const int64_t *bt_row = p.bt + static_cast<int64_t>(seq) * p.bt_stride;

  f32x16_t acc[VC];
#pragma unroll
  for (int c = 0; c < VC; ++c) acc[c] = f32x16_t{};
  float m_run = -INFINITY, l_run = 0.f;

  // The wave's tiles are wave, wave + kWaves, ...; lane 2u + s holds the block
  // id of span s (16 keys) of its tile kb + u, kb a multiple of 32 (-1: out of
  // range; spans past the last key repeat its block).
  int64_t ids = 0;
  auto load_ids = [&](int kb) __attribute__((always_inline)) {
    const int64_t key =
        static_cast<int64_t>(wave + kWaves * (kb + (lane >> 1))) * kBNF + 16 * (lane & 1);
    const int64_t id = bt_row[(key < kv_end ? static_cast<int>(key) : kv_end - 1) >> bs_log2];
    ids = id >= 0 && id < p.num_blocks ? id : -1;
  };
  struct TileAt {
    int64_t slot[2];  // first row of each span in the pool (0 when bad)
    int last[2];      // its last row that the workgroup needs
    bool bad[2];
    uint32_t vbytes[2];  // bytes of its V rows under a buffer resource (0 when bad)
  };
  auto tile_at = [&](int k) __attribute__((always_inline)) -> TileAt {
    TileAt t;
    const int key0 = (wave + kWaves * k) * kBNF;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int src = 2 * (k & 31) + s;
      const int64_t id = static_cast<int64_t>(
          static_cast<uint64_t>(static_cast<uint32_t>(
              __builtin_amdgcn_readlane(static_cast<int>(ids), src))) |
          (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(
               static_cast<int>(ids >> 32), src)))
           << 32));
      // A span wholly past the last key re-reads that key's row.
      const int key = min(key0 + 16 * s, kv_end - 1);
      t.bad[s] = id < 0;
      t.slot[s] = ((id < 0 ? 0 : id) << bs_log2) + (id < 0 ? 0 : key & bs_mask);
      t.last[s] = id < 0 ? 0 : min(15, kv_end - 1 - key);
      t.vbytes[s] = id < 0 ? 0u : static_cast<uint32_t>(t.last[s]) * row_bytes + 4u * d;
    }
    return t;
  };
  f32x4_t kf[QK];
  vec_t vf[16];
  auto load_k = [&](const TileAt &t) __attribute__((always_inline)) {
    const int s = m >> 4;
    const int64_t row = (s ? t.slot[1] : t.slot[0]) + min(m & 15, s ? t.last[1] : t.last[0]);
    const char *krow = reinterpret_cast<const char *>(kc + row * row_elems) + k_lane;
#pragma unroll
    for (int j = 0; j < QK; ++j) {
      const int e = 8 * j + 4 * half;
      kf[j] = *reinterpret_cast<const f32x4_t *>(krow + (kPad && e >= d ? -4 * (e - 8 * j) : 32 * j));
    }
  };
  // V rows through a buffer resource per span that ends with its last needed
  // row: rows past it, and all rows of a bad block, read as zeros.
  auto load_v = [&](const TileAt &t) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float *>(vc + t.slot[s] * row_elems), 0, t.vbytes[s], 0x00020000);
#pragma unroll
      for (int i = 0; i < 8; ++i) {  // keys 8 (i / 4) + 4 half + i % 4 of the span
        const uint32_t row = (8u * (i >> 2) + (i & 3)) * row_bytes;
        if constexpr (VC == 1)
          vf[8 * s + i] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(r, v_lane, row, 0));
        else if constexpr (VC == 2)
          vf[8 * s + i] = __builtin_bit_cast(
              vec_t, __builtin_amdgcn_raw_buffer_load_b64(r, v_lane, row, 0));
        else
          vf[8 * s + i] = __builtin_bit_cast(
              vec_t, __builtin_amdgcn_raw_buffer_load_b128(r, v_lane, row, 0));
      }
    }
  };

  // V rows of the last tile and the one before it (no other is masked) that are
  // not finite, bit r for row r, where this wave has the tile.
  uint32_t late[2] = {0, 0};
  const int nk = ntiles > wave ? (ntiles - wave + kWaves - 1) / kWaves : 0;
  TileAt cur{};
  if (nk > 0) {  // uniform per wave
    load_ids(0);
    cur = tile_at(0);
    load_k(cur);
    load_v(cur);
  }
  for (int k = 0; k < nk; ++k) {
    const int key0 = (wave + kWaves * k) * kBNF;
    TileAt next = cur;
    if (k + 1 < nk) {
      if (((k + 1) & 31) == 0) load_ids(k + 1);
      next = tile_at(k + 1);
    }
    if constexpr (kPad) {  // dims past the head
#pragma unroll
      for (int j = 0; j < QK; ++j)
        if (8 * j + 4 * half >= d) kf[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    // S^T of the tile.
    f32x16_t s = f32x16_t{};
    if constexpr (kPad) {
      // Four chains: the generic kernel these head sizes ran on adds a score in
      // eight parts, and one chain of D/2 steps was further from 64 bits than
      // that at short contexts (2.5e-7 against 1.5e-7 at head size 96).
      f32x16_t part[4];
#pragma unroll
      for (int j = 0; j < QK; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          part[j & 3] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              kf[j][e], qf[j][e], j < 4 && e == 0 ? f32x16_t{} : part[j & 3], 0, 0, 0);
      s = (part[0] + part[1]) + (part[2] + part[3]);  // times c2 below
    } else {
#pragma unroll
      for (int j = 0; j < QK; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j][e], qf[j][e], s, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (k + 1 < nk) load_k(next);
    __builtin_amdgcn_sched_barrier(0);
    // Mask: keys past the query's position, and all keys of a bad block.
    const bool bad = cur.bad[0] || cur.bad[1];
    if (bad || key0 + kBNF - 1 > first_masked) {  // uniform
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (cur.bad[i >> 3] || key0 + 8 * (i >> 2) + 4 * half + (i & 3) > qpos) s[i] = -INFINITY;
      // A masked key's probability is 0, but 0 times an infinity or NaN is NaN:
      // V rows that are not finite count as zeros in the MFMAs of a masked tile
      // and are added after the last one, for the queries that see them.
      float none[2] = {0.f, 0.f};  // NaN if the lane's part of some row is not finite
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int c = 0; c < VC; ++c) {
          if constexpr (VC == 1) none[i & 1] = fmaf(vf[i], 0.f, none[i & 1]);
          else none[i & 1] = fmaf(vf[i][c], 0.f, none[i & 1]);
        }
      const float any_off = none[0] + none[1];
      if (__builtin_expect(key0 + kBNF - 1 > first_masked && __any(any_off != any_off), 0)) {
        uint32_t rows = 0;  // bit r: row r of the tile
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          bool off = false;
#pragma unroll
          for (int c = 0; c < VC; ++c) {
            float v;
            if constexpr (VC == 1) v = vf[i];
            else v = vf[i][c];
            off |= !(fabsf(v) < INFINITY);
          }
          const uint64_t lanes = __ballot(off);
          const int r = 8 * (i >> 2) + (i & 3);
          if (static_cast<uint32_t>(lanes) != 0) rows |= 1u << r;
          if (static_cast<uint32_t>(lanes >> 32) != 0) rows |= 16u << r;
        }
        // A span past the last key holds that key's row again: zeros as well,
        // but not a key to look up in the block table.
        const int keys = kv_end - key0;
        if (keys <= kBNF) late[0] = rows & (~0u >> (kBNF - keys));
        else late[1] = rows;
        uint32_t own = rows >> (4 * half);
        asm volatile("" : "+v"(own));
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (own & (1u << (8 * (i >> 2) + (i & 3)))) vf[i] = vec_t(0.f);
      }
    }
    // Online softmax (base 2). The reference point stays 0 until the query
    // has seen a key, so masked scores give exactly zero probabilities.
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = other_half_max(mx);
    const float m_new = fmaxf(m_run, kPad ? mx * c2 : mx);
    const float ref = m_new == -INFINITY ? 0.f : m_new;
    if (__any(m_new > m_run)) {
      const float alpha = __builtin_amdgcn_exp2f(m_run - ref);  // 0 while m_run is -inf
      l_run *= alpha;
#pragma unroll
      for (int c = 0; c < VC; ++c) acc[c] *= alpha;
    }
    m_run = m_new;
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if constexpr (kPad)  // the max keeps a masked score's small term finite
        s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], c2, -ref) + fmaxf(s[i], -1e30f) * c2_lo);
      else
        s[i] = __builtin_amdgcn_exp2f(s[i] - ref);
      sum[i & 3] += s[i];
    }
    l_run += (sum[0] + sum[1]) + (sum[2] + sum[3]);
    // O^T += V^T P^T.
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int c = 0; c < VC; ++c) {
        float v;
        if constexpr (VC == 1) v = vf[i];
        else v = vf[i][c];
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, s[i], acc[c], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
    if (k + 1 < nk) load_v(next);
    __builtin_amdgcn_sched_barrier(0);
    cur = next;
  }

  // Out of line: a branch over it costs an instruction fetch.
  if (__builtin_expect((late[0] | late[1]) != 0, 0)) {
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
      const int key0 = (ntiles - 1 - t) * kBNF;
#pragma unroll 1
      for (uint32_t left = t == 0 ? late[0] : late[1]; left != 0; left &= left - 1) {  // uniform
        const int key = key0 + __builtin_ctz(left);
        // A uniform row under buffer resources, as in the main loop (an address in
        // vector registers here would move the pools' there too). Dims past the
        // head read as zeros.
        const int64_t id = bt_row[key >> bs_log2];
        const int64_t block = static_cast<int64_t>(
            static_cast<uint64_t>(static_cast<uint32_t>(
                __builtin_amdgcn_readfirstlane(static_cast<int>(id)))) |
            (static_cast<uint64_t>(static_cast<uint32_t>(
                 __builtin_amdgcn_readfirstlane(static_cast<int>(id >> 32))))
             << 32));
        const int64_t at = ((block << bs_log2) + (key & bs_mask)) * row_elems;
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(kc + at), 0, 4u * d, 0x00020000);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(vc + at), 0, 4u * d, 0x00020000);
        uint32_t hf = half;  // opaque: nothing of this is kept across the main loop
        asm volatile("" : "+v"(hf));
        float x = 0.f;  // the query's score for the key: a half-wave's dims, then both
#pragma unroll
        for (int j = 0; j < QK; ++j) {
          const f32x4_t k = __builtin_bit_cast(
              f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, 32 * j + 16 * hf, 0, 0));
#pragma unroll
          for (int i = 0; i < 4; ++i) x = fmaf(qf[j][i], k[i], x);
        }
        x += __shfl_xor(x, 32);
        const float ref = m_run == -INFINITY ? 0.f : m_run;
        const float pr = __builtin_amdgcn_exp2f(kPad ? fmaf(x, c2, -ref) + x * c2_lo : x - ref);
#pragma unroll
        for (int i = 0; i < 16; ++i) {  // dims VC * (8 (i / 4) + 4 half + i % 4) and on
          const uint32_t off = 4u * VC * (8 * (i >> 2) + (i & 3)) + 16u * VC * hf;
          vec_t v;
          if constexpr (VC == 1)
            v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, off, 0, 0));
          else if constexpr (VC == 2)
            v = __builtin_bit_cast(vec_t, __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0));
          else
            v = __builtin_bit_cast(vec_t, __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0));
#pragma unroll
          for (int c = 0; c < VC; ++c) {
            float y;
            if constexpr (VC == 1) y = v;
            else y = v[c];
            acc[c][i] += key <= qpos ? pr * y : 0.f;
          }
        }
      }
    }
  }

  // The waves' parts: (O^T, m, l) of each, lane-major, then wave w adds and
  // stores the registers w, w + kWaves, ... (acc[c][i] = O[query m][dim
  // VC * (8 (i / 4) + 4 half + i % 4) + c]).
  constexpr int A = 16 * VC;
  __shared__ float part[kWaves][A][64];
  __shared__ float m_s[kWaves][64], l_s[kWaves][64];
#pragma unroll
  for (int c = 0; c < VC; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) part[wave][i * VC + c][lane] = acc[c][i];
  m_s[wave][lane] = m_run;
  l_s[wave][lane] = l_run;
  __syncthreads();
  float mx = m_s[0][lane];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, m_s[w][lane]);
  const float ref = mx == -INFINITY ? 0.f : mx;
  float f[kWaves], l = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    f[w] = __builtin_amdgcn_exp2f(m_s[w][lane] - ref);  // 0 for a wave without keys
    l += f[w] * (l_s[w][lane] + l_s[w][lane ^ 32]);
  }
  if (!q_ok) return;
  const float inv = 1.f / l;
  float *orow = static_cast<float *>(p.out) + (rg.q0 + qi) * p.o_st +
                static_cast<int64_t>(h) * p.o_sh;
  // Register i of every accumulator: VC consecutive dims, one store.
#pragma unroll
  for (int u = 0; u < 16 / kWaves; ++u) {
    const int i = wave + kWaves * u;
    const int e = VC * (8 * (i >> 2) + 4 * half + (i & 3));
    if (kPad && e >= d) continue;
    vec_t o;
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      float x = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) x += f[w] * part[w][i * VC + c][lane];
      if constexpr (VC == 1) o = x * inv;
      else o[c] = x * inv;
    }
    *reinterpret_cast<vec_t *>(orow + e) = o;
  }
}

template <int D, int kWaves, bool kPad>
int launch_waves(const PrefillParams &q, int64_t blocks, hipStream_t stream) {
  prefill_f32_mfma<D, kWaves, kPad>
      <<<dim3(static_cast<unsigned>(blocks)), 64 * kWaves, 0, stream>>>(q);
  return check_launch("mlr_paged_prefill(fp32 mfma)");
}

template <int D, bool kPad>
int launch_f32(const PrefillParams &p, int64_t max_query_len, hipStream_t stream) {
  PrefillParams q = p;
  q.n_qtiles = static_cast<int>(ceil_div(max_query_len, kBMF));
  const int64_t items = static_cast<int64_t>(q.num_seqs) * q.n_qtiles;
  const int64_t blocks = ceil_div(items, 8) * 8 * q.hq;
  if (blocks > INT32_MAX)
    return set_error(MLR_ERR_UNSUPPORTED, "mlr_paged_prefill: too many work items");
  const int64_t groups = items * q.hq, cus = current_device_cus();
  if constexpr (D < 128) {
    // A grid of fewer workgroups than CUs: eight waves each, half the keys a
    // wave (at 128 their registers would spill).
    if (groups <= cus) return launch_waves<D, 8, kPad>(q, blocks, stream);
  }
  // Short contexts in a grid that fills the GPU: fewer waves, so that each has
  // some tiles between its first load and the merge. us per call with 1 / 2 /
  // 4 waves: 16 x 200 tokens (7 tiles), 28/4 heads of 128 88 / 109 / 160; 4 x 300
  // (10 tiles) 54 / 53 / 70; 300 after 1000 (41 tiles) x 4 300 / 252 / 240.
  const int64_t context = p.qsl != nullptr ? p.max_blocks * p.block_size : p.s_ctx;
  if (groups >= 4 * cus && context <= 8 * kBNF) return launch_waves<D, 1, kPad>(q, blocks, stream);
  if (groups >= 4 * cus && context <= 16 * kBNF) return launch_waves<D, 2, kPad>(q, blocks, stream);
  return launch_waves<D, 4, kPad>(q, blocks, stream);
}

}  // namespace

bool prefill_f32_eligible(const PrefillParams &p, int dtype) {
  const bool aligned = (reinterpret_cast<uintptr_t>(p.q) & 15u) == 0 &&
                       (reinterpret_cast<uintptr_t>(p.kc) & 15u) == 0 &&
                       (reinterpret_cast<uintptr_t>(p.vc) & 15u) == 0 &&
                       (reinterpret_cast<uintptr_t>(p.out) & 15u) == 0 &&
                       p.q_st % 4 == 0 && p.q_sh % 4 == 0 && p.o_st % 4 == 0 &&
                       p.o_sh % 4 == 0;
  // Positions are 32-bit inside the kernel. Where the scale multiplies the score
  // (the padded form), it must not round to 0 in FP32: 0 times a masked score of
  // -inf would be NaN. Smaller scales stay on the generic kernel.
  constexpr int64_t k2g = int64_t(1) << 31;
  const bool padded = p.d != 64 && p.d != 128;
  return dtype == MLR_DTYPE_F32 && p.d % 4 == 0 && p.d <= 128 && aligned && p.bs_log2 >= 4 &&
         p.max_blocks * p.block_size < k2g && 16 * static_cast<int64_t>(p.hkv) * p.d * 4 < k2g &&
         p.scale > (padded ? 1e-30 : 0.0) && p.scale < 1e30;
}

int launch_prefill_f32(const PrefillParams &p, int64_t max_query_len, hipStream_t stream) {
  if (p.d <= 32) return launch_f32<32, true>(p, max_query_len, stream);
  if (p.d == 64) return launch_f32<64, false>(p, max_query_len, stream);
  if (p.d < 64) return launch_f32<64, true>(p, max_query_len, stream);
  if (p.d == 128) return launch_f32<128, false>(p, max_query_len, stream);
  return launch_f32<128, true>(p, max_query_len, stream);
}

}  // namespace mlr
