// int4 K cache: quantize/pack, static channel subset, subset slab, and the
// decode scoring kernel fused with block max-pooling.
//
// The reference scores fp32 over GQA-expanded bf16 K (qabs_cuda_kernels.py:
// 63-158) and keeps a transposed bf16 K copy for it (evaluate_qwen3_top2_
// head_limit3_ppl.py:2018-2042).  Here the scored stream is an int4 slab of
// S channels per token (S/2 bytes + one fp16 scale), read once with 128-bit
// loads; the dot is v_dot4_i32_i8 on nibbles shifted into the high half of
// each byte, so no sign-extension or bias pass is needed.
//
// Built with -ffp-contract=off: the ranking key fp32(scale) * fp32(I) is a
// single IEEE multiply, identical to the CPU oracle.
#include <algorithm>

#include "common.h"

#include "score.h"
#include "window.h"

#ifndef QKV_SCORE_TARGET_WGS
#define QKV_SCORE_TARGET_WGS 4096
#endif

namespace qkv {
namespace {

constexpr int kThreads = 256;

// Exact fp16 value times 2^24 (every finite fp16 is a multiple of 2^-24).
__device__ __forceinline__ uint64_t fp16_fixed24(uint32_t bits) {
  uint32_t e = (bits >> 10) & 0x1Fu;
  uint32_t m = bits & 0x3FFu;
  if (e == 0) return m;
  return static_cast<uint64_t>(1024u + m) << (e - 1);
}

// Eight bf16 (or, with F16, fp16) channels of a 16-byte load, widened exactly.
template <bool F16>
__device__ __forceinline__ void halfx8(const uint4& raw, float* x) {
  x[0] = half_lo<F16>(raw.x); x[1] = half_hi<F16>(raw.x);
  x[2] = half_lo<F16>(raw.y); x[3] = half_hi<F16>(raw.y);
  x[4] = half_lo<F16>(raw.z); x[5] = half_hi<F16>(raw.z);
  x[6] = half_lo<F16>(raw.w); x[7] = half_hi<F16>(raw.w);
}

// The fp16 scale of a group with amax `a` >= 0: fp16(fp32(a / 7)), saturated.
// a holds at most 11 significant bits, so a / 7 is either exactly an fp16
// rounding boundary or at least 2^-15 (relative) away from every one: one
// Newton step on a * fp32(1/7) (exact where the quotient is representable)
// rounds to the same fp16 as the IEEE division, in 3 instructions.
__device__ __forceinline__ uint32_t group_scale(float a) {
  a = fminf(a, 3.4028235e38f);   // (an infinite amax saturates as it did)
  const float r7 = 1.0f / 7.0f;
  const float q = a * r7;
  return f32_to_f16bits_sat(__builtin_fmaf(__builtin_fmaf(-7.0f, q, a), r7, q));
}

// Reciprocal of a scale for codes8, 0 for the all-zero group's scale 0.
__device__ __forceinline__ float code_rcp(float s) { return s != 0.0f ? __builtin_amdgcn_rcpf(s) : 0.0f; }

// Eight codes clamp(rint_even(x / s), -8, 7) as one little-endian word of
// nibbles (channel i at bits 4i..4i+3), rs ~ 1/s.  x and s have at most 11
// significant bits, so x / s is either exactly half-way between two integers
// or at least 2^-13.1 away from every such point (below 128 in magnitude).
// fma(x, rs, 384) rounds the quotient to multiples of 2^-15: an approximate
// quotient of a tie lands exactly on it, any other stays on its side.  Adding
// 1.5 * 2^23 - 384 rounds to the nearest integer, ties to even, leaving
// 0x4B400000 + code in the bits; the codes are gathered by shift-and-add
// (the constants' sum is known) as (code + 8) nibbles, then xor 8.  4.3
// instructions a value; the IEEE division with rint, conversion and masking
// took about 20 and bound the pack kernel.  The scale 0 (rs = 0) gives code 0
// for every value, and a NaN under another scale -8 (the median of a NaN and
// the bounds is the lower one), as the division with its clamp did.
__device__ __forceinline__ uint32_t codes8(const float* x, float rs) {
  uint32_t acc = 0;
#pragma unroll
  for (int i = 7; i >= 0; --i) {
    const float t = __builtin_fmaf(x[i], rs, 384.0f) + (12582912.0f - 384.0f);
    const float c = __builtin_amdgcn_fmed3f(t, 12582904.0f, 12582919.0f);
    acc = (acc << 4) + __float_as_uint(c);
  }
  constexpr uint32_t kBias = 0x4B400000u + (0x4B400000u << 4) + (0x4B400000u << 8);   // higher terms vanish mod 2^32
  return rs != 0.0f ? (acc - kBias + 0x88888888u) ^ 0x88888888u : 0u;
}

// Max over the LANES (4, 8 or 16) lanes of an aligned group, on the bit
// patterns of non-negative floats.
template <int LANES>
__device__ __forceinline__ float group_max(float x) {
  static_assert(LANES == 2 || LANES == 4 || LANES == 8 || LANES == 16, "lanes of a DPP row");
  uint32_t v = __float_as_uint(x);
  v = max(v, dpp_mov<0xB1>(v, v));
  if constexpr (LANES >= 4) v = max(v, dpp_mov<0x4E>(v, v));
  if constexpr (LANES >= 8) v = max(v, dpp_mov<0x141>(v, v));
  if constexpr (LANES >= 16) v = max(v, dpp_mov<0x140>(v, v));
  return __uint_as_float(v);
}

// ---------------------------------------------------------------------------
// Pack: one thread per 8 channels of a token; GROUP/8 lanes share a scale.
// A workgroup takes kPackIter * 256 * 8 / D tokens of one row, every thread's
// kPackIter 16-byte loads issued before the first is used.  Bound by HBM: 2 x 8
// rows x 32768 tokens (134 MB of K in, 38 MB out) took 60 us with one load a
// thread and a division per code, 30 us now (5.7 TB/s).
// ---------------------------------------------------------------------------
constexpr int kPackIter = 2;   // (1.4 us slower at 4 loads a thread, 2.6 at 8, 134 MB of K)

template <int GROUP, bool F16>
__global__ __launch_bounds__(kThreads) void pack_kernel(
    const uint16_t* __restrict__ key, int64_t ksb, int64_t ksh, int64_t kst, int kv_heads,
    int t_begin, int t_end, int tpt_log2, unsigned tiles, uint8_t* __restrict__ packed,
    uint16_t* __restrict__ scales, int64_t capacity) {
  constexpr int TPG = GROUP / 8;
  const unsigned r = blockIdx.x / tiles, tile = blockIdx.x - r * tiles;
  const int b = static_cast<int>(r / static_cast<unsigned>(kv_heads));
  const int h = static_cast<int>(r) - b * kv_heads;
  const int c8 = threadIdx.x & ((1 << tpt_log2) - 1);
  const int step = kThreads >> tpt_log2;   // tokens per load of the workgroup
  const int t0 = t_begin + static_cast<int>(tile) * kPackIter * step + static_cast<int>(threadIdx.x >> tpt_log2);
  const uint16_t* row = key + b * ksb + h * ksh + c8 * 8;
  uint4 raw[kPackIter];
#pragma unroll
  for (int it = 0; it < kPackIter; ++it) {
    raw[it] = make_uint4(0, 0, 0, 0);
    if (t0 + it * step < t_end)
      raw[it] = *reinterpret_cast<const uint4*>(row + static_cast<int64_t>(t0 + it * step) * kst);
  }
#pragma unroll
  for (int it = 0; it < kPackIter; ++it) {
    const int t = t0 + it * step;
    float x[8];
    halfx8<F16>(raw[it], x);
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) a = fmaxf(a, fabsf(x[i]));
    const uint32_t sbits = group_scale(group_max<TPG>(a));
    const uint32_t word = codes8(x, code_rcp(f16bits_to_f32(sbits)));
    if (t < t_end) {
      const int64_t tok = static_cast<int64_t>(r) * capacity + t;
      reinterpret_cast<uint32_t*>(packed)[(tok << tpt_log2) + c8] = word;
      if (c8 % TPG == 0) scales[((tok << tpt_log2) + c8) / TPG] = static_cast<uint16_t>(sbits);
    }
  }
}

// ---------------------------------------------------------------------------
// Channel statistic: sum_t |code| * F(scale), exact in uint64 (order-free).
// A workgroup sums one chunk of a row's tokens: a thread takes 16 channels of
// a token (8 bytes), four tokens' loads in flight; the threads' sums meet in
// LDS.  With `part` the chunk's sums are stored there (no atomics, no zeroed
// memory) for select_channels_kernel to add up; else they are added to
// `stats` by atomics (integers, so the result does not depend on the order).
// Bound by the reads of the packed copy (38 MB at 16 rows x 32768 tokens,
// mostly cached from the packing): 125 us with code-by-code 64-bit sums and
// atomics, about 12 us now.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void zero_u64_kernel(uint64_t* p, int64_t n) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i < n) p[i] = 0;
}

// |code| of eight nibbles at once (8 for code -8).
__device__ __forceinline__ uint32_t nibble_abs(uint32_t w) {
  const uint32_t s = w & 0x88888888u, one = s >> 3;
  return (w ^ (s | (s - one))) + one;
}

__global__ __launch_bounds__(kThreads) void channel_stats_kernel(
    const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scales, int tokens,
    int64_t capacity, int head_dim, int group, int chunk, uint64_t* __restrict__ part,
    uint64_t* __restrict__ stats) {
  constexpr int kPad = kThreads + 8;   // channels k and k + 1 of a slot 16 banks apart
  __shared__ uint64_t sums[16 * kPad];
  const int r = blockIdx.y;
  const int lpt = head_dim / 16;         // threads per token
  const int step = kThreads / lpt;       // tokens per load of the workgroup
  const int slot = threadIdx.x % lpt, tl = threadIdx.x / lpt;
  const int t0 = blockIdx.x * chunk, t1 = min(tokens, t0 + chunk);
  const int spt = head_dim / group;
  const uint2* words = reinterpret_cast<const uint2*>(packed) + static_cast<int64_t>(r) * capacity * lpt + slot;
  const uint16_t* sc = scales + static_cast<int64_t>(r) * capacity * spt + (slot * 16) / group;
  uint64_t acc[16] = {};
  constexpr int U = 4;
  for (int t = t0 + tl; t < t1; t += U * step) {
    uint2 w[U];
    uint32_t sb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {   // tokens past the chunk: scale 0 adds nothing
      const int64_t tu = min(t + u * step, t1 - 1);
      w[u] = words[tu * lpt];
      sb[u] = sc[tu * spt];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t f = t + u * step < t1 ? fp16_fixed24(sb[u]) : 0;
      const uint32_t flo = static_cast<uint32_t>(f), fhi = static_cast<uint32_t>(f >> 32);
      const uint32_t a[2] = {nibble_abs(w[u].x), nibble_abs(w[u].y)};
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] += static_cast<uint64_t>(flo) * ((a[i >> 3] >> (4 * (i & 7))) & 0xFu);
      if (__any(fhi)) {   // scales of 256 and more
#pragma unroll
        for (int i = 0; i < 16; ++i)
          acc[i] += static_cast<uint64_t>(fhi * ((a[i >> 3] >> (4 * (i & 7))) & 0xFu)) << 32;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) sums[i * kPad + threadIdx.x] = acc[i];
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < head_dim) {
    const int cs = threadIdx.x % lpt, ck = threadIdx.x / lpt;   // channel 16 * cs + ck
    uint64_t s = 0;
#pragma unroll 8
    for (int j = 0; j < step; ++j) s += sums[ck * kPad + cs + lpt * j];
    const int c = cs * 16 + ck;
    if (part)
      part[(static_cast<int64_t>(r) * gridDim.x + blockIdx.x) * head_dim + c] = s;
    else if (s)
      atomicAdd(reinterpret_cast<unsigned long long*>(stats + static_cast<int64_t>(r) * head_dim + c),
                static_cast<unsigned long long>(s));
  }
}

// One workgroup of 1024 threads per row: the statistic summed from the row's
// `n_part` partial sums (written to `stats`), or read from `stats` (n_part =
// 0); rank(c) = #{e : st[e] > st[c] or (st[e] == st[c] and e < c)}; the
// channels of rank < S are written in ascending channel order.  1024 / D
// threads share a channel's sums and its rank's compares.  Bound by latency,
// one load round and one rank pass: 8.8 us with one thread per channel, 5 now.
__global__ __launch_bounds__(1024) void select_channels_kernel(const uint64_t* __restrict__ part, int n_part,
                                                               uint64_t* __restrict__ stats, int head_dim,
                                                               int selected, int32_t* __restrict__ chan_idx) {
  __shared__ uint64_t psum[1024];
  __shared__ uint64_t st[256];
  __shared__ int rank_s[256];
  __shared__ int wcnt[4];
  const int r = blockIdx.x, tid = threadIdx.x;
  const int c = tid & (head_dim - 1), q = tid / head_dim, nq = 1024 / head_dim;
  uint64_t v = 0;
  if (n_part) {
    const uint64_t* p = part + static_cast<int64_t>(r) * n_part * head_dim + c;
#pragma unroll 4
    for (int i = q; i < n_part; i += nq) v += p[static_cast<int64_t>(i) * head_dim];
  } else if (q == 0) {
    v = stats[static_cast<int64_t>(r) * head_dim + c];
  }
  psum[tid] = v;
  if (tid < 256) rank_s[tid] = 0;
  __syncthreads();
  if (tid < head_dim) {
    uint64_t t = 0;
    for (int j = 0; j < nq; ++j) t += psum[j * head_dim + tid];
    st[tid] = t;
    if (n_part) stats[static_cast<int64_t>(r) * head_dim + tid] = t;
  }
  __syncthreads();
  const uint64_t own = st[c];
  int rank = 0;
  const int per = head_dim / nq;   // compares of this thread: 4 (D = 64), 16 or 64
#pragma unroll 4
  for (int i = 0; i < per; ++i) {
    const int e = q * per + i;
    rank += (st[e] > own) || (st[e] == own && e < c);
  }
  if (rank) atomicAdd(&rank_s[c], rank);
  __syncthreads();
  const bool sel = tid < head_dim && rank_s[c] < selected;
  const uint64_t mask = __ballot(sel);
  if (tid < head_dim && (tid & 63) == 0) wcnt[tid >> 6] = __popcll(mask);
  __syncthreads();
  if (sel) {
    int pos = __popcll(mask & ((1ull << (tid & 63)) - 1ull));
    for (int w = 0; w < (tid >> 6); ++w) pos += wcnt[w];
    chan_idx[static_cast<int64_t>(r) * selected + pos] = c;
  }
}

// ---------------------------------------------------------------------------
// Subset slab: S/8 lanes per token, each gathers 8 selected channels.
//
// The slab's codes are stored in tiles of 4096 bytes = 64 lanes x 4 chunks of
// 16 bytes, one tile per 8192/S keys.  Lane l of a tile owns the 128/S
// consecutive keys [l * 128/S, (l+1) * 128/S), i.e. 64 logical bytes; its
// logical byte b sits at tile offset (64 * (b / 16) + l) * 16 + b % 16.  A
// wave reading chunk 64j + l in load j therefore issues fully coalesced
// 16-byte loads and still ends with whole, consecutive keys in each lane.
// ---------------------------------------------------------------------------

// Byte offset, within a row's slab, of logical code byte x of key t.
template <int S>
__device__ __forceinline__ int64_t slab_offset(int64_t t, int x) {
  constexpr int KPLN = 128 / S;            // keys per lane
  const int64_t tile = t / slab_tile_keys(S);
  const int k = static_cast<int>(t - tile * slab_tile_keys(S));
  const int lane = k / KPLN;
  const int b = (k - lane * KPLN) * (S / 2) + x;
  return tile * 4096 + (64 * (b >> 4) + lane) * 16 + (b & 15);
}
// Rows of K 16-byte aligned: one wave takes 64 tokens of a row.  The tokens'
// whole rows are loaded with 16-byte loads, all in flight (every 128-byte
// line of K holds selected channels, so nothing is read in vain), and staged
// in LDS; then lane l owns token l, reads its S channels from LDS (the
// channel ids are wave-uniform) and writes its S/2 bytes in 16-byte pieces,
// so the scale and the codes need no other lane.  LDS rows are 16 bytes
// longer than K's: a read's 64 lanes fall on 16 banks, 4 lanes each.  Bound
// by HBM: 2 x 8 rows x 32768 tokens (134 MB of K) took 89 us with 2-byte loads
// (build_slab_kernel, which stays for rows these loads cannot read), 27 now.
template <int S, int D, bool F16>
__global__ __launch_bounds__(64) void build_slab_rows_kernel(
    const uint16_t* __restrict__ key, int64_t ksb, int64_t ksh, int64_t kst, int kv_heads,
    int t_begin, int t_end, unsigned tiles, const int32_t* __restrict__ chan_idx,
    uint8_t* __restrict__ slab, uint16_t* __restrict__ slab_scales, int64_t capacity) {
  constexpr int kLds = D / 8 + 1;            // 16-byte pieces of an LDS row
  constexpr int kTok = 512 / D;              // tokens per load of the wave
  constexpr int kLoads = 64 / kTok;
  constexpr int kBatch = kLoads < 16 ? kLoads : 16;
  __shared__ uint4 rows[64 * kLds];
  const unsigned r = blockIdx.x / tiles, tile = blockIdx.x - r * tiles;
  const int b = static_cast<int>(r / static_cast<unsigned>(kv_heads));
  const int h = static_cast<int>(r) - b * kv_heads;
  const int lane = threadIdx.x;
  const int t0 = t_begin + static_cast<int>(tile) * 64;
  const int piece = lane % (D / 8), tl = lane / (D / 8);
  const uint16_t* base = key + b * ksb + h * ksh + piece * 8;
#pragma unroll
  for (int i0 = 0; i0 < kLoads; i0 += kBatch) {
    uint4 raw[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int k = (i0 + i) * kTok + tl;
      raw[i] = make_uint4(0, 0, 0, 0);
      if (t0 + k < t_end) raw[i] = *reinterpret_cast<const uint4*>(base + static_cast<int64_t>(t0 + k) * kst);
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) rows[((i0 + i) * kTok + tl) * kLds + piece] = raw[i];
  }
  __syncthreads();
  const int t = t0 + lane;
  const uint16_t* own = reinterpret_cast<const uint16_t*>(rows + lane * kLds);
  const int32_t* idx = chan_idx + static_cast<int64_t>(r) * S;
  float x[S];
  float a = 0.0f;
#pragma unroll
  for (int i = 0; i < S; ++i) {
    // channel ids come from qkv_int4_select_channels; clamping keeps a bad id in the row
    x[i] = half_to_f32<F16>(own[min(max(idx[i], 0), D - 1)]);
    a = fmaxf(a, fabsf(x[i]));
  }
  const uint32_t sbits = group_scale(a);
  const float rs = code_rcp(f16bits_to_f32(sbits));
  uint32_t w[S / 8];
#pragma unroll
  for (int j = 0; j < S / 8; ++j) w[j] = codes8(x + 8 * j, rs);
  if (t >= t_end) return;
  uint8_t* out = slab + static_cast<int64_t>(r) * capacity * (S / 2);
  if constexpr (S == 16) {
    *reinterpret_cast<uint2*>(out + slab_offset<S>(t, 0)) = make_uint2(w[0], w[1]);
  } else {
#pragma unroll
    for (int j = 0; j < S / 32; ++j)
      *reinterpret_cast<uint4*>(out + slab_offset<S>(t, 16 * j)) =
          make_uint4(w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]);
  }
  slab_scales[static_cast<int64_t>(r) * capacity + t] = static_cast<uint16_t>(sbits);
}

// Any alignment: S/8 lanes per token, 2-byte loads of the selected channels.
template <int S, bool F16>
__global__ __launch_bounds__(kThreads) void build_slab_kernel(
    const uint16_t* __restrict__ key, int64_t ksb, int64_t ksh, int64_t kst, int kv_heads,
    int t_begin, int ntok, int head_dim, const int32_t* __restrict__ chan_idx,
    uint8_t* __restrict__ slab, uint16_t* __restrict__ slab_scales, int64_t capacity, int64_t total) {
  constexpr int TPT = S / 8;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const bool active = gid < total;
  const int64_t g = active ? gid : 0;
  const int64_t tok_lin = g / TPT;
  const int jj = static_cast<int>(g - tok_lin * TPT);
  const int64_t r = tok_lin / ntok;
  const int t = t_begin + static_cast<int>(tok_lin - r * ntok);
  const int b = static_cast<int>(r / kv_heads), h = static_cast<int>(r % kv_heads);
  float x[8];
  const uint16_t* row = key + b * ksb + h * ksh + static_cast<int64_t>(t) * kst;
  const int32_t* idx = chan_idx + r * S + jj * 8;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = min(max(active ? idx[i] : 0, 0), head_dim - 1);
    x[i] = active ? half_to_f32<F16>(row[c]) : 0.0f;
  }
  float a = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) a = fmaxf(a, fabsf(x[i]));
  const uint32_t sbits = group_scale(group_max<TPT>(a));
  const uint32_t word = codes8(x, code_rcp(f16bits_to_f32(sbits)));
  if (active) {
    const int64_t tok = r * capacity + t;
    *reinterpret_cast<uint32_t*>(slab + r * capacity * (S / 2) + slab_offset<S>(t, 4 * jj)) = word;
    if (jj == 0) slab_scales[tok] = static_cast<uint16_t>(sbits);
  }
}

// The row's query words as a table: qwords[2d] = qlo[d], qwords[2d+1] = qhi[d].
template <int S, bool F16>
__global__ __launch_bounds__(64) void query_words_kernel(
    const uint16_t* __restrict__ query, int q_heads, int kv_heads, int head_dim,
    const int32_t* __restrict__ chan_idx, uint32_t* __restrict__ qwords, float* __restrict__ qscale_out) {
  const int r = blockIdx.x, lane = threadIdx.x;
  uint32_t qlo[S / 8], qhi[S / 8];
  float qs;
  const RowQueryLoads<S> ql = row_query_load<S>(query, q_heads, kv_heads, head_dim, chan_idx, r);
  row_query_finish<S, F16>(ql, query, q_heads, kv_heads, head_dim, r, qlo, qhi, &qs);
  uint32_t* out = qwords + static_cast<int64_t>(r) * (S / 4);
#pragma unroll
  for (int d = 0; d < S / 8; ++d) {
    if (lane == 2 * d) out[2 * d] = qlo[d];
    if (lane == 2 * d + 1) out[2 * d + 1] = qhi[d];
  }
  if (qscale_out && lane == 0) qscale_out[r] = qs;
}

template <int S, bool DEBUG, bool F16>
__global__ __launch_bounds__(kScoreThreads) void decode_scores_kernel(
    const uint16_t* __restrict__ query, int q_heads, int kv_heads, int head_dim,
    const int32_t* __restrict__ chan_idx, const uint8_t* __restrict__ slab,
    const uint16_t* __restrict__ slab_scales, int64_t capacity, int tokens, int block,
    int chunk, float* __restrict__ bmax, int nb, int32_t* __restrict__ isum,
    float* __restrict__ keys_out, float* __restrict__ qscale_out) {
  score_chunk<S, DEBUG, F16>(query, q_heads, kv_heads, head_dim, chan_idx, slab, slab_scales, capacity, tokens,
                               block, chunk, bmax, nb, isum, keys_out, qscale_out, blockIdx.y, blockIdx.x);
}

template <bool DEBUG, bool F16>
int launch_scores(int S, dim3 grid, hipStream_t st, const uint16_t* q, int hq, int hkv, int d,
                  const int32_t* ci, const uint8_t* slab, const uint16_t* ss, int64_t cap, int T,
                  int block, int chunk, float* bmax, int nb, int32_t* isum, float* keys, float* qs) {
  switch (S) {
#define QKV_CASE(SS)                                                                               \
  case SS:                                                                                         \
    decode_scores_kernel<SS, DEBUG, F16><<<grid, kScoreThreads, 0, st>>>(q, hq, hkv, d, ci, slab, ss, cap, T, \
                                                               block, chunk, bmax, nb, isum, keys, \
                                                               qs);                                \
    break;
    QKV_CASE(16) QKV_CASE(32) QKV_CASE(64) QKV_CASE(128)
#undef QKV_CASE
    default: return fail(QKV_ERR_UNSUPPORTED, "selected channel count %d not built", S);
  }
  return check_launch("qkv_int4_decode_scores");
}

// Decode scoring of qkv_int4_decode_topk: token scores (block 1), one
// workgroup per 4096-key chunk of the long-row top-k, each key also counted
// in the chunk's 12-bit histogram in LDS, and the chunk's counts added to its
// row's histogram (row_hist) -- or, where the selection works on chunk lists,
// the chunk's top-k window (chunk_window) written where qkv_topk_ws's
// histogram pass would write it.
// win_waves: the chunk's waves, every wave stage one whole slab tile.
constexpr int win_waves(int s) {
  return kStageChunk / slab_tile_keys(s) >= 16 ? 16 : static_cast<int>(kStageChunk / slab_tile_keys(s));
}

template <int S, bool F16>
__global__ __launch_bounds__(64 * win_waves(S)) void decode_scores_win_kernel(
    const uint16_t* __restrict__ query, int q_heads, int kv_heads, int head_dim,
    const int32_t* __restrict__ chan_idx, const uint8_t* __restrict__ slab,
    const uint16_t* __restrict__ slab_scales, int64_t capacity, int tokens, int k, float* __restrict__ scores,
    int n_chunks, int32_t* __restrict__ win, int* __restrict__ row_hist, int64_t hist_stride,
    float* __restrict__ qscale_out) {
  constexpr int NWV = win_waves(S), NT = 64 * NWV;
  static_assert(kStageChunk % (NWV * slab_tile_keys(S)) == 0, "a chunk is whole workgroup stages");
  __shared__ uint32_t h[kHistBins];
  __shared__ int wsum[NWV];
  __shared__ int t_sh;
#pragma unroll
  for (int i = 0; i < kHistBins / NT; ++i) h[threadIdx.x + NT * i] = 0;
  if (threadIdx.x == 0) t_sh = 0;
  __syncthreads();
  score_chunk<S, false, F16, NWV>(query, q_heads, kv_heads, head_dim, chan_idx, slab, slab_scales, capacity, tokens,
                                  1, kStageChunk, scores, tokens, nullptr, nullptr, qscale_out, blockIdx.y,
                                  blockIdx.x, h);
  __syncthreads();
  if (row_hist) {   // uniform: counted into the row's histogram instead
    flush_row_hist<NT>(h, row_hist + blockIdx.y * hist_stride);
    return;
  }
  const int len = min(kStageChunk, tokens - static_cast<int>(blockIdx.x) * kStageChunk);
  chunk_window<NT, false>(h, min(k, len), win + (static_cast<int64_t>(blockIdx.y) * n_chunks + blockIdx.x) * kWinWords,
                          wsum, &t_sh);
}

bool pow2(int64_t v) { return v > 0 && (v & (v - 1)) == 0; }

}  // namespace
}  // namespace qkv

using namespace qkv;

QKV_EXPORT int qkv_int4_pack_k(const void* key, const int64_t* k_strides, int64_t batch,
                               int64_t kv_heads, int64_t t_begin, int64_t t_end, int64_t head_dim,
                               int64_t group, uint8_t* packed, uint16_t* scales, int64_t capacity,
                               int dtype, void* stream) {
  if (!key || !k_strides || !packed || !scales) return fail(QKV_ERR_INVALID, "qkv_int4_pack_k: null pointer");
  bool f16;
  if (int rc = half_dtype(dtype, "qkv_int4_pack_k", &f16)) return rc;
  if (batch <= 0 || kv_heads <= 0 || t_begin < 0 || t_end < t_begin || t_end > capacity)
    return fail(QKV_ERR_INVALID, "qkv_int4_pack_k: bad token range [%lld, %lld) for capacity %lld",
                (long long)t_begin, (long long)t_end, (long long)capacity);
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return fail(QKV_ERR_UNSUPPORTED, "qkv_int4_pack_k: head_dim must be 64, 128 or 256");
  if ((group != 32 && group != 64 && group != 128) || head_dim % group)
    return fail(QKV_ERR_INVALID, "qkv_int4_pack_k: group must be 32, 64 or 128 and divide head_dim");
  if (!aligned(key, 16) || (k_strides[0] | k_strides[1] | k_strides[2]) % 8)
    return fail(QKV_ERR_INVALID, "qkv_int4_pack_k: K rows must be 16-byte aligned");
  if (capacity % 64 || !aligned(packed, 16) || !aligned(scales, 16))
    return fail(QKV_ERR_INVALID, "qkv_int4_pack_k: capacity must be a multiple of 64 and outputs 16-byte aligned");
  const int64_t ntok = t_end - t_begin;
  if (ntok == 0) return QKV_OK;
  const int tpt_log2 = head_dim == 64 ? 3 : head_dim == 128 ? 4 : 5;
  const int64_t tiles = cdiv(ntok, kPackIter * (kThreads >> tpt_log2));
  if (batch * kv_heads * tiles > 0x7FFFFFFF) return fail(QKV_ERR_INVALID, "qkv_int4_pack_k: too many tokens");
  dim3 grid(static_cast<unsigned>(batch * kv_heads * tiles));
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* k = static_cast<const uint16_t*>(key);
#define QKV_PACK(GG, FF)                                                                              \
  pack_kernel<GG, FF><<<grid, kThreads, 0, st>>>(k, k_strides[0], k_strides[1], k_strides[2],        \
                                                 static_cast<int>(kv_heads), static_cast<int>(t_begin), \
                                                 static_cast<int>(t_end), tpt_log2,                   \
                                                 static_cast<unsigned>(tiles), packed, scales, capacity)
  if (f16) {
    if (group == 32) QKV_PACK(32, true);
    else if (group == 64) QKV_PACK(64, true);
    else QKV_PACK(128, true);
  } else {
    if (group == 32) QKV_PACK(32, false);
    else if (group == 64) QKV_PACK(64, false);
    else QKV_PACK(128, false);
  }
#undef QKV_PACK
  return check_launch("qkv_int4_pack_k");
}

// Token chunks of the channel statistic: about 1024 workgroups over the rows
// (of the whole cache build at 16 rows of 32768: 73.6 us, at 2048 75.4, at 512 75.0),
// chunks of at least 128 tokens (one round of four loads at D = 128) and at
// most 128 a row, so that the partial sums stay a small share of the read.
static int64_t stats_chunk(int64_t rows, int64_t tokens) {
  const int64_t want = std::min<int64_t>(128, std::max<int64_t>(1, 1024 / rows));
  return std::max<int64_t>(128, cdiv(cdiv(tokens, want), 128) * 128);
}

static int check_select(const uint8_t* packed, const uint16_t* scales, int64_t rows, int64_t tokens,
                        int64_t capacity, int64_t head_dim, int64_t group, int64_t selected, const uint64_t* stats,
                        const int32_t* chan_idx) {
  if (!packed || !scales || !stats || !chan_idx)
    return fail(QKV_ERR_INVALID, "qkv_int4_select_channels: null pointer");
  if (rows <= 0 || rows > 65535 || tokens <= 0 || tokens > capacity || tokens > (int64_t(1) << 20))
    return fail(QKV_ERR_INVALID, "qkv_int4_select_channels: need 1 <= tokens <= min(capacity, 2^20), rows <= 65535");
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return fail(QKV_ERR_UNSUPPORTED, "qkv_int4_select_channels: head_dim must be 64, 128 or 256");
  if ((group != 32 && group != 64 && group != 128) || head_dim % group)
    return fail(QKV_ERR_INVALID, "qkv_int4_select_channels: bad group");
  if (selected < 1 || selected > head_dim)
    return fail(QKV_ERR_INVALID, "qkv_int4_select_channels: selected must be in [1, head_dim]");
  if (capacity % 64) return fail(QKV_ERR_INVALID, "qkv_int4_select_channels: capacity must be a multiple of 64");
  return QKV_OK;
}

// The statistic and the selection; `part` (may be null) holds the chunks' sums.
static int run_select(const uint8_t* packed, const uint16_t* scales, int64_t rows, int64_t tokens, int64_t capacity,
                      int64_t head_dim, int64_t group, int64_t selected, uint64_t* part, uint64_t* stats,
                      int32_t* chan_idx, hipStream_t st) {
  const int64_t chunk = stats_chunk(rows, tokens);
  dim3 grid(static_cast<unsigned>(cdiv(tokens, chunk)), static_cast<unsigned>(rows));
  if (!part) {
    const int64_t n = rows * head_dim;
    zero_u64_kernel<<<static_cast<unsigned>(cdiv(n, kThreads)), kThreads, 0, st>>>(stats, n);
    if (int rc = check_launch("qkv_int4_select_channels(zero)")) return rc;
  }
  channel_stats_kernel<<<grid, kThreads, 0, st>>>(packed, scales, static_cast<int>(tokens), capacity,
                                                  static_cast<int>(head_dim), static_cast<int>(group),
                                                  static_cast<int>(chunk), part, stats);
  if (int rc = check_launch("qkv_int4_select_channels(stats)")) return rc;
  select_channels_kernel<<<static_cast<unsigned>(rows), 1024, 0, st>>>(
      part, part ? static_cast<int>(grid.x) : 0, stats, static_cast<int>(head_dim), static_cast<int>(selected),
      chan_idx);
  return check_launch("qkv_int4_select_channels(select)");
}

QKV_EXPORT int qkv_int4_select_channels(const uint8_t* packed, const uint16_t* scales, int64_t rows,
                                        int64_t tokens, int64_t capacity, int64_t head_dim,
                                        int64_t group, int64_t selected, uint64_t* stats,
                                        int32_t* chan_idx, void* stream) {
  if (int rc = check_select(packed, scales, rows, tokens, capacity, head_dim, group, selected, stats, chan_idx))
    return rc;
  return run_select(packed, scales, rows, tokens, capacity, head_dim, group, selected, nullptr, stats, chan_idx,
                    static_cast<hipStream_t>(stream));
}

QKV_EXPORT int64_t qkv_int4_select_channels_workspace_bytes(int64_t rows, int64_t tokens, int64_t head_dim) {
  if (rows <= 0 || tokens <= 0 || head_dim <= 0) return -1;
  return rows * cdiv(tokens, stats_chunk(rows, tokens)) * head_dim * 8;
}

QKV_EXPORT int qkv_int4_select_channels_ws(const uint8_t* packed, const uint16_t* scales, int64_t rows,
                                           int64_t tokens, int64_t capacity, int64_t head_dim, int64_t group,
                                           int64_t selected, uint64_t* stats, int32_t* chan_idx, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
  if (int rc = check_select(packed, scales, rows, tokens, capacity, head_dim, group, selected, stats, chan_idx))
    return rc;
  const int64_t need = qkv_int4_select_channels_workspace_bytes(rows, tokens, head_dim);
  if (!workspace || workspace_bytes < need || !aligned(workspace, 8))
    return fail(QKV_ERR_INVALID, "qkv_int4_select_channels_ws: workspace needs %lld bytes (8-byte aligned), got %lld",
                (long long)need, (long long)workspace_bytes);
  return run_select(packed, scales, rows, tokens, capacity, head_dim, group, selected,
                    static_cast<uint64_t*>(workspace), stats, chan_idx, static_cast<hipStream_t>(stream));
}

QKV_EXPORT int qkv_int4_build_slab(const void* key, const int64_t* k_strides, int64_t batch,
                                   int64_t kv_heads, int64_t t_begin, int64_t t_end,
                                   int64_t head_dim, const int32_t* chan_idx, int64_t selected,
                                   uint8_t* slab, uint16_t* slab_scales, int64_t capacity,
                                   int dtype, void* stream) {
  if (!key || !k_strides || !chan_idx || !slab || !slab_scales)
    return fail(QKV_ERR_INVALID, "qkv_int4_build_slab: null pointer");
  bool f16;
  if (int rc = half_dtype(dtype, "qkv_int4_build_slab", &f16)) return rc;
  if (batch <= 0 || kv_heads <= 0 || t_begin < 0 || t_end < t_begin || t_end > capacity)
    return fail(QKV_ERR_INVALID, "qkv_int4_build_slab: bad token range");
  if (selected != 16 && selected != 32 && selected != 64 && selected != 128)
    return fail(QKV_ERR_UNSUPPORTED, "qkv_int4_build_slab: selected must be 16, 32, 64 or 128");
  if (selected > head_dim) return fail(QKV_ERR_INVALID, "qkv_int4_build_slab: selected > head_dim");
  if (capacity % slab_tile_keys(static_cast<int>(selected)) || !aligned(slab, 16) || !aligned(slab_scales, 16))
    return fail(QKV_ERR_INVALID, "qkv_int4_build_slab: capacity must be a multiple of %lld and outputs 16-byte aligned",
                (long long)slab_tile_keys(static_cast<int>(selected)));
  const int64_t ntok = t_end - t_begin;
  if (ntok == 0) return QKV_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* k = static_cast<const uint16_t*>(key);
  const int64_t tiles = cdiv(ntok, 64);
  if (aligned(key, 16) && (k_strides[0] | k_strides[1] | k_strides[2]) % 8 == 0 &&
      (head_dim == 64 || head_dim == 128 || head_dim == 256) && batch * kv_heads * tiles <= 0x7FFFFFFF) {
    const unsigned rgrid = static_cast<unsigned>(batch * kv_heads * tiles);
    auto launch = [&](auto sc, auto dc) {
      constexpr int SS = decltype(sc)::value, DD = decltype(dc)::value;
      if constexpr (SS <= DD) {
        return with_half(f16, [&](auto fc) {
          build_slab_rows_kernel<SS, DD, decltype(fc)::value><<<rgrid, 64, 0, st>>>(
              k, k_strides[0], k_strides[1], k_strides[2], static_cast<int>(kv_heads), static_cast<int>(t_begin),
              static_cast<int>(t_end), static_cast<unsigned>(tiles), chan_idx, slab, slab_scales, capacity);
          return check_launch("qkv_int4_build_slab");
        });
      } else {
        return fail(QKV_ERR_INVALID, "qkv_int4_build_slab: selected > head_dim");
      }
    };
    auto with_d = [&](auto sc) {
      if (head_dim == 64) return launch(sc, std::integral_constant<int, 64>{});
      if (head_dim == 128) return launch(sc, std::integral_constant<int, 128>{});
      return launch(sc, std::integral_constant<int, 256>{});
    };
    switch (selected) {
      case 16: return with_d(std::integral_constant<int, 16>{});
      case 32: return with_d(std::integral_constant<int, 32>{});
      case 64: return with_d(std::integral_constant<int, 64>{});
      default: return with_d(std::integral_constant<int, 128>{});
    }
  }
  const int64_t total = batch * kv_heads * ntok * (selected / 8);
  dim3 grid(static_cast<unsigned>(cdiv(total, kThreads)));
#define QKV_SLAB(SS, FF)                                                                             \
  build_slab_kernel<SS, FF><<<grid, kThreads, 0, st>>>(k, k_strides[0], k_strides[1], k_strides[2], \
                                                       static_cast<int>(kv_heads), static_cast<int>(t_begin), \
                                                       static_cast<int>(ntok), static_cast<int>(head_dim), \
                                                       chan_idx, slab, slab_scales, capacity, total)
#define QKV_SLAB_ALL(FF)                  \
  switch (selected) {                     \
    case 16: QKV_SLAB(16, FF); break;     \
    case 32: QKV_SLAB(32, FF); break;     \
    case 64: QKV_SLAB(64, FF); break;     \
    default: QKV_SLAB(128, FF); break;    \
  }
  if (f16) QKV_SLAB_ALL(true) else QKV_SLAB_ALL(false)
#undef QKV_SLAB_ALL
#undef QKV_SLAB
  return check_launch("qkv_int4_build_slab");
}

// Shared argument checks of the query side (scoring and query words).
static int check_query(const void* query, int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
                const int32_t* chan_idx, int64_t selected, const char* what) {
  if (!query || !chan_idx) return fail(QKV_ERR_INVALID, "%s: null query pointer", what);
  if (batch <= 0 || kv_heads <= 0 || q_heads % kv_heads)
    return fail(QKV_ERR_INVALID, "%s: q_heads must be a multiple of kv_heads", what);
  if (batch * kv_heads > 65535) return fail(QKV_ERR_INVALID, "%s: too many rows", what);
  if (head_dim != 64 && head_dim != 128) return fail(QKV_ERR_UNSUPPORTED, "%s: head_dim must be 64 or 128", what);
  if (selected != 16 && selected != 32 && selected != 64 && selected != 128)
    return fail(QKV_ERR_UNSUPPORTED, "%s: selected must be 16, 32, 64 or 128", what);
  if (selected > head_dim) return fail(QKV_ERR_INVALID, "%s: selected > head_dim", what);
  if (!aligned(query, 4)) return fail(QKV_ERR_INVALID, "%s: query must be 4-byte aligned", what);
  return QKV_OK;
}

QKV_EXPORT int qkv_int4_query_words(const void* query, int64_t batch, int64_t q_heads,
                                    int64_t kv_heads, int64_t head_dim, const int32_t* chan_idx,
                                    int64_t selected, uint32_t* qwords, float* qscale, int dtype,
                                    void* stream) {
  if (int rc = check_query(query, batch, q_heads, kv_heads, head_dim, chan_idx, selected, "qkv_int4_query_words"))
    return rc;
  bool f16;
  if (int rc = half_dtype(dtype, "qkv_int4_query_words", &f16)) return rc;
  if (!qwords) return fail(QKV_ERR_INVALID, "qkv_int4_query_words: null qwords pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned grid = static_cast<unsigned>(batch * kv_heads);
  const uint16_t* q = static_cast<const uint16_t*>(query);
  const int hq = static_cast<int>(q_heads), hkv = static_cast<int>(kv_heads), hd = static_cast<int>(head_dim);
#define QKV_QW(SS, FF) query_words_kernel<SS, FF><<<grid, 64, 0, st>>>(q, hq, hkv, hd, chan_idx, qwords, qscale)
#define QKV_QW_ALL(FF)                \
  switch (selected) {                 \
    case 16: QKV_QW(16, FF); break;   \
    case 32: QKV_QW(32, FF); break;   \
    case 64: QKV_QW(64, FF); break;   \
    default: QKV_QW(128, FF); break;  \
  }
  if (f16) QKV_QW_ALL(true) else QKV_QW_ALL(false)
#undef QKV_QW_ALL
#undef QKV_QW
  return check_launch("qkv_int4_query_words");
}

QKV_EXPORT int qkv_int4_decode_scores(const void* query, int64_t batch, int64_t q_heads,
                                      int64_t kv_heads, int64_t head_dim, const int32_t* chan_idx,
                                      int64_t selected, const uint8_t* slab,
                                      const uint16_t* slab_scales, int64_t capacity, int64_t tokens,
                                      int64_t block, float* bmax, int32_t* isum, float* keys,
                                      float* qscale, int dtype, void* stream) {
  if (int rc = check_query(query, batch, q_heads, kv_heads, head_dim, chan_idx, selected,
                           "qkv_int4_decode_scores"))
    return rc;
  bool f16;
  if (int rc = half_dtype(dtype, "qkv_int4_decode_scores", &f16)) return rc;
  if (!slab || !slab_scales) return fail(QKV_ERR_INVALID, "qkv_int4_decode_scores: null slab pointer");
  if (!bmax && !(isum && keys))
    return fail(QKV_ERR_INVALID, "qkv_int4_decode_scores: need bmax or both isum and keys");
  if ((isum == nullptr) != (keys == nullptr))
    return fail(QKV_ERR_INVALID, "qkv_int4_decode_scores: isum and keys go together");
  if (tokens <= 0 || tokens > capacity || tokens >= (int64_t(1) << 30))
    return fail(QKV_ERR_INVALID, "qkv_int4_decode_scores: need 1 <= tokens <= capacity");
  if (!aligned(slab, 16) || !aligned(slab_scales, 16))
    return fail(QKV_ERR_INVALID, "qkv_int4_decode_scores: slab and scales must be 16-byte aligned");
  if (capacity % slab_tile_keys(static_cast<int>(selected)))
    return fail(QKV_ERR_INVALID, "qkv_int4_decode_scores: capacity must be a multiple of %lld for %lld channels",
                (long long)slab_tile_keys(static_cast<int>(selected)), (long long)selected);
  const int stage = static_cast<int>(slab_tile_keys(static_cast<int>(selected)));   // keys per wave stage
  if (!pow2(block) || block > stage)
    return fail(QKV_ERR_INVALID, "qkv_int4_decode_scores: block must be a power of two <= %d", stage);
  const int64_t rows = batch * kv_heads;
  const int stage_wg = kScoreWaves * stage;   // keys one workgroup stage covers
  int64_t chunk = cdiv(rows * tokens, QKV_SCORE_TARGET_WGS);
  chunk = std::max<int64_t>(stage_wg, cdiv(chunk, stage_wg) * stage_wg);
  dim3 grid(static_cast<unsigned>(cdiv(tokens, chunk)), static_cast<unsigned>(rows));
  const int nb = static_cast<int>(cdiv(tokens, block));
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint16_t* q = static_cast<const uint16_t*>(query);
  const int hq = static_cast<int>(q_heads), hkv = static_cast<int>(kv_heads), hd = static_cast<int>(head_dim);
#define QKV_SC(DBG, FF, IS, KS)                                                                      \
  return launch_scores<DBG, FF>(static_cast<int>(selected), grid, st, q, hq, hkv, hd, chan_idx, slab,  \
                                slab_scales, capacity, static_cast<int>(tokens), static_cast<int>(block), \
                                static_cast<int>(chunk), bmax, nb, IS, KS, qscale)
  if (isum) {
    if (f16) QKV_SC(true, true, isum, keys);
    QKV_SC(true, false, isum, keys);
  }
  if (f16) QKV_SC(false, true, nullptr, nullptr);
  QKV_SC(false, false, nullptr, nullptr);
#undef QKV_SC
}

namespace qkv {
int topk_filtered(const float* values, int64_t rows, int64_t n, int64_t ld, int64_t k, int32_t* out,
                  void* workspace, hipStream_t st, bool given);
bool topk_takes_windows(int64_t n, int64_t k);
bool topk_takes_row_hist(int64_t rows, int64_t n, int64_t k, const void* workspace, int64_t bytes, bool counted,
                         bool kept);
int64_t topk_hist_stride();
int topk_big_clear(int64_t rows, int64_t n, void* workspace, hipStream_t st, int** hist, int64_t* stride);
int topk_big_finish(const float* values, int64_t rows, int64_t n, int64_t ld, int64_t k, int32_t* out,
                    void* workspace, int* state, hipStream_t st);
void topk_state_clear(int64_t rows, int* state, hipStream_t st);
}  // namespace qkv

QKV_EXPORT int qkv_int4_decode_topk(const void* query, int64_t batch, int64_t q_heads, int64_t kv_heads,
                                    int64_t head_dim, const int32_t* chan_idx, int64_t selected,
                                    const uint8_t* slab, const uint16_t* slab_scales, int64_t capacity,
                                    int64_t tokens, int64_t k, float* scores, int32_t* out, void* workspace,
                                    int64_t workspace_bytes, int dtype, void* stream) {
  return qkv_int4_decode_topk_state(query, batch, q_heads, kv_heads, head_dim, chan_idx, selected, slab, slab_scales,
                                    capacity, tokens, k, scores, out, workspace, workspace_bytes, nullptr, 0, dtype,
                                    stream);
}

QKV_EXPORT int qkv_int4_decode_topk_state(const void* query, int64_t batch, int64_t q_heads, int64_t kv_heads,
                                          int64_t head_dim, const int32_t* chan_idx, int64_t selected,
                                          const uint8_t* slab, const uint16_t* slab_scales, int64_t capacity,
                                          int64_t tokens, int64_t k, float* scores, int32_t* out, void* workspace,
                                          int64_t workspace_bytes, void* state, int64_t state_bytes, int dtype,
                                          void* stream) {
  static const char* what = "qkv_int4_decode_topk";
  if (int rc = check_query(query, batch, q_heads, kv_heads, head_dim, chan_idx, selected, what)) return rc;
  bool f16;
  if (int rc = half_dtype(dtype, what, &f16)) return rc;
  if (!slab || !slab_scales || !scores || !out) return fail(QKV_ERR_INVALID, "%s: null pointer", what);
  if (tokens <= 0 || tokens > capacity || tokens >= (int64_t(1) << 30))
    return fail(QKV_ERR_INVALID, "%s: need 1 <= tokens <= capacity", what);
  if (k < 1 || k > tokens) return fail(QKV_ERR_INVALID, "%s: need 1 <= k <= tokens", what);
  if (!aligned(slab, 16) || !aligned(slab_scales, 16))
    return fail(QKV_ERR_INVALID, "%s: slab and scales must be 16-byte aligned", what);
  if (capacity % slab_tile_keys(static_cast<int>(selected)))
    return fail(QKV_ERR_INVALID, "%s: capacity must be a multiple of %lld for %lld channels", what,
                (long long)slab_tile_keys(static_cast<int>(selected)), (long long)selected);
  const int64_t rows = batch * kv_heads;
  const int64_t need = topk_least_bytes(rows, tokens, k);
  if (need < 0 || workspace_bytes < need || (need > 0 && !workspace))
    return fail(QKV_ERR_INVALID, "%s: workspace needs %lld bytes, got %lld", what, (long long)need,
                (long long)workspace_bytes);
  if (need > 0 && !aligned(workspace, 16)) return fail(QKV_ERR_INVALID, "%s: workspace must be 16-byte aligned", what);
  const bool row_hist = topk_takes_row_hist(rows, tokens, k, workspace, workspace_bytes, true, state != nullptr);
  if (!(topk_takes_windows(tokens, k) || row_hist) || rows > 65535) {   // the scores, then qkv_topk_ws as it stands
    if (int rc = qkv_int4_decode_scores(query, batch, q_heads, kv_heads, head_dim, chan_idx, selected, slab,
                                        slab_scales, capacity, tokens, 1, scores, nullptr, nullptr, nullptr, dtype,
                                        stream))
      return rc;
    return qkv_topk_ws(scores, rows, tokens, tokens, k, out, workspace, workspace_bytes, stream);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int n_chunks = static_cast<int>(cdiv(tokens, kStageChunk));
  dim3 grid(static_cast<unsigned>(n_chunks), static_cast<unsigned>(rows));
  const uint16_t* q = static_cast<const uint16_t*>(query);
  int32_t* win = static_cast<int32_t*>(workspace);   // qkv_topk_ws's window region
  int* hist = nullptr;
  int64_t hist_stride = 0;
  const bool kept = row_hist && state;   // a zero-filled state the caller keeps: nothing to clear
  if (row_hist) {
    if (kept) {
      const int64_t need_state = qkv_topk_state_bytes(rows, tokens, k);
      if (state_bytes < need_state || !aligned(state, 16))
        return fail(QKV_ERR_INVALID, "%s: the state needs %lld bytes (16-byte aligned), got %lld", what,
                    (long long)need_state, (long long)state_bytes);
      hist = static_cast<int*>(state);
      hist_stride = topk_hist_stride();
    } else if (int rc = topk_big_clear(rows, tokens, workspace, st, &hist, &hist_stride)) {
      return rc;
    }
  }
  auto launch = [&](auto sc, auto fc) {
    constexpr int SS = decltype(sc)::value;
    constexpr bool FF = decltype(fc)::value;
    decode_scores_win_kernel<SS, FF><<<grid, 64 * win_waves(SS), 0, st>>>(
        q, static_cast<int>(q_heads), static_cast<int>(kv_heads), static_cast<int>(head_dim), chan_idx, slab,
        slab_scales, capacity, static_cast<int>(tokens), static_cast<int>(k), scores, n_chunks, win, hist,
        hist_stride, nullptr);
    return check_launch(what);
  };
  auto with_f = [&](auto sc) {
    return f16 ? launch(sc, std::true_type{}) : launch(sc, std::false_type{});
  };
  int rc;
  switch (selected) {
    case 16: rc = with_f(std::integral_constant<int, 16>{}); break;
    case 32: rc = with_f(std::integral_constant<int, 32>{}); break;
    case 64: rc = with_f(std::integral_constant<int, 64>{}); break;
    case 128: rc = with_f(std::integral_constant<int, 128>{}); break;
    default: return fail(QKV_ERR_UNSUPPORTED, "%s: selected channel count %lld not built", what, (long long)selected);
  }
  if (!rc && row_hist)
    rc = topk_big_finish(scores, rows, tokens, tokens, k, out, workspace, kept ? hist : nullptr, st);
  if (rc && kept) topk_state_clear(rows, hist, st);   // the scores may have been counted
  if (rc || row_hist) return rc;
  return topk_filtered(scores, rows, tokens, tokens, k, out, workspace, st, true);
}
