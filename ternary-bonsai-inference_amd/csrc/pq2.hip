// PQ2_0 embedding gather-dequant for gfx950, alone and fused with RMSNorm.
//
//   bh_pq2_embed_gather      batched Weights::row_f32 on token_embd.weight
//                            (src/weights.rs:333-349, src/prefill.rs:143-154)
//                            = kernels::decode_pq2_0_row per id (src/kernels.rs:214-229)
//   bh_pq2_embed_gather_rms  + the first rms_norm (src/forward.rs:691, 701-702)
//
// PQ2_0 layout (src/kernels.rs:204-229): a row of ne0 weights is ceil(ne0/128)
// blocks of 34 bytes: a little-endian f16 scale, then 32 bytes holding 128
// 2-bit codes, LSB first (weight j of the block: byte j/4, bits 2*(j%4)).
// Weight = (code - 1) * scale.
//
// Design.  One float4 of output per lane over the flat [n_ids][ne0/4]
// range: the lane reads its 128-block's f16 scale (an aligned halfword:
// blocks start on even bytes) and one code byte -- exactly the 4 weights of
// its float4 -- and stores 16 bytes.  The output (20 KB per row) dominates the
// traffic; the packed read (1360 B per row, cache-resident across the 320
// lanes that share it) is 1/15 of it.
//
// Fused RMSNorm, bit-exact.  The reference sums the 5120 squares of a row
// one after another in f32 (src/kernels.rs:65-68); on quantised embedding
// rows that sequence drifts ~1e-5 from any tree-ordered sum, so the fused
// kernels reproduce the sequence itself.  On ternary codes a 128-block adds
// d*d as many times as it has codes other than 1, a run that seqsum.hpp
// evaluates exactly without its additions.  Up to 16 rows per CU one launch:
// a workgroup per row, one wave taking the row's runs by turns (a lane per
// block; code 3 adds 4 d*d, see wave_row_ss) under the embedding stores, then
// the norm row.  Its time is the launch, the row's first touch and about 16
// turns: T = 1 8.4 us, 256 11.5, 2048 17.2 (5.0 TB/s of 86.7 MB); a chain of
// the 5120 additions, a lane per row, took 22.7, 27.8 and 29.5.  Longer
// batches: two launches of flat writers (below), the sums walked a lane per
// row under the stores.
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "common.hpp"
#include "seqsum.hpp"

namespace bh {
namespace {

constexpr int kBlock = 256;
constexpr int kPq2Block = 34;
constexpr size_t kMaxSeqSmem = 128 * 1024;  // LDS cap of a fused block (gfx950: 160 KB per CU)


struct GatherArgs {
  const uint8_t *table;
  const uint32_t *ids;
  float *out;       // embedding rows
  float *out_norm;  // norm rows
  const float *w;
  uint32_t *bad_id;
  int row_bytes, ne0, n_ids;
  uint32_t n_rows;
  float eps;
};

// Decodes float4 f of the packed row at `rowb` straight from global memory
// (the scale halfword and one code byte; a block starts on an even byte, so
// the halfword load is aligned).
__device__ __forceinline__ float4 decode4_global(const uint8_t *rowb, int f) {
  const uint8_t *blk = rowb + (f >> 5) * kPq2Block;
  const uint32_t h = *reinterpret_cast<const uint16_t *>(blk);
  const uint32_t c = blk[2 + (f & 31)];
  const float scale = __uint_as_float(half_bits_to_f32_bits(h));
  const bool finite = (h & 0x7c00u) != 0x7c00u;
  return make_float4(pq2_weight(c & 3u, scale, finite), pq2_weight((c >> 2) & 3u, scale, finite),
                     pq2_weight((c >> 4) & 3u, scale, finite),
                     pq2_weight((c >> 6) & 3u, scale, finite));
}

// ---------------------------------------------------------------------------
// Gather + RMSNorm, one workgroup per row: wave 0 forms the row's sum of
// squares -- one lane per 128-block (windows of 64 blocks), by turns -- while
// the other waves write the embedding row; then all write the norm row.
// ---------------------------------------------------------------------------
constexpr int kRowThreads = 256;

// Inclusive prefix sum over the wave's 64 lanes (all active): DPP row shifts,
// then the last lane of each 16-lane row and of the lower half passed on.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
  auto add = [&](auto ctrl, auto rows) {
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), decltype(ctrl)::value,
                                                           decltype(rows)::value, 0xF, false));
  };
  add(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xF>{});  // row_shr:1
  add(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xF>{});
  add(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xF>{});
  add(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xF>{});
  add(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});  // row_bcast:15
  add(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});  // row_bcast:31
  return v;
}

// LDS of a wave that adds blocks weight by weight: the window's codes, eight
// words a block, and one block's squares.
struct HandLds {
  uint32_t codes[64 * 8];
  float sq[128];
};

// Adds the `valid` squares of block f of the window, whose scale bits are h, to
// s in order, on one whole wave.  They pass through LDS, from where every lane
// reads the same four at a time; squares past `valid` are +0, which leaves any
// sum of squares as it is.
__device__ __forceinline__ float wave_block_ss(float s, HandLds &m, int f, uint32_t h, int valid) {
  const int lane = threadIdx.x & 63;
  const float d = __uint_as_float(half_bits_to_f32_bits(h));
  const bool finite = (h & 0x7c00u) != 0x7c00u;
#pragma unroll
  for (int j = lane; j < 128; j += 64) {
    const float v = pq2_weight((m.codes[8 * f + (j >> 4)] >> (2 * (j & 15))) & 3u, d, finite);
    m.sq[j] = j < valid ? v * v : 0.0f;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const float4 *q4 = reinterpret_cast<const float4 *>(m.sq);
#pragma unroll 8
  for (int j = 0; j < 32; ++j) {
    const float4 q = q4[j];
    s += q.x;  // src/kernels.rs:65-68
    s += q.y;
    s += q.z;
    s += q.w;
  }
  return s;
}

// The reference's sequential f32 sum of squares of the packed row, bit for
// bit, on one whole wave.  A block with code 3 holds squares of d d and of 4 d d;
// it is added in closed form where it stays in the sum's binade and weight by
// weight where not (a fifth of the blocks of four codes; a block of a
// non-finite scale always).  Rows of four codes, T = 1 / 256 / 2048: 11.8 / 15.5
// / 20.3 us, against 9.6 / 12.4 / 18.7 for three codes and 23.0 / 27.7 / 30.4 by
// a chain of all 5120 additions; with every block of code 3 weight by weight
// 29.5 / 31.1 / 39.0.
__device__ __forceinline__ float wave_row_ss(const uint8_t *row, int ne0, int nblk, HandLds &hl) {
  const int lane = threadIdx.x & 63;
  float s = 0.0f;
  for (int b0 = 0; b0 < nblk; b0 += 64) {
    const int b = b0 + lane;
    float x = 0.0f;
    uint32_t n = 0, n4 = 0, h = 0;  // squares of d d and of 4 d d still to add
    bool finite = true;
    if (b < nblk) {
      // the block's 34 bytes as eight aligned words and a halfword
      const bool even = (b & 1) == 0;
      const uint8_t *blk = row + static_cast<size_t>(b) * kPq2Block;
      const uint32_t *w32 = reinterpret_cast<const uint32_t *>(blk + (even ? 0 : 2));
      const uint32_t h16 = *reinterpret_cast<const uint16_t *>(blk + (even ? 32 : 0));
      uint32_t dw[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) dw[k] = w32[k];
      h = even ? (dw[0] & 0xffffu) : h16;
      const int valid = ne0 - b * 128 < 128 ? ne0 - b * 128 : 128;
      uint32_t ones = 0, threes = 0, w[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {  // 16 codes a word
        const uint32_t nx = k < 7 ? dw[k < 7 ? k + 1 : 0] : h16;
        w[k] = even ? ((dw[k] >> 16) | (nx << 16)) : dw[k];
        const int lo = valid - 16 * k;
        const uint32_t mask =
            lo >= 16 ? 0x55555555u : (lo <= 0 ? 0u : 0x55555555u & ((1u << (2 * lo)) - 1u));
        const uint32_t t = w[k] ^ 0x55555555u;  // code 1 -> 00
        ones += __popc(~(t | (t >> 1)) & mask);
        threes += __popc(w[k] & (w[k] >> 1) & mask);
      }
      const float d = __uint_as_float(half_bits_to_f32_bits(h));
      x = d * d;
      finite = (h & 0x7c00u) != 0x7c00u;
      if (x != 0.0f) {  // d = 0: squares of +0
        n = static_cast<uint32_t>(valid) - ones - threes;
        n4 = threes;
      }
      if (!finite || n4 != 0u) {
        n = finite ? n : 1u;
        uint4 *c = reinterpret_cast<uint4 *>(hl.codes + 8 * lane);
        c[0] = make_uint4(w[0], w[1], w[2], w[3]);
        c[1] = make_uint4(w[4], w[5], w[6], w[7]);
      }
    }
    const uint64_t hand = __ballot(!finite || n4 != 0u);
    // HAND: the window has blocks of code 3 or a non-finite scale
    auto turns = [&](auto hand_c) {
      constexpr bool HAND = decltype(hand_c)::value;
      for (;;) {
        const uint32_t sb = __builtin_amdgcn_readfirstlane(__float_as_uint(s));
        const int es = static_cast<int>(sb >> 23);
        const SeqUnits u = seq_units(es, x);
        const SeqUnits u4 = HAND ? seq_units(es, 4.0f * x) : u;
        const uint32_t inc =
            HAND ? (finite ? seq_mixed_added(n, u, n4, u4) : 0u) : (n != 0u ? seq_units_added(n, u) : 0u);
        const uint32_t upto = wave_prefix(inc);
        const uint32_t start = sb + (upto - inc);
        const SeqStep step = seq_step(start, x, n, u);
        bool whole = n == 0u || step.whole;
        if constexpr (HAND) {
          if (n4 != 0u) whole = seq_mixed_whole(start, inc, n, u, n4, u4);
          whole = whole && (finite || n == 0u);
        }
        const uint64_t stay = __ballot(!whole);
        if (stay == 0u) {
          s = __uint_as_float(sb + __builtin_amdgcn_readlane(upto, 63));
          break;
        }
        const int f = __builtin_ctzll(stay);
        uint32_t left = 0;
        if (HAND && ((hand >> f) & 1u) != 0u) {
          const int rest = ne0 - (b0 + f) * 128;
          s = wave_block_ss(__uint_as_float(__builtin_amdgcn_readlane(start, f)), hl, f,
                            __builtin_amdgcn_readlane(h, f), rest < 128 ? rest : 128);
        } else {
          s = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(step.s), f));
          left = __builtin_amdgcn_readlane(step.left, f);
        }
        n = lane < f ? 0u : (lane == f ? left : n);
        if constexpr (HAND) n4 = lane <= f ? 0u : n4;
      }
    };
    if (hand != 0u)
      turns(std::true_type{});
    else
      turns(std::false_type{});
  }
  return s;
}

template <int T>
__global__ __launch_bounds__(T) void pq2_gather_row_kernel(GatherArgs a) {
  __shared__ float row_scale;
  __shared__ __attribute__((aligned(16))) HandLds hand;
  const size_t t = blockIdx.x;
  const uint32_t id = a.ids[t];
  const int n4 = a.ne0 >> 2;
  float4 *oe = reinterpret_cast<float4 *>(a.out) + t * n4;
  float4 *on = reinterpret_cast<float4 *>(a.out_norm) + t * n4;
  if (id >= a.n_rows) {
    if (threadIdx.x == 0 && a.bad_id != nullptr) *a.bad_id = id;
    for (int f = threadIdx.x; f < n4; f += T) {
      store_stream(oe + f, make_float4(0.f, 0.f, 0.f, 0.f));
      store_stream(on + f, make_float4(0.f, 0.f, 0.f, 0.f));
    }
    return;
  }
  const uint8_t *row = a.table + static_cast<size_t>(id) * a.row_bytes;
  if (threadIdx.x < 64) {
    __builtin_amdgcn_s_setprio(3);  // the other waves wait for this one
    const float ss = wave_row_ss(row, a.ne0, a.row_bytes / kPq2Block, hand);
    // src/kernels.rs:69-70: mean = ss / n; scale = 1 / sqrt(mean + eps)
    if (threadIdx.x == 0) row_scale = 1.0f / sqrtf(ss / static_cast<float>(a.ne0) + a.eps);
    __builtin_amdgcn_s_setprio(0);
  } else {
    for (int f = threadIdx.x - 64; f < n4; f += T - 64) store_stream(oe + f, decode4_global(row, f));
  }
  __syncthreads();
  const float rs = row_scale;
  for (int f = threadIdx.x; f < n4; f += T) {
    const float4 wv = reinterpret_cast<const float4 *>(a.w)[f];
    const float4 v = decode4_global(row, f);
    // src/kernels.rs:71-73
    store_stream(on + f, make_float4((v.x * rs) * wv.x, (v.y * rs) * wv.y, (v.z * rs) * wv.z,
                                     (v.w * rs) * wv.w));
  }
}

// ---------------------------------------------------------------------------
// Gather + RMSNorm in two launches with flat writers.
// ---------------------------------------------------------------------------
// Launch 1 (pq2_scale_embed_kernel): its first blocks compute every row's
// 1 / sqrt(ss / n + eps)
// with ss the reference's sequential f32 sum of squares, bit for bit, without
// decoding the row: on a block of ternary codes (0, 1, 2) every square is d*d
// or +0, and +0 leaves the sum unchanged, so the block adds d*d as many times
// as it has codes other than 1 -- a run that repeat_add_f32 evaluates in
// closed form.  A block holding code 3 (square 4*d*d) or a non-finite scale
// is added weight by weight instead.  One lane walks one row, so the walk is
// a chain of ~55 dependent steps (one per block plus one per binade the sum
// crosses, ~20 us); the launch's other blocks write the embedding rows from a
// flat grid meanwhile.  Launch 2 (pq2_norm_write_kernel) writes the norm rows
// from a flat grid.  Both writers keep the streaming-store shape: no block
// stores a region longer than 4 KB.
constexpr int kScaleRows = 16;  // rows per scale block: one per lane of its walk

// Logical block of physical block p when a grid of 8 * per blocks is
// numbered XCD-contiguously: the hardware hands block p to XCD p % 8, and
// that XCD takes logical blocks [(p % 8) * per, (p % 8 + 1) * per) in order.
// (Only the speed depends on that dispatch order, never the results.)
__device__ __forceinline__ unsigned xcd_block(unsigned p, unsigned per) {
  return (p & 7u) * per + (p >> 3);
}

// Sum-of-squares summary of one 128-weight block of a staged row: the run
// value d*d (f32 bits) and the run length, or the fallback flag.
struct BlockRun {
  uint32_t xbits;
  uint32_t n;  // bit 31: add this block weight by weight
};

// Scale block `sblk` of launch 1: rows sblk*kScaleRows .. (+kScaleRows).
__device__ __forceinline__ void row_scale_block(const GatherArgs &a, float *row_scale,
                                                unsigned sblk, BlockRun *runs) {
  const int nblk = a.row_bytes / kPq2Block;
  const int tid = threadIdx.x;
  const size_t row0 = static_cast<size_t>(sblk) * kScaleRows;
  const int nr = (a.n_ids - static_cast<int>(row0)) < kScaleRows ? a.n_ids - static_cast<int>(row0)
                                                                 : kScaleRows;
  // one lane per (row, block), straight from the table: count the codes
  // other than 1 among the block's valid weights, flag code 3 and
  // non-finite scales.  The block's 34 bytes start on an even byte: eight
  // aligned words and one halfword cover them without reading past it.
  // A lane takes up to kScalePairs pairs per round and issues all their
  // loads (ids, then table words) before it uses any: under the writers'
  // HBM traffic a load round trip is long, and the walk waits for this.
  constexpr int kScalePairs = 4;
  const int total = nr * nblk;
  for (int base = 0; base < total; base += 256 * kScalePairs) {
    uint32_t idp[kScalePairs];
#pragma unroll
    for (int p = 0; p < kScalePairs; ++p) {
      const int i = base + p * 256 + tid;
      idp[p] = i < total ? a.ids[row0 + i / nblk] : a.n_rows;
    }
    uint32_t dw[kScalePairs][8];
    uint32_t h16[kScalePairs];
#pragma unroll
    for (int p = 0; p < kScalePairs; ++p) {
      const int i = base + p * 256 + tid;
      const int b = i - (i / nblk) * nblk;
      const bool even = (b & 1) == 0;  // block start 4-aligned (rows are 16-aligned)
      h16[p] = 0u;
#pragma unroll
      for (int k = 0; k < 8; ++k) dw[p][k] = 0u;
      if (idp[p] < a.n_rows) {
        const uint8_t *blk = a.table + static_cast<size_t>(idp[p]) * a.row_bytes + b * kPq2Block;
        const uint32_t *w32 = reinterpret_cast<const uint32_t *>(blk + (even ? 0 : 2));
        h16[p] = *reinterpret_cast<const uint16_t *>(blk + (even ? 32 : 0));
#pragma unroll
        for (int k = 0; k < 8; ++k) dw[p][k] = w32[k];
      }
    }
#pragma unroll
    for (int p = 0; p < kScalePairs; ++p) {
      const int i = base + p * 256 + tid;
      if (idp[p] >= a.n_rows) continue;  // past the pairs, or a bad id (no scale)
      const int b = i - (i / nblk) * nblk;
      const bool even = (b & 1) == 0;
      const uint32_t h = even ? (dw[p][0] & 0xffffu) : h16[p];
      const int valid = (a.ne0 - b * 128) < 128 ? a.ne0 - b * 128 : 128;
      uint32_t ones = 0, threes = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k) {  // 16 codes per 32-bit word
        const uint32_t w =
            even ? ((dw[p][k] >> 16) | ((k < 7 ? dw[p][k < 7 ? k + 1 : 0] : h16[p]) << 16)) : dw[p][k];
        const int lo = valid - 16 * k;
        const uint32_t mask = lo >= 16 ? 0x55555555u : (lo <= 0 ? 0u : 0x55555555u & ((1u << (2 * lo)) - 1u));
        const uint32_t t = w ^ 0x55555555u;  // code 1 -> 00
        ones += __popc(~(t | (t >> 1)) & mask);
        threes |= w & (w >> 1) & mask;
      }
      const bool finite = (h & 0x7c00u) != 0x7c00u;
      const float d = __uint_as_float(half_bits_to_f32_bits(h));
      BlockRun br;
      br.xbits = __float_as_uint(d * d);
      br.n = static_cast<uint32_t>(valid) - ones;
      if (threes != 0u || !finite) br.n |= 0x80000000u;
      runs[i] = br;
    }
  }
  __syncthreads();
  if (tid >= nr) return;
  const uint32_t id = a.ids[row0 + tid];
  if (id >= a.n_rows) return;
  // the walk is the launch's latency-critical path: its wave goes first
  // when it shares a SIMD with the writer waves
  __builtin_amdgcn_s_setprio(3);
  const BlockRun *rr = runs + tid * nblk;
  // Each lane walks its own row's blocks; one repeat_add_step_f32 per loop
  // trip, and a lane whose block is done moves to its next one in the same
  // trip, so the wave's trips are the most any of its rows needs rather
  // than the sum of per-block maxima.
  float ss = 0.0f;
  int b = 0;
  BlockRun cur = rr[0];
  BlockRun next = rr[nblk > 1 ? 1 : 0];  // an index select: both from LDS
  while (b < nblk) {
    uint32_t left = cur.n;
    if (left & 0x80000000u) {
      // weight by weight, as src/kernels.rs:65-68 (code 3 or a non-finite scale)
      const uint8_t *blk = a.table + static_cast<size_t>(id) * a.row_bytes + b * kPq2Block;
      const uint32_t h = *reinterpret_cast<const uint16_t *>(blk);
      const float sc = __uint_as_float(half_bits_to_f32_bits(h));
      const bool finite = (h & 0x7c00u) != 0x7c00u;
      const int valid = (a.ne0 - b * 128) < 128 ? a.ne0 - b * 128 : 128;
      for (int j = 0; j < valid; ++j) {
        const uint32_t code = (static_cast<uint32_t>(blk[2 + (j >> 2)]) >> ((j & 3) * 2)) & 3u;
        const float v = pq2_weight(code, sc, finite);
        ss += v * v;  // no contraction: built with -ffp-contract=off
      }
      left = 0u;
    } else if (left != 0u && cur.xbits != 0u) {
      left = repeat_add_step_f32(ss, __uint_as_float(cur.xbits), left);
    } else {
      left = 0u;  // d = 0 or only code 1: the squares are all +0
    }
    cur.n = left;
    if (left == 0u) {
      ++b;
      cur = next;
      if (b + 1 < nblk) next = rr[b + 1];
    }
  }
  // src/kernels.rs:69-70: mean = ss / n; scale = 1 / sqrt(mean + eps)
  row_scale[row0 + tid] = 1.0f / sqrtf(ss / static_cast<float>(a.ne0) + a.eps);
}

// Launch 1: blocks [0, n_scale) compute the row scales (dispatched first, so
// their walks run under the stores), the rest write the embedding rows, one
// float4 per lane over the flat [n_ids][ne0/4] range.
__global__ __launch_bounds__(256) void pq2_scale_embed_kernel(GatherArgs a, float *row_scale,
                                                              unsigned n_scale, unsigned s_per,
                                                              unsigned e_per) {
  extern __shared__ BlockRun runs[];  // [kScaleRows][nblk]
  if (blockIdx.x < n_scale) {
    // scale blocks in the same XCD-contiguous order as the writers, so a
    // row's summary pass runs on the XCD that writes it
    const unsigned sblk = xcd_block(blockIdx.x, s_per);
    if (sblk * kScaleRows < static_cast<unsigned>(a.n_ids)) row_scale_block(a, row_scale, sblk, runs);
    return;
  }
  // one float4 per lane; the writer blocks are numbered XCD-contiguously:
  // the blocks one XCD runs (every 8th) write one contiguous range of rows,
  // so each gathered row is fetched into one XCD's L2 (and its address
  // translations warmed there) instead of the five XCDs its 5 blocks would
  // otherwise spread over
  const uint32_t n4 = static_cast<uint32_t>(a.ne0) >> 2;
  const uint32_t idx = xcd_block(blockIdx.x - n_scale, e_per) * 256u + threadIdx.x;
  if (idx >= static_cast<uint32_t>(a.n_ids) * n4) return;
  const uint32_t t = idx / n4;
  const uint32_t f = idx - t * n4;
  const uint32_t id = a.ids[t];
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (id < a.n_rows) {
    v = decode4_global(a.table + static_cast<size_t>(id) * a.row_bytes, f);
  } else if (f == 0 && a.bad_id != nullptr) {
    *a.bad_id = id;
  }
  store_stream(reinterpret_cast<float4 *>(a.out) + idx, v);
}

size_t scale_smem_bytes(size_t row_bytes) {
  return kScaleRows * (row_bytes / kPq2Block) * sizeof(BlockRun);
}

// Plain gather: one float4 of output per lane over the flat [n_ids][ne0/4]
// range (fits 32 bits: checked by the host).
__global__ __launch_bounds__(256) void pq2_rows_write_kernel(GatherArgs a, unsigned per) {
  const uint32_t n4 = static_cast<uint32_t>(a.ne0) >> 2;
  // XCD-contiguous block order: a row's blocks share one XCD's L2
  const uint32_t idx = xcd_block(blockIdx.x, per) * 256u + threadIdx.x;
  if (idx >= static_cast<uint32_t>(a.n_ids) * n4) return;
  const uint32_t t = idx / n4;
  const uint32_t f = idx - t * n4;
  const uint32_t id = a.ids[t];
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  if (id < a.n_rows) {
    o = decode4_global(a.table + static_cast<size_t>(id) * a.row_bytes, f);
  } else if (f == 0 && a.bad_id != nullptr) {
    *a.bad_id = id;
  }
  store_stream(reinterpret_cast<float4 *>(a.out) + idx, o);
}

// Launch 2: the norm rows (v * scale) * w (src/kernels.rs:71-73), one float4
// per lane over the flat [n_ids][ne0/4] range, with the row scales of
// launch 1 (bad ids: zeros, as the embedding rows).
__global__ __launch_bounds__(256) void pq2_norm_write_kernel(GatherArgs a, const float *row_scale,
                                                             unsigned per) {
  const uint32_t n4 = static_cast<uint32_t>(a.ne0) >> 2;
  const uint32_t idx = xcd_block(blockIdx.x, per) * 256u + threadIdx.x;  // as launch 1
  if (idx >= static_cast<uint32_t>(a.n_ids) * n4) return;
  const uint32_t t = idx / n4;
  const uint32_t f = idx - t * n4;
  const uint32_t id = a.ids[t];
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  if (id < a.n_rows) {
    const float rs = row_scale[t];
    const float4 wv = reinterpret_cast<const float4 *>(a.w)[f];
    const float4 v = decode4_global(a.table + static_cast<size_t>(id) * a.row_bytes, f);
    o = make_float4((v.x * rs) * wv.x, (v.y * rs) * wv.y, (v.z * rs) * wv.z, (v.w * rs) * wv.w);
  }
  store_stream(reinterpret_cast<float4 *>(a.out_norm) + idx, o);
}

// Any ne0 / alignment: byte reads straight from the table.
template <bool NORM>
__global__ __launch_bounds__(kBlock) void pq2_gather_loop_kernel(
    const uint8_t *__restrict__ table, size_t row_bytes, int ne0, uint32_t n_rows,
    const uint32_t *__restrict__ ids, float *__restrict__ out, const float *__restrict__ w,
    float eps, float *__restrict__ out_norm, uint32_t *bad_id) {
  __shared__ float lds[kBlock / 64];
  const size_t t = blockIdx.x;
  const uint32_t id = ids[t];
  float *orow = out + t * ne0;
  if (id >= n_rows) {
    if (bad_id != nullptr && threadIdx.x == 0) *bad_id = id;
    for (int j = threadIdx.x; j < ne0; j += kBlock) {
      orow[j] = 0.0f;
      if constexpr (NORM) out_norm[t * ne0 + j] = 0.0f;
    }
    return;
  }
  const uint8_t *rowb = table + static_cast<size_t>(id) * row_bytes;
  auto weight = [&](int j) {
    const uint8_t *blk = rowb + (j >> 7) * kPq2Block;
    const uint32_t h = static_cast<uint32_t>(blk[0]) | (static_cast<uint32_t>(blk[1]) << 8);
    const int jj = j & 127;
    const uint32_t code = (static_cast<uint32_t>(blk[2 + (jj >> 2)]) >> ((jj & 3) * 2)) & 3u;
    return pq2_weight(code, __uint_as_float(half_bits_to_f32_bits(h)), (h & 0x7c00u) != 0x7c00u);
  };
  for (int j = threadIdx.x; j < ne0; j += kBlock) orow[j] = weight(j);
  if constexpr (NORM) {
    // the reference's sequential f32 sum (src/kernels.rs:65-68), one lane;
    // this path only serves layouts the staged kernels cannot take
    __syncthreads();
    if (threadIdx.x == 0) {
      float ss = 0.0f;
      for (int j = 0; j < ne0; ++j) ss += orow[j] * orow[j];
      lds[0] = 1.0f / sqrtf(ss / static_cast<float>(ne0) + eps);
    }
    __syncthreads();
    const float scale = lds[0];
    for (int j = threadIdx.x; j < ne0; j += kBlock)
      out_norm[t * ne0 + j] = (weight(j) * scale) * w[j];
  }
}

int gather_impl(const uint8_t *table, size_t ne0, size_t n_rows, const uint32_t *ids,
                size_t n_ids, const float *w, float eps, float *out, float *out_norm,
                uint32_t *bad_id, hipStream_t st, bool norm) {
  if (n_ids == 0 || ne0 == 0) return ok();
  if (ne0 > 0x7fffffffu || n_ids > 0x7fffffffu)
    return fail(BH_ERR_SHAPE, "pq2 gather: ne0 or n_ids exceeds 2^31-1");
  if (n_rows > 0xffffffffu) return fail(BH_ERR_SHAPE, "pq2 gather: n_rows exceeds 2^32-1");
  const size_t row_bytes = bh_pq2_row_bytes(ne0);
  const unsigned grid = static_cast<unsigned>(n_ids);
  const uint32_t nr = static_cast<uint32_t>(n_rows);
  // writers: one float4 per lane (16-byte stores, halfword table loads); the
  // two-launch form stages rows with 16-byte loads
  const bool rows_ok = (ne0 % 4 == 0) && n_ids * (ne0 / 4) < 0xfffff000u && aligned16(table) &&
                       aligned16(out) && (!norm || (aligned16(out_norm) && aligned16(w)));
  const unsigned wgrid = static_cast<unsigned>((n_ids * (ne0 / 4) + 255) / 256);
  GatherArgs ga{};
  ga.table = table;
  ga.ids = ids;
  ga.out = out;
  ga.out_norm = out_norm;
  ga.w = w;
  ga.bad_id = bad_id;
  ga.row_bytes = static_cast<int>(row_bytes);
  ga.ne0 = static_cast<int>(ne0);
  ga.n_ids = static_cast<int>(n_ids);
  ga.n_rows = nr;
  ga.eps = eps;
  if (rows_ok && !norm) {
    const unsigned per = (wgrid + 7) / 8;
    BH_LAUNCH(pq2_rows_write_kernel, 8 * per, 256, 0, st, ga, per);
    return ok();
  }
  const size_t cus = device_cu_count();
  if (rows_ok && norm && row_bytes % 16 == 0 && n_ids >= 16 * cus &&
      scale_smem_bytes(row_bytes) <= kMaxSeqSmem) {
    // Long batches: row scales + embedding rows, then the norm rows (two flat
    // writers, which stream faster than a workgroup's two rows one after the
    // other).  Measured against the kernel below (us): T = 4096 36 / 34, 6000
    // 43 / 49, 8192 56 / 66.
    float *scales = static_cast<float *>(device_scratch(n_ids * sizeof(float), kScratchGather, st));
    if (scales == nullptr) return BH_ERR_HIP;
    const size_t smem = scale_smem_bytes(row_bytes);
    if (int e = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(pq2_scale_embed_kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(smem)),
                          "hipFuncSetAttribute"))
      return e;
    const unsigned scale_blocks = static_cast<unsigned>((n_ids + kScaleRows - 1) / kScaleRows);
    const unsigned s_per = (scale_blocks + 7) / 8;
    const unsigned e_per = (wgrid + 7) / 8;
    BH_LAUNCH(pq2_scale_embed_kernel, 8 * s_per + 8 * e_per, 256, smem, st, ga, scales, 8 * s_per,
              s_per, e_per);
    BH_LAUNCH(pq2_norm_write_kernel, 8 * e_per, 256, 0, st, ga, scales, e_per);
    return ok();
  }
  if (rows_ok && norm && row_bytes % 4 == 0) {  // a block's codes are whole aligned words
    // More rows than the CUs hold workgroups of 256 lanes (8 each): short ones
    // take 128, so that all of them are under way at once.  2048 columns, us at
    // 2560 / 3072 / 4095 rows of three codes: 17.1 / 18.4 / 21.7 with 256 lanes,
    // 14.6 / 14.8 / 18.8 with 128; at 2048 rows 13.0 / 13.4, and 3072 columns at
    // 4095 rows 22.8 / 25.3, so both lines stay there.  (A wave a row and a chain
    // of all additions, a lane a row, were 22.3 and 17.0; that chain is the
    // faster one on 1024 columns too, 11.4 for 15.1 at 4095 rows.)
    if (n_ids > 8 * cus && ne0 <= 2048)
      BH_LAUNCH((pq2_gather_row_kernel<128>), grid, 128, 0, st, ga);
    else
      BH_LAUNCH((pq2_gather_row_kernel<kRowThreads>), grid, kRowThreads, 0, st, ga);
  } else {
    if (norm) {
      BH_LAUNCH((pq2_gather_loop_kernel<true>), grid, kBlock, 0, st, table, row_bytes,
                static_cast<int>(ne0), nr, ids, out, w, eps, out_norm, bad_id);
    } else {
      BH_LAUNCH((pq2_gather_loop_kernel<false>), grid, kBlock, 0, st, table, row_bytes,
                static_cast<int>(ne0), nr, ids, out, w, eps, out_norm, bad_id);
    }
  }
  return ok();
}

}  // namespace
}  // namespace bh

using namespace bh;

extern "C" int bh_pq2_embed_gather(const uint8_t *table, size_t ne0, size_t n_rows,
                                   const uint32_t *ids, size_t n_ids, float *out,
                                   uint32_t *bad_id, bh_stream stream) {
  if (n_ids && ne0 && (!table || !ids || !out))
    return fail(BH_ERR_ARG, "pq2_embed_gather: null pointer");
  return gather_impl(table, ne0, n_rows, ids, n_ids, nullptr, 0.0f, out, nullptr, bad_id,
                     as_stream(stream), false);
}

extern "C" int bh_pq2_embed_gather_rms(const uint8_t *table, size_t ne0, size_t n_rows,
                                       const uint32_t *ids, size_t n_ids, const float *w,
                                       size_t w_len, float eps, float *out_embed,
                                       float *out_norm, uint32_t *bad_id, bh_stream stream) {
  if (w_len != ne0)
    return fail(BH_ERR_SHAPE, "pq2_embed_gather_rms: weight len " + std::to_string(w_len) +
                                  " != ne0 " + std::to_string(ne0));
  if (n_ids && ne0 && (!table || !ids || !out_embed || !out_norm || !w))
    return fail(BH_ERR_ARG, "pq2_embed_gather_rms: null pointer");
  return gather_impl(table, ne0, n_rows, ids, n_ids, w, eps, out_embed, out_norm, bad_id,
                     as_stream(stream), true);
}
