// PQ2_0 products of many tokens on the block-scaled FP6 x FP4 matrix cores.
//
// Reference: kernels::pq2_matmul_n (src/kernels.rs:340-423), whose row dot
// (:633-653) adds scale * block_sum over a row's 128-weight blocks.
//
// v_mfma_scale_f32_32x32x64_f8f6f4 (D = A * B + C on a 32 x 32 tile) runs
// e2m3 x e2m1 products at four times the f16 rate, with one power-of-two
// scale (E8M0 byte) per row and 32 k-slots of A, and per column and 32
// k-slots of B:
//   B = weights: the values code - 1 in {-1, 0, 1, 2}, halved, are exact in
//       e2m1, so a block is multiplied as it is and the sum needs no
//       correction for the code's offset (a weight of 0 adds exactly 0, though
//       a large x there coarsens the step of its group's other columns);
//   A = x: each 32 columns of a token are scaled by the power of two that
//       puts their largest |x| in [2^23, 2^24), rounded to integers X and
//       written as five signed base-32 digits (-16 .. 16, exact in e2m3 as
//       digit / 8): a step of 2^-24 of the power of two above the group's
//       largest |x|, which is 24 bits for that one (what f32 itself holds) and
//       k fewer for a column 2^-k as large (the integer form: 22 bits of the
//       largest of 128 columns; the f16 form: 22 of each column).  The group's
//       power of two is the A scale, the digit's 2^(5 j) the B scale, so all
//       ten products of a 128-block (two k halves, five digits) accumulate
//       into one f32 tile and leave x in its own units;
//   then acc += d * block tile, one FMA per output and block, as the
//   reference adds scale * block_sum.
// Error against 64-bit sums (2-norm): 1.1e-7 .. 2.1e-7 on the model's shapes;
// the integer form's 22-bit x gives 3.0e-7 .. 3.5e-7.
//
// Bound: the FP6 x FP4 products themselves.  On random operands a register
// loop of this instruction reaches 5.3 .. 5.8 P products/s here (7.8 on zeros:
// the clock gives way), a fifth of that is 1.06 .. 1.16 P useful ones; int8 in
// three digits would reach 1.2 but leaves i32 sums to be combined per block
// (5 VALU operations an output against 1), f16 hi + lo 0.85.  The 16 x 16 x
// 128 form runs at half the rate.
//
// Measured (us a call, N tokens; integer form before / this now):
//   [17408 x 5120]  N=17  31 / 25    61  49 / 35   256 127 / 105  512 243 / 145
//                   1024 458 / 243   2048 906 / 440 (0.83 P useful products/s)
//   [5120 x 17408]  N=17  87 / 27    61  89 / 36   256 150 / 85   512 253 / 150
//                   2048 954 / 462
//   [248320 x 5120] N=32 251 / 146
// At 2048 tokens the products take 396 us of the 440 (350 with every load
// replaced by a repeated one), unpacking 22, the digits 20, the parts 8.
//
// Lane layout (lane l, n = l % 32, g = l / 32): A[n][32 g + e] and
// B[32 g + e][n] are k-slots e = 0 .. 31 of the lane, D[8 (i / 4) + 4 g +
// i % 4][n] its output i.  A block is two MFMA steps ("halves" h); k-slot
// e = 8 r + i of half h is block column 64 g + 32 h + 16 (r / 2) + 2 i + r % 2
// on both sides: lane group g owns 16 bytes of a block's codes, operand dword
// r holds the codes of one parity of one dword of them, a nibble each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "common.hpp"
#include "pq2_mx.hpp"
#include "pq2_mx_plan.hpp"

namespace bh {
namespace {

constexpr int kBlkBytes = 34;
constexpr int kDigits = 5;
typedef int i8v __attribute__((ext_vector_type(8)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

// x record of one (32-token tile, 128-block): 2 x 5 operand planes [h][digit]
// of 64 lanes, first the lanes' dwords 0-3, then dwords 4-5, then a dword a
// lane with the A scale bytes of h = 0, 1; rounded up to whole 16 KB.
constexpr int kXHi = 2 * kDigits * 1024;
constexpr int kXScale = kXHi + 2 * kDigits * 512;
constexpr int kXRec = kMxXRec;
// weight record of one (32-row tile, 128-block): operand planes [h] of 64
// lanes x 16 bytes; the f32 block scales stand in an array of their own.
constexpr int kWRec = kMxWRec;

// Column of a lane's 32 of a half that k-slot e stands for.
__host__ __device__ constexpr int mx_column(int e) {
  return 16 * (e >> 4) + 2 * (e & 7) + ((e >> 3) & 1);
}

struct XPrepArgs {
  const float *x;  // [n_tok][ne0]
  uint8_t *rec;    // [tiles][nblk] records
  int ne0, n_tok, nblk;
  size_t items;    // tiles * nblk * 2
};

// One wave per (32-token tile, block, k half); lane (n, g) turns the 32
// columns of its token and lane group into digits.  Bound by the integer
// work (about 30 operations an element).
__global__ __launch_bounds__(256) void pq2_mx_xprep_kernel(XPrepArgs a) {
  const size_t item = static_cast<size_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (item >= a.items) return;
  const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
  const int h = static_cast<int>(item & 1);
  const size_t tb = item >> 1;
  const size_t tile = tb / static_cast<size_t>(a.nblk);
  const int b = static_cast<int>(tb - tile * a.nblk);
  const size_t t = tile * 32 + n;
  float f[32];
  if (t < static_cast<size_t>(a.n_tok)) {
    const float4 *xr = reinterpret_cast<const float4 *>(a.x + t * a.ne0 + 128 * b + 64 * g + 32 * h);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float4 v = xr[q];
      f[4 * q] = v.x;
      f[4 * q + 1] = v.y;
      f[4 * q + 2] = v.z;
      f[4 * q + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int q = 0; q < 32; ++q) f[q] = 0.0f;
  }
  // largest magnitude through its bits: a NaN or an infinity comes out on top
  uint32_t mx = 0;
#pragma unroll
  for (int c = 0; c < 32; ++c) {
    const uint32_t m = __float_as_uint(f[c]) & 0x7fffffffu;
    mx = m > mx ? m : mx;
  }
  const bool bad = mx >= 0x7f800000u;
  // |x| < 2^k; groups below 2^-120 keep an absolute step of 2^-144
  int k = static_cast<int>(mx >> 23) - 126;
  k = k < -120 ? -120 : k;
  uint32_t dg[kDigits][6];
#pragma unroll
  for (int d = 0; d < kDigits; ++d)
#pragma unroll
    for (int r = 0; r < 6; ++r) dg[d][r] = 0;
  const int up = 24 - k;
#pragma unroll
  for (int e = 0; e < 32; ++e) {
    const float v = bad ? 0.0f : f[mx_column(e)];
    const int X = static_cast<int>(__builtin_rintf(__builtin_ldexpf(v, up)));  // |X| <= 2^24
    // X + 16 (1 + 32 + 32^2 + 32^3): the four low base-32 digits with 16
    // added to each; flipping a field's top bit takes the 16 off again
    const uint32_t V = static_cast<uint32_t>(X + 0x84210) ^ 0x84210u;
    const int bit = 6 * e, r = bit >> 5, s = bit & 31;
#pragma unroll
    for (int d = 0; d < kDigits; ++d) {
      // -16 .. 15; the top one -16 .. 16
      const int dgt = d < 4 ? static_cast<int>(V << (27 - 5 * d)) >> 27 : static_cast<int>(V) >> 20;
      const int neg = -dgt;
      // e2m3 of digit / 8: the magnitude as it is, the sign in bit 5
      const uint32_t code = static_cast<uint32_t>(neg > dgt ? neg : dgt) |
                            (static_cast<uint32_t>(dgt) & 32u);
      dg[d][r] |= code << s;
      if (s > 26) dg[d][r + 1] |= code >> (32 - s);
    }
  }
  uint8_t *rec = a.rec + tb * kXRec;
#pragma unroll
  for (int d = 0; d < kDigits; ++d) {
    const int p = h * kDigits + d;
    *reinterpret_cast<uint4 *>(rec + p * 1024 + lane * 16) =
        make_uint4(dg[d][0], dg[d][1], dg[d][2], dg[d][3]);
    *reinterpret_cast<uint2 *>(rec + kXHi + p * 512 + lane * 8) = make_uint2(dg[d][4], dg[d][5]);
  }
  // A scale 2^(k - 2) (255: NaN, which takes every product of the token with it)
  rec[kXScale + lane * 4 + h] = static_cast<uint8_t>(bad ? 255 : 125 + k);
}

// (code - 1) / 2 as e2m1 nibbles: -0.5 = 1001, 0 = 1000, 0.5 = 0001, 1 = 0010
// for codes 0 .. 3.  Even codes of the dword (bits 0-1 of each nibble):
__device__ __forceinline__ uint32_t mx_even(uint32_t w) {
  return (~w & 0x11111111u) | (~(w << 2) & 0x88888888u) | (w & (w << 1) & 0x22222222u);
}

struct WPrepArgs {
  const uint8_t *w;  // first row, 4-byte aligned
  uint8_t *rec;      // [tiles][nblk] records
  float *scale;      // [tiles][nblk][32]
  size_t row_bytes;
  int n_rows, nblk, chunks;
};

// One workgroup per (32-row tile, chunk of 8 blocks): the rows' packed bytes
// through LDS (dword loads along each row), then the operand nibbles of each
// (block, half, lane).
constexpr int kWChunk = 8;
constexpr int kWRowWords = kWChunk * kBlkBytes / 4;  // 68
constexpr int kWPitch = kWRowWords + 1;              // odd: the 32 rows of a column in 32 banks
__global__ __launch_bounds__(256) void pq2_mx_wprep_kernel(WPrepArgs a) {
  __shared__ uint32_t s[32 * kWPitch + 1];
  const int tile = blockIdx.x / a.chunks, chunk = blockIdx.x % a.chunks;
  const int b0 = chunk * kWChunk;
  const int nb = a.nblk - b0 < kWChunk ? a.nblk - b0 : kWChunk;
  const int words = nb * kBlkBytes / 4;  // nblk is even, so chunks hold whole dwords
  for (int i = threadIdx.x; i < 32 * kWRowWords; i += 256) {
    const int r = i / kWRowWords, c = i - r * kWRowWords;
    const int row = tile * 32 + r;
    if (c < words && row < a.n_rows)
      s[r * kWPitch + c] = *reinterpret_cast<const uint32_t *>(
          a.w + static_cast<size_t>(row) * a.row_bytes + static_cast<size_t>(b0) * kBlkBytes + 4 * c);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
  const bool live = tile * 32 + n < a.n_rows;
  for (int i = threadIdx.x >> 6; i < 2 * nb; i += 4) {
    const int b = i >> 1, h = i & 1;
    // codes of (g, h): 8 bytes from byte 34 b + 2 + 16 g + 8 h of the row
    const int byte = kBlkBytes * b + 2 + 16 * g + 8 * h;
    const uint32_t *p = s + n * kWPitch + (byte >> 2);
    const uint32_t e0 = p[0], e1 = p[1], e2 = p[2];
    const int sh = byte & 3;  // 0 or 2
    const uint32_t c0 = sh ? __builtin_amdgcn_alignbyte(e1, e0, 2) : e0;
    const uint32_t c1 = sh ? __builtin_amdgcn_alignbyte(e2, e1, 2) : e1;
    uint4 v = make_uint4(mx_even(c0), mx_even(c0 >> 2), mx_even(c1), mx_even(c1 >> 2));
    if (!live) v = make_uint4(0, 0, 0, 0);
    const size_t tb = static_cast<size_t>(tile) * a.nblk + b0 + b;
    *reinterpret_cast<uint4 *>(a.rec + tb * kWRec + h * 1024 + lane * 16) = v;
    if (h == 0 && g == 0) {
      const int sb = kBlkBytes * b;
      const uint32_t d = s[n * kWPitch + (sb >> 2)] >> (8 * (sb & 3));
      a.scale[tb * 32 + n] =
          live ? __uint_as_float(half_bits_to_f32_bits(d & 0xffffu)) : 0.0f;
    }
  }
}

struct GemmArgs {
  const uint8_t *xrec, *wrec;
  const float *wscale;
  float *y;      // [n_tok][y_stride]
  float4 *part;  // partial tiles of the split units
  int n_rows, n_tok, nblk, y_stride;
  int row_tiles, tok_tiles;  // of 32
  int panels, tsets;         // workgroup tiles along rows and tokens
  int full;                  // units that are whole tiles; the rest are parts
  int split;                 // parts of each remaining tile
};

constexpr int kRT = 4;          // row tiles (of 32) of a wave
constexpr int kWR = 4, kWT = 2;  // waves of a workgroup along rows and tokens
constexpr int kThreads = 64 * kWR * kWT;
constexpr int kPanelRows = 32 * kRT * kWR, kSetTok = 32 * kWT;
static_assert(kPanelRows == kMxPanelRows && kSetTok == kMxSetTok, "the plan's tile");

// Tile q of the walk: 8 row panels by token sets, so that the tiles of
// neighbouring units share their panels' and sets' records in L2.
__device__ __forceinline__ void unit_tile(int q, int panels, int tsets, int &panel, int &tset) {
  const int grp = q / (8 * tsets);
  const int p0 = grp * 8;
  const int np = panels - p0 < 8 ? panels - p0 : 8;
  const int i = q - grp * 8 * tsets;
  tset = i / np;
  panel = p0 + i - tset * np;
}

// B scale of digit j: 2^(5 j - 18) (x = X 2^(k - 24), digit = 8 v, code - 1 =
// 2 w, and the A scale carries 2^(k - 2)).
constexpr int mx_digit_scale(int j) { return 127 - 18 + 5 * j; }

// Half H of a block: the five digits of x (LDS record xb) times the operands
// of R row tiles; half 0 starts the block's tiles.  The lowest digits first:
// each sum is rounded at its final size.
template <int H, int R>
__device__ __forceinline__ void mx_block(std::integral_constant<int, H>, const uint8_t *xb, int lane,
                                         int xs, int ws03, int ws4, const u4v (&wh)[R],
                                         f16v (&blk)[R]) {
  auto digit = [&](auto jc) {
    constexpr int J = decltype(jc)::value;
    constexpr int p = H * kDigits + J;
    const u4v lo = *reinterpret_cast<const u4v *>(xb + p * 1024 + lane * 16);
    const uint2 hi = *reinterpret_cast<const uint2 *>(xb + kXHi + p * 512 + lane * 8);
    const i8v x = {static_cast<int>(lo.x), static_cast<int>(lo.y), static_cast<int>(lo.z),
                   static_cast<int>(lo.w), static_cast<int>(hi.x), static_cast<int>(hi.y), 0, 0};
#pragma unroll
    for (int r = 0; r < R; ++r) {
      f16v c;
      if constexpr (H == 0 && J == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) c[i] = 0.0f;
      } else {
        c = blk[r];
      }
      const i8v w = {static_cast<int>(wh[r].x), static_cast<int>(wh[r].y),
                     static_cast<int>(wh[r].z), static_cast<int>(wh[r].w), 0, 0, 0, 0};
      // A scale: byte H of xs; B scale: byte J of ws03, or ws4
      if constexpr (J < 4)
        blk[r] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, w, c, 2, 4, H, xs, J, ws03);
      else
        blk[r] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, w, c, 2, 4, H, xs, 0, ws4);
    }
  };
  digit(std::integral_constant<int, 0>{});
  digit(std::integral_constant<int, 1>{});
  digit(std::integral_constant<int, 2>{});
  digit(std::integral_constant<int, 3>{});
  digit(std::integral_constant<int, 4>{});
}

// A workgroup multiplies 512 rows by 64 tokens over blocks [kb, ke): 4 x 2
// waves of 128 rows x 32 tokens.  Four row tiles a wave keep the reads of x
// from LDS at 48 bytes a cycle of the 128 there are (a fragment serves four
// products); 8 : 1 in rows to tokens matches x records 7.5 times the weights'
// size per row.  256 x 64 and 512 x 32 tiles of 4 waves, two workgroups a CU,
// measured the same to 6 % slower, 128 x 128 2.2 times slower.  The token sets' x records go through a
// double-buffered LDS stage (block b + 1 written while block b is
// multiplied, block b + 2 in flight in registers), each wave's weight
// operands come straight from their records half a block ahead.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void pq2_mx_gemm_kernel(GemmArgs a) {
  extern __shared__ u4v smem[];
  constexpr int kBuf = kWT * kXRec;  // bytes of one stage
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave % kWR, wt = wave / kWR;
  // unit -> tile and block range; whole tiles are dealt so that an XCD (unit
  // id mod 8) takes a contiguous run of the walk
  int q, kb = 0, ke = a.nblk, slot = -1;
  const int u = blockIdx.x;
  if (u < a.full) {
    q = (u & 7) * (a.full >> 3) + (u >> 3);
  } else {
    const int v = u - a.full, part = v % a.split;
    q = a.full + v / a.split;
    kb = static_cast<int>(static_cast<int64_t>(a.nblk) * part / a.split);
    ke = static_cast<int>(static_cast<int64_t>(a.nblk) * (part + 1) / a.split);
    if (a.split > 1) slot = v;
  }
  int panel, tset;
  unit_tile(q, a.panels, a.tsets, panel, tset);
  const int tt0 = tset * kWT;
  const int rt0 = (panel * kWR + wr) * kRT;

  // x copy: thread i moves uint4 i, i + 512, .. of the stage
  constexpr int kCopy = kBuf / 16 / kThreads;
  const u4v *xsrc[kWT];
#pragma unroll
  for (int i = 0; i < kWT; ++i) {
    int tt = tt0 + i;
    tt = tt < a.tok_tiles ? tt : a.tok_tiles - 1;  // a tile past the end is read, never stored
    xsrc[i] = reinterpret_cast<const u4v *>(a.xrec + (static_cast<size_t>(tt) * a.nblk + kb) * kXRec) +
              threadIdx.x;
  }
  u4v xr[kCopy];
  auto xload = [&](int s) {  // block kb + s
#pragma unroll
    for (int i = 0; i < kCopy; ++i)
      xr[i] = xsrc[i * kThreads * 16 / kXRec][static_cast<size_t>(s) * (kXRec / 16) +
                                              i * kThreads % (kXRec / 16)];
  };
  auto xstore = [&](int s) {
#pragma unroll
    for (int i = 0; i < kCopy; ++i) smem[(s & 1) * (kBuf / 16) + i * kThreads + threadIdx.x] = xr[i];
  };
  // weight operands and scales of the wave's row tiles
  const uint8_t *wsrc[kRT];
  const float *dsrc[kRT];
#pragma unroll
  for (int r = 0; r < kRT; ++r) {
    int rt = rt0 + r;
    rt = rt < a.row_tiles ? rt : a.row_tiles - 1;
    const size_t tb = static_cast<size_t>(rt) * a.nblk + kb;
    wsrc[r] = a.wrec + tb * kWRec + lane * 16;
    dsrc[r] = a.wscale + tb * 32 + (lane & 31);
  }
  u4v w0[kRT], w1[kRT];  // halves 0 and 1 of a block
  float d[kRT];
  auto wload = [&](u4v(&w)[kRT], int hs) {  // half step hs = 2 s + h
#pragma unroll
    for (int r = 0; r < kRT; ++r)
      w[r] = *reinterpret_cast<const u4v *>(wsrc[r] + static_cast<size_t>(hs) * 1024);
  };
  auto dload = [&](int s) {
#pragma unroll
    for (int r = 0; r < kRT; ++r) d[r] = dsrc[r][s * 32];
  };

  f16v acc[kRT];
#pragma unroll
  for (int r = 0; r < kRT; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[r][i] = 0.0f;
  const int ws03 = mx_digit_scale(0) | mx_digit_scale(1) << 8 | mx_digit_scale(2) << 16 |
                   mx_digit_scale(3) << 24;
  const int ws4 = mx_digit_scale(4);

  const int n = ke - kb;
  xload(0);
  wload(w0, 0);
  xstore(0);
  xload(n > 1 ? 1 : 0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  for (int s = 0; s < n; ++s) {
    // loads past the last block repeat it: no branches around them
    const int s1 = s + 1 < n ? s + 1 : s, s2 = s + 2 < n ? s + 2 : s1;
    xstore(s + 1);  // the other buffer's readers passed the last barrier
    wload(w1, 2 * s + 1);
    dload(s);
    xload(s2);
    __builtin_amdgcn_sched_barrier(0);  // the loads are issued before the products
    const uint8_t *xb = reinterpret_cast<const uint8_t *>(smem) + (s & 1) * kBuf + wt * kXRec;
    const int xs = *reinterpret_cast<const int *>(xb + kXScale + lane * 4);
    f16v blk[kRT];
    mx_block(std::integral_constant<int, 0>{}, xb, lane, xs, ws03, ws4, w0, blk);
    __builtin_amdgcn_sched_barrier(0);
    wload(w0, 2 * s1);
    __builtin_amdgcn_sched_barrier(0);
    mx_block(std::integral_constant<int, 1>{}, xb, lane, xs, ws03, ws4, w1, blk);
#pragma unroll
    for (int r = 0; r < kRT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][i] = __builtin_fmaf(blk[r][i], d[r], acc[r][i]);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }

  if (slot >= 0) {  // a part: the lanes' sums as they are, 16 bytes a lane
    float4 *dst = a.part + (static_cast<size_t>(slot) * (kWR * kWT) + wave) * kRT * 4 * 64 + lane;
#pragma unroll
    for (int r = 0; r < kRT; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dst[(r * 4 + i) * 64] =
            make_float4(acc[r][4 * i], acc[r][4 * i + 1], acc[r][4 * i + 2], acc[r][4 * i + 3]);
    return;
  }
  const int t0 = (tt0 + wt) * 32 + 4 * (lane >> 5);
#pragma unroll
  for (int r = 0; r < kRT; ++r) {
    const int row = (rt0 + r) * 32 + (lane & 31);
    if (row < a.n_rows) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = t0 + 8 * (i >> 2) + (i & 3);
        if (t < a.n_tok) a.y[static_cast<size_t>(t) * a.y_stride + row] = acc[r][i];
      }
    }
  }
}

// Adds the parts of the split tiles in order: one lane per four outputs.
__global__ __launch_bounds__(256) void pq2_mx_fold_kernel(GemmArgs a) {
  constexpr int kLanes = kWR * kWT * kRT * 4 * 64;  // float4 of a tile
  const int tile = blockIdx.x / (kLanes / 256);
  const int i = blockIdx.x % (kLanes / 256) * 256 + threadIdx.x;
  const float4 *src = a.part + static_cast<size_t>(tile) * a.split * kLanes + i;
  float4 v = src[0];
  for (int p = 1; p < a.split; ++p) {
    const float4 e = src[static_cast<size_t>(p) * kLanes];
    v.x += e.x;
    v.y += e.y;
    v.z += e.z;
    v.w += e.w;
  }
  int panel, tset;
  unit_tile(a.full + tile, a.panels, a.tsets, panel, tset);
  const int lane = i & 63, quad = (i >> 6) & 3, r = (i >> 8) % kRT, wave = i / (kRT * 4 * 64);
  const int row = ((panel * kWR + wave % kWR) * kRT + r) * 32 + (lane & 31);
  const int t = (tset * kWT + wave / kWR) * 32 + 8 * quad + 4 * (lane >> 5);
  if (row >= a.n_rows) return;
  const float o[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (t + k < a.n_tok) a.y[static_cast<size_t>(t + k) * a.y_stride + row] = o[k];
}

// ---------------------------------------------------------------------------
// Few tokens: the weights are read once or twice, so they are multiplied from
// the packed rows as they are.  A workgroup is W waves of R row tiles on one
// token tile.  Each wave stages two blocks of its rows (68 bytes a row: four
// 16-byte loads and a dword) in an LDS area of its own, the next four in
// flight in registers.  A row's 17 dwords go to slots 0-8 and 12-19 of 20: the two
// blocks' lane-group halves then start on 16 bytes (slots 0, 4, 12, 16), and
// eight rows of a 16-byte read lie in distinct banks.  A short call is bound
// by its three launches (of 25 us at 17 tokens on [17408 x 5120] the digits
// take 5, the products 13, the parts 5), a wide one by the overlap of loads,
// decoding and products in two waves a SIMD (of 146 us on [248320 x 5120] 93
// stay with every load removed, 74 without the products too; the packed rows
// alone take 50).  Three or four row tiles a wave spill or lose a wave, two
// token tiles a wave, 4-wave workgroups with a barrier a block and a rolled
// block loop were no faster.
// ---------------------------------------------------------------------------
constexpr int kRawPitch = 20;  // dwords
typedef u4v u4v_a4 __attribute__((aligned(4)));

struct RawArgs {
  const uint8_t *w;  // first row, 4-byte aligned
  const uint8_t *xrec;
  float *y;
  float4 *part;
  size_t row_bytes;
  int n_rows, n_tok, nblk;
  int tok_tiles, split;
};

template <int W, int R>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2)))
void pq2_mx_raw_kernel(RawArgs a) {
  extern __shared__ u4v smem[];
  constexpr int kThr = 64 * W;
  constexpr int kBuf = 2 * kXRec;  // bytes of one x stage: a pair of blocks
  constexpr int kRows = 32 * R;        // rows of a wave
  constexpr int kCopy = kBuf / 16 / kThr;
  static_assert(kThr <= 1024 && kBuf % (16 * kThr) == 0, "whole copies");
  const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t *stage = reinterpret_cast<uint32_t *>(smem) + 2 * kBuf / 4 + wave * kRows * kRawPitch;
  const int unit = blockIdx.x;
  const int part = unit % a.split, tile = unit / a.split;
  const int panel = tile / a.tok_tiles, tt = tile - panel * a.tok_tiles;
  const int pairs = a.nblk / 2;
  const int pb = static_cast<int>(static_cast<int64_t>(pairs) * part / a.split);
  const int pe = static_cast<int>(static_cast<int64_t>(pairs) * (part + 1) / a.split);
  const int row0 = (panel * W + wave) * kRows;

  const u4v *xsrc =
      reinterpret_cast<const u4v *>(a.xrec + static_cast<size_t>(tt) * a.nblk * kXRec) + threadIdx.x;
  u4v xr[kCopy];
  auto xload = [&](int p) {  // block pair p
    p = p < pe ? p : pe - 1;
#pragma unroll
    for (int i = 0; i < kCopy; ++i)
      xr[i] = xsrc[static_cast<size_t>(p) * (kBuf / 16) + i * kThr];
  };
  auto xstore = [&](int p) {
#pragma unroll
    for (int i = 0; i < kCopy; ++i) smem[((p - pb) & 1) * (kBuf / 16) + i * kThr + threadIdx.x] = xr[i];
  };
  // rows through the stage: lane 4 i + j moves piece j (dwords 0, 4, 9, 13 on)
  // of rows i, i + 16, ..; the ninth dword of rows lane, lane + 64, ..
  const int pj = lane & 3;
  const int rfirst = row0 < a.n_rows ? row0 : a.n_rows - 1;
  const uint32_t rlast = static_cast<uint32_t>(a.n_rows - 1 - rfirst);  // rows past the end repeat it
  const uint8_t *wbase = a.w + static_cast<size_t>(rfirst) * a.row_bytes;
  constexpr int kMid = (kRows + 63) / 64;
  u4v wra[2 * R], wrb[2 * R];  // the next pair and the one after it
  uint32_t wma[kMid], wmb[kMid];
  auto wload = [&](u4v(&wr)[2 * R], uint32_t(&wm)[kMid], int p) {  // block pair p of the row
    p = p < pe ? p : pe - 1;
    const uint8_t *src = wbase + static_cast<size_t>(p) * (2 * kBlkBytes);
    const uint32_t r0 = static_cast<uint32_t>(lane >> 2), o = 16 * pj + 4 * (pj >> 1);
#pragma unroll
    for (int k = 0; k < 2 * R; ++k)
      wr[k] = *reinterpret_cast<const u4v_a4 *>(src + (min(16 * k + r0, rlast) * a.row_bytes + o));
#pragma unroll
    for (int k = 0; k < kMid; ++k)
      wm[k] = *reinterpret_cast<const uint32_t *>(
          src + (min(64u * k + static_cast<uint32_t>(lane), rlast) * a.row_bytes + 32));
  };
  auto wstore = [&](const u4v(&wr)[2 * R], const uint32_t(&wm)[kMid]) {
#pragma unroll
    for (int k = 0; k < 2 * R; ++k)
      *reinterpret_cast<u4v *>(stage + (16 * k + (lane >> 2)) * kRawPitch + 4 * pj + 4 * (pj >> 1)) = wr[k];
#pragma unroll
    for (int k = 0; k < kMid; ++k)
      if (kRows >= 64 || lane < kRows) stage[(64 * k + lane) * kRawPitch + 8] = wm[k];
  };

  f16v acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[r][i] = 0.0f;
  const int ws03 = mx_digit_scale(0) | mx_digit_scale(1) << 8 | mx_digit_scale(2) << 16 |
                   mx_digit_scale(3) << 24;
  const int ws4 = mx_digit_scale(4);

  xload(pb);
  wload(wra, wma, pb);
  wload(wrb, wmb, pb + 1);
  xstore(pb);
  xload(pb + 1);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  auto pair = [&](int p, u4v(&wr)[2 * R], uint32_t(&wm)[kMid]) {
    wstore(wr, wm);  // this wave read the previous pair before its last barrier
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    xstore(p + 1);  // the other buffer's readers passed the last barrier
    xload(p + 2);
    wload(wr, wm, p + 2);  // behind the x loads: waiting for those leaves these in flight
    __builtin_amdgcn_sched_barrier(0);  // the loads are issued before the products
    auto block = [&](auto odd) {
      constexpr int O = decltype(odd)::value;
      u4v w0[R], w1[R];
      float d[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint32_t *sp = stage + (32 * r + n) * kRawPitch;
        u4v q = *reinterpret_cast<const u4v *>(sp + (O ? 12 : 0) + 4 * g);
        uint32_t sc = sp[O ? 8 : 0];
        if constexpr (O == 0) {  // codes start two bytes into a dword
          const uint32_t e = sp[4 * g + 4];
          q = u4v{__builtin_amdgcn_alignbyte(q.y, q.x, 2), __builtin_amdgcn_alignbyte(q.z, q.y, 2),
                  __builtin_amdgcn_alignbyte(q.w, q.z, 2), __builtin_amdgcn_alignbyte(e, q.w, 2)};
        } else {
          sc >>= 16;
        }
        d[r] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(sc)));
        w0[r] = u4v{mx_even(q.x), mx_even(q.x >> 2), mx_even(q.y), mx_even(q.y >> 2)};
        w1[r] = u4v{mx_even(q.z), mx_even(q.z >> 2), mx_even(q.w), mx_even(q.w >> 2)};
      }
      const uint8_t *xb = reinterpret_cast<const uint8_t *>(smem) + ((p - pb) & 1) * kBuf + O * kXRec;
      const int xs = *reinterpret_cast<const int *>(xb + kXScale + lane * 4);
      f16v blk[R];
      mx_block(std::integral_constant<int, 0>{}, xb, lane, xs, ws03, ws4, w0, blk);
      mx_block(std::integral_constant<int, 1>{}, xb, lane, xs, ws03, ws4, w1, blk);
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][i] = __builtin_fmaf(blk[r][i], d[r], acc[r][i]);
    };
    block(std::integral_constant<int, 0>{});
    block(std::integral_constant<int, 1>{});
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  for (int p = pb; p < pe; p += 2) {
    pair(p, wra, wma);
    if (p + 1 < pe) pair(p + 1, wrb, wmb);
  }

  if (a.split > 1) {  // a part: the lanes' sums as they are, 16 bytes a lane
    float4 *dst = a.part + (static_cast<size_t>(unit) * W + wave) * R * 4 * 64 + lane;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dst[(r * 4 + i) * 64] =
            make_float4(acc[r][4 * i], acc[r][4 * i + 1], acc[r][4 * i + 2], acc[r][4 * i + 3]);
    return;
  }
  const int t0 = tt * 32 + 4 * g;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int row = row0 + 32 * r + n;
    if (row < a.n_rows) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = t0 + 8 * (i >> 2) + (i & 3);
        if (t < a.n_tok) a.y[static_cast<size_t>(t) * a.n_rows + row] = acc[r][i];
      }
    }
  }
}

// Adds the parts of every tile in order: one lane per four outputs.
template <int W, int R>
__global__ __launch_bounds__(256) void pq2_mx_raw_fold_kernel(RawArgs a) {
  constexpr int kLanes = W * R * 4 * 64;  // float4 of a tile
  const int tile = blockIdx.x / (kLanes / 256);
  const int i = blockIdx.x % (kLanes / 256) * 256 + threadIdx.x;
  const int panel = tile / a.tok_tiles, tt = tile - panel * a.tok_tiles;
  const int lane = i & 63, quad = (i >> 6) & 3, r = (i >> 8) % R, wave = i / (R * 4 * 64);
  const int row = (panel * W + wave) * 32 * R + 32 * r + (lane & 31);
  const int t = tt * 32 + 8 * quad + 4 * (lane >> 5);
  if (row >= a.n_rows || t >= a.n_tok) return;
  const float4 *src = a.part + static_cast<size_t>(tile) * a.split * kLanes + i;
  float4 v = src[0];
  for (int p = 1; p < a.split; ++p) {
    const float4 e = src[static_cast<size_t>(p) * kLanes];
    v.x += e.x;
    v.y += e.y;
    v.z += e.z;
    v.w += e.w;
  }
  const float o[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (t + k < a.n_tok) a.y[static_cast<size_t>(t + k) * a.n_rows + row] = o[k];
}

int xprep(const float *x, size_t ne0, size_t n_tok, uint8_t *rec, hipStream_t st) {
  const size_t nblk = ne0 / 128;
  const XPrepArgs a{x, rec, static_cast<int>(ne0), static_cast<int>(n_tok), static_cast<int>(nblk),
                    (n_tok + 31) / 32 * nblk * 2};
  BH_LAUNCH(pq2_mx_xprep_kernel, static_cast<unsigned>((a.items + 3) / 4), 256, 0, st, a);
  return ok();
}

template <int R>
int launch_raw(const uint8_t *w, size_t ne0, size_t n_rows, const float *x, size_t n_tok, float *y,
               size_t split, char *scratch, const MxScratch &m, hipStream_t st) {
  constexpr int W = kMxRawWaves;
  const size_t nblk = ne0 / 128, tok_tiles = (n_tok + 31) / 32;
  const size_t panels = (n_rows + 32 * W * R - 1) / (32 * W * R), tiles = panels * tok_tiles;
  uint8_t *rec = reinterpret_cast<uint8_t *>(scratch);
  if (int e = xprep(x, ne0, n_tok, rec, st)) return e;
  const RawArgs a{w, rec, y, reinterpret_cast<float4 *>(scratch + m.x), bh_pq2_row_bytes(ne0),
                  static_cast<int>(n_rows), static_cast<int>(n_tok), static_cast<int>(nblk),
                  static_cast<int>(tok_tiles), static_cast<int>(split)};
  constexpr int lds = 4 * kXRec + 32 * W * R * kRawPitch * 4;
  if (int e = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(pq2_mx_raw_kernel<W, R>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                        "hipFuncSetAttribute"))
    return e;
  BH_LAUNCH((pq2_mx_raw_kernel<W, R>), static_cast<unsigned>(tiles * split), 64 * W, lds, st, a);
  if (split > 1)
    BH_LAUNCH((pq2_mx_raw_fold_kernel<W, R>), static_cast<unsigned>(tiles * (W * R)), 256, 0, st, a);
  return ok();
}

}  // namespace

int pq2_mx_gemm(const uint8_t *w, size_t ne0, size_t n_rows, const float *x, size_t n_tok, float *y,
                hipStream_t st) {
  const size_t nblk = ne0 / 128, slots = device_cu_count();
  const MxPlan plan = mx_plan(n_rows, n_tok, nblk, slots);
  const MxScratch m = mx_scratch_of(plan, n_rows, n_tok, nblk, slots);
  char *scratch = static_cast<char *>(
      device_scratch(mx_reserve_bytes(n_rows, n_tok, nblk), kScratchMatmul, st, m.total()));
  if (scratch == nullptr) return BH_ERR_HIP;
  if (plan.R == 1) return launch_raw<1>(w, ne0, n_rows, x, n_tok, y, plan.split, scratch, m, st);
  if (plan.R == 2) return launch_raw<2>(w, ne0, n_rows, x, n_tok, y, plan.split, scratch, m, st);

  const size_t pass_rows = mx_pass_rows(nblk), tok_tiles = (n_tok + 31) / 32;
  const size_t tsets = (n_tok + kSetTok - 1) / kSetTok;
  uint8_t *rec = reinterpret_cast<uint8_t *>(scratch);
  if (int e = xprep(x, ne0, n_tok, rec, st)) return e;
  constexpr int lds = 2 * kWT * kXRec;
  if (int e = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(pq2_mx_gemm_kernel),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                        "hipFuncSetAttribute"))
    return e;
  for (size_t r0 = 0; r0 < n_rows; r0 += pass_rows) {
    const size_t rows = std::min(n_rows - r0, pass_rows), row_tiles = (rows + 31) / 32;
    const size_t panels = (rows + kPanelRows - 1) / kPanelRows;
    const MxPlan p = mx_pass_plan(rows, n_tok, nblk, slots);
    const size_t rest = panels * tsets - p.full;
    const size_t row_bytes = bh_pq2_row_bytes(ne0);
    const WPrepArgs wa{w + r0 * row_bytes, rec + m.x,
                       reinterpret_cast<float *>(scratch + m.x + m.w), row_bytes,
                       static_cast<int>(rows), static_cast<int>(nblk),
                       static_cast<int>((nblk + kWChunk - 1) / kWChunk)};
    BH_LAUNCH(pq2_mx_wprep_kernel, static_cast<unsigned>(row_tiles * wa.chunks), 256, 0, st, wa);
    const GemmArgs a{rec, wa.rec, wa.scale, y + r0,
                     reinterpret_cast<float4 *>(scratch + m.x + m.w + m.d),
                     static_cast<int>(rows), static_cast<int>(n_tok), static_cast<int>(nblk),
                     static_cast<int>(n_rows), static_cast<int>(row_tiles),
                     static_cast<int>(tok_tiles), static_cast<int>(panels), static_cast<int>(tsets),
                     static_cast<int>(p.full), static_cast<int>(p.split)};
    BH_LAUNCH(pq2_mx_gemm_kernel, static_cast<unsigned>(p.full + rest * p.split), kThreads, lds, st, a);
    if (p.split > 1) {
      constexpr int kPerTile = kWR * kWT * kRT * 4 * 64 / 256;
      BH_LAUNCH(pq2_mx_fold_kernel, static_cast<unsigned>(rest * kPerTile), 256, 0, st, a);
    }
  }
  return ok();
}

}  // namespace bh
