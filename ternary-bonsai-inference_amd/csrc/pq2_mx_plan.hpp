// How a PQ2_0 product of many tokens is cut (pq2_mx.hip), and what scratch it
// reserves.  Host arithmetic only: no HIP.
#pragma once

#include <algorithm>
#include <cstddef>

namespace bh {

// x record of one (32-token tile, 128-block) and weight record of one (32-row
// tile, 128-block), and the rows and tokens of an unpacked workgroup.
constexpr size_t kMxXRec = 16384;
constexpr size_t kMxWRec = 2048;
constexpr size_t kMxPanelRows = 512, kMxSetTok = 64;
constexpr size_t kMxRawWaves = 8;

// Unpacked weights of one pass over the rows: bounds the scratch that a wide
// matrix (the vocabulary) would take, at 68 bytes a row and block.
constexpr size_t kMxUnpackBytes = 96 << 20;
// Partial sums of the parts: no call of the model's shapes wants more than 48
// MB of them, and past this they cost more than the parts give.
constexpr size_t kMxPartBytes = 96 << 20;
// Fewer tokens never take the unpacked kernel (the cost model first picks it
// at 131), so they don't reserve its scratch.
constexpr size_t kMxUnpackTok = 129;

// How a call is cut: the raw kernel with R row tiles a wave (R = 1, 2), or the
// unpacked kernel (R = 0), each with its tiles' blocks in `split` parts, and
// the time that this is expected to take.  The times were fitted to calls of
// 16 to 2048 tokens on [17408 x 5120], [5120 x 17408] and [6144 x 5120]
// (within about 15 %): a turn of two blocks takes a round of raw workgroups
// 1.9 us (R = 1) or 2.9 us (R = 2), a block takes a round of unpacked ones 2.3
// us; a round costs 4 us besides; unpacking runs at 1.3 TB/s of packed bytes;
// parts cost a launch and their sums through memory.
struct MxPlan {
  int R;
  size_t full, split;
  double us;
};

constexpr size_t mx_ceil(size_t a, size_t b) { return (a + b - 1) / b; }
constexpr size_t mx_raw_rows(int R) { return 32 * kMxRawWaves * static_cast<size_t>(R); }
// f32 sums of one raw or unpacked workgroup
constexpr size_t mx_raw_part(int R) { return mx_raw_rows(R) * 32 * 4; }
constexpr size_t kMxUnpackPart = kMxPanelRows * kMxSetTok * 4;

inline void mx_raw_plan(size_t n_rows, size_t tok_tiles, size_t nblk, size_t slots, MxPlan &best) {
  const size_t pairs = nblk / 2;
  for (int R = 1; R <= 2; ++R) {
    const size_t rows = mx_raw_rows(R), tiles = mx_ceil(n_rows, rows) * tok_tiles;
    for (size_t s = 1; s <= std::min<size_t>(pairs, 32); ++s) {
      if (s > 1 && tiles * s * mx_raw_part(R) > kMxPartBytes) break;
      const double rounds = static_cast<double>(mx_ceil(tiles * s, slots));
      const double turns = static_cast<double>(mx_ceil(pairs, s));
      double us = rounds * (turns * (R == 1 ? 1.9 : 2.9) + 4.0);
      if (s > 1) us += 5.0 + static_cast<double>(tiles * s * rows * 32 * 8) / 3e6;
      if (us < best.us) best = MxPlan{R, 0, s, us};
    }
  }
}

// Whole rounds of tiles over the CUs (one workgroup each), then the rest in
// parts that fill shorter rounds.
inline void mx_unpacked_plan(size_t n_rows, size_t n_tok, size_t nblk, size_t slots, MxPlan &best) {
  const size_t tiles = mx_ceil(n_rows, kMxPanelRows) * mx_ceil(n_tok, kMxSetTok);
  const size_t full = slots % 8 == 0 ? tiles / slots * slots : 0, rest = tiles - full;
  const double base = static_cast<double>(n_rows * nblk * 34) / 1.3e6 + 5.0 +
                      static_cast<double>(full / slots) * (static_cast<double>(nblk) * 2.3 + 4.0);
  if (rest == 0) {
    if (base < best.us) best = MxPlan{0, full, 1, base};
    return;
  }
  for (size_t s = 1; s <= std::min<size_t>(nblk / 2, 16); ++s) {
    if (s > 1 && rest * s * kMxUnpackPart > kMxPartBytes) break;
    const double rounds = static_cast<double>(mx_ceil(rest * s, slots));
    double us = base + rounds * (static_cast<double>(mx_ceil(nblk, s)) * 2.3 + 4.0);
    if (s > 1) us += 5.0 + static_cast<double>(rest * s * kMxPanelRows * kMxSetTok * 8) / 3e6;
    if (us < best.us) best = MxPlan{0, full, s, us};
  }
}

inline MxPlan mx_plan(size_t n_rows, size_t n_tok, size_t nblk, size_t slots) {
  MxPlan p{1, 0, 1, 1e30};
  mx_raw_plan(n_rows, mx_ceil(n_tok, 32), nblk, slots, p);
  if (n_tok >= kMxUnpackTok) mx_unpacked_plan(n_rows, n_tok, nblk, slots, p);
  return p;
}

// The unpacked kernel's passes over the rows, and the plan of one of `rows`.
inline size_t mx_pass_rows(size_t nblk) {
  return std::max<size_t>(1, kMxUnpackBytes / (nblk * (kMxWRec / 32 + 4)) / kMxPanelRows) * kMxPanelRows;
}
inline MxPlan mx_pass_plan(size_t rows, size_t n_tok, size_t nblk, size_t slots) {
  MxPlan p{0, 0, 1, 1e30};
  mx_unpacked_plan(rows, n_tok, nblk, slots, p);
  return p;
}

// Scratch: x records, unpacked records, their scales, partial sums.
struct MxScratch {
  size_t x, w, d, parts;
  size_t total() const { return x + w + d + parts; }
};
inline MxScratch mx_scratch_of(const MxPlan &plan, size_t n_rows, size_t n_tok, size_t nblk, size_t slots) {
  MxScratch m{mx_ceil(n_tok, 32) * nblk * kMxXRec, 0, 0, 0};
  if (plan.R != 0) {
    const size_t tiles = mx_ceil(n_rows, mx_raw_rows(plan.R)) * mx_ceil(n_tok, 32);
    if (plan.split > 1) m.parts = tiles * plan.split * mx_raw_part(plan.R);
    return m;
  }
  const size_t pass = std::min(n_rows, mx_pass_rows(nblk)), tiles0 = mx_ceil(pass, 32);
  m.w = tiles0 * nblk * kMxWRec;
  m.d = mx_ceil(tiles0 * nblk * 32 * 4, 256) * 256;
  for (const size_t rows : {pass, n_rows % pass}) {
    if (rows == 0) continue;
    const MxPlan p = mx_pass_plan(rows, n_tok, nblk, slots);
    const size_t rest = mx_ceil(rows, kMxPanelRows) * mx_ceil(n_tok, kMxSetTok) - p.full;
    if (p.split > 1) m.parts = std::max(m.parts, rest * p.split * kMxUnpackPart);
  }
  return m;
}

// What a call reserves: enough for itself and for every call of fewer tokens
// on the same matrix, whose plans may have more parts than its own.  So one
// call at the largest batch prepares a stream capture of any smaller one,
// which must not allocate.
inline size_t mx_reserve_bytes(size_t n_rows, size_t n_tok, size_t nblk) {
  const size_t tok_tiles = mx_ceil(n_tok, 32), pairs = nblk / 2;
  size_t parts = 0;
  if (pairs > 1)
    for (int R = 1; R <= 2; ++R)
      parts = std::max(parts, mx_ceil(n_rows, mx_raw_rows(R)) * tok_tiles * std::min<size_t>(pairs, 32) *
                                  mx_raw_part(R));
  size_t unpacked = 0;
  if (n_tok >= kMxUnpackTok) {
    const size_t pass = std::min(n_rows, mx_pass_rows(nblk)), tiles0 = mx_ceil(pass, 32);
    unpacked = tiles0 * nblk * kMxWRec + mx_ceil(tiles0 * nblk * 32 * 4, 256) * 256;
    if (pairs > 1)
      parts = std::max(parts, mx_ceil(pass, kMxPanelRows) * mx_ceil(n_tok, kMxSetTok) *
                                  std::min<size_t>(pairs, 16) * kMxUnpackPart);
  }
  return tok_tiles * nblk * kMxXRec + unpacked + std::min(parts, kMxPartBytes);
}

}  // namespace bh
