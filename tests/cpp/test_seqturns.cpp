// CPU check of the turn-wise evaluation of a whole row's runs (csrc/seqsum.hpp:
// seq_units, seq_step, seq_units_added) against the plain loop of sequential
// f32 additions.  Built with g++ by tests/test_seqturns.py (x86-64 SSE
// arithmetic: IEEE f32, round to nearest even, no contraction).
#define __host__
#define __device__
// the GPU's reciprocal is within 1 ulp: also built one ulp down and up
#include <cmath>
#ifndef RCP_ULP
#define RCP_ULP 0
#endif
static inline float test_rcp(float v) {
  float r = 1.0f / v;
  if (RCP_ULP < 0) r = std::nextafter(r, 0.0f);
  if (RCP_ULP > 0) r = std::nextafter(r, 2.0f * r);
  return r;
}
#define BH_SEQ_RCP(v) test_rcp(v)
#include "../../ternary-bonsai-inference_amd/csrc/seqsum.hpp"

#include <cstdint>
#include <cstdio>
#include <initializer_list>

namespace {

uint64_t g_state = 0x9e3779b97f4a7c15ull;
uint32_t below(uint32_t n) {  // splitmix64
  uint64_t z = (g_state += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return static_cast<uint32_t>((z ^ (z >> 31)) % n);
}

// f16 value of bits h (finite), widened exactly
float half_val(uint32_t h) {
  const uint32_t e = (h >> 10) & 0x1f, m = h & 0x3ff;
  return e == 0 ? static_cast<float>(m) * bh::seq_u2f(0x33800000u)  // m * 2^-24
                : bh::seq_u2f(((e + 112u) << 23) | (m << 13));
}

// Windows of `lanes` runs, one lane each, as a wave takes them: units from the
// binade of the turn's sum, each lane's start by the prefix sum of the lanes
// before it (all of them, as the wave forms it), the first that does not stay.
float by_turns(const float *x, const uint32_t *runs, int n_runs, int lanes, int &turns) {
  float s = 0.0f;
  for (int w = 0; w < n_runs; w += lanes) {
    const int nl = n_runs - w < lanes ? n_runs - w : lanes;
    uint32_t n[64];
    for (int l = 0; l < nl; ++l) n[l] = x[w + l] != 0.0f ? runs[w + l] : 0u;
    for (;;) {
      ++turns;
      const uint32_t sb = bh::seq_f2u(s);
      uint32_t at = sb;
      int f = -1;
      bh::SeqStep first{};
      for (int l = 0; l < nl; ++l) {
        const bh::SeqUnits u = bh::seq_units(static_cast<int>(sb >> 23), x[w + l]);
        const bh::SeqStep step = bh::seq_step(at, x[w + l], n[l], u);
        if (n[l] != 0 && !step.whole && f < 0) {
          f = l;
          first = step;
        }
        at += n[l] != 0 ? bh::seq_units_added(n[l], u) : 0u;
      }
      if (f < 0) {
        s = bh::seq_u2f(at);
        break;
      }
      s = first.s;
      for (int l = 0; l < f; ++l) n[l] = 0;
      n[f] = first.left;
    }
  }
  return s;
}

// Blocks of squares x and 4 x in a drawn order, a lane each, as a wave takes
// them: in closed form where the block stays in the binade, square by square
// (in its order) where it does not.
struct Mixed {
  float x;
  uint32_t n1, n4;
  uint64_t four[2];  // place j holds 4 x (of the first n1 + n4)
};
float add_in_order(float s, const Mixed &b) {
  volatile float acc = s;
  for (uint32_t j = 0; j < b.n1 + b.n4; ++j)
    acc = acc + (((b.four[j >> 6] >> (j & 63)) & 1u) ? 4.0f * b.x : b.x);
  return acc;
}
float mixed_by_turns(const Mixed *b, int n_blk, int &turns) {
  float s = 0.0f;
  for (int done = 0; done < n_blk;) {
    ++turns;
    const uint32_t sb = bh::seq_f2u(s);
    const int es = static_cast<int>(sb >> 23);
    uint32_t at = sb;
    int l = done;
    for (; l < n_blk; ++l) {
      const bh::SeqUnits u = bh::seq_units(es, b[l].x), u4 = bh::seq_units(es, 4.0f * b[l].x);
      const uint32_t inc = bh::seq_mixed_added(b[l].n1, u, b[l].n4, u4);
      if (b[l].n1 + b[l].n4 != 0 && !bh::seq_mixed_whole(at, inc, b[l].n1, u, b[l].n4, u4)) break;
      at += inc;
    }
    s = bh::seq_u2f(at);
    if (l < n_blk) s = add_in_order(s, b[l++]);
    done = l;
  }
  return s;
}

// A row whose second run's last addition lands exactly on the upper end of the
// sum's binade (a rounded-up step: m = q + 1 divides the gap), with more runs
// behind it, which have to be added in the next binade's units.  Random rows
// land about once in a million.  Returns the number of blocks.
int landing_row(float *x, uint32_t *n) {
  for (;;) {
    const uint32_t e = 3 + below(24);
    const float d0 = half_val((e << 10) | below(1024));
    x[0] = d0 * d0;
    n[0] = 1 + below(100);
    volatile float s = 0.0f;
    for (uint32_t i = 0; i < n[0]; ++i) s = s + x[0];
    const uint32_t sb = bh::seq_f2u(s);
    const uint32_t gap = (1u << 24) - ((sb & 0x7fffffu) | 0x800000u);
    for (int tries = 0; tries < 400; ++tries) {
      const uint32_t down = below(6);
      if (e < 1 + down) continue;
      const float d = half_val(((e - down) << 10) | below(1024));
      x[1] = d * d;
      const bh::SeqUnits u = bh::seq_units(static_cast<int>(sb >> 23), x[1]);
      if (u.m != u.q + 1 || u.tie || gap % u.m != 0 || gap / u.m > 128) continue;
      n[1] = gap / u.m;
      const int nblk = 3 + static_cast<int>(below(38));
      for (int b = 2; b < nblk; ++b) {
        const uint32_t de = below(6);
        const float db = half_val(((e > de ? e - de : 1) << 10) | below(1024));
        x[b] = db * db;
        n[b] = below(129);
      }
      return nblk;
    }
  }
}

}  // namespace

int main() {
  long rows = 0, turns40 = 0, rows40 = 0;
  int fail = 0;
  for (int it = 0; it < 60000; ++it) {
    const int kind = it % 6;
    const int nblk = kind == 5 ? 1 + static_cast<int>(below(150)) : 40;
    const uint32_t base = below(28);
    float x[160];
    uint32_t n[160];
    float loop = 0.0f;
    for (int b = 0; b < nblk; ++b) {
      uint32_t h;
      switch (kind) {
        case 0: h = below(0x7c00u); break;                                // any scale
        case 1: h = (5 + below(20)) << 10; break;                         // powers of two: ties
        case 2: h = b == 0 ? 0x7000u + below(0x400u) : 1 + below(0x1000u); break;  // big, then tiny
        case 3: h = 0x3c00u; break;                                       // whole sums
        default: h = ((base + below(3)) << 10) | below(1024);             // a few binades
      }
      const float d = half_val(h);
      x[b] = d * d;
      n[b] = below(7) == 0 ? 128u * below(2) : below(129);
      volatile float acc = loop;
      for (uint32_t i = 0; i < n[b]; ++i) acc = acc + x[b];
      loop = acc;
    }
    for (int lanes : {64, 40, 7}) {
      int turns = 0;
      const float got = by_turns(x, n, nblk, lanes, turns);
      if (kind == 4 && lanes == 64) {
        turns40 += turns;
        ++rows40;
      }
      if (bh::seq_f2u(got) != bh::seq_f2u(loop)) {
        if (fail < 10)
          std::printf("MISMATCH row %d kind %d lanes %d: loop %08x turns %08x\n", it, kind, lanes,
                      bh::seq_f2u(loop), bh::seq_f2u(got));
        ++fail;
      }
      ++rows;
    }
  }
  {  // two such rows as they were found: 1 + 124 + 77 and 40-block data's first six runs
    const float d0 = half_val(0x3c45u), d1 = half_val(0x2d55u);
    const float xa[3] = {d0 * d0, d1 * d1, d1 * d1};
    const uint32_t na[3] = {1, 124, 77};
    const float xb[6] = {0.0879898667f, 0.00947723165f, 1.09186172f, 0.109112799f, 7.55140209e-05f, 0.342179298f};
    const uint32_t nb[6] = {118, 83, 100, 70, 85, 75};
    int turns = 0;
    const float a = by_turns(xa, na, 3, 64, turns), b = by_turns(xb, nb, 6, 64, turns);
    if (a != 2.53446317f || b != 153.663376f) {
      std::printf("MISMATCH literal rows: %.9g %.9g\n", a, b);
      ++fail;
    }
  }
  for (int it = 0; it < 1000; ++it) {
    float x[160];
    uint32_t n[160];
    const int nblk = landing_row(x, n);
    volatile float loop = 0.0f;
    for (int b = 0; b < nblk; ++b)
      for (uint32_t i = 0; i < n[b]; ++i) loop = loop + x[b];
    for (int lanes : {64, 7}) {
      int turns = 0;
      const float got = by_turns(x, n, nblk, lanes, turns);
      if (bh::seq_f2u(got) != bh::seq_f2u(loop)) {
        if (fail < 10)
          std::printf("MISMATCH landing row %d lanes %d: loop %08x turns %08x\n", it, lanes,
                      bh::seq_f2u(loop), bh::seq_f2u(got));
        ++fail;
      }
      ++rows;
    }
  }
  long by_hand = 0, mixed_rows = 0;
  for (int it = 0; it < 12000; ++it) {  // rows of blocks of two kinds of squares
    Mixed b[64];
    const uint32_t base = below(28);
    const int nblk = 1 + static_cast<int>(below(64));
    volatile float loop = 0.0f;
    for (int l = 0; l < nblk; ++l) {
      uint32_t h;
      switch (it % 4) {
        case 0: h = 1 + below(0x7bffu); break;                // any scale
        case 1: h = (5 + below(20)) << 10; break;             // powers of two: ties
        case 2: h = 0x3c00u + (below(4) << 8); break;         // whole sums, ends on binades
        default: h = ((base + below(3)) << 10) | below(1024);  // a few binades
      }
      const float d = half_val(h);
      b[l].x = d * d;
      b[l].n1 = b[l].n4 = 0;
      b[l].four[0] = b[l].four[1] = 0;
      const uint32_t n = below(5) == 0 ? below(3) : below(129);
      for (uint32_t j = 0; j < n; ++j) {
        const bool four = below(3) == 0;
        b[l].four[j >> 6] |= static_cast<uint64_t>(four) << (j & 63);
        ++(four ? b[l].n4 : b[l].n1);
      }
      loop = add_in_order(loop, b[l]);
    }
    int turns = 0;
    const float got = mixed_by_turns(b, nblk, turns);
    if (it % 4 == 3) by_hand += turns - 1, mixed_rows += nblk;
    if (bh::seq_f2u(got) != bh::seq_f2u(loop)) {
      if (fail < 10)
        std::printf("MISMATCH mixed row %d: loop %08x turns %08x\n", it, bh::seq_f2u(loop), bh::seq_f2u(got));
      ++fail;
    }
    ++rows;
  }
  std::printf("mixed blocks of a few binades: %.2f of them by hand\n",
              static_cast<double>(by_hand) / static_cast<double>(mixed_rows));
  std::printf("%ld rows, %d mismatches, %.1f turns a row of 40 blocks\n", rows, fail,
              static_cast<double>(turns40) / static_cast<double>(rows40));
  return fail != 0;
}
