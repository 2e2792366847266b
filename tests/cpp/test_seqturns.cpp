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
  std::printf("%ld rows, %d mismatches, %.1f turns a row of 40 blocks\n", rows, fail,
              static_cast<double>(turns40) / static_cast<double>(rows40));
  return fail != 0;
}
