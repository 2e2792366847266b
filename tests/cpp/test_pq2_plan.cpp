// CPU checks of how PQ2_0 products of many tokens are cut (csrc/pq2_mx_plan.hpp),
// built with g++ by tests/test_pq2_plan.py.
//   test_pq2_plan                     scratch checks over drawn shapes
//   test_pq2_plan ne0 n_rows n_tok    the plan on 256 CUs: R (0: unpacked), parts
//                                     of a split tile, passes over the rows
#include "../../ternary-bonsai-inference_amd/csrc/pq2_mx_plan.hpp"

#include <cstdint>
#include <cstdio>
#include <cstdlib>

namespace {

uint64_t g_state = 1;
uint32_t below(uint32_t n) {  // splitmix64
  uint64_t z = (g_state += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return static_cast<uint32_t>((z ^ (z >> 31)) % n);
}

// One matrix from 1 token to `top`: every call's own need is reserved, and
// nothing that a smaller batch reserves is missing at a larger one.
int check(size_t nblk, size_t n_rows, size_t top, size_t slots) {
  size_t last = 0;
  for (size_t t = 1; t <= top; ++t) {
    const bh::MxPlan p = bh::mx_plan(n_rows, t, nblk, slots);
    const size_t need = bh::mx_scratch_of(p, n_rows, t, nblk, slots).total();
    const size_t got = bh::mx_reserve_bytes(n_rows, t, nblk);
    if (need > got || got < last) {
      std::printf("FAIL nblk %zu rows %zu tokens %zu: needs %zu, reserves %zu, smaller batch %zu\n", nblk,
                  n_rows, t, need, got, last);
      return 1;
    }
    last = got;
  }
  return 0;
}

}  // namespace

int main(int argc, char **argv) {
  if (argc == 4) {
    const size_t nblk = std::strtoull(argv[1], nullptr, 10) / 128;
    const size_t n_rows = std::strtoull(argv[2], nullptr, 10), n_tok = std::strtoull(argv[3], nullptr, 10);
    const bh::MxPlan p = bh::mx_plan(n_rows, n_tok, nblk, 256);
    std::printf("%d %zu %zu\n", p.R, p.split, p.R ? 1 : bh::mx_ceil(n_rows, bh::mx_pass_rows(nblk)));
    return 0;
  }
  int fail = 0;
  const size_t rows[] = {17408, 5120, 6144, 12288, 1024, 48, 248320};
  for (const size_t n : rows)
    for (const size_t nblk : {40, 48, 136}) fail += check(nblk, n, 2100, 256);
  for (int it = 0; it < 60; ++it)
    fail += check(2 * (1 + below(it % 2 ? 80 : 8)), size_t{1} << below(17) | below(64), 700,
                  it % 3 ? 256 : 80 + below(230));
  std::printf("%d failures\n", fail);
  return fail != 0;
}
