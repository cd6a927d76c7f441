// Host run of finish_top (qblas_amd/csrc/finish_top.hpp) against finish_reg_top (exact.hpp): the same
// result and the same bound, bit for bit, on random, cancelling, tied, short, special and extreme
// operands.  Usage: finish_top_host_check <seed> <cases>
#include <stdio.h>
#include <stdlib.h>
#include "../../qblas_amd/csrc/finish_top.hpp"

using namespace qb;

static uint64_t st;
static uint64_t rnd() {
  uint64_t z = (st += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
static int in(int lo, int hi) { return lo + (int)(rnd() % (uint64_t)(hi - lo + 1)); }
static q128 rq(int lo, int hi) {
  q128 v = q_make(rnd(), ((rnd() & 1) << 63) | ((uint64_t)in(lo, hi) << 48) | (rnd() & FRAC_HI_MASK));
  switch (rnd() % 6) {
    case 0: v.lo = 0; v.hi &= ~0xffffffffull; break;  // few bits
    case 1: v.lo = 0; break;
    case 2: v.lo = ~0ull; break;
  }
  return v;
}
template <int N>
static long run(long cases, const char *name) {
  long bad = 0;
  for (long c = 0; c < cases; ++c) {
    uint32_t M[N];
    const int msb = rnd() % 4 ? in(32 * N / 2, 32 * N - 1) : in(0, 32 * N - 1), kind = (int)(rnd() % 10);
    for (int i = 0; i < N; ++i) {
      uint32_t w = (uint32_t)rnd();
      if (kind == 6 && 32 * i + 31 < msb - 60) w = 0;   // short
      if (kind == 7) w = rnd() % 3 ? 0u : ~0u;
      if (32 * i > msb) w = 0;
      else if (msb - 32 * i < 31) w &= (2u << (msb - 32 * i)) - 1u;
      M[i] = w;
    }
    M[msb >> 5] |= 1u << (msb & 31);
    const int lsb = (kind == 9 ? (rnd() & 1 ? in(-16500, -16300) : in(16200, 16390)) : in(-60, 60)) - msb;
    const uint32_t sS = (uint32_t)(rnd() & 1);
    q128 alpha = rq(16383 - 3, 16383 + 3), beta = rq(16383 - 3, 16383 + 3), y = rq(16383 - 70, 16383 + 70);
    if (kind == 0) beta = q_zero(rnd() & 1);
    if (kind == 1) y = q_zero(rnd() & 1);
    if (kind <= 2 && rnd() % 2) alpha = q_make(0, ((rnd() & 1) << 63) | 0x3fff000000000000ull);
    if (kind == 3) {  // beta y against alpha M: exact or near cancellation
      const q128 s = finish_reg_t<N>(M, lsb, sS, 0u, 0u, false, q_one(), q_zero(0), q_zero(0));
      beta = alpha;
      y = s;
      y.hi ^= 1ull << 63;
      if (rnd() & 1) y.lo ^= 1ull << (rnd() % 64);
      if (rnd() & 1) y.hi ^= 1ull << (rnd() % 48);
    }
    if (kind == 4) beta = rq(1, 0x7ffe);
    if (kind == 5) y = rq(0, 0x7ffe);
    if (kind == 8) alpha = rq(0, 0x7ffe);
    if (q_iszero(alpha)) continue;
    int t0, t1;
    const q128 want = finish_reg_top<N>(M, lsb, sS, alpha, beta, y, t0), got = finish_top<N>(M, lsb, sS, alpha, beta, y, t1);
    if (want.lo != got.lo || want.hi != got.hi || t0 != t1)
      if (bad++ < 5)
        printf("N %d kind %d msb %d lsb %d: got %016lx%016lx (%d) want %016lx%016lx (%d)\n", N, kind, msb, lsb, got.hi, got.lo, t1,
               want.hi, want.lo, t0);
  }
  printf("%s: cases %ld mismatches %ld\n", name, cases, bad);
  return bad;
}
int main(int argc, char **argv) {
  st = strtoull(argv[1], 0, 10);
  const long n = atol(argv[2]);
  return run<6>(n, "6 words") + run<9>(n, "9 words") + run<11>(n, "11 words") ? 1 : 0;
}
