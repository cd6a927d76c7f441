// Host build of the accumulating FMA chain (qblas_amd/csrc/chain.hpp) against fma_packed, bit for bit
// after every step, over chains of many kinds of operands.  Usage: chain_host_check <seed> <chains>
// -> prints "steps <n> slow <n> mismatches <n>" per kind and exits 1 on any mismatch.
#include <stdio.h>
#include <stdlib.h>
#include "../../qblas_amd/csrc/chain.hpp"

using namespace qb;
static uint64_t st;
static uint64_t rnd() {
  uint64_t z = (st += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
static q128 mk(uint64_t s, int be, uint64_t fh, uint64_t fl) {
  return q_make(fl, (s << 63) | ((uint64_t)be << 48) | (fh & FRAC_HI_MASK));
}
static q128 full(int be) { return mk(rnd() & 1, be, rnd(), rnd()); }
static q128 shorty(int be, int bits) {  // `bits` leading fraction bits, the rest zero
  uint64_t fh = rnd() & FRAC_HI_MASK, fl = rnd();
  const int drop = 112 - bits;
  if (drop >= 64) {
    fl = 0;
    fh = drop >= 112 ? 0 : (fh >> (drop - 64)) << (drop - 64);
  } else if (drop > 0) {
    fl = (fl >> drop) << drop;
  }
  return mk(rnd() & 1, be, fh, fl);
}
static q128 extreme() {  // all ones, powers of two, one ulp off
  switch (rnd() % 4) {
    case 0: return mk(rnd() & 1, 16383 + (int)(rnd() % 5) - 2, ~0ull, ~0ull);
    case 1: return mk(rnd() & 1, 16383 + (int)(rnd() % 5) - 2, 0, 0);
    case 2: return mk(rnd() & 1, 16383 + (int)(rnd() % 5) - 2, 0, 1);
    default: return mk(rnd() & 1, 16383 + (int)(rnd() % 5) - 2, ~0ull, ~0ull << (rnd() % 64));
  }
}
static const char *kinds[] = {"uniform", "wide",     "double", "integer", "extreme",  "offsets",
                              "ends",    "specials", "cancel", "short",   "subnormal"};
static q128 prev_a, prev_b;
static void operands(int kind, int i, q128 &a, q128 &b) {
  auto geo = [] { int e = 0; while (e < 60 && (rnd() & 1)) ++e; return e; };
  switch (kind) {
    case 0: a = full(16382 - geo()); b = full(16382 - geo()); break;
    case 1: a = full(16353 + (int)(rnd() % 60)); b = full(16353 + (int)(rnd() % 60)); break;
    case 2: a = shorty(16382 - geo(), 52); b = shorty(16382 - geo(), 52); break;
    case 3: a = shorty(16383 + (int)(rnd() % 6), (int)(rnd() % 6)); b = shorty(16383 + (int)(rnd() % 4), (int)(rnd() % 4)); break;
    case 4: a = extreme(); b = extreme(); break;
    case 5: a = full(16383 + (int)(rnd() % 340) - 170); b = rnd() & 1 ? extreme() : full(16383); break;
    case 6: {
      const int top = (int)(rnd() & 1);
      a = full(top ? 0x7ffe - (int)(rnd() % 200) : 1 + (int)(rnd() % 200));
      b = full(16383 + (int)(rnd() % 300) - 150);
      break;
    }
    case 7:
      a = full(16383);
      b = full(16383);
      switch (rnd() % 24) {
        case 0: a = q_zero(rnd() & 1); break;
        case 1: b = q_zero(rnd() & 1); break;
        case 2: a = mk(rnd() & 1, 0, rnd(), rnd()); break;
        case 3: if (i > 20) a = q_inf(rnd() & 1); break;
        case 4: if (i > 30) b = q_nan(); break;
      }
      break;
    case 8:  // pairs that cancel exactly or to the last bits
      if (i & 1) {
        a = prev_a;
        b = prev_b;
        a.hi ^= 1ull << 63;
        if (rnd() & 1) a.lo ^= rnd() & 3;
      } else {
        a = full(16383 + (int)(rnd() % 80));
        b = full(16383 + (int)(rnd() % 8));
      }
      break;
    case 9: a = shorty(16383 + (int)(rnd() % 120) - 60, (int)(rnd() % 113)); b = shorty(16383, (int)(rnd() % 113)); break;
    default: a = full(1 + (int)(rnd() % 300)); b = full(16383 - (int)(rnd() % 260)); break;
  }
  prev_a = a;
  prev_b = b;
}
static bool same(q128 x, q128 y) { return x.lo == y.lo && x.hi == y.hi; }
int main(int argc, char **argv) {
  st = strtoull(argv[1], 0, 10);
  const int chains = atoi(argv[2]);
  long bad = 0;
  for (int kind = 0; kind < (int)(sizeof(kinds) / sizeof(*kinds)); ++kind) {
    long steps = 0, slow = 0, wrong = 0;
    for (int c = 0; c < chains; ++c) {
      q128 ref = q_zero(0);
      cacc acc;
      cacc_init(acc);
      if (rnd() % 3 == 0) {  // a chain that starts from a value (column-major gemv: beta * y)
        q128 a, b;
        operands(kind, 0, a, b);
        ref = rnd() % 8 ? a : q_zero(1);
        cacc_set(acc, ref);
      }
      for (int i = 0; i < 200; ++i) {
        q128 a, b;
        operands(kind, i, a, b);
        ref = fma_packed(a, b, ref);
        ++steps;
        const cop A = cop_unpack(a), B = cop_unpack(b);
        if (i == 0) cacc_first(acc, A, B);
        if (!cacc_step(acc, A, B)) {
          ++slow;
          chain_slow(acc, a, b);
        }
        const q128 got = cacc_get(acc);
        if (!same(got, ref)) {
          if (wrong < 5)
            printf("%s step %d: a %016lx%016lx b %016lx%016lx got %016lx%016lx want %016lx%016lx\n", kinds[kind], i,
                   a.hi, a.lo, b.hi, b.lo, got.hi, got.lo, ref.hi, ref.lo);
          ++wrong;
          cacc_set(acc, ref);
        }
      }
    }
    printf("%s: steps %ld slow %ld mismatches %ld\n", kinds[kind], steps, slow, wrong);
    bad += wrong;
  }
  return bad ? 1 : 0;
}
