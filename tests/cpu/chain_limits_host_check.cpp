// Host build of the accumulating FMA chain (qblas_amd/csrc/chain.hpp) where chain_host_check does not go: the limits of the fast
// step (operands next to 2^+-8100, accumulators next to +-CH_EMAX), and matrices with many zeros, whose steps chain_zero and
// chain_rest take, against fma_packed, bit for bit after every step.  Usage: chain_limits_host_check <seed> <chains>
// -> per kind "steps <n> slow <n> mismatches <n>"; exits 1 on a mismatch.
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
static q128 mk(uint64_t s, int e, uint64_t fh, uint64_t fl) {  // exponent e
  return q_make(fl, (s << 63) | ((uint64_t)(e + QBIAS) << 48) | (fh & FRAC_HI_MASK));
}
static q128 full(int e) { return mk(rnd() & 1, e, rnd(), rnd()); }
static const char *kinds[] = {"top", "bottom", "topcancel", "bottomcancel", "zeros", "signedzeros", "zerospecials"};
static q128 first(int kind) {
  switch (kind) {
    case 0: case 2: return full(16240 + (int)(rnd() % 140));
    case 1: case 3: return full(-16240 - (int)(rnd() % 140));
    default: return rnd() & 1 ? q_zero(rnd() & 1) : full(-(int)(rnd() % 40));
  }
}
static void operands(int kind, int i, q128 &a, q128 &b) {
  static q128 pa, pb;
  const int sign = kind & 1 ? -1 : 1;
  auto zero = [](int in) { return rnd() % in ? full(-(int)(rnd() % 4)) : q_zero(rnd() & 1); };
  switch (kind) {
    case 0: case 1: a = full(sign * (8040 + (int)(rnd() % 64))); b = full(sign * (8040 + (int)(rnd() % 64))); break;
    case 2: case 3:  // the same, every second product the one before but for its last bits, negated
      a = full(sign * (8040 + (int)(rnd() % 61)));
      b = full(sign * (8040 + (int)(rnd() % 61)));
      if (i & 1) {
        a = pa;
        b = pb;
        a.hi ^= 1ull << 63;
        a.lo ^= (rnd() & 7) << (rnd() % 40);
      }
      break;
    case 4: a = zero(2); b = zero(2); break;
    case 5: a = rnd() % 8 ? q_zero(rnd() & 1) : full(0); b = rnd() % 8 ? q_zero(rnd() & 1) : full(0); break;
    default:
      a = zero(2);
      b = zero(2);
      if (i > 40 && rnd() % 60 == 0) a = rnd() & 1 ? q_inf(rnd() & 1) : mk(rnd() & 1, -QBIAS, rnd(), rnd());
      if (i > 150 && rnd() % 60 == 0) b = q_nan();
  }
  pa = a;
  pb = b;
}
int main(int argc, char **argv) {
  st = strtoull(argv[1], 0, 10);
  const int chains = atoi(argv[2]);
  long bad = 0;
  for (int kind = 0; kind < (int)(sizeof(kinds) / sizeof(*kinds)); ++kind) {
    long steps = 0, slow = 0, wrong = 0;
    for (int c = 0; c < chains; ++c) {
      q128 ref = rnd() & 1 ? q_zero(0) : first(kind);
      cacc acc;
      cacc_set(acc, ref);
      for (int i = 0; i < 200; ++i, ++steps) {
        q128 a, b;
        operands(kind, i, a, b);
        ref = fma_packed(a, b, ref);
        const cop A = cop_unpack(a), B = cop_unpack(b);
        if (i == 0) cacc_first(acc, A, B);
        if (!cacc_step(acc, A, B)) {
          ++slow;
          // the two forms that kernels use
          if (c & 1) chain_rest(acc, a, b);
          else if ((A.zero | B.zero) != 1u || !chain_zero(acc, A.neg ^ B.neg)) chain_slow(acc, a, b);
        }
        const q128 got = cacc_get(acc);
        if (got.lo != ref.lo || got.hi != ref.hi) {
          if (wrong++ < 3)
            printf("%s step %d: a %016lx%016lx b %016lx%016lx got %016lx%016lx want %016lx%016lx\n", kinds[kind], i, a.hi, a.lo, b.hi, b.lo,
                   got.hi, got.lo, ref.hi, ref.lo);
          cacc_set(acc, ref);
        }
      }
    }
    printf("%s: steps %ld slow %ld mismatches %ld\n", kinds[kind], steps, slow, wrong);
    bad += wrong;
  }
  return bad ? 1 : 0;
}
