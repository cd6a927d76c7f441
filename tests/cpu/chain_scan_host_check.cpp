// Host build of the wave-wide FMA chain (qblas_amd/csrc/chain_scan.hpp): its blocks of 64 lanes with
// the lanes' prefix sums as loops, against serial fma_packed, bit for bit, over chains of many kinds
// of operands.  Usage: chain_scan_host_check <seed> <chains>
// -> per kind "steps <n> blocks <n> fixes <n> single <n> wrong chains <n>"; exits 1 on a wrong chain.
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "../../qblas_amd/csrc/chain_scan.hpp"

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
static q128 shorty(int be, int bits) {
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
static const char *kinds[] = {"uniform", "wide", "double", "integer", "ones", "positive", "sparse",
                              "ties",    "ends", "special", "cancel", "extreme", "edges", "drift"};
static int geo() {
  int e = 0;
  while (e < 60 && (rnd() & 1)) ++e;
  return e;
}
static void operands(int kind, int i, q128 &a, q128 &b) {
  static q128 pa, pb;
  switch (kind) {
    case 0: a = full(16382 - geo()); b = full(16382 - geo()); break;
    case 1: a = full(16353 + (int)(rnd() % 60)); b = full(16353 + (int)(rnd() % 60)); break;
    case 2: a = shorty(16382 - geo(), 52); b = shorty(16382 - geo(), 52); break;
    case 3: a = shorty(16383 + (int)(rnd() % 6), (int)(rnd() % 6)); b = shorty(16383 + (int)(rnd() % 4), (int)(rnd() % 4)); break;
    case 4: a = q_one(); b = q_one(); break;
    case 5: a = full(16382 - geo()); b = full(16382 - geo()); a.hi &= ~0ull >> 1; b.hi &= ~0ull >> 1; break;
    case 6: a = rnd() % 4 ? q_zero(rnd() & 1) : full(16382 - geo()); b = full(16382 - geo()); break;
    case 7: a = shorty(16383 - (int)(rnd() % 4), 52 + (int)(rnd() % 4)); b = shorty(16383 - (int)(rnd() % 12), 52); break;
    case 8: a = full(rnd() & 1 ? 0x7ffe - (int)(rnd() % 200) : 1 + (int)(rnd() % 200)); b = full(16383 + (int)(rnd() % 300) - 150); break;
    case 9:
      a = full(16383);
      b = full(16383);
      switch (rnd() % 40) {
        case 0: a = q_zero(rnd() & 1); break;
        case 1: b = q_zero(rnd() & 1); break;
        case 2: a = mk(rnd() & 1, 0, rnd(), rnd()); break;
        case 3: if (i > 200) a = q_inf(rnd() & 1); break;
        case 4: if (i > 250) b = q_nan(); break;
      }
      break;
    case 10:
      if (i & 1) {
        a = pa;
        b = pb;
        a.hi ^= 1ull << 63;
        if (rnd() & 1) a.lo ^= rnd() & 3;
      } else {
        a = full(16383 + (int)(rnd() % 80));
        b = full(16383 + (int)(rnd() % 8));
      }
      break;
    case 11:
      a = mk(rnd() & 1, 16383 + (int)(rnd() % 3) - 1, rnd() & 1 ? ~0ull : 0, rnd() & 1 ? ~0ull : rnd() & 1);
      b = mk(rnd() & 1, 16383 + (int)(rnd() % 3) - 1, rnd() & 1 ? ~0ull : 0, rnd() & 1 ? ~0ull : rnd() & 1);
      break;
    case 12:  // sums next to powers of two, with runs of zero products
      a = rnd() % 3 == 0 ? q_zero(rnd() & 1) : mk(rnd() & 1, 16383 - 20 * (int)(rnd() % 7), rnd() & 1 ? ~0ull : 0, rnd() & 1 ? ~0ull : 0);
      b = q_one();
      break;
    default: a = full(16383 + i / 16 % 40); b = full(16383 - i / 40 % 20); break;
  }
  pa = a;
  pb = b;
}
static long blocks, fixes, packed;
static q128 chain64(q128 init, const std::vector<q128> &a, const std::vector<q128> &b) {
  sstate s;
  sstate_set(s, init);
  const int64_t n = (int64_t)a.size();
  for (int64_t pos = 0; pos < n;) {
    const int cnt = (int)(n - pos < 64 ? n - pos : 64);
    sprod p[64];
    for (int i = 0; i < 64; ++i)
      p[i] = i < cnt ? sc_product(a[pos + i], b[pos + i]) : sc_product(q_zero(0), q_zero(0));
    int lo = 0;
    while (lo < cnt) {
      int cut = lo;
      if (s.kind == 2 && s.b == QBIAS + 1) {
        if (q_isnan(sstate_get(s))) return q_nan();
        while (cut < cnt && q_bexp(a[pos + cut]) != 0x7fff && q_bexp(b[pos + cut]) != 0x7fff) ++cut;
      } else if (s.kind != 2) {
        ++blocks;
        int first = -1;
        for (int i = 63; i >= 0; --i)
          if (p[i].Ep != -SC_BIG && !p[i].bad) first = i;
        const int32_t b0 = s.kind == 0 ? s.b : (first >= 0 ? p[first].Ep : 0), bmin = b0 - SC_LOW;
        slane l[64];
        uint32_t S[64][4];
        double d = sc_first(s), sum = 0;
        int32_t bp = s.kind == 0 ? s.b : SC_BIG;
        uint32_t T[4] = {0, 0, 0, 0};
        if (s.kind == 0) {
          uint32_t c = s.neg & 1u;
          for (int w = 0; w < 4; ++w) T[w] = ch_addc(0u, s.w[w] ^ s.neg, c, c);
        }
        bool usable = true;
        for (int i = 0; i < 64; ++i) {
          sum += sc_value(p[i], b0);
          const int32_t bi = sc_binade(sum + d, b0);
          l[i] = sc_round(p[i], bi, bp, bmin);
          if (p[i].Ep != -SC_BIG) bp = bi;
          uint32_t c = 0;
          for (int w = 0; w < 4; ++w) S[i][w] = T[w] = ch_addc(T[w], l[i].v[w], c, c);
        }
        for (int f = 0; f < 64; ++f) {
          usable = usable && !(p[f].bad || (p[f].Ep != -SC_BIG && !l[f].live));
          if (!l[f].fix || !usable) continue;
          ++fixes;
          const int32_t D = sc_fix(l[f], S[f][0]);
          for (int i = f; i < 64; ++i) {
            uint32_t c = 0;
            S[i][0] = ch_addc(S[i][0], (uint32_t)D, c, c);
            for (int w = 1; w < 4; ++w) S[i][w] = ch_addc(S[i][w], (uint32_t)(D >> 31), c, c);
          }
        }
        cut = 0;
        while (cut < 64 && !p[cut].bad && (p[cut].Ep == -SC_BIG || (l[cut].live && sc_inside(S[cut][3], l[cut].k)))) ++cut;
        if (cut > lo) sstate_from_sum(s, S[cut - 1], bmin);
      }
      lo = cut;
      if (cut < cnt) {
        ++packed;
        sstate_step(s, a[pos + cut], b[pos + cut]);
        for (int i = 0; i <= cut; ++i) sc_clear(p[i]);
        lo = cut + 1;
        if (lo > 32) break;
      }
    }
    pos += lo >= cnt ? 64 : lo;
  }
  return sstate_get(s);
}
int main(int argc, char **argv) {
  st = strtoull(argv[1], 0, 10);
  const int chains = atoi(argv[2]);
  long bad = 0;
  for (int kind = 0; kind < (int)(sizeof(kinds) / sizeof(*kinds)); ++kind) {
    long steps = 0, wrong = 0;
    blocks = fixes = packed = 0;
    for (int c = 0; c < chains; ++c) {
      const int n = c % 8 == 0 ? 1 + (int)(rnd() % 200) : 1 + (int)(rnd() % 1500);
      std::vector<q128> a(n), b(n);
      q128 init = q_zero(0);
      if (rnd() % 3 == 0) {
        q128 x;
        operands(kind, 0, init, x);
        if (rnd() % 8 == 0) init = q_zero(1);
      }
      q128 ref = init;
      for (int i = 0; i < n; ++i) {
        operands(kind, i, a[i], b[i]);
        ref = fma_packed(a[i], b[i], ref);
      }
      const q128 got = chain64(init, a, b);
      steps += n;
      if (got.lo != ref.lo || got.hi != ref.hi) {
        if (wrong++ < 3) printf("%s n %d got %016lx%016lx want %016lx%016lx\n", kinds[kind], n, got.hi, got.lo, ref.hi, ref.lo);
      }
    }
    printf("%s: steps %ld blocks %ld fixes %ld single %ld wrong chains %ld\n", kinds[kind], steps, blocks, fixes, packed, wrong);
    bad += wrong;
  }
  return bad ? 1 : 0;
}
