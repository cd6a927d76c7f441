// Host build of both forms of the scanned FMA chain (qblas_amd/csrc/chain_scan.hpp), the wave's 64 steps at a time
// and the workgroup's 2048, with lanes and prefix sums as loops, against serial fma_packed, bit for bit.
// Usage: chain_group_host_check <seed> <chains>
// -> per kind, of chains by a wave and by a workgroup, the steps, the passes over a block, the steps taken alone, and the chains
// that went on with exact blocks or were left; and "wrong chains <n>".  Exits 1 on a wrong chain.
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
static q128 head(int be, int bits) {  // at most 64 leading fraction bits
  const uint64_t f = bits ? rnd() >> (64 - bits) << (64 - bits) : 0;
  return mk(rnd() & 1, be, f >> 16, f << 48);
}
static int geo() {
  int e = 0;
  while (e < 60 && (rnd() & 1)) ++e;
  return e;
}
static q128 whole(int v) {  // the integer v
  if (v == 0) return q_zero(0);
  const int m = v < 0 ? -v : v, e = 31 - __builtin_clz(m);
  return q_make(0, ((uint64_t)(v < 0) << 63) | ((uint64_t)(16383 + e) << 48) | ((uint64_t)(m - (1 << e)) << (48 - e)));
}
static const char *kinds[] = {"uniform", "wide", "double", "positive", "sparse", "ties", "drift", "special", "extreme", "edges",
                              "ones", "signs", "alternating", "twos", "integer", "difference", "zeroed", "cancel", "subnormal", "ends", "nearends", "brink", "far"};
static void operands(int kind, int i, q128 &a, q128 &b) {
  static q128 pa, pb;
  switch (kind) {
    case 0: a = full(16382 - geo()); b = full(16382 - geo()); break;
    case 1: a = full(16353 + (int)(rnd() % 60)); b = full(16353 + (int)(rnd() % 60)); break;
    case 2: a = head(16382 - geo(), 52); b = head(16382 - geo(), 52); break;
    case 3: a = full(16382 - geo()); b = full(16382 - geo()); a.hi &= ~0ull >> 1; b.hi &= ~0ull >> 1; break;
    case 4: a = rnd() % 4 ? q_zero(rnd() & 1) : full(16382 - geo()); b = full(16382 - geo()); break;
    case 5: a = head(16383 - (int)(rnd() % 4), 52 + (int)(rnd() % 4)); b = head(16383 - (int)(rnd() % 12), 52); break;
    case 6: a = full(16383 + i / 16 % 40); b = full(16383 - i / 40 % 20); break;
    case 7:
      a = full(16383);
      b = full(16383);
      switch (rnd() % 400) {
        case 0: a = q_zero(rnd() & 1); break;
        case 1: b = q_zero(rnd() & 1); break;
        case 2: a = mk(rnd() & 1, 0, rnd(), rnd()); break;
        case 3: if (i > 5000) a = q_inf(rnd() & 1); break;
        case 4: if (i > 7000) b = q_nan(); break;
      }
      break;
    case 8:
      a = mk(rnd() & 1, 16383 + (int)(rnd() % 3) - 1, rnd() & 1 ? ~0ull : 0, rnd() & 1 ? ~0ull : rnd() & 1);
      b = mk(rnd() & 1, 16383 + (int)(rnd() % 3) - 1, rnd() & 1 ? ~0ull : 0, rnd() & 1 ? ~0ull : rnd() & 1);
      break;
    case 9:  // sums next to powers of two, with runs of zero products
      a = rnd() % 3 == 0 ? q_zero(rnd() & 1) : mk(rnd() & 1, 16383 - 20 * (int)(rnd() % 7), rnd() & 1 ? ~0ull : 0, rnd() & 1 ? ~0ull : 0);
      b = q_one();
      break;
    case 10: a = b = q_one(); break;
    case 11: a = whole(rnd() & 1 ? 1 : -1); b = q_one(); break;
    case 12: a = whole(i & 1 ? -1 : 1); b = q_one(); break;
    case 13: a = whole(i & 2 ? -1 : 1); b = q_one(); break;
    case 14: a = whole((int)(rnd() % 17) - 8); b = whole((int)(rnd() % 9) - 4); break;
    case 15: a = whole(i % 3 == 1 ? -2 : 1); b = head(16383, 20); if (i % 3) b = pb; break;  // x - 2x + x
    case 16:  // x, -x
      a = full(16382 - geo());
      b = q_one();
      if (i & 1) {
        a = pa;
        a.hi ^= 1ull << 63;
      }
      break;
    case 17:
      a = full(16383 + (int)(rnd() % 80));
      b = full(16383 + (int)(rnd() % 8));
      if (i & 1) {
        a = pa;
        b = pb;
        a.hi ^= 1ull << 63;
        if (rnd() & 1) a.lo ^= rnd() & 3;
      }
      break;
    case 18: a = mk(rnd() & 1, 0, rnd(), rnd()); b = full(16382 - geo()); break;
    case 19: a = full(rnd() & 1 ? 0x7ffe - (int)(rnd() % 200) : 1 + (int)(rnd() % 200)); b = full(16383 + (int)(rnd() % 300) - 150); break;
    case 21: a = i ? full(16383 - 20 - (int)(rnd() % 60)) : mk(0, 16383 + 58, (rnd() & 1 ? ~0ull : 0) ^ (rnd() & 0x3ffff), rnd()); b = i ? full(16383) : q_one(); break;
    case 22: a = full(12383 + (int)(rnd() % 8000)); b = full(12383 + (int)(rnd() % 8000)); break;
    default: {  // products next to +-SC_EMAX of operands that are not special
      const int top = i / 512 & 1 ? 1 : -1;
      a = full(16383 + top * (8040 + (int)(rnd() % 60)));
      b = full(16383 + top * (8040 + (int)(rnd() % 60)));
    }
  }
  pa = a;
  pb = b;
}

typedef std::vector<q128> vec;
static long passes, group_passes, alone;
template <bool LOSSLESS>
static bool final(const sprod &p, const slane &l, const uint32_t (&S)[4], uint32_t before) {
  return !p.bad && (p.Ep == -SC_BIG || (LOSSLESS ? sc_final(l, S, before) : l.live && sc_inside(S[3], l.k)));
}
static void add(uint32_t (&x)[4], const uint32_t (&y)[4]) {
  uint32_t c = 0;
  for (int i = 0; i < 4; ++i) x[i] = ch_addc(x[i], y[i], c, c);
}
static void add(uint32_t (&x)[4], int32_t y) {
  const uint32_t e = (uint32_t)(y >> 31), w[4] = {(uint32_t)y, e, e, e};
  add(x, w);
}
// the state in units of 2^(bmin - 112)
static void units(uint32_t (&T)[4], const sstate &s, int32_t bmin) {
  unsigned __int128 v = 0;
  if (s.kind == 0) {
    for (int i = 3; i >= 0; --i) v = (v << 32) | s.w[i];
    const int up = s.b - bmin - SC_LOW;
    v = up >= 0 ? v << up : v >> -up;
    if (s.neg) v = -v;
  }
  for (int i = 0; i < 4; ++i) T[i] = (uint32_t)(v >> (32 * i));
}
template <bool LOSSLESS>
static int64_t wave(sstate &s, const vec &a, const vec &b, int64_t pos, int64_t n) {
  int poor = 0;
  while (pos < n) {
    const int cnt = (int)(n - pos < 64 ? n - pos : 64);
    sprod p[64];
    for (int i = 0; i < 64; ++i) p[i] = i < cnt ? sc_product(a[pos + i], b[pos + i]) : sc_product(q_zero(0), q_zero(0));
    int lo = 0;
    while (lo < cnt) {
      int cut = lo;
      if (s.kind == 2 && s.b == QBIAS + 1) {
        if (q_isnan(sstate_get(s))) {
          sstate_set(s, q_nan());
          return n;
        }
        while (cut < cnt && q_bexp(a[pos + cut]) != 0x7fff && q_bexp(b[pos + cut]) != 0x7fff) ++cut;
      } else if (s.kind != 2) {
        ++passes;
        int first = -1;
        for (int i = 63; i >= 0; --i)
          if (p[i].Ep != -SC_BIG && !p[i].bad) first = i;
        const int32_t b0 = s.kind == 0 ? s.b : (first >= 0 ? p[first].Ep : 0), bmin = b0 - SC_LOW;
        slane l[64];
        uint32_t S[64][4], T[4], S0;
        units(T, s, bmin);
        S0 = T[0];
        double sum = 0;
        int32_t bp = s.kind == 0 ? s.b : SC_BIG;
        bool usable = true;
        for (int i = 0; i < 64; ++i) {
          sum += sc_value(p[i], b0);
          const int32_t bi = sc_binade(sum + sc_first(s), b0, LOSSLESS ? p[i].Ep : SC_BIG);
          l[i] = sc_round<LOSSLESS>(p[i], bi, bp, bmin);
          if (p[i].Ep != -SC_BIG) bp = bi;
          add(T, l[i].v);
          for (int w = 0; w < 4; ++w) S[i][w] = T[w];
        }
        for (int f = 0; f < 64; ++f) {
          usable = usable && !(p[f].bad || (p[f].Ep != -SC_BIG && !l[f].live));
          if (!l[f].fix || !usable) continue;
          const int32_t D = sc_fix(l[f], S[f][0]);
          for (int i = f; i < 64; ++i) add(S[i], D);
        }
        cut = 0;
        while (cut < 64 && final<LOSSLESS>(p[cut], l[cut], S[cut], cut ? S[cut - 1][0] : S0)) ++cut;
        if (cut > lo) sstate_from_sum(s, S[cut - 1], bmin, LOSSLESS);
      }
      const int from = lo;
      lo = cut;
      if (cut < cnt) {
        if (LOSSLESS) return pos + cut;
        sstate_step(s, a[pos + cut], b[pos + cut]);
        for (int i = 0; i <= cut; ++i) sc_clear(p[i]);
        lo = cut + 1;
        poor = cut - from < 16 ? poor + 1 : 0;
        if (poor == SC_POOR) return pos + lo;
        if (lo > 32) break;
      }
    }
    if (lo >= cnt) poor = 0;
    pos += lo >= cnt ? 64 : lo;
  }
  return n;
}
static void wave_lossless(sstate &s, int &short_blocks, const vec &a, const vec &b, int64_t pos, int64_t n) {
  while (pos < n) {
    const int64_t at = wave<true>(s, a, b, pos, n);
    if (at >= n) return;
    const int by = sc_pace(short_blocks, at - pos);
    pos = n - at < by ? n : at + by;
    cacc acc;
    cacc_set(acc, sstate_get(s));
    for (int64_t i = at; i < pos; ++i) {
      ++alone;
      if (!cacc_step(acc, cop_unpack(a[i]), cop_unpack(b[i]))) chain_slow(acc, a[i], b[i]);
    }
    sstate_set(s, cacc_get(acc));
  }
}
// wave_chain_or_not
static bool wave_or_not(sstate &s, const vec &a, const vec &b, int64_t pos, int64_t n, bool leave) {
  int short_blocks = 0;
  while (pos < n) {
    const int64_t at = wave<true>(s, a, b, pos, n);
    if (at >= n) break;
    const int by = sc_pace(short_blocks, at - pos);
    if (leave && short_blocks == SC_POOR) return false;
    pos = n - at < by ? n : at + by;
    for (int64_t i = at; i < pos; ++i) sstate_step(s, a[i], b[i]);
  }
  return true;
}
template <bool LOSSLESS>
static int64_t group(sstate &s, const vec &a, const vec &b, int64_t pos) {
  const int64_t n = (int64_t)a.size();
  bool single = true;
  int poor = 0;
  int64_t solo = 64;
  int short_blocks = 0;
  while (pos < n) {
    if (single || s.kind != 0) {
      const int64_t by = LOSSLESS ? solo : 64, to = n - pos < by ? n : pos + by;
      if (LOSSLESS) {
        wave_lossless(s, short_blocks, a, b, pos, to);
        pos = to;
      } else {
        pos = wave<false>(s, a, b, pos, to);
        if (pos < to) return pos;
      }
      if (s.kind == 2 && q_isnan(sstate_get(s))) return n;
      single = false;
      continue;
    }
    ++group_passes;
    static sprod p[SG_STEPS];
    static slane l[SG_STEPS];
    static uint32_t S[SG_STEPS][4];
    double end[SG_WAVES], d[SG_STEPS], sum = 0;
    for (int i = 0; i < SG_STEPS; ++i) {
      p[i] = pos + i < n ? sc_product(a[pos + i], b[pos + i]) : sc_product(q_zero(0), q_zero(0));
      d[i] = (sum += sc_value(p[i], s.b)) + sc_first(s);
      end[i / SG_SPAN] = d[i];
    }
    int32_t top = s.b;
    for (double e : end) {
      const int32_t t = sc_binade(e, s.b, s.b);
      if (t > top) top = t;
    }
    int32_t bmin = top + 2 - SC_WIN;
    if (bmin > s.b) bmin = s.b - SC_LOW;
    uint32_t T[4], S0;
    units(T, s, bmin);
    S0 = T[0];
    int32_t bp = -SC_BIG;
    std::vector<sg_fix> list;
    for (int i = 0; i < SG_STEPS; ++i) {
      if (i % SG_SPAN == 0) bp = -SC_BIG;  // a wave does not know the binade before
      const int32_t bi = sc_binade(d[i], s.b, LOSSLESS ? p[i].Ep : SC_BIG);
      l[i] = sc_round<LOSSLESS>(p[i], bi, bp, bmin);
      if (p[i].Ep != -SC_BIG) bp = bi;
      add(T, l[i].v);
      for (int w = 0; w < 4; ++w) S[i][w] = T[w];
      if (l[i].fix) list.push_back(sg_make_fix(l[i], T[0]));
    }
    std::vector<int32_t> corr;
    uint32_t E = 0;
    for (const sg_fix &f : list) {
      const uint32_t z = f.A + E, add = (1u << (f.k - 1)) - (f.odd ? 1u : 0u), grid = 0u - (1u << f.k);
      E = ((z + add + ((z & f.odd) ? 1u : 0u)) & grid) - f.after;
      corr.push_back((int32_t)E >> 1);
    }
    int done = 0, at = 0;
    uint32_t before = S0;
    for (; done < SG_STEPS; ++done) {
      at += l[done].fix;
      add(S[done], at ? corr[at - 1] : 0);
      if (!final<LOSSLESS>(p[done], l[done], S[done], before)) break;
      before = S[done][0];
    }
    if (done) sstate_from_sum(s, S[done - 1], bmin, LOSSLESS);
    pos += done;
    single = done < SG_STEPS;
    poor = done < 128 ? poor + 1 : 0;
    if (!LOSSLESS && poor == 3) return pos;
    solo = poor < 2 ? 64 : solo < 8192 ? 2 * solo : 8192;
  }
  return n;
}
int main(int argc, char **argv) {
  st = strtoull(argv[1], 0, 10);
  const int chains = atoi(argv[2]);
  long bad = 0;
  for (int kind = 0; kind < (int)(sizeof(kinds) / sizeof(*kinds)); ++kind) {
    long steps[2] = {0, 0}, wrong = 0;
    passes = group_passes = alone = 0;
    long wave_passes = 0, wave_alone = 0, turned[2] = {0, 0}, left = 0;
    for (int c = 0; c < chains; ++c) {
      const int groups = c % 4 == 0;
      const int n = 1 + (int)(rnd() % (groups ? 9000 : 1500));
      vec a(n), b(n);
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
      const long were = passes, were_alone = alone;
      sstate s;
      sstate_set(s, init);
      const int64_t at = groups ? group<false>(s, a, b, 0) : wave<false>(s, a, b, 0, n);
      if (at < n) {
        ++turned[groups];
        if (groups) {
          group<true>(s, a, b, at);
        } else {
          sstate t = s;
          const long are = passes;
          if (!wave_or_not(t, a, b, at, n, true)) {
            ++left;
            t = s;
            wave_or_not(t, a, b, at, n, false);
          }
          const q128 got = sstate_get(t);
          wrong += got.lo != ref.lo || got.hi != ref.hi;
          passes = are;
          int short_blocks = 0;
          wave_lossless(s, short_blocks, a, b, at, n);
        }
      }
      const q128 got = sstate_get(s);
      if (!groups) wave_passes += passes - were, wave_alone += alone - were_alone;
      steps[groups] += n;
      if (got.lo != ref.lo || got.hi != ref.hi) {
        if (wrong++ < 3)
          printf("%s groups %d n %d got %016lx%016lx want %016lx%016lx\n", kinds[kind], groups, n, got.hi, got.lo, ref.hi, ref.lo);
      }
    }
    printf("%s: steps %ld passes %ld alone %ld exact %ld left %ld group steps %ld passes %ld alone %ld exact %ld wrong chains %ld\n", kinds[kind],
           steps[0], wave_passes, wave_alone, turned[0], left, steps[1], group_passes, alone - wave_alone, turned[1], wrong);
    bad += wrong;
  }
  return bad ? 1 : 0;
}
