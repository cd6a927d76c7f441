// chain_scan.hpp -- one long FMA chain S_i = RN(S_{i-1} + a_i b_i) by a whole wave, 64 steps at a
// time, the same values bit for bit as 64 serial steps.
//
// A serial chain is a latency: about 0.6 us a step for one wave of 64 chains, whatever the chip has
// idle.  But while the binade of the partial sums is known, a step is an integer addition: with
// u_i = 2^(b_i - 112), the unit in the last place of S_i,
//     S_i = S_{i-1} + RN_{u_i}(a_i b_i)      when S_{i-1} is a multiple of u_i,
// which holds unless the step climbs into a higher binade (b_i > b_{i-1}), and RN does not depend on
// S_{i-1} unless a_i b_i is a tie of the grid u_i.  So a block of 64 steps, one per lane, is
//   1. the exact products, as frames (chain.hpp), and their values in double precision;
//   2. a prefix sum in double precision, which predicts every b_i;
//   3. every product rounded to its grid u_i, and a 128-bit prefix sum of the integers;
//   4. for the climbing steps and the ties, in order, the rounding done again from the low bits of
//      the exact S_{i-1}: a difference of at most a few units, added to all later sums;
//   5. a check that every S_i lies strictly inside its predicted binade.  The sums before the first
//      lane that fails are final; that lane's step is done by itself and the lanes after it are taken
//      again from there.
// Sums of small integers, of +-1, of terms that cancel pass zero and powers of two all the time, and fail: a pass a
// step, and a single step besides.  After SC_POOR short passes in a row a chain goes on with blocks that also take
// the steps that round nothing (LOSSLESS): with S_{i-1} and the product multiples of u_i their sum is a binary128 value
// wherever it lies below 2^(b_i + 1).  Entries +-1, 8192 x 2048 row-major gemv: 0.33 ms, 3.9 ms without; dot of 2^20: 0.24
// and 17 ms.  A copy of the code, as the few instructions more cost other chains 3 to 6%.
// Where those blocks fail too (sums that fall by more binades than a block has, subnormal numbers), steps go one at a
// time: by all lanes (lane_steps), 2 us each, or, in a launch of many chains, a chain a lane in a kernel of its
// own (wave_chain_or_not): subnormal entries, 8192 x 2048, 2.5 ms, 14 ms a wave a chain.
// Integers are in units of 2^(bmin - 112) with bmin = b - 7 for the b of the block's first sum, so
// binades bmin .. bmin + 13 fit 128 bits.  A product of zero leaves S as it is; steps that are done
// count as such products.
#pragma once
#include <utility>

#include "chain.hpp"

namespace qb {

constexpr int SC_WIN = 14;      // binades of a block
constexpr int SC_LOW = 7;       // of them below the first sum's
// Passes in a row that end within 16 steps before a chain goes on with lossless blocks, and of those before it is left to a
// lane (wave_chain_or_not).  The first sums of a chain climb and fall through many binades: of 10000 chains of log-uniform
// terms 78% have two such passes in a row, 11% four, 2.6% five, one eight.  Few chains that turn hold a launch up: with
// five, column-major 8192^2 takes 0.86 ms, not 0.77, as the rows of a cache line part.
constexpr int SC_POOR = 8;
constexpr int32_t SC_BIG = 1 << 20;
constexpr int32_t SC_EMAX = 16200;

// the chain's value between blocks
struct sstate {
  uint32_t w[4];  // kind 0: |S| with the leading bit at bit 112 + SC_LOW; kind 2: the packed value
  int32_t b;      // kind 0: exponent of the leading bit
  uint32_t neg;   // kind 0: 0 or ~0
  int32_t kind;   // 0: finite; 1: +0; 2: Inf, NaN, -0, or an exponent beyond +-SC_EMAX
};
QB_HD void sstate_set(sstate &s, q128 v) {
  s.w[0] = (uint32_t)v.lo;
  s.w[1] = (uint32_t)(v.lo >> 32);
  s.w[2] = (uint32_t)v.hi;
  s.w[3] = (uint32_t)(v.hi >> 32);
  s.b = (int32_t)q_bexp(v) - QBIAS;
  s.neg = (uint32_t)((int32_t)s.w[3] >> 31);
  s.kind = 2;
  if ((s.w[0] | s.w[1] | s.w[2] | s.w[3]) == 0) s.kind = 1;
  if (s.b >= -SC_EMAX && s.b <= SC_EMAX) {
    const uint64_t mh = (v.hi & FRAC_HI_MASK) | HIDDEN;
    const uint64_t lo = v.lo << SC_LOW, hi = (mh << SC_LOW) | (v.lo >> (64 - SC_LOW));
    s.w[0] = (uint32_t)lo;
    s.w[1] = (uint32_t)(lo >> 32);
    s.w[2] = (uint32_t)hi;
    s.w[3] = (uint32_t)(hi >> 32);
    s.kind = 0;
  }
}
QB_HD q128 sstate_get(const sstate &s) {
  const uint64_t lo = ((uint64_t)s.w[1] << 32) | s.w[0], hi = ((uint64_t)s.w[3] << 32) | s.w[2];
  if (s.kind == 1) return q_zero(0);
  if (s.kind == 2) return q_make(lo, hi);
  return q_make((lo >> SC_LOW) | (hi << (64 - SC_LOW)),
                ((uint64_t)(s.neg & 1u) << 63) | ((uint64_t)(s.b + QBIAS) << 48) | ((hi >> SC_LOW) & FRAC_HI_MASK));
}
// S (two's complement, units of 2^(bmin - 112)) as the state; S is a binary128 value or zero, its leading bit in
// 112..125, or, any: anywhere below
QB_HD void sstate_from_sum(sstate &s, const uint32_t (&S)[4], int32_t bmin, bool any = false) {
  const uint32_t x = (uint32_t)((int32_t)S[3] >> 31);
  uint64_t lo = (((uint64_t)S[1] << 32) | S[0]) ^ (((uint64_t)x << 32) | x);
  uint64_t hi = (((uint64_t)S[3] << 32) | S[2]) ^ (((uint64_t)x << 32) | x);
  lo += x & 1u;
  hi += (x & 1u) & (lo == 0);
  s.neg = x;
  if ((lo | hi) == 0) {
    s.kind = 1;
    s.w[0] = s.w[1] = s.w[2] = s.w[3] = 0;
    return;
  }
  if (any && hi == 0) {
    hi = lo;
    lo = 0;
    bmin -= 64;
  }
  // the leading bit to bit 48 + SC_LOW of hi
  const int lz = clz64(hi), L = lz - (15 - SC_LOW);
  s.b = bmin + 15 - lz;
  if (L >= 0) {
    hi = shl_fill(hi, lo, L);
    lo <<= L;
  } else {  // a multiple of its unit in the last place: exact
    lo = shr_fill(hi, lo, -L);
    hi >>= -L;
  }
  s.w[0] = (uint32_t)lo;
  s.w[1] = (uint32_t)(lo >> 32);
  s.w[2] = (uint32_t)hi;
  s.w[3] = (uint32_t)(hi >> 32);
  s.kind = (s.b >= -SC_EMAX && s.b <= SC_EMAX) ? 0 : 2;
  if (s.kind == 2) {
    s.kind = 0;
    sstate t = s;
    const q128 v = sstate_get(t);
    sstate_set(s, v);
  }
}

// one step by itself
QB_HD void sstate_step(sstate &s, q128 a, q128 b) {
  if (s.kind != 2) {
    cacc acc;
    cacc_init(acc);
    if (s.kind == 0) {  // the leading bit at frame bit 32 + 112 + SC_LOW
      uint32_t c = s.neg & 1u;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc.w[i] = ch_addc(s.w[i] ^ s.neg, 0u, c, c);
      acc.E = s.b + 8 - SC_LOW;
    }
    const cop A = cop_unpack(a), B = cop_unpack(b);
    cacc_first(acc, A, B);
    if (cacc_step(acc, A, B)) {
      sstate_from_sum(s, acc.w, acc.E - 8);
      return;
    }
  }
  sstate_set(s, fma_packed(a, b, sstate_get(s)));
}

// one lane's product: |a b| = F 2^(Ep - 157) and lower bits, the leading one at bit 157 or 158
struct sprod {
  uint32_t F[5];
  int32_t Ep;    // -SC_BIG for a zero product
  uint32_t neg;  // 0 or ~0
  int32_t tz;    // trailing zero bits of the 226-bit product
  bool bad;      // an operand is Inf, NaN or subnormal, or the exponent is beyond +-SC_EMAX
};
QB_HD void sc_clear(sprod &p) {  // a product of zero
  p.Ep = -SC_BIG;
  p.bad = false;
  p.tz = SC_BIG;
#pragma unroll
  for (int i = 0; i < 5; ++i) p.F[i] = 0;
}
QB_HD sprod sc_product(q128 qa, q128 qb) {
  sprod r;
  const cop a = cop_unpack(qa), b = cop_unpack(qb);
  uint64_t c[7];
  cop_columns(c, a, b);
  r.F[0] = (((uint32_t)c[2] >> 9) & 0xfffffu) | ((uint32_t)c[3] << 20);
  r.F[1] = (((uint32_t)c[3] >> 12) & 0x1ffffu) | ((uint32_t)c[4] << 17);
  r.F[2] = (((uint32_t)c[4] >> 15) & 0x3fffu) | ((uint32_t)c[5] << 14);
  r.F[3] = (((uint32_t)c[5] >> 18) & 0x7ffu) | ((uint32_t)c[6] << 11);
  r.F[4] = ch_alignbit((uint32_t)(c[6] >> 32), (uint32_t)c[6], 21);
  r.neg = a.neg ^ b.neg;
  r.tz = a.tz + b.tz + 72;
  const uint32_t ea = q_bexp(qa), eb = q_bexp(qb);
  r.Ep = (int32_t)(ea + eb) - 2 * QBIAS;
  r.bad = r.Ep < -SC_EMAX || r.Ep > SC_EMAX;
  if (ea - 1u > 0x7ffdu || eb - 1u > 0x7ffdu) {
    const bool fin = q_bexp(qa) != 0x7fffu && q_bexp(qb) != 0x7fffu;
    const bool zero = fin && (q_iszero(qa) || q_iszero(qb));
    sc_clear(r);
    r.bad = !zero;
  }
  return r;
}
QB_HD double sc_ldexp(double x, int e) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_ldexp(x, e);
#else
  return __builtin_ldexp(x, e);
#endif
}
// the product's value over 2^eref
QB_HD double sc_value(const sprod &p, int32_t eref) {
  const double m = sc_ldexp((double)p.F[4] * 0x1p32 + (double)p.F[3], p.Ep - 61 - eref);
  return p.neg ? -m : m;
}
QB_HD double sc_first(const sstate &s) {  // S over 2^b
  const double m = ((double)s.w[3] * 0x1p32 + (double)s.w[2]) * (1.0 / (double)(1ull << (48 + SC_LOW)));
  return s.kind == 1 ? 0.0 : (s.neg ? -m : m);
}
// exponent of the leading bit of s 2^eref, `zero` for zero
QB_HD int32_t sc_binade(double s, int32_t eref, int32_t zero = SC_BIG) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int e = __builtin_amdgcn_frexp_exp(s);
#else
  int e;
  (void)__builtin_frexp(s, &e);
#endif
  return s == 0.0 ? zero : e - 1 + eref;
}

// one lane's step on the grid of its predicted binade
struct slane {
  uint32_t v[4];  // RN_u(product), signed, units of 2^(bmin - 112)
  uint32_t x0, x1;  // the signed product's floor: 32 bits below the unit, and the lowest word
  int32_t k;      // b - bmin
  bool lost;      // product bits below x0
  bool live;      // a nonzero product on a grid of the window
  bool fix;       // climbs into a higher binade, or a tie
};
// LOSSLESS: a product that is a multiple of the lowest grid is live also where the sum is predicted below it
template <bool LOSSLESS = false>
QB_HD slane sc_round(const sprod &p, int32_t b, int32_t bprev, int32_t bmin) {
  slane r;
  const int32_t k = b - bmin;
  r.live = !p.bad && p.Ep != -SC_BIG && (uint32_t)k < (uint32_t)SC_WIN && p.Ep <= bmin + SC_WIN - 1;
  r.k = r.live ? k : 0;
  int32_t sh = bmin - p.Ep + 13;
  sh = sh < 0 ? 0 : (sh > 159 ? 159 : sh);
  const uint32_t m4 = ch_mask<7>((uint32_t)sh), m2 = ch_mask<6>((uint32_t)sh), m1 = ch_mask<5>((uint32_t)sh);
  uint32_t U[5], V[5], Q[6];
  U[0] = ch_sel(m4, p.F[4], p.F[0]);
#pragma unroll
  for (int i = 1; i < 5; ++i) U[i] = p.F[i] & ~m4;
  V[0] = ch_sel(m2, U[2], U[0]);
  V[1] = ch_sel(m2, U[3], U[1]);
  V[2] = ch_sel(m2, U[4], U[2]);
  V[3] = U[3] & ~m2;
  V[4] = U[4] & ~m2;
#pragma unroll
  for (int i = 0; i < 4; ++i) Q[i] = ch_sel(m1, V[i + 1], V[i]);
  Q[4] = V[4] & ~m1;
  Q[5] = 0;
  uint32_t X[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) X[i] = ch_alignbit(Q[i + 1], Q[i], (uint32_t)sh);
  r.lost = p.tz < 67 + sh;
  // + half a unit of the grid, bits below the grid cleared
  const uint64_t half = 0x80000000ull << r.k;
  uint32_t c = 0;
  const uint32_t y0 = ch_addc(X[0], (uint32_t)half, 0u, c);
  const uint32_t y1 = ch_addc(X[1], (uint32_t)(half >> 32), c, c);
  const uint32_t y2 = ch_addc(X[2], 0u, c, c), y3 = ch_addc(X[3], 0u, c, c), y4 = ch_addc(X[4], 0u, c, c);
  const uint32_t below = (1u << r.k) - 1u;
  const bool tie = (y0 | (y1 & below)) == 0 && !r.lost;  // exactly half a unit
  if (LOSSLESS) r.live = r.live || (k < 0 && !p.bad && p.Ep != -SC_BIG && p.Ep <= bmin + SC_WIN - 1 && X[0] == 0 && !r.lost);
  const uint32_t on = r.live ? ~0u : 0u;
  const uint32_t neg = p.neg & on;
  c = neg & 1u;
  r.v[0] = ch_addc((y1 & ~below & on) ^ neg, 0u, c, c);
  r.v[1] = ch_addc((y2 & on) ^ neg, 0u, c, c);
  r.v[2] = ch_addc((y3 & on) ^ neg, 0u, c, c);
  r.v[3] = ch_addc((y4 & on) ^ neg, 0u, c, c);
  // floor of the signed product: -(X + fraction) is ~X when something is lost, else ~X + 1
  c = (neg & 1u) & (uint32_t)!r.lost;
  r.x0 = ch_addc(X[0] ^ neg, 0u, c, c);
  r.x1 = ch_addc(X[1] ^ neg, 0u, c, c);
  r.fix = r.live && (b > bprev || tie);
  return r;
}
// what the lane's sum S (its lowest word) has to be corrected by: RN of the exact S_{i-1} + product
// on the grid, from the low 64 bits
QB_HD int32_t sc_fix(const slane &l, uint32_t S0) {
  const uint64_t z = (((uint64_t)(S0 - l.v[0]) << 32) + (((uint64_t)l.x1 << 32) | l.x0)) | (uint64_t)l.lost;
  const uint64_t lsb = (z >> (32 + l.k)) & 1u;
  const uint64_t n = z + ((0x80000000ull << l.k) - 1u + lsb);
  return (int32_t)(((uint32_t)(n >> 32) & ~((1u << l.k) - 1u)) - S0);
}
// S lies strictly inside the binade bmin + k (values next to its ends count as outside)
QB_HD bool sc_inside(uint32_t S3, int32_t k) {
  const uint32_t h = S3 ^ (uint32_t)((int32_t)S3 >> 31);
  const uint32_t f = (h + 1u) & ((1u << (16 + k)) - 1u);
  return (h >> (16 + k)) == 1u && f > 1u;
}
// LOSSLESS: S lies inside the binade bmin + k, with its lower words looked at (a chain may stay next to the end of a binade
// for hundreds of steps), or the step is exact: the product and the sum before (its lowest word) are multiples of
// the unit, and |S| is below the end of the binade.
QB_HD bool sc_final(const slane &l, const uint32_t (&S)[4], uint32_t before) {
  const uint32_t h = S[3] ^ (uint32_t)((int32_t)S[3] >> 31), t = h >> (16 + l.k), unit = (1u << l.k) - 1u;
  const bool inside = t == 1u && ((h & ((1u << (16 + l.k)) - 1u)) | S[0] | S[1] | S[2]) != 0;
  const bool exact = t <= 1u && !l.lost && (l.x0 | ((l.x1 | before) & unit)) == 0;
  return l.live && (inside || exact);
}

// How many steps a chain takes one at a time after a block that ended early: one, or ever more, up to 512, where blocks
// go on ending within 16 steps (short: their number in a row)
QB_HD int sc_pace(int &short_blocks, int64_t done) {
  short_blocks = done >= 16 ? 0 : short_blocks < 13 ? short_blocks + 1 : 13;
  return short_blocks <= 4 ? 1 : 1 << (short_blocks - 4);
}

// a chain by a workgroup (group_chain)
constexpr int SG_WAVES = 8;  // at most 16: a row of lanes holds a value of each
constexpr int SG_PER = 4;    // two prefix sums for 256 steps of a wave
constexpr int SG_SPAN = 64 * SG_PER;
constexpr int SG_STEPS = SG_SPAN * SG_WAVES;
// sc_fix as a step E -> ((A + E + add + ((A + E) & odd ? 1 : 0)) & grid) - after on the corrections so far, E, in
// halves of 2^(bmin - 112): A is the exact sum before the step plus the product's floor; what lies below A
// takes the tie's place of the odd bit
struct sg_fix {
  uint32_t A, odd, after;
  int32_t k;
};
QB_HD sg_fix sg_make_fix(const slane &l, uint32_t S0) {
  const uint64_t z = ((uint64_t)(S0 - l.v[0]) << 32) + (((uint64_t)l.x1 << 32) | l.x0);
  const bool low = l.lost || ((uint32_t)z & 0x7fffffffu) != 0;
  sg_fix r;
  r.A = (uint32_t)(z >> 31);
  r.k = l.k + 1;
  r.odd = low ? 0u : 1u << r.k;
  r.after = S0 << 1;
  return r;
}

#if defined(__HIPCC__)
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t sc_dpp(uint32_t x) {  // 0 where there is no source lane
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, ROWS == 0xf);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ void sc_scan_step(uint32_t (&v)[4]) {
  uint32_t t[4], c = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i] = sc_dpp<CTRL, ROWS>(v[i]);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = ch_addc(v[i], t[i], c, c);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ void sc_scan_step(double &v) {
  const uint64_t u = __double_as_longlong(v);
  const uint32_t lo = sc_dpp<CTRL, ROWS>((uint32_t)u), hi = sc_dpp<CTRL, ROWS>((uint32_t)(u >> 32));
  v += __longlong_as_double(((uint64_t)hi << 32) | lo);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ void sc_scan_step(uint32_t &v) {
  v += sc_dpp<CTRL, ROWS>(v);
}
// inclusive prefix sum over the wave: rows of 16 lanes by shifts, then the rows' totals
template <typename X>
__device__ __forceinline__ void sc_scan_row(X &v) {
  sc_scan_step<0x111, 0xf>(v);
  sc_scan_step<0x112, 0xf>(v);
  sc_scan_step<0x114, 0xf>(v);
  sc_scan_step<0x118, 0xf>(v);
}
template <typename X>
__device__ __forceinline__ void sc_scan(X &v) {
  sc_scan_row(v);
  sc_scan_step<0x142, 0xa>(v);  // row_bcast:15
  sc_scan_step<0x143, 0xc>(v);  // row_bcast:31
}
__device__ __forceinline__ uint32_t sc_lane(uint32_t x, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)x, l);
}
__device__ __forceinline__ q128 sc_load(const q128 *p) {
  const uint4 v = *reinterpret_cast<const uint4 *>(p);
  return q_make(((uint64_t)v.y << 32) | v.x, ((uint64_t)v.w << 32) | v.z);
}

__device__ __forceinline__ void sstate_uniform(sstate &s) {
#pragma unroll
  for (int i = 0; i < 4; ++i) s.w[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)s.w[i]);
  s.b = __builtin_amdgcn_readfirstlane(s.b);
  s.neg = (uint32_t)__builtin_amdgcn_readfirstlane((int)s.neg);
  s.kind = __builtin_amdgcn_readfirstlane(s.kind);
}
// a_i = p[i stride], and a constant
struct sc_strided {
  const q128 *p;
  int64_t stride;
  __device__ __forceinline__ q128 operator()(int64_t i) const { return sc_load(p + i * stride); }
};
struct sc_const {
  q128 v;
  __device__ __forceinline__ q128 operator()(int64_t) const { return v; }
};

// S = RN(S + a(i) b(i)) for i = pos..n-1 by one whole wave.  s (in scalar registers), a, b, pos and n are
// the same in all lanes.  Returns the first step not done: n, or, where SC_POOR passes in a row were short, or, LOSSLESS,
// where a pass fails.
template <bool LOSSLESS, typename LA, typename LB>
__device__ __forceinline__ int64_t wave_steps(sstate &s, const LA a, const LB b, int64_t pos, int64_t n) {
  int poor = 0;  // passes in a row
  const int lane = (int)(threadIdx.x & 63);
  q128 qa = q_zero(0), qb_ = q_zero(0);
  if (pos + lane < n) {
    qa = a(pos + lane);
    qb_ = b(pos + lane);
  }
  while (pos < n) {
    const int cnt = (int)((n - pos < 64) ? n - pos : 64);
    // the next block's operands (read again below if this block ends early)
    q128 na = q_zero(0), nb = q_zero(0);
    const int64_t nx = pos + 64 + lane;
    if (nx < n) {
      na = a(nx);
      nb = b(nx);
    }
    sprod p = sc_product(qa, qb_);
    if (lane >= cnt) sc_clear(p);
    int lo = 0;  // steps of the block that are done
    while (lo < cnt) {
      int cut = lo;  // steps before it are final after this pass; step `cut` is done by itself
      if (s.kind == 2 && s.b == QBIAS + 1) {  // Inf or NaN
        if (q_isnan(sstate_get(s))) {
          sstate_set(s, q_nan());
          sstate_uniform(s);
          return n;
        }
        // an infinity stays until an operand is not finite
        const int64_t at = pos + lane;
        const uint64_t odd =
            __ballot(lane >= lo && lane < cnt && (q_bexp(a(at < n ? at : 0)) == 0x7fffu || q_bexp(b(at < n ? at : 0)) == 0x7fffu));
        cut = odd ? __ffsll((unsigned long long)odd) - 1 : 64;
      } else if (s.kind != 2) {
        const uint64_t nz = __ballot(p.Ep != -SC_BIG && !p.bad);
        const int32_t b0 = s.kind == 0 ? s.b : (nz ? (int32_t)sc_lane((uint32_t)p.Ep, __ffsll((unsigned long long)nz) - 1) : 0);
        const int32_t bmin = b0 - SC_LOW;
        double d = sc_value(p, b0);
        sc_scan(d);
        d += sc_first(s);
        const int32_t bi = sc_binade(d, b0, LOSSLESS ? p.Ep : SC_BIG);
        // the binade before: of the last lane below with a product (whose own check covers it), S's for
        // the first one (a zero S is a multiple of every unit)
        const uint64_t below = __ballot(p.Ep != -SC_BIG) & ((1ull << lane) - 1);
        int32_t bp = __builtin_amdgcn_ds_bpermute(4 * (63 - clz64(below)), bi);
        if (below == 0) bp = s.kind == 0 ? s.b : SC_BIG;
        const slane l = sc_round<LOSSLESS>(p, bi, bp, bmin);
        uint32_t S[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) S[i] = l.v[i];
        sc_scan(S);
        {
          uint32_t c = s.neg & 1u;
          const uint32_t z = s.kind == 0 ? ~0u : 0u, ng = s.neg & z;
          c &= z;
#pragma unroll
          for (int i = 0; i < 4; ++i) S[i] = ch_addc(S[i], (s.w[i] & z) ^ ng, c, c);
        }
        // no lane from the first unusable one on counts
        const uint64_t dead = __ballot(p.bad || (p.Ep != -SC_BIG && !l.live));
        for (uint64_t fm = __ballot(l.fix) & (dead ? (dead & -dead) - 1 : ~0ull); fm; fm &= fm - 1) {
          const int f = __ffsll((unsigned long long)fm) - 1;
          const int32_t D = (int32_t)sc_lane((uint32_t)sc_fix(l, S[0]), f);
          const int32_t e = lane >= f ? D : 0;
          const uint32_t x = (uint32_t)(e >> 31);
          uint32_t c = 0;
          S[0] = ch_addc(S[0], (uint32_t)e, c, c);
#pragma unroll
          for (int i = 1; i < 4; ++i) S[i] = ch_addc(S[i], x, c, c);
        }
        bool ok;
        if constexpr (LOSSLESS) {
          const uint32_t first = s.kind == 0 ? (s.w[0] ^ s.neg) - s.neg : 0u;  // of the sum before the block
          const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)S[0], 0x138, 0xf, 0xf, false);  // wave_shr:1
          ok = !p.bad && (p.Ep == -SC_BIG || sc_final(l, S, before));
        } else {
          ok = !p.bad && (p.Ep == -SC_BIG || (l.live && sc_inside(S[3], l.k)));
        }
        const uint64_t badm = ~__ballot(ok);
        cut = badm ? __ffsll((unsigned long long)badm) - 1 : 64;
        if (cut > lo) {
          uint32_t T[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) T[i] = sc_lane(S[i], cut - 1);
          sstate_from_sum(s, T, bmin, LOSSLESS);
        }
      }
      const int from = lo;
      lo = cut;
      if constexpr (LOSSLESS) {
        if (cut < cnt) return pos + cut;
      } else if (cut < cnt) {
        sstate_step(s, a(pos + cut), b(pos + cut));  // loaded again: seldom
        sstate_uniform(s);
        if (lane <= cut) sc_clear(p);
        lo = cut + 1;
        poor = cut - from < 16 ? poor + 1 : 0;
        if (poor == SC_POOR) return pos + lo;
        if (lo > 32) break;  // few lanes left: the next block begins here
      }
    }
    if (lo >= cnt) {
      poor = 0;
      pos += 64;
      qa = na;
      qb_ = nb;
    } else {
      pos += lo;
      const int64_t i = pos + lane;
      if (i < n) {
        qa = a(i);
        qb_ = b(i);
      }
    }
  }
  return n;
}
// S = RN(S + a(i) b(i)) for i = pos..to-1, a step at a time by all lanes: where blocks fail.  Lanes load and unpack
// LANE_SPAN operands at once, the next ones on their way meanwhile.  Vector instructions, as the operands come from
// LDS: as scalar ones a step takes several times as long.
constexpr int LANE_SPAN = 16;
struct alignas(16) lane_lds {
  cop a[LANE_SPAN], b[LANE_SPAN];
  q128 pa[LANE_SPAN], pb[LANE_SPAN];
};
template <typename LA, typename LB>
__device__ __forceinline__ q128 lane_steps(q128 v, const LA a, const LB b, int64_t pos, int64_t to, lane_lds &lds) {
  const int lane = (int)(threadIdx.x & 63);
  const bool mine = lane < LANE_SPAN;
  cacc acc;
  cacc_set(acc, v);
  q128 x = q_zero(0), y = q_zero(0);
  if (mine && pos + lane < to) {
    x = a(pos + lane);
    y = b(pos + lane);
  }
  for (; pos < to; pos += LANE_SPAN) {
    __builtin_amdgcn_wave_barrier();  // the reads of the operands before are done
    if (mine) {
      lds.a[lane] = cop_unpack(x);
      lds.b[lane] = cop_unpack(y);
      lds.pa[lane] = x;
      lds.pb[lane] = y;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int cnt = (int)(to - pos < LANE_SPAN ? to - pos : LANE_SPAN);
    if (mine && pos + LANE_SPAN + lane < to) {
      x = a(pos + LANE_SPAN + lane);
      y = b(pos + LANE_SPAN + lane);
    }
    cop A = lds.a[0], B = lds.b[0];
    for (int q = 0; q < cnt; ++q) {
      const int nq = (q + 1) % LANE_SPAN;
      const cop nA = lds.a[nq], nB = lds.b[nq];
      if (!cacc_step(acc, A, B)) chain_rest(acc, lds.pa[q], lds.pb[q]);
      A = nA;
      B = nB;
    }
  }
  return cacc_get(acc);
}
// a chain's steps pos..n-1 with lossless blocks
template <typename LA, typename LB>
__device__ __forceinline__ void wave_lossless_steps(sstate &s, int &short_blocks, const LA a, const LB b, int64_t pos, int64_t n,
                                                 lane_lds &lds) {
  while (pos < n) {
    const int64_t at = wave_steps<true>(s, a, b, pos, n);
    if (at >= n) return;
    const int by = sc_pace(short_blocks, at - pos);
    pos = n - at < by ? n : at + by;
    sstate_set(s, lane_steps(sstate_get(s), a, b, at, pos, lds));
    sstate_uniform(s);
  }
}
// a whole chain of n steps from init; every lane returns the result
template <typename LA, typename LB>
__device__ __forceinline__ q128 wave_chain(q128 init, const LA a, const LB b, int64_t n, lane_lds &lds) {
  sstate s;
  sstate_set(s, init);
  sstate_uniform(s);
  const int64_t pos = wave_steps<false>(s, a, b, 0, n);
  if (pos < n) {
    int short_blocks = 0;
    wave_lossless_steps(s, short_blocks, a, b, pos, n, lds);
  }
  return sstate_get(s);
}

// The same in a launch of many chains, with fewer registers: steps alone are scalar ones.  False where the result is not there,
// as blocks go on failing and the chain may be left (leave): a step alone takes a wave as many instructions as 64
// chains of a wave, and 16 waves a SIMD of them took 7 to 15 times as long as those.
template <typename LA, typename LB>
__device__ __forceinline__ bool wave_chain_or_not(q128 &v, const LA a, const LB b, int64_t n, bool leave) {
  sstate s;
  sstate_set(s, v);
  sstate_uniform(s);
  int64_t pos = wave_steps<false>(s, a, b, 0, n);
  int short_blocks = 0;
  while (pos < n) {
    const int64_t at = wave_steps<true>(s, a, b, pos, n);
    if (at >= n) break;
    const int by = sc_pace(short_blocks, at - pos);
    if (leave && short_blocks == SC_POOR) return false;
    pos = n - at < by ? n : at + by;
    for (int64_t i = at; i < pos; ++i) {
      sstate_step(s, a(i), b(i));
      sstate_uniform(s);
    }
  }
  v = sstate_get(s);
  return true;
}

// The same by a workgroup of SG_WAVES waves, SG_PER consecutive steps a lane and SG_STEPS at a time, for a
// launch of fewer chains than the chip has CUs.  Each wave does its steps as above from the predicted sum
// before them; the exact sums before a wave are the state and the totals of the waves before it, and the
// rounding done again at climbs and ties goes through one list in step order, by the first wave.  A wave does
// not know the binade that the one before ends in, so its first product counts as a climb.  The window of
// binades lies below the largest of the sums at the waves' ends (the state's rule where that would cut the
// state itself).  Where a sum leaves the window, or the state is not of kind 0, the next 64 steps are one
// wave's work, which every wave does for itself.  Every barrier is met by all waves: what decides is the same
// in all of them.
struct sg_lds {
  double dsum[16];         // the waves' sums of products, in double precision
  uint4 total[16];         // of rounded products
  uint32_t fixes[16];      // roundings to be done again
  union {
    uint4 list[SG_STEPS];        // of each: sum + product below the grid, doubled (sg_fix)
    lane_lds lanes[SG_WAVES];    // the waves' single steps, between passes
  };
  uint32_t corr[SG_STEPS]; // the correction of the sums from there on
  uint4 end[16];           // the sum after the wave's last good step
  int cut[16];             // good steps
};
// The fixes of lanes F0 .. F0 + 7, z = A + E of the first one in, (E + after) of the last one out; the next
// one's z is (E + after) + C.  Inline assembly: the condition of the AND is the addition's carry, which the
// compiler makes with two compares and a select, and a lane is written by its number.
template <int F0, int... F>
__device__ __forceinline__ void sg_fix_eight(uint32_t &z, uint32_t &kept, uint32_t C, uint32_t odd, uint32_t add,
                                             uint32_t grid, std::integer_sequence<int, F...>) {
  (([&] {
     uint32_t r = z;
     if (F0 + F > 0) r += sc_lane(C, F0 + F);
     asm("s_and_b32 %0, %1, %2\n\ts_addc_u32 %0, %1, %3"
         : "=&s"(z)
         : "s"(r), "s"(sc_lane(odd, F0 + F)), "s"(sc_lane(add, F0 + F))
         : "scc");
     z &= sc_lane(grid, F0 + F);
     asm("v_writelane_b32 %0, %1, %2" : "+v"(kept) : "s"(z), "n"(F0 + F));
   }()),
   ...);
}
template <int... G>
__device__ __forceinline__ void sg_fix_lanes(uint32_t &z, uint32_t &kept, uint32_t C, uint32_t odd, uint32_t add,
                                             uint32_t grid, int cnt, std::integer_sequence<int, G...>) {
  (void)((8 * G < cnt &&
          (sg_fix_eight<8 * G>(z, kept, C, odd, add, grid, std::make_integer_sequence<int, 8>{}), true)) &&
         ...);
}
// Steps pos..n-1; returns the first one not done: n, or, not LOSSLESS, where the chain
// gets on poorly: three passes in a row end within 128 steps, or wave_steps gives up.
template <bool LOSSLESS, typename LA, typename LB>
__device__ __forceinline__ int64_t group_steps(sstate &s, const LA a, const LB b, int64_t pos, int64_t n, sg_lds &lds) {
  const int lane = (int)(threadIdx.x & 63), wl = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  q128 qa[SG_PER], qb_[SG_PER];
  auto fetch = [&](int64_t at) {
    const int64_t i = at + SG_PER * (int)threadIdx.x;
#pragma unroll
    for (int r = 0; r < SG_PER; ++r) {
      qa[r] = qb_[r] = q_zero(0);
      if (i + r < n) {
        qa[r] = a(i + r);
        qb_[r] = b(i + r);
      }
    }
  };
  fetch(pos);
  int poor = 0;  // passes in a row
  int64_t alone = 64;
  int short_blocks = 0;
  for (bool single = true; pos < n;) {  // the first sums climb and fall through many binades
    if (single || s.kind != 0) {
      const int64_t by = LOSSLESS ? alone : 64, to = n - pos < by ? n : pos + by;
      if constexpr (LOSSLESS) {
        wave_lossless_steps(s, short_blocks, a, b, pos, to, lds.lanes[wv]);
        pos = to;
      } else {
        pos = wave_steps<false>(s, a, b, pos, to);
        if (pos < to) return pos;
      }
      if (s.kind == 2 && q_isnan(sstate_get(s))) return n;
      fetch(pos);
      single = false;
      continue;
    }
    sprod p[SG_PER];
    double d[SG_PER];  // sums of the lane's products
    bool any = false;  // the lane has a product
#pragma unroll
    for (int r = 0; r < SG_PER; ++r) {
      p[r] = sc_product(qa[r], qb_[r]);
      if (pos + SG_PER * (int)threadIdx.x + r >= n) sc_clear(p[r]);
      any |= p[r].Ep != -SC_BIG;
      const double v = sc_value(p[r], s.b);
      d[r] = r ? d[r ? r - 1 : 0] + v : v;
    }
    fetch(pos + SG_STEPS);  // the next steps' operands (read again below if these end early)
    double dt = d[SG_PER - 1];
    sc_scan(dt);
    if (lane == 63) lds.dsum[wv] = dt;
    __syncthreads();
    // the sum before the wave, and the largest binade at a wave's end
    double before = lds.dsum[wl];
    sc_scan_row(before);
    before += sc_first(s);
    int32_t top = sc_binade(before, s.b, s.b);
#pragma unroll
    for (int i = 1; i < 16; i <<= 1) top = max(top, __shfl_xor(top, i));
    top = max(__builtin_amdgcn_readfirstlane(top), s.b);
    int32_t bmin = top + 2 - SC_WIN;
    if (bmin > s.b) bmin = s.b - SC_LOW;
    const uint64_t bu = __double_as_longlong(before);
    const int wp = wv ? wv - 1 : 0;  // the wave before
    const double d0 =
        wv ? __longlong_as_double(((uint64_t)sc_lane((uint32_t)(bu >> 32), wp) << 32) | sc_lane((uint32_t)bu, wp)) : sc_first(s);
    // the sums before the lane: exact differences do not matter, only that a lane's own are used throughout
    const double dl = (dt - d[SG_PER - 1]) + d0;
    int32_t bi[SG_PER], last = 0;
#pragma unroll
    for (int r = 0; r < SG_PER; ++r) {
      bi[r] = sc_binade(dl + d[r], s.b, LOSSLESS ? p[r].Ep : SC_BIG);
      last = p[r].Ep != -SC_BIG ? bi[r] : last;
    }
    const uint64_t lanes_below = (1ull << lane) - 1;
    const uint64_t below = __ballot(any) & lanes_below;
    int32_t bp = __builtin_amdgcn_ds_bpermute(4 * (63 - clz64(below)), last);
    if (below == 0) bp = -SC_BIG;  // unknown: a climb
    slane l[SG_PER];
    uint32_t V[SG_PER][4];  // sums of the lane's rounded products
    int at = 0, mine = 0, all = 0;  // fixes before the lane, of the lane, of the wave
#pragma unroll
    for (int r = 0; r < SG_PER; ++r) {
      l[r] = sc_round<LOSSLESS>(p[r], bi[r], bp, bmin);
      bp = p[r].Ep != -SC_BIG ? bi[r] : bp;
      uint32_t c = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) V[r][i] = r ? ch_addc(V[r ? r - 1 : 0][i], l[r].v[i], c, c) : l[r].v[i];
      const uint64_t fm = __ballot(l[r].fix);
      at += __popcll(fm & lanes_below);
      all += __popcll(fm);
    }
    uint32_t S[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) S[i] = V[SG_PER - 1][i];
    sc_scan(S);
    if (lane == 63) {
      lds.total[wv] = make_uint4(S[0], S[1], S[2], S[3]);
      lds.fixes[wv] = (uint32_t)all;
    }
    __syncthreads();
    uint32_t fx = lds.fixes[wl];
    sc_scan_row(fx);
    at += wv ? (int)sc_lane(fx, wp) : 0;
    const int fixes = (int)sc_lane(fx, 15);
    {
      const uint4 t = lds.total[wl];
      uint32_t B[4] = {t.x, t.y, t.z, t.w};
      sc_scan_row(B);
      // the state in units of 2^(bmin - 112): s.b - bmin is 0..SC_WIN - 2, the leading bit of w at 112 + SC_LOW
      const int up = s.b - bmin - SC_LOW;
      uint64_t lo = ((uint64_t)s.w[1] << 32) | s.w[0], hi = ((uint64_t)s.w[3] << 32) | s.w[2];
      if (up >= 0) {
        hi = shl_fill(hi, lo, up);
        lo <<= up;
      } else {  // the bits below the leading 113 are zero
        lo = shr_fill(hi, lo, -up);
        hi >>= -up;
      }
      const uint32_t w[4] = {(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
      uint32_t c = s.neg & 1u, c2 = 0, c3 = 1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // the sum before the lane
        const uint32_t base = ch_addc(w[i] ^ s.neg, wv ? sc_lane(B[i], wp) : 0u, c, c);
        S[i] = ch_addc(S[i], base, c2, c2);
        S[i] = ch_addc(S[i], ~V[SG_PER - 1][i], c3, c3);
      }
    }
#pragma unroll
    for (int r = 0; r < SG_PER; ++r) {
      if (l[r].fix) {
        const sg_fix f = sg_make_fix(l[r], S[0] + V[r][0]);
        lds.list[at + mine] = make_uint4(f.A, f.odd, f.after, (uint32_t)f.k);
        ++mine;
      }
    }
    __syncthreads();
    if (wv == 0) {  // one by one, in scalar registers
      uint32_t E = 0;
      for (int f0 = 0; f0 < fixes; f0 += 64) {
        const int cnt = fixes - f0 < 64 ? fixes - f0 : 64;
        const uint4 u = lds.list[f0 + (lane < cnt ? lane : 0)];
        const uint32_t add = (1u << (u.w - 1)) - (u.y ? 1u : 0u), grid = 0u - (1u << u.w);
        const uint32_t C = u.x - (uint32_t)__shfl_up((int)u.z, 1);
        uint32_t z = sc_lane(u.x, 0) + E, kept = 0;  // kept: (E + after) of the lane's fix
        sg_fix_lanes(z, kept, C, u.y, add, grid, cnt, std::make_integer_sequence<int, 8>{});
        E = z - sc_lane(u.z, 63);
        if (lane < cnt) lds.corr[f0 + lane] = (uint32_t)((int32_t)(kept - u.z) >> 1);
      }
    }
    __syncthreads();
    // the sums of the lane's steps, checked: `good` of them are final, the last of those in S
    uint32_t corr = at ? lds.corr[at - 1] : 0u, prev = S[0] + corr;
    uint32_t G[4];
    int good = 0;
    bool still = true;
#pragma unroll
    for (int i = 0; i < 4; ++i) G[i] = 0;
#pragma unroll
    for (int r = 0; r < SG_PER; ++r) {
      if (l[r].fix) corr = lds.corr[at++];
      const uint32_t x = (uint32_t)((int32_t)corr >> 31);
      uint32_t c = 0, c2 = 0, X[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        X[i] = ch_addc(S[i], V[r][i], c, c);
        X[i] = ch_addc(X[i], i ? x : corr, c2, c2);
      }
      still = still && !p[r].bad && (p[r].Ep == -SC_BIG || (LOSSLESS ? sc_final(l[r], X, prev) : l[r].live && sc_inside(X[3], l[r].k)));
      prev = X[0];
      good += still ? 1 : 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) G[i] = still ? X[i] : G[i];
    }
    const uint64_t badm = ~__ballot(good == SG_PER);
    const int bl = badm ? __ffsll((unsigned long long)badm) - 1 : 64;  // the first lane that fails
    const int bg = bl < 64 ? (int)sc_lane((uint32_t)good, bl & 63) : 0;
    const int el = bg ? bl : bl - 1;  // the lane of the last good step
    if (lane == (el < 0 ? 0 : el)) {
      lds.end[wv] = make_uint4(G[0], G[1], G[2], G[3]);
      lds.cut[wv] = SG_PER * bl + bg;
    }
    __syncthreads();
    const uint64_t early = __ballot(lane < SG_WAVES && lds.cut[wl] < SG_SPAN);
    const int w = early ? __ffsll((unsigned long long)early) - 1 : SG_WAVES - 1;
    const int cut = __builtin_amdgcn_readfirstlane(lds.cut[w]);
    const int done = SG_SPAN * w + cut;
    if (done) {
      const uint4 t = lds.end[cut ? w : w - 1];
      const uint32_t T[4] = {t.x, t.y, t.z, t.w};
      sstate_from_sum(s, T, bmin, LOSSLESS);
      sstate_uniform(s);
    }
    pos += done;
    single = done < SG_STEPS;
    poor = done < 128 ? poor + 1 : 0;
    if constexpr (LOSSLESS) alone = poor < 2 ? 64 : alone < 8192 ? 2 * alone : 8192;
    else if (poor == 3) return pos;
  }
  return n;
}
// a whole chain of n steps from init; every lane returns the result
template <typename LA, typename LB>
__device__ __forceinline__ q128 group_chain(q128 init, const LA a, const LB b, int64_t n, sg_lds &lds) {
  if (threadIdx.x < 16) {  // waves that the workgroup does not have
    lds.dsum[threadIdx.x] = 0.0;
    lds.total[threadIdx.x] = make_uint4(0, 0, 0, 0);
    lds.fixes[threadIdx.x] = 0;
    lds.cut[threadIdx.x] = SG_SPAN;
  }
  __syncthreads();
  sstate s;
  sstate_set(s, init);
  sstate_uniform(s);
  const int64_t pos = group_steps<false>(s, a, b, 0, n, lds);
  if (pos < n) group_steps<true>(s, a, b, pos, n, lds);
  return sstate_get(s);
}
#endif  // __HIPCC__

}  // namespace qb
