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
// Integers are in units of 2^(bmin - 112) with bmin = b - 7 for the b of the block's first sum, so
// binades bmin .. bmin + 13 fit 128 bits.  A product of zero leaves S as it is; steps that are done
// count as such products.
#pragma once
#include "chain.hpp"

namespace qb {

constexpr int SC_WIN = 14;      // binades of a block
constexpr int SC_LOW = 7;       // of them below the first sum's
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
// S (two's complement, units of 2^(bmin - 112)) as the state; S is a binary128 value or zero
QB_HD void sstate_from_sum(sstate &s, const uint32_t (&S)[4], int32_t bmin) {
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
  // the leading bit lies in 112..125, at bit 48..61 of hi: to bit 48 + SC_LOW
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
  r.Ep = a.e + b.e;
  r.bad = r.Ep < -SC_EMAX || r.Ep > SC_EMAX;  // CH_ESPECIAL operands among them
  if (a.e == CH_ESPECIAL || b.e == CH_ESPECIAL) {
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
// exponent of the leading bit of s 2^eref, SC_BIG for zero
QB_HD int32_t sc_binade(double s, int32_t eref) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int e = __builtin_amdgcn_frexp_exp(s);
#else
  int e;
  (void)__builtin_frexp(s, &e);
#endif
  return s == 0.0 ? SC_BIG : e - 1 + eref;
}

// one lane's step on the grid of its predicted binade
struct slane {
  uint32_t v[4];  // RN_u(product), signed, units of 2^(bmin - 112)
  uint32_t x0, x1;  // the signed product's floor: 32 bits below the unit, and the lowest word
  int32_t k;      // b - bmin
  bool lost;      // product bits below x0
  bool live;      // a nonzero product whose grid is in the window
  bool fix;       // climbs into a higher binade, or a tie
};
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

#if defined(__HIPCC__)
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t sc_dpp(uint32_t x) {  // 0 where there is no source lane
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
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
// inclusive prefix sum over the wave: rows of 16 lanes by shifts, then the rows' totals
template <typename X>
__device__ __forceinline__ void sc_scan(X &v) {
  sc_scan_step<0x111, 0xf>(v);
  sc_scan_step<0x112, 0xf>(v);
  sc_scan_step<0x114, 0xf>(v);
  sc_scan_step<0x118, 0xf>(v);
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

// S = RN(S + a(i) b(i)) for i = 0..n-1 by one whole wave; every lane returns the result.  init, a, b
// and n are the same in all lanes.
template <typename LA, typename LB>
__device__ __forceinline__ q128 wave_chain(q128 init, const LA a, const LB b, int64_t n) {
  const int lane = (int)(threadIdx.x & 63);
  sstate s;  // the same in all lanes, in scalar registers
  sstate_set(s, init);
  sstate_uniform(s);
  q128 qa = q_zero(0), qb_ = q_zero(0);
  if (lane < n) {
    qa = a(lane);
    qb_ = b(lane);
  }
  int64_t pos = 0;
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
        if (q_isnan(sstate_get(s))) return q_nan();
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
        const int32_t bi = sc_binade(d, b0);
        // the binade before: of the last lane below with a product (whose own check covers it), S's for
        // the first one (a zero S is a multiple of every unit)
        const uint64_t below = __ballot(p.Ep != -SC_BIG) & ((1ull << lane) - 1);
        int32_t bp = __builtin_amdgcn_ds_bpermute(4 * (63 - clz64(below)), bi);
        if (below == 0) bp = s.kind == 0 ? s.b : SC_BIG;
        const slane l = sc_round(p, bi, bp, bmin);
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
        const bool ok = !p.bad && (p.Ep == -SC_BIG || (l.live && sc_inside(S[3], l.k)));
        const uint64_t badm = ~__ballot(ok);
        cut = badm ? __ffsll((unsigned long long)badm) - 1 : 64;
        if (cut > lo) {
          uint32_t T[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) T[i] = sc_lane(S[i], cut - 1);
          sstate_from_sum(s, T, bmin);
        }
      }
      lo = cut;
      if (cut < cnt) {
        sstate_step(s, a(pos + cut), b(pos + cut));  // loaded again: seldom
        sstate_uniform(s);
        if (lane <= cut) sc_clear(p);
        lo = cut + 1;
        if (lo > 32) break;  // few lanes left: the next block begins here
      }
    }
    if (lo >= cnt) {
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
  return sstate_get(s);
}
#endif  // __HIPCC__

}  // namespace qb
