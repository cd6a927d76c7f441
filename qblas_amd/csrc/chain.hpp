// chain.hpp -- accumulating correctly rounded FMA chains, acc = RN(a*b + acc), the step of every
// REFERENCE-order kernel (the serial loops of include/quadblas/algorithms/level1.hpp:20-25,
// level2.hpp:35-44,69-80, level3.hpp:200-210).  Same values as fma_packed on packed operands, bit
// for bit, with the accumulator and the operands held in forms the step needs no shifting for.
//
//   cop   an operand, unpacked once: four 29-bit limbs of the 113-bit significand (so the columns
//         of a product, sums of at most four 58-bit products, fit 64 bits), exponent, sign as a
//         mask and the number of trailing zero bits.  Zero, subnormal, Inf and NaN operands, and
//         exponents beyond +-CH_OMAX, carry the exponent CH_ESPECIAL, which no step takes.
//   cacc  the accumulator: a 160-bit two's complement frame W (five 32-bit words, the lowest always
//         zero between steps) with value W 2^(E-152).  The leading bit lies anywhere in bits
//         146..158, so a step that moves it by a few bits needs no renormalisation.
//
// One step: the product's columns (16 v_mad_u64_u32, each column's carry the next one's addend), its
// bits 72.. as a frame with leading bit 152/153 at exponent ea + eb; the frame with the lower
// exponent is shifted right onto the other one's grid (the product by whole words with bit masks, then
// a funnel; the accumulator by the funnel), added in two's complement, and rounded in place at the
// 113th bit below the leading one.  Bits of the product below the grid act through a sticky bit only,
// which its trailing zeros (the sum of the operands') decide without looking at them: floor(x) plus a
// sticky bit rounds x correctly, as the grid lies at least 34 bits below the rounding position.
// About 85 VALU instructions, 105 with a product 2^32 below the accumulator in the wave; 401 with sign
// and magnitude in 64-bit words and a case per exponent order.  gemm 2048^3: 21.9 ms on uniform entries
// (27.7 ms with both operands' shifts in every step).
// Left to the packed operation (chain_slow): special operands, exponents near the ends of the range, a
// zero accumulator without cacc_first, one more than 31 bits below the product's grid, and sums that
// cancel by 26 bits or more.
#pragma once
#include "q128.hpp"

namespace qb {

constexpr int32_t CH_ESPECIAL = 1 << 22;  // exponent of an operand the step does not take
constexpr int32_t CH_APACKED = 1 << 24;   // exponent of an accumulator that is held packed
constexpr int32_t CH_EZERO = -(1 << 24);  // exponent of a zero accumulator
constexpr int32_t CH_OMAX = 8100;         // |exponent| of an operand: a product's lies within 16200
constexpr int32_t CH_EMAX = 16300;        // |exponent| of an accumulator's frame: every sum is a normal number
constexpr uint32_t CH_DRANGE = 1u << 17;  // exponent differences of a step: -31 .. 2^17 - 31

struct cop {
  uint32_t l[4];  // significand = sum l[i] 2^(29 i)
  int32_t e;      // value = (-1)^neg significand 2^(e - 112)
  uint32_t neg;   // 0 or ~0
  int32_t tz;     // trailing zero bits of the significand, less 36 (a product's frame begins at bit 72)
  uint32_t zero;  // 1: zero; 2: Inf or NaN
};
struct cacc {
  uint32_t w[4];  // words 1..4 of the frame (word 0 is zero); the packed value if E == CH_APACKED
  int32_t E;
};

QB_HD uint32_t ch_alignbit(uint32_t hi, uint32_t lo, uint32_t s) {  // (hi:lo) >> (s & 31), low word
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_alignbit(hi, lo, s);
#else
  return (uint32_t)((((uint64_t)hi << 32) | lo) >> (s & 31));
#endif
}
// leading bits equal to the sign bit (0xffffffff when all are)
QB_HD uint32_t ch_signbits(uint32_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t r;
  asm("v_ffbh_i32 %0, %1" : "=v"(r) : "v"(x));
  return r;
#else
  const uint32_t v = x ^ (uint32_t)((int32_t)x >> 31);
  return v ? (uint32_t)__builtin_clz(v) : 0xffffffffu;
#endif
}
// bit B of x as a mask.  Inline assembly on the device: seen as a sign, the compiler turns selects by
// the mask into a compare and two or three instructions each instead of one v_bfi_b32
template <int B>
QB_HD uint32_t ch_mask(uint32_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t r;
  asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(r) : "v"(x), "n"(B));
  return r;
#else
  return 0u - ((x >> B) & 1u);
#endif
}
QB_HD bool ch_any(bool x) {  // of the wave's active lanes: a branch the whole wave takes or skips
#if defined(__HIP_DEVICE_COMPILE__)
  return __ballot(x) != 0;
#else
  return x;
#endif
}
QB_HD int32_t ch_clamp(int32_t x, int32_t lo, int32_t hi) { return x < lo ? lo : (x > hi ? hi : x); }
QB_HD uint32_t ch_sel(uint32_t mask, uint32_t a, uint32_t b) { return (mask & a) | (~mask & b); }
QB_HD uint32_t ch_addc(uint32_t a, uint32_t b, uint32_t ci, uint32_t &co) {
#if defined(__clang__)
  uint32_t c;
  const uint32_t r = __builtin_addc(a, b, ci, &c);
  co = c;
  return r;
#else
  const uint64_t r = (uint64_t)a + b + ci;
  co = (uint32_t)(r >> 32);
  return (uint32_t)r;
#endif
}
QB_HD int ch_ctz64(uint64_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __ffsll((unsigned long long)x) - 1;
#else
  return __builtin_ctzll(x);
#endif
}

QB_HD cop cop_unpack(q128 a) {
  cop r;
  const uint32_t be = q_bexp(a);
  const uint64_t mh = (a.hi & FRAC_HI_MASK) | HIDDEN;
  r.l[0] = (uint32_t)a.lo & 0x1fffffffu;
  r.l[1] = (uint32_t)(a.lo >> 29) & 0x1fffffffu;
  r.l[2] = ch_alignbit((uint32_t)mh, (uint32_t)(a.lo >> 32), 26) & 0x1fffffffu;
  r.l[3] = (uint32_t)(mh >> 23);
  r.e = (int32_t)be - QBIAS;
  if ((uint32_t)(r.e + CH_OMAX) > (uint32_t)(2 * CH_OMAX)) r.e = CH_ESPECIAL;
  r.neg = (uint32_t)((int32_t)(uint32_t)(a.hi >> 32) >> 31);
  r.tz = (a.lo ? ch_ctz64(a.lo) : 64 + ch_ctz64(mh)) - 36;
  r.zero = be == 0x7fffu ? 2u : (be == 0 && (a.lo | (a.hi << 1)) == 0) ? 1u : 0u;
  return r;
}

QB_HD void cacc_init(cacc &c) {
  c.w[0] = c.w[1] = c.w[2] = c.w[3] = 0;
  c.E = CH_EZERO;
}
QB_HD void cacc_set(cacc &c, q128 v) {
  const int32_t e = (int32_t)q_bexp(v) - QBIAS;
  if ((e < 50 - CH_EMAX && !q_iszero(v)) || e > CH_EMAX - 50) {
    c.w[0] = (uint32_t)v.lo;
    c.w[1] = (uint32_t)(v.lo >> 32);
    c.w[2] = (uint32_t)v.hi;
    c.w[3] = (uint32_t)(v.hi >> 32);
    c.E = CH_APACKED;
    return;
  }
  const uq u = unpack_finite(v);
  if ((u.mh | u.ml) == 0) {
    cacc_init(c);
    c.w[0] = u.s;  // the sign of a zero: below every grid it is shifted to
    return;
  }
  // leading bit (112 of m) to bit 153: words 1..4 hold m << 9
  const uint64_t lo = u.ml << 9, hi = (u.mh << 9) | (u.ml >> 55);
  const uint64_t x = u.s ? ~0ull : 0ull;
  const uint64_t l2 = (lo ^ x) + (x & 1), h2 = (hi ^ x) + ((x & 1) & (lo == 0));
  c.w[0] = (uint32_t)l2;
  c.w[1] = (uint32_t)(l2 >> 32);
  c.w[2] = (uint32_t)h2;
  c.w[3] = (uint32_t)(h2 >> 32);
  c.E = u.e - 1;
}
QB_HD q128 cacc_get(const cacc &c) {
  uint64_t lo = ((uint64_t)c.w[1] << 32) | c.w[0], hi = ((uint64_t)c.w[3] << 32) | c.w[2];
  if (c.E == CH_APACKED) return q_make(lo, hi);
  if (c.E == CH_EZERO) return q_zero(c.w[0]);
  const uint64_t x = (uint64_t)((int64_t)hi >> 63);
  lo = (lo ^ x) + (x & 1);
  hi = (hi ^ x) + ((x & 1) & (lo == 0));
  const int lz = clz64(hi) - 1;  // the leading bit lies in 114..126 of (hi:lo): one to bit 126
  uq u;
  const uint64_t h = shl_fill(hi, lo, lz), l = lo << lz;
  u.mh = h >> 14;
  u.ml = shr_fill(h, l, 14);
  u.e = c.E + 6 - lz;  // bit 126 of (hi:lo) is bit 158 of the frame
  u.s = (uint32_t)(x & 1);
  return pack(u);
}

// columns of the product of two significands: column k at bit 29 k, each one's carry over 29 bits
// added into the next (the digits are the low 29 bits of columns 0..5 and all of column 6)
QB_HD void cop_columns(uint64_t (&c)[7], const cop &a, const cop &b) {
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const int lo = k < 4 ? 0 : k - 3, hi = k < 4 ? k : 3;
    uint64_t t = k ? c[k - 1] >> 29 : 0;
#pragma unroll
    for (int i = lo; i <= hi; ++i) {
      t += (uint64_t)a.l[i] * b.l[k - i];
#if defined(__HIP_DEVICE_COMPILE__)
      asm("" : "+v"(t));  // keep the carry the first addend: reassociated, it costs an addition of its own
#endif
    }
    c[k] = t;
  }
}
// P >> (sh & ~31), zeros from above, for sh < 160: taken by the wave only when a lane needs it
QB_HD void ch_shift_words(uint32_t (&P)[5], uint32_t sh) {
  if (!ch_any(sh >= 32)) return;
  const uint32_t m4 = ch_mask<7>(sh), m2 = ch_mask<6>(sh), m1 = ch_mask<5>(sh);
  uint32_t Q[5];
  Q[0] = ch_sel(m4, P[4], P[0]);
#pragma unroll
  for (int i = 1; i < 5; ++i) Q[i] = P[i] & ~m4;
  P[0] = ch_sel(m2, Q[2], Q[0]);
  P[1] = ch_sel(m2, Q[3], Q[1]);
  P[2] = ch_sel(m2, Q[4], Q[2]);
  P[3] = Q[3] & ~m2;
  P[4] = Q[4] & ~m2;
#pragma unroll
  for (int i = 0; i < 4; ++i) P[i] = ch_sel(m1, P[i + 1], P[i]);
  P[4] &= ~m1;
}
// bits 72.. of a product as a frame, its leading bit at 152 or 153
QB_HD void ch_frame(uint32_t (&P)[5], const uint64_t (&k)[7]) {
  P[0] = (((uint32_t)k[2] >> 14) & 0x7fffu) | ((uint32_t)k[3] << 15);
  P[1] = (((uint32_t)k[3] >> 17) & 0xfffu) | ((uint32_t)k[4] << 12);
  P[2] = (((uint32_t)k[4] >> 20) & 0x1ffu) | ((uint32_t)k[5] << 9);
  P[3] = (((uint32_t)k[5] >> 23) & 0x3fu) | ((uint32_t)k[6] << 6);
  P[4] = ch_alignbit((uint32_t)(k[6] >> 32), (uint32_t)k[6], 26);
}
// acc = RN(a*b + acc).  Returns false, leaving acc as it was, when the packed operation has to do it.
QB_HD bool cacc_step(cacc &acc, const cop &a, const cop &b) {
  uint64_t k[7];
  cop_columns(k, a, b);
  uint32_t P[5];
  ch_frame(P, k);
  const int32_t Ep = a.e + b.e;
  const int32_t d = acc.E - Ep;
  // d > 0: the product moves right onto the accumulator's grid, by a funnel, after whole words where a
  // lane has a product 2^32 and more below (none has with entries of one scale)
  const int32_t sh = ch_clamp(d, 0, 159);
  ch_shift_words(P, (uint32_t)sh);
  // its sign is applied as a complement; the missing +1 goes in as the sum's carry when no bit of the
  // product lies below the grid
  const uint32_t neg = a.neg ^ b.neg;
#pragma unroll
  for (int i = 0; i < 4; ++i) P[i] = ch_alignbit(P[i + 1], P[i], (uint32_t)sh) ^ neg;
  P[4] = (P[4] >> (sh & 31)) ^ neg;
  const bool st = a.tz + b.tz < sh;
  // d < 0: the accumulator moves onto the product's grid, by at most 31 bits (word 0 takes them)
  uint32_t A[5] = {0, acc.w[0], acc.w[1], acc.w[2], acc.w[3]};
  if (ch_any(d < 0)) {
    const uint32_t sa = (uint32_t)(d < 0 ? -d : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) A[i] = ch_alignbit(A[i + 1], A[i], sa);
    A[4] = (uint32_t)((int32_t)A[4] >> (sa & 31));
  }
  uint32_t F[5], c = (uint32_t)((neg != 0) & !st);
#pragma unroll
  for (int i = 0; i < 5; ++i) F[i] = ch_addc(P[i], A[i], c, c);
  int32_t E = Ep > acc.E ? Ep : acc.E;
  uint32_t fb = ch_signbits(F[4]);
  uint32_t w0 = F[0] | (uint32_t)st;
  if (((uint32_t)(d + 31) > CH_DRANGE) | (fb - 2u > 11u)) {
    // special or far apart; a sum in words 0..3 only; else the leading bit left 146..157: to 153
    if (((uint32_t)(d + 31) > CH_DRANGE) | (fb > 31u)) return false;
    if (fb < 2u) {
      const uint32_t r = 6 - fb;
      const uint32_t lost = w0 << (32 - r);
      w0 = ch_alignbit(F[1], w0, r) | (uint32_t)(lost != 0);
#pragma unroll
      for (int i = 1; i < 4; ++i) F[i] = ch_alignbit(F[i + 1], F[i], r);
      F[4] = (uint32_t)((int32_t)F[4] >> r);
    } else {
      const uint32_t r = 32 - (fb - 6);
#pragma unroll
      for (int i = 4; i > 1; --i) F[i] = ch_alignbit(F[i], F[i - 1], r);
      F[1] = ch_alignbit(F[1], w0, r);
      w0 = (w0 << (32 - r)) | (w0 & 1u);  // the sticky bit stays at the bottom
    }
    E += 6 - (int32_t)fb;
    if ((uint32_t)(E + CH_EMAX) > (uint32_t)(2 * CH_EMAX)) return false;
    fb = 6;
  }
  // round to nearest even at bit 47 - fb, bit 15 - fb of word 1: half less one unit is added, and one
  // unit more if anything lies below word 1 or the result is odd
  c = (uint32_t)((w0 | ((F[1] >> (15u - fb)) & 1u)) != 0);
  acc.w[0] = ch_addc(F[1], 0x3fffu >> fb, c, c) & ~(0x7fffu >> fb);
  acc.w[1] = ch_addc(F[2], 0u, c, c);
  acc.w[2] = ch_addc(F[3], 0u, c, c);
  acc.w[3] = ch_addc(F[4], 0u, c, c);
  acc.E = E;
  return true;
}
// before a chain's first step: a zero accumulator takes the product's grid, so the step is an ordinary one
QB_HD void cacc_first(cacc &acc, const cop &a, const cop &b) {
  if (acc.E == CH_EZERO && a.e != CH_ESPECIAL && b.e != CH_ESPECIAL) {
    acc.w[0] = 0;  // -0 + x = x
    acc.E = a.e + b.e;
  }
}
QB_HD void chain_slow(cacc &acc, q128 a, q128 b) { cacc_set(acc, fma_packed(a, b, cacc_get(acc))); }
// A product of zero (neg: its sign) leaves a sum that is not zero as it is.  False: for the packed operation.
// A matrix with many zeros brings one to some lane of a wave at nearly every step, and the wave does not wait for the
// packed operation then: 1000 x 1000 x 300, nine of ten entries zero, 1.5 ms, 2.4 ms with it; gemv 65536 x 300
// column-major 0.26 and 0.39 ms.
QB_HD bool chain_zero(cacc &acc, uint32_t neg) {
  if (acc.E == CH_EZERO) acc.w[0] &= neg;  // the sum of two zeros is -0 where both are
  return acc.E != CH_APACKED;
}
QB_HD void chain_rest(cacc &acc, q128 a, q128 b) {  // a step that cacc_step does not take
  const bool zero = (q_iszero(a) && q_bexp(b) != 0x7fffu) || (q_iszero(b) && q_bexp(a) != 0x7fffu);
  if (zero && chain_zero(acc, (uint32_t)((a.hi ^ b.hi) >> 63))) return;
  chain_slow(acc, a, b);
}

QB_HD q128 chain_mul(q128 a, q128 b) {  // mul_packed(a, b)
  const cop A = cop_unpack(a), B = cop_unpack(b);
  cacc z;
  cacc_init(z);
  z.w[0] = 1;  // -0
  cacc_first(z, A, B);
  if (!cacc_step(z, A, B)) chain_slow(z, a, b);
  return cacc_get(z);
}
// acc = RN(a*b + acc) for packed a, b, with b's unpacked form at hand
QB_HD void chain_fma(cacc &acc, q128 a, q128 b, const cop &B) {
  const cop A = cop_unpack(a);
  if (!cacc_step(acc, A, B)) chain_slow(acc, a, b);
}
QB_HD void chain_fma(cacc &acc, q128 a, q128 b) { chain_fma(acc, a, b, cop_unpack(b)); }

// y_i = fma(alpha, sum, mul(beta, y_i)) with sum = c0 + c1 (two chains), the odd tail's fma applied;
// the four operations as one loop, so the step's code is there once
QB_HD q128 gemv_row_end(q128 c0, q128 c1, int pair, int odd, q128 ta, q128 tx, q128 alpha,
                                             q128 beta, q128 y) {
  q128 by = q_zero(1), sum = c0;
#pragma unroll 1
  for (int op = 0; op < 4; ++op) {
    if ((op == 1 && !pair) || (op == 2 && !odd)) continue;
    const q128 a = op == 0 ? beta : op == 1 ? c1 : op == 2 ? ta : alpha;
    const q128 b = op == 0 ? y : op == 1 ? q_one() : op == 2 ? tx : sum;
    cacc acc;
    cacc_set(acc, (op == 0 || op == 3) ? by : sum);
    chain_fma(acc, a, b);
    const q128 r = cacc_get(acc);
    if (op == 0 || op == 3) by = r;
    else sum = r;
  }
  return by;
}
#if defined(__HIPCC__)
// One chain per lane along a row of a matrix, all lanes of a wave against the same vector:
//   ch = RN(a[s sa] x(s per + par) + ch)   for s = 0..steps-1
// with per = 1, or 2 when lanes of odd and even par (0 or 1) take every other element.  The wave unpacks
// 32 elements of x at a time into its own LDS; every lane of the wave calls (live: it has a chain), and
// steps, per and x are the same in all of them.  Elements of a are loaded four steps at a time, a group
// ahead, and pass through the lane's LDS slots, so the step's code is there once: a row's lane pair then
// asks for a whole 128-byte line at once.  With a load per step the lines of a wave's 32 rows were
// fetched again and again (13.8 GB for the 9.0 GB of a batch of 2048 gemv problems).
constexpr int LC_GROUP = 4;
struct chain_lds {
  cop u[32];
  q128 p[32];
  uint4 a[LC_GROUP][64];
};
template <typename X>
__device__ __forceinline__ void lane_chain(cacc &ch, bool live, const q128 *__restrict__ a, int64_t sa, int64_t steps,
                                           int per, int par, const X x, chain_lds &lds) {
  const int lane = (int)(threadIdx.x & 63), span = 32 / per;
  uint4 v[LC_GROUP];
#pragma unroll
  for (int g = 0; g < LC_GROUP; ++g) {
    v[g] = make_uint4(0, 0, 0, 0);
    if (live && g < steps) v[g] = *reinterpret_cast<const uint4 *>(a + g * sa);
  }
  for (int64_t s0 = 0; s0 < steps; s0 += span) {
    const int cnt = (int)((steps - s0 < span) ? steps - s0 : span);
    __builtin_amdgcn_wave_barrier();  // the wave's reads of the span before are done
    if (lane < cnt * per) {
      const q128 e = x(s0 * per + lane);
      lds.p[lane] = e;
      lds.u[lane] = cop_unpack(e);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (!live) continue;
    for (int q0 = 0; q0 < cnt; q0 += LC_GROUP) {
#pragma unroll
      for (int g = 0; g < LC_GROUP; ++g) lds.a[g][lane] = v[g];
      a += LC_GROUP * sa;
#pragma unroll
      for (int g = 0; g < LC_GROUP; ++g)
        if (s0 + q0 + LC_GROUP + g < steps) v[g] = *reinterpret_cast<const uint4 *>(a + g * sa);
      const int ge = cnt - q0 < LC_GROUP ? cnt - q0 : LC_GROUP;
      for (int g = 0; g < ge; ++g) {
        const uint4 w = lds.a[g][lane];
        const q128 e = q_make(((uint64_t)w.y << 32) | w.x, ((uint64_t)w.w << 32) | w.z);
        const int k = (q0 + g) * per + par;
        const cop E = cop_unpack(e);
        if (s0 + q0 + g == 0) cacc_first(ch, E, lds.u[k]);
        if (!cacc_step(ch, E, lds.u[k])) chain_rest(ch, e, lds.p[k]);
      }
    }
  }
}

// The chains t = sum over l in [kk, ke) of A(i, l) B(l, j) of a TM x TN tile of C at (i0, j0), one per thread of 256,
// rows fastest.  Per step of KT values of l the workgroup loads the tile's TM x KT elements of A and
// KT x TN of B once (coalesced along the contiguous dimension), unpacks them into LDS, and every thread
// runs its chain over the step from LDS, in the order l = kk, kk + 1, ...  A special operand that is not zero is taken
// from memory again.  Every thread of the workgroup calls; threads outside m x n return zero.
template <int TM, int TN, int KT>
__device__ __forceinline__ q128 tile_chain(int colmajor, int64_t m, int64_t n, const q128 *__restrict__ A, int64_t lda,
                                           const q128 *__restrict__ B, int64_t ldb, int64_t i0, int64_t j0, int64_t kk,
                                           int64_t ke, cop *sA, cop *sB) {
  static_assert(TM * TN == 256, "256 threads");
  const int64_t as_i = colmajor ? 1 : lda, as_l = colmajor ? lda : 1;
  const int64_t bs_l = colmajor ? 1 : ldb, bs_j = colmajor ? ldb : 1;
  const int ti = (int)threadIdx.x % TM, tj = (int)threadIdx.x / TM;
  const bool live = i0 + ti < m && j0 + tj < n;
  const q128 *ap = A + (i0 + ti) * as_i;
  const q128 *bp = B + (j0 + tj) * bs_j;
  auto load = [](const q128 *p) {
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    return q_make(((uint64_t)v.y << 32) | v.x, ((uint64_t)v.w << 32) | v.z);
  };
  cacc ch;
  cacc_init(ch);
  for (int64_t l0 = kk; l0 < ke; l0 += KT) {
    const int lt = (int)((ke - l0 < KT) ? ke - l0 : KT);
    __syncthreads();  // the previous step's operands are no longer read
#pragma unroll
    for (int e0 = 0; e0 < TM * KT; e0 += 256) {
      const int e = e0 + (int)threadIdx.x;  // rows contiguous: r fastest; l contiguous: q fastest
      const int r = colmajor ? e % TM : e / KT, q = colmajor ? e / TM : e % KT;
      if (e < TM * KT && q < lt && i0 + r < m) sA[q * TM + r] = cop_unpack(load(A + (i0 + r) * as_i + (l0 + q) * as_l));
    }
#pragma unroll
    for (int e0 = 0; e0 < TN * KT; e0 += 256) {
      const int e = e0 + (int)threadIdx.x;
      const int c = colmajor ? e / KT : e % TN, q = colmajor ? e % KT : e / TN;
      if (e < TN * KT && q < lt && j0 + c < n) sB[q * TN + c] = cop_unpack(load(B + (l0 + q) * bs_l + (j0 + c) * bs_j));
    }
    __syncthreads();
    if (live) {
      if (l0 == kk) cacc_first(ch, sA[ti], sB[tj]);
      for (int q = 0; q < lt; ++q)
        if (const cop &a = sA[q * TM + ti], &b = sB[q * TN + tj]; !cacc_step(ch, a, b))
          if ((a.zero | b.zero) != 1u || !chain_zero(ch, a.neg ^ b.neg))
            chain_slow(ch, load(ap + (l0 + q) * as_l), load(bp + (l0 + q) * bs_l));
    }
  }
  return cacc_get(ch);
}
#endif  // __HIPCC__

}  // namespace qb
