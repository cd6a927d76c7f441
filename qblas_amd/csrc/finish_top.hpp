// finish_top.hpp -- the epilogue RN(alpha M 2^lsb + beta y) of the OZAKI finishes: finish_reg_top
// (exact.hpp), same result and same bound, on 29-bit limbs and 160-bit frames (chain.hpp).
//
// M is cut to its top 128 bits H; alpha H (241 bits) and beta y (226 bits) become frames of 160 bits
// with their leading bits at 152 or 153, the lower one shifted onto the other one's grid, complemented
// for a negative sign and added.  Both were rounded down to the grid, so the exact sum lies 0 to 2 grid
// units above the frame's, and rounds as the frame does unless the bits below the rounding position
// (34 of them at least) come within that of a half: then, and for special operands, sums that cancel
// deeply and exponents near the ends of the range, finish_reg_top decides.
// About 300 VALU instructions in place of 1100 (the 12-word frame of finish_reg_top): the finish of a batch of
// 4096 products 2.11 -> 1.58 ms (1.30 ms with the descriptors by scalar loads).
#pragma once
#include "chain.hpp"
#include "exact.hpp"

namespace qb {

template <int N>
QB_HD q128 finish_top(const uint32_t (&M)[N], int lsb, uint32_t sS, q128 alpha, q128 beta, q128 yv, int &terr) {
  static_assert(N >= 6, "top five words");
  const cop a = cop_unpack(alpha), b = cop_unpack(beta), y = cop_unpack(yv);
  const bool z2 = q_iszero(beta) | q_iszero(yv);
  bool ok = a.e != CH_ESPECIAL && (z2 || (b.e != CH_ESPECIAL && y.e != CH_ESPECIAL));
  // leading bit to the top of the top word
  uint32_t W[N];
#pragma unroll
  for (int i = 0; i < N; ++i) W[i] = M[i];
  int up = 0;
#pragma unroll
  for (int step = 4; step >= 1; step >>= 1) {
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < step; ++i) top |= W[N - 1 - i];
    if (ch_any(top == 0)) {
      up += top == 0 ? 32 * step : 0;
#pragma unroll
      for (int i = N - 1; i >= 0; --i) W[i] = top == 0 ? (i >= step ? W[i - step] : 0u) : W[i];
    }
  }
  ok = ok && W[N - 1] != 0;
  const int lz = clz64((uint64_t)W[N - 1]) & 31;
  uint32_t H[4], cut = W[N - 5] << lz;
#pragma unroll
  for (int i = 0; i < 4; ++i) H[i] = (uint32_t)(((((uint64_t)W[N - 4 + i] << 32) | W[N - 5 + i]) << lz) >> 32);
#pragma unroll
  for (int i = 0; i < N - 5; ++i) cut |= W[i];
  const int sh = 32 * N - 128 - up - lz;
  const bool one = (a.l[0] | a.l[1] | a.l[2]) == 0 && a.l[3] == (1u << 25) && a.e == 0;
  terr = (cut && !(z2 && one)) ? lsb + sh + a.e + 1 : INT_MIN;
  // alpha H: bits 87.. as a frame
  uint32_t F[5], P[5];
  {
    const uint32_t h[5] = {H[0] & 0x1fffffffu, ch_alignbit(H[1], H[0], 29) & 0x1fffffffu,
                           ch_alignbit(H[2], H[1], 26) & 0x1fffffffu, ch_alignbit(H[3], H[2], 23) & 0x1fffffffu, H[3] >> 20};
    uint64_t c[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      uint64_t t = k ? c[k - 1] >> 29 : 0;
#pragma unroll
      for (int i = (k < 4 ? 0 : k - 3); i <= (k < 5 ? k : 4); ++i) t += (uint64_t)h[i] * a.l[k - i];
      c[k] = t;
    }
    F[0] = ((uint32_t)c[3] & 0x1fffffffu) | ((uint32_t)c[4] << 29);
    F[1] = (((uint32_t)c[4] >> 3) & 0x3ffffffu) | ((uint32_t)c[5] << 26);
    F[2] = (((uint32_t)c[5] >> 6) & 0x7fffffu) | ((uint32_t)c[6] << 23);
    F[3] = (((uint32_t)c[6] >> 9) & 0xfffffu) | ((uint32_t)c[7] << 20);
    F[4] = (uint32_t)(c[7] >> 12);
  }
  const int32_t E1 = lsb + sh + a.e + 127, E2 = z2 ? E1 - 200 : b.e + y.e, d = E1 - E2;
  {
    uint64_t k[7];
    cop_columns(k, b, y);
    ch_frame(P, k);
  }
  const uint32_t s1 = (uint32_t)ch_clamp(-d, 0, 159), s2 = (uint32_t)ch_clamp(d, 0, 159);
  const uint32_t n1 = (0u - sS) ^ a.neg, n2 = z2 ? 0u : b.neg ^ y.neg;
  ch_shift_words(F, s1);
  ch_shift_words(P, s2);
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const uint32_t f = i < 4 ? ch_alignbit(F[i + 1], F[i], s1) : F[4] >> (s1 & 31);
    const uint32_t p = z2 ? 0u : (i < 4 ? ch_alignbit(P[i + 1], P[i], s2) : P[4] >> (s2 & 31));
    F[i] = ch_addc(f ^ n1, p ^ n2, c, c);
  }
  int32_t E = E1 > E2 ? E1 : E2;
  uint32_t fb = ch_signbits(F[4]), near = 2;
  if (fb - 2u > 11u) {  // the leading bit to 153 (chain.hpp); zeros from below when it moves up
    ok = ok && fb <= 31u;
    const uint32_t f = fb <= 31u ? fb : 6u;
    if (f < 2u) {
      const uint32_t r = 6 - f;
#pragma unroll
      for (int i = 0; i < 4; ++i) F[i] = ch_alignbit(F[i + 1], F[i], r);
      F[4] = (uint32_t)((int32_t)F[4] >> r);
    } else if (f > 6u) {
      const uint32_t r = 32 - (f - 6);
#pragma unroll
      for (int i = 4; i > 0; --i) F[i] = ch_alignbit(F[i], F[i - 1], r);
      F[0] <<= 32 - r;
      near = 2u << (f - 6);
    }
    E += 6 - (int32_t)f;
    fb = 6;
  }
  // bits below the rounding position (bit 15 - fb of word 1), less than `near` below a half or on it
  const uint64_t below = (((uint64_t)F[1] << 32) | F[0]) & ((1ull << (47 - fb)) - 1);
  ok = ok && ((1ull << (46 - fb)) - below) > near && (uint32_t)(E + CH_EMAX) <= (uint32_t)(2 * CH_EMAX);
  if (!ok) return finish_reg_top<N>(M, lsb, sS, alpha, beta, yv, terr);
  cacc r;
  c = 0;
  r.w[0] = ch_addc(F[1], 0x4000u >> fb, c, c) & ~(0x7fffu >> fb);
  r.w[1] = ch_addc(F[2], 0u, c, c);
  r.w[2] = ch_addc(F[3], 0u, c, c);
  r.w[3] = ch_addc(F[4], 0u, c, c);
  r.E = E;
  return cacc_get(r);
}

}  // namespace qb
