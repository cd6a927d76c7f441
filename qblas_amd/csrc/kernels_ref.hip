// kernels_ref.hip -- reference-order ("bit-exact") kernels for dot, gemv and gemm, plus the seeded
// input generators.
//
// Each kernel reproduces the evaluation order of the reference routine it cites, with correctly
// rounded binary128 operations (q128.hpp), so on the same inputs it returns the reference's
// result bit for bit:
//   dot  : include/quadblas/algorithms/level1.hpp:14-137
//   gemv : include/quadblas/algorithms/level2.hpp:15-99
//   gemm : include/quadblas/algorithms/level3.hpp:187-336 (kc from detail/blocking.hpp:17-67)
// Every reference chain is a serial order of rounded steps.  Where there are chains enough to fill the
// chip one lane owns one (chain.hpp); where there are few, a wave does a chain's steps 64 at a time
// with the same results (chain_scan.hpp).  The other forms (kernels_exact.hip, kernels_dd.hip,
// kernels_ozaki.hip) trade the reference order for exact or wider accumulation.
#include <algorithm>

#include "chain_scan.hpp"
#include "kernels.h"

using namespace qb;

namespace qbk {

__device__ __forceinline__ q128 ld(const q128 *p) {
  const uint4 v = *reinterpret_cast<const uint4 *>(p);
  return q_make(((uint64_t)v.y << 32) | v.x, ((uint64_t)v.w << 32) | v.z);
}
__device__ __forceinline__ void st(q128 *p, q128 v) {
  uint4 w;
  w.x = (uint32_t)v.lo;
  w.y = (uint32_t)(v.lo >> 32);
  w.z = (uint32_t)v.hi;
  w.w = (uint32_t)(v.hi >> 32);
  *reinterpret_cast<uint4 *>(p) = w;
}

// ------------------------------------------------------------------------------------------
// dot (level1.hpp)
// ------------------------------------------------------------------------------------------

// Chunk t of T: [t*chunk, t == T-1 ? n : (t+1)*chunk), chunk = n / T  (level1.hpp:47,58-59).
__device__ __forceinline__ void chunk_range(int64_t n, int T, int t, int64_t &s, int64_t &e) {
  const int64_t chunk = n / T;
  s = (int64_t)t * chunk;
  e = (t == T - 1) ? n : s + chunk;
}

// a contiguous chunk's value from its two chains' and, of an odd length, its last element (at e - 1)
__device__ __forceinline__ q128 dot_pair_end(q128 r, q128 a, const q128 *__restrict__ x, const q128 *__restrict__ y,
                                             int64_t e, int odd) {
  q128 b = q_one();
#pragma unroll 1
  for (int op = 0; op < 1 + odd; ++op) {
    cacc acc;
    cacc_set(acc, r);
    chain_fma(acc, a, b);
    r = cacc_get(acc);
    a = ld(x + e - 1);
    b = ld(y + e - 1);
  }
  return r;
}

// Contiguous: chunk t is two chains, lane p's over elements start+p, start+p+2, ... for i < len/2
// (dot_kernel_vectorized, level1.hpp:20-25), combined by horizontal_sum (quad_vector.hpp:141-150) and
// the odd tail's fma (level1.hpp:29-32).  Strided: one serial chain per chunk (level1.hpp:111-114,
// :130-133).  There are only T or 2T chains, so each gets a whole wave, 64 elements at a time
// (chain_scan.hpp); a workgroup is one chunk.  part[t] receives the chunk's value, or, with one
// chunk, out the result ('direct': n < 500 returns the kernel's value without the final
// "0 + partial" sum, level1.hpp:40-43, :128-134).
// Bound by the latency of a block of 64 steps, about 1.8 us.
__global__ void __launch_bounds__(128) k_dot_ref_chunks(const q128 *__restrict__ x, int64_t incx,
                                                        const q128 *__restrict__ y, int64_t incy, int64_t n, int T,
                                                        int direct, q128 *__restrict__ part, q128 *__restrict__ out) {
  __shared__ q128 second;
  __shared__ lane_lds lds[2];
  const int t = (int)blockIdx.x, pair = blockDim.x > 64;  // two waves: contiguous
  const int p = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int64_t s, e;
  chunk_range(n, T, t, s, e);
  const int64_t len = e > s ? e - s : 0, step = 1 + pair;
  const q128 *xc = x + (s + p) * incx, *yc = y + (s + p) * incy;
  q128 r = wave_chain(q_zero(0), sc_strided{xc, step * incx}, sc_strided{yc, step * incy}, len / step, lds[p]);
  if (pair) {
    if (threadIdx.x == 64) second = r;
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  if (pair && len) r = dot_pair_end(r, second, x, y, e, (int)(len & 1));
  if (T == 1)
    st(out, direct ? r : add_packed(q_zero(0), r));
  else
    st(part + t, r);
}
// Long chunks: a workgroup per chain (group_chain), whose values k_dot_ref_sum puts together.  2048 steps take
// 6.3 us with the operands in L2, 9 us in the dot of 2^20, of VALU issue, barriers and waits for operands, and a climb or
// tie 0.05 us more (120 cycles).  A chain of 32768 uniform terms takes 17.4 such passes, 1.4 of them ended early by a sum
// near zero and followed by 64 steps of a wave, and has 570 climbs; of log-uniform ones 16.3 and 150.  2^20 elements,
// T = 16: 0.25 ms (0.94 ms with a wave per chain; log-uniform 0.165 ms, 0.78 ms).
__global__ void __launch_bounds__(64 * SG_WAVES) k_dot_ref_group(const q128 *__restrict__ x, int64_t incx,
                                                                 const q128 *__restrict__ y, int64_t incy, int64_t n,
                                                                 int T, int pair, q128 *__restrict__ part) {
  __shared__ sg_lds lds;
  const int t = (int)blockIdx.x >> pair, p = (int)blockIdx.x & pair;
  int64_t s, e;
  chunk_range(n, T, t, s, e);
  const int64_t step = 1 + pair;
  const q128 r = group_chain(q_zero(0), sc_strided{x + (s + p) * incx, step * incx},
                             sc_strided{y + (s + p) * incy, step * incy}, (e - s) / step, lds);
  if (threadIdx.x == 0) st(part + blockIdx.x, r);
}
// the chunks' values summed from +0 in chunk order (level1.hpp:67-71, :117-120): one more chain.  PAIR: part holds the
// values of a chunk's two chains (dot_pair_end)
template <bool PAIR>
__global__ void __launch_bounds__(64) k_dot_ref_sum(const q128 *__restrict__ x, const q128 *__restrict__ y, int64_t n, int T,
                                                    q128 *__restrict__ part, q128 *__restrict__ out) {
  __shared__ lane_lds lds;
  if constexpr (PAIR) {
    for (int t = threadIdx.x; t < T; t += 64) {
      int64_t s, e;
      chunk_range(n, T, t, s, e);
      st(part + 2 * t, dot_pair_end(ld(part + 2 * t), ld(part + 2 * t + 1), x, y, e, (int)((e - s) & 1)));
    }
    __syncthreads();
  }
  const q128 r = wave_chain(q_zero(0), sc_strided{part, 1 + PAIR}, sc_const{q_one()}, T, lds);
  if (threadIdx.x == 0) st(out, r);
}

// ------------------------------------------------------------------------------------------
// gemv (level2.hpp)
// ------------------------------------------------------------------------------------------

// RowMajor, incx == 1: row i's two lane chains run on lanes 2i and 2i+1 (dot_kernel_vectorized
// on the row, level2.hpp:35-38); the pair is combined with a lane exchange, the odd tail applied,
// then y_i = fma(alpha, sum, mul(beta, y_i)) (level2.hpp:48).
// RowMajor, incx != 1: one chain per row (level2.hpp:41-44).
__global__ void __launch_bounds__(64) k_gemv_row_ref(int64_t m, int64_t n, q128 alpha, const q128 *__restrict__ A,
                                                     int64_t lda, const q128 *__restrict__ x, int64_t incx, q128 beta,
                                                     q128 *__restrict__ y, int64_t incy, const int *__restrict__ only) {
  __shared__ __attribute__((aligned(16))) chain_lds lds;
  const int pair = incx == 1, lane = (int)threadIdx.x, p = lane & pair;
  const int64_t i = (int64_t)blockIdx.x * (64 >> pair) + (lane >> pair);
  const bool live = i < m && (!only || only[i]);  // all rows, or those that the kernel below left
  if (!__ballot(live)) return;
  const q128 *row = A + i * lda;
  cacc ch;
  cacc_init(ch);
  lane_chain(ch, live, row + p, 1 + pair, n >> pair, 1 + pair, p, [=](int64_t j) { return ld(x + j * incx); }, lds);
  const q128 mine = cacc_get(ch);
  const uint64_t olo = (uint64_t)__shfl_xor((unsigned long long)mine.lo, 1);
  const uint64_t ohi = (uint64_t)__shfl_xor((unsigned long long)mine.hi, 1);
  if (!live || p != 0) return;
  const int odd = pair && (n & 1);
  q128 *yi = y + i * incy;
  st(yi, gemv_row_end(mine, q_make(olo, ohi), pair, odd, odd ? ld(row + n - 1) : q_zero(0),
                      odd ? ld(x + n - 1) : q_zero(0), alpha, beta, ld(yi)));
}
// Few rows: one wave per chain, 64 columns at a time (chain_scan.hpp); rows of a workgroup share x.
// A pair's chains are neighbouring waves, the first of which ends the row.  MANY: in a launch of many chains, a row
// that blocks of 64 fail on is left, marked in left[] unless that is null, for the kernel above.
template <bool MANY>
__global__ void __launch_bounds__(256) k_gemv_row_ref_scan(int64_t m, int64_t n, q128 alpha, const q128 *__restrict__ A,
                                                           int64_t lda, const q128 *__restrict__ x, int64_t incx,
                                                           q128 beta, q128 *__restrict__ y, int64_t incy,
                                                           int *__restrict__ left) {
  __shared__ q128 other[4];
  __shared__ int s_left[4];
  const int pair = incx == 1;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t c = (int64_t)blockIdx.x * 4 + w;
  const int64_t i = pair ? c >> 1 : c;
  const int p = pair ? (int)(c & 1) : 0;
  q128 r = q_zero(0);
  bool leave = false;
  if (i < m) {
    const sc_strided a{A + i * lda + p, 1 + pair}, b{x + p, pair ? 2 : incx};
    if constexpr (MANY) {
      leave = !wave_chain_or_not(r, a, b, n >> pair, left != nullptr);
    } else {
      __shared__ lane_lds lds[4];
      r = wave_chain(r, a, b, n >> pair, lds[w]);
    }
  }
  if ((threadIdx.x & 63) == 0) {
    other[w] = r;
    s_left[w] = leave;
  }
  __syncthreads();
  if (i < m && p == 0 && (threadIdx.x & 63) == 0) {
    if constexpr (MANY) {
      leave = s_left[w] || s_left[w ^ pair];
      if (left) left[i] = leave;
      if (leave) return;
    }
    const int odd = pair && (n & 1);
    q128 *yi = y + i * incy;
    st(yi, gemv_row_end(r, other[w ^ pair], pair, odd, odd ? ld(A + i * lda + n - 1) : q_zero(0),
                        odd ? ld(x + n - 1) : q_zero(0), alpha, beta, ld(yi)));
  }
}

// ColMajor: ax[j] = mul(alpha, x_j) once per column (level2.hpp:71).
__global__ void k_scale_vec(int64_t n, q128 alpha, const q128 *__restrict__ x, int64_t incx,
                            q128 *__restrict__ ax) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += stride)
    st(ax + j, chain_mul(alpha, ld(x + j * incx)));
}
// ColMajor: y_i = mul(beta, y_i) (level2.hpp:63-66), then y_i = fma(A_ij, ax_j, y_i) for
// j = 0..n-1 (level2.hpp:69-80); lane i owns row i, so loads of A columns coalesce.
__global__ void __launch_bounds__(64) k_gemv_col_ref(int64_t m, int64_t n, const q128 *__restrict__ A, int64_t lda,
                                                     const q128 *__restrict__ ax, q128 beta, q128 *__restrict__ y,
                                                     int64_t incy, const int *__restrict__ only) {
  __shared__ __attribute__((aligned(16))) chain_lds lds;
  for (int64_t i0 = (int64_t)blockIdx.x * 64; i0 < m; i0 += (int64_t)gridDim.x * 64) {
    const int64_t i = i0 + threadIdx.x;
    const bool live = i < m && (!only || only[i]);  // all rows, or those that the kernel below left
    if (!__ballot(live)) continue;
    q128 *yi = y + i * incy;
    cacc ch;
    cacc_set(ch, live ? chain_mul(beta, ld(yi)) : q_zero(0));
    lane_chain(ch, live, A + i, lda, n, 1, 0, [=](int64_t j) { return ld(ax + j); }, lds);
    if (live) st(yi, cacc_get(ch));
  }
}
// Few rows: one wave per row; the eight rows of a workgroup share the 128-byte lines of A's columns.  MANY: as above.
template <bool MANY>
__global__ void __launch_bounds__(512) k_gemv_col_ref_scan(int64_t m, int64_t n, const q128 *__restrict__ A,
                                                           int64_t lda, const q128 *__restrict__ ax, q128 beta,
                                                           q128 *__restrict__ y, int64_t incy, int *__restrict__ left) {
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t i = (int64_t)blockIdx.x * 8 + w;
  if (i >= m) return;
  q128 *yi = y + i * incy;
  q128 r = chain_mul(beta, ld(yi));
  const sc_strided a{A + i, lda}, b{ax, 1};
  bool leave = false;
  if constexpr (MANY) {
    leave = !wave_chain_or_not(r, a, b, n, left != nullptr);
    if (left && (threadIdx.x & 63) == 0) left[i] = leave;
  } else {
    __shared__ lane_lds lds[8];
    r = wave_chain(r, a, b, n, lds[w]);
  }
  if (!leave && (threadIdx.x & 63) == 0) st(yi, r);
}

// ------------------------------------------------------------------------------------------
// gemm (level3.hpp)
// ------------------------------------------------------------------------------------------

// One lane per C element.  k is processed in blocks of kc; each block is a fresh chain t and
// C = fma(alpha, t, mul(first ? beta : 1, C)) (level3.hpp:297-300 with the micro-kernel's
// epilogue :102-109; gemm_simple :200-210 is the single-block case); the product with 1 changes
// nothing, so C = fma(alpha, t, C) over the blocks is one more chain, from beta * C.  Layout-aware indexing for
// both layouts.  A workgroup computes a 16 x 16 tile of C (tile_chain).
// Bound by VALU issue: 85 to 105 instructions per wave and multiply-add (chain.hpp).  4096^3
// log-uniform: 214 ms = 643 quad GFLOP/s (577 ms with a 401-instruction step); 2048^3 uniform 21.9 ms.
// part == null: the workgroup takes all blocks of k.  Else it takes block kb0 + blockIdx.z and writes its t to
// part[(blockIdx.z n + j) m + i], for k_gemm_ref_fold: the blocks' chains do not depend on each other,
// so a C of few tiles still fills the chip: 500 x 333 x 700 326 us against 454, 64 x 64 x 2000 70 us against 823.
// The latter's 256 workgroups are one wave a SIMD: bound by a step's latency of 0.46 us, which 85 instructions in place of
// 105 did not shorten (68 us then), as the chain of dependent additions stayed as long.
// KT: values of k staged at a time, 1 KB of LDS each.  32 let five workgroups share a CU, 16 eight: with more
// workgroups than five a CU 16 is faster (1000^3 2734 us against 2850, 500 x 333 x 700 363 against 377), with
// fewer the barriers cost more than there is to overlap them with (100 x 100 x 900 78 us against 75).
constexpr int64_t GR_FIVE = 5 * 256;
template <int KT>
__global__ void __launch_bounds__(256) k_gemm_ref(int colmajor, int64_t m, int64_t n, int64_t k, int64_t kc,
                                                  q128 alpha, const q128 *__restrict__ A, int64_t lda,
                                                  const q128 *__restrict__ B, int64_t ldb, q128 beta,
                                                  q128 *__restrict__ C, int64_t ldc, int64_t kb0,
                                                  q128 *__restrict__ part) {
  __shared__ __attribute__((aligned(16))) cop sA[KT * 16];
  __shared__ __attribute__((aligned(16))) cop sB[KT * 16];
  const int ti = threadIdx.x & 15, tj = threadIdx.x >> 4;
  const int64_t i0 = (int64_t)blockIdx.y * 16, j0 = (int64_t)blockIdx.x * 16;
  const int64_t i = i0 + ti, j = j0 + tj;
  const bool live = i < m && j < n;  // every thread takes part in the loads and barriers
  q128 *ci = C + (colmajor ? j * ldc + i : i * ldc + j);
  const int64_t k0 = part ? (kb0 + blockIdx.z) * kc : 0, k1 = part ? (k0 + kc < k ? k0 + kc : k) : k;
  cacc c;
  if (!part) cacc_set(c, live ? chain_mul(beta, ld(ci)) : q_zero(0));
  for (int64_t kk = k0; kk < k1; kk += kc) {
    const int64_t ke = (kk + kc < k1) ? kk + kc : k1;
    const q128 t = tile_chain<16, 16, KT>(colmajor, m, n, A, lda, B, ldb, i0, j0, kk, ke, sA, sB);
    if (live) {
      if (!part) chain_fma(c, alpha, t);
      else st(part + ((int64_t)blockIdx.z * n + j) * m + i, t);
    }
  }
  if (!part && live) st(ci, cacc_get(c));
}
// C = fma(alpha, t, C) over blocks kb0 .. kb0 + nb - 1, C = beta * C before block 0
__global__ void __launch_bounds__(256) k_gemm_ref_fold(int colmajor, int64_t m, int64_t n, int64_t kb0, int64_t nb,
                                                       q128 alpha, q128 beta, const q128 *__restrict__ part,
                                                       q128 *__restrict__ C, int64_t ldc) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= m * n) return;
  const int64_t j = e / m, i = e - j * m;
  q128 *ci = C + (colmajor ? j * ldc + i : i * ldc + j);
  cacc c;
  cacc_set(c, kb0 == 0 ? mul_packed(beta, ld(ci)) : ld(ci));
  const cop al = cop_unpack(alpha);
  for (int64_t b = 0; b < nb; ++b) chain_fma(c, ld(part + b * m * n + e), alpha, al);
  st(ci, cacc_get(c));
}

// ------------------------------------------------------------------------------------------
// seeded generators (same definitions as the CPU oracle's or_fill / or_fill_pair_y)
// ------------------------------------------------------------------------------------------

__device__ __forceinline__ uint64_t rand64(uint64_t seed, uint64_t idx) {
  uint64_t z = seed + (idx + 1) * 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double u11(uint64_t r) { return (double)(r >> 11) * 0x1p-52 - 1.0; }
__device__ __forceinline__ q128 full_uniform(uint64_t seed, uint64_t i) {
  const double a = u11(rand64(seed, 2 * i)), b = u11(rand64(seed, 2 * i + 1));
  // b * 2^-60 is exact; the sum is one correctly rounded binary128 add
  return add_packed(from_double(a), mul_packed(from_double(b), from_double(0x1p-60)));
}

// value number i of generator kind (0..4)
__device__ q128 gen_value(int kind, uint64_t seed, int64_t i, int lo_exp, int hi_exp) {
  q128 v;
  if (kind == 0) {
    v = full_uniform(seed, (uint64_t)i);
  } else if (kind == 1) {
    const uint64_t r0 = rand64(seed, 3 * (uint64_t)i), r1 = rand64(seed, 3 * (uint64_t)i + 1),
                   r2 = rand64(seed, 3 * (uint64_t)i + 2);
    const uint32_t span = (uint32_t)(hi_exp - lo_exp);
    const int e = lo_exp + (int)((uint32_t)r0 % span);
    v = q_make(r2, (r0 & (1ull << 63)) | ((uint64_t)(e + QBIAS) << 48) | (r1 >> 16));
  } else if (kind == 2 || kind == 4) {
    const int64_t p = i & ~(int64_t)1;
    if ((p % 8) < 2) {
      const double u = 1.0 + (double)(rand64(seed, (uint64_t)p) >> 12) * 0x1p-52;
      v = mul_packed(from_double(u), from_double(kind == 4 ? 1e22 : 1e20));
      if (i & 1) v.hi ^= 1ull << 63;
    } else {
      v = full_uniform(seed, (uint64_t)i);
    }
  } else {  // kind 3: y vector of the cancellation variant (own stream; equal values on each pair)
    const int64_t p0 = i & ~(int64_t)1;
    const int64_t p = ((p0 % 8) < 2) ? p0 : i;
    v = full_uniform(seed + 1, (uint64_t)p);
  }
  return v;
}

__global__ void k_fill(int kind, uint64_t seed, int64_t n, int lo_exp, int hi_exp, q128 *__restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    st(out + i, gen_value(kind, seed, i, lo_exp, hi_exp));
}

// value number r*cols + c of the generator stored at element (r, c) of a rows x cols matrix
// (RowMajor r*ld + c or ColMajor r + c*ld)
__global__ void k_fill_2d(int kind, uint64_t seed, int64_t rows, int64_t cols, int64_t ld, int colmajor, int lo_exp,
                          int hi_exp, q128 *__restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < rows * cols; g += stride) {
    // walk the storage order so that writes coalesce
    const int64_t r = colmajor ? g % rows : g / cols, c = colmajor ? g / rows : g % cols;
    st(out + (colmajor ? r + c * ld : r * ld + c), gen_value(kind, seed, r * cols + c, lo_exp, hi_exp));
  }
}

// ------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------

// Whether a dot's chains get a workgroup each instead of a wave (a workgroup's registers take a CU).  Measured,
// us (workgroup, wave): 32 chains of 512 41, 32; 1024 47, 56; 4096 60, 160; 32768 288, 949; 256 chains of 512
// 52, 43; 1024 54, 60 (48, 45 log-uniform); 1536 70, 83 (53, 57); 4096 95, 164.
static bool group_chains(int64_t chains, int64_t len) { return chains <= 256 && len >= 1280; }

hipError_t launch_dot_ref(const q128 *x, int64_t incx, const q128 *y, int64_t incy, int64_t n, int T,
                          q128 *part, q128 *out, hipStream_t st) {
  const int contiguous = (incx == 1 && incy == 1);
  int Teff = T, direct = 0;
  if (n < 500) {  // level1.hpp:40-43 (contiguous) and :128-134 (strided): one chain set, no sum
    Teff = 1;
    direct = 1;
  }
  if (group_chains(Teff << contiguous, (n / Teff) >> contiguous)) {
    hipLaunchKernelGGL(k_dot_ref_group, dim3((unsigned)(Teff << contiguous)), dim3(64 * SG_WAVES), 0, st, x, incx, y,
                       incy, n, Teff, contiguous, part);
    hipLaunchKernelGGL(contiguous ? k_dot_ref_sum<true> : k_dot_ref_sum<false>, dim3(1), dim3(64), 0, st, x, y, n, Teff, part, out);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_dot_ref_chunks, dim3(Teff), dim3(contiguous ? 128 : 64), 0, st, x, incx, y, incy, n, Teff, direct,
                     part, out);
  if (Teff > 1) hipLaunchKernelGGL(k_dot_ref_sum<false>, dim3(1), dim3(64), 0, st, x, y, n, Teff, part, out);
  return hipGetLastError();
}

// Whether a gemv's chains go to a wave each (chain_scan.hpp) or to a lane each (lane_chain).  A lane's
// step is a latency of about 0.5 us until the lanes fill the chip; a wave's block of 64 steps costs a
// fixed amount and about 9 instructions a step.  Measured, uniform entries, us (wave each, lane each):
// row-major 1500^2 69, 359; 8192^2 797, 1932; 16384 x 2048 (32768 chains) 457, 519; 65536 x 1000 980, 316;
// column-major 2049 x 777 63, 366; 8192^2 1061, 3738; 32768 x 1024 476, 510; 4608 x 16 20, 16.
static bool few_chains(int64_t chains, int64_t len) {
  return chains <= 32768 && chains * ((len + 63) / 64 * 64 + 128) <= 36864 * len;
}

// Whether there are so many chains of a wave each that they may be left to a lane each.  With more than four waves a SIMD, steps one at a time
// wait for each other: subnormal entries, 8192 x 2048 row-major, 2.5 ms left, 14 ms not; with fewer they do not (1500^2
// 1.7 ms left, 2.3 ms not), and the second launch costs other calls 2.5 us of 66.
static bool many_chains(int64_t chains) { return chains > 4096; }
size_t gemv_ref_left(int colmajor, int64_t m, int64_t n, int64_t incx) {
  const int pair = !colmajor && incx == 1;
  return few_chains(m << pair, n >> pair) && many_chains(m << pair) ? (size_t)m * sizeof(int) : 0;
}

hipError_t launch_gemv_ref(int colmajor, int64_t m, int64_t n, q128 alpha, const q128 *A, int64_t lda,
                           const q128 *x, int64_t incx, q128 beta, q128 *y, int64_t incy, q128 *ax, int *left,
                           hipStream_t st) {
  const int threads = 64;
  const int pair = !colmajor && incx == 1;
  const bool scan = few_chains(m << pair, n >> pair);
  if (!colmajor) {
    const int64_t lanes = m << pair;
    if (scan) {
      const auto f = many_chains(lanes) ? k_gemv_row_ref_scan<true> : k_gemv_row_ref_scan<false>;
      hipLaunchKernelGGL(f, dim3((unsigned)((lanes + 3) / 4)), dim3(256), 0, st, m, n, alpha, A, lda, x, incx, beta, y,
                         incy, left);
      if (!left) return hipGetLastError();
    }
    const int64_t blocks = (lanes + threads - 1) / threads;
    if (!grid_fits(blocks, threads)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gemv_row_ref, dim3((unsigned)blocks), dim3(threads), 0, st, m, n, alpha, A, lda, x,
                       incx, beta, y, incy, left);
  } else {
    hipLaunchKernelGGL(k_scale_vec, dim3(stride_blocks(n, 256)), dim3(256), 0, st, n, alpha, x, incx, ax);
    if (scan) {
      const auto f = many_chains(m) ? k_gemv_col_ref_scan<true> : k_gemv_col_ref_scan<false>;
      hipLaunchKernelGGL(f, dim3((unsigned)((m + 7) / 8)), dim3(512), 0, st, m, n, A, lda, ax, beta, y, incy, left);
      if (!left) return hipGetLastError();
    }
    hipLaunchKernelGGL(k_gemv_col_ref, dim3(stride_blocks(m, threads)), dim3(threads), 0, st, m, n,
                       A, lda, ax, beta, y, incy, left);
  }
  return hipGetLastError();
}

// Workspace for splitting the blocks of k over workgroups (0: not split): a workgroup of four waves is
// a tile, and the chip takes 5 or 8 of them per CU at a time (LDS), so below about 2048 tiles it is idle in
// part or for the last wave.  Rounds of at most 64 MB of t.
size_t gemm_ref_ws(int64_t m, int64_t n, int64_t k, int64_t kc) {
  const int64_t nb = (k + kc - 1) / kc, tm = (m + 15) / 16, tn = (n + 15) / 16;
  if (nb < 2 || tm > 2048 || tn > 2048 || tm * tn >= 2048) return 0;
  const int64_t t = 16 * m * n, fit = std::min<int64_t>((int64_t)(64 << 20) / t, 32768);
  return (size_t)(t * std::min(nb, fit));
}

hipError_t launch_gemm_ref(int colmajor, int64_t m, int64_t n, int64_t k, int64_t kc, q128 alpha, const q128 *A,
                           int64_t lda, const q128 *B, int64_t ldb, q128 beta, q128 *C, int64_t ldc, q128 *part,
                           hipStream_t st) {
  if (!grid_fits((n + 15) / 16, 256)) return hipErrorInvalidValue;
  const unsigned tn = (unsigned)((n + 15) / 16), tm = (unsigned)((m + 15) / 16);
  const int64_t tiles = (int64_t)tn * tm;
  if (!part) {
    const auto f = tiles > GR_FIVE ? k_gemm_ref<16> : k_gemm_ref<32>;
    hipLaunchKernelGGL(f, dim3(tn, tm), dim3(256), 0, st, colmajor, m, n, k, kc, alpha, A, lda, B, ldb, beta,
                       C, ldc, (int64_t)0, part);
    return hipGetLastError();
  }
  const int64_t nb = (k + kc - 1) / kc, zb = (int64_t)(gemm_ref_ws(m, n, k, kc) / (size_t)(16 * m * n));
  for (int64_t z = 0; z < nb; z += zb) {
    const int64_t c = nb - z < zb ? nb - z : zb;
    const auto f = tiles * c > GR_FIVE ? k_gemm_ref<16> : k_gemm_ref<32>;
    hipLaunchKernelGGL(f, dim3(tn, tm, (unsigned)c), dim3(256), 0, st, colmajor, m, n, k, kc, alpha, A, lda, B,
                       ldb, beta, C, ldc, z, part);
    hipLaunchKernelGGL(k_gemm_ref_fold, dim3((unsigned)((m * n + 255) / 256)), dim3(256), 0, st, colmajor, m, n, z, c,
                       alpha, beta, part, C, ldc);
  }
  return hipGetLastError();
}

__global__ void k_zero(q128 *__restrict__ p, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) st(p + i, q_zero(0));
}
hipError_t launch_zero(q128 *p, int64_t n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero, dim3(stride_blocks(n, 256)), dim3(256), 0, st, p, n);
  return hipGetLastError();
}

hipError_t launch_fill(int kind, uint64_t seed, int64_t n, int lo_exp, int hi_exp, q128 *out, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill, dim3(stride_blocks(n, 256)), dim3(256), 0, st, kind, seed, n, lo_exp, hi_exp,
                     out);
  return hipGetLastError();
}


hipError_t launch_fill_2d(int kind, uint64_t seed, int64_t rows, int64_t cols, int64_t ld, int colmajor, int lo_exp,
                          int hi_exp, q128 *out, hipStream_t st) {
  const int64_t n = rows * cols;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_2d, dim3(stride_blocks(n, 256)), dim3(256), 0, st, kind, seed, rows, cols, ld,
                     colmajor, lo_exp, hi_exp, out);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// axpy and the square root of nrm2 (level1.hpp:139-223, c_interface.hpp:34-59)
// ------------------------------------------------------------------------------------------
// y_i = fma(alpha, x_i, y_i): one correctly rounded FMA per element, independent of order and
// chunking (axpy_kernel_vectorized's lanes and tail compute the same per-element FMA)
__global__ void k_axpy(int64_t n, q128 alpha, const q128 *__restrict__ x, int64_t incx, q128 *__restrict__ y,
                       int64_t incy) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    st(y + i * incy, fma_packed(alpha, ld(x + i * incx), ld(y + i * incy)));
}
__global__ void k_sqrt1(q128 *p) {
  if (threadIdx.x == 0) st(p, sqrt_packed(ld(p)));
}

hipError_t launch_axpy(int64_t n, q128 alpha, const q128 *x, int64_t incx, q128 *y, int64_t incy, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_axpy, dim3((unsigned)blocks), dim3(256), 0, st, n, alpha, x, incx, y, incy);
  return hipGetLastError();
}
hipError_t launch_sqrt1(q128 *p, hipStream_t st) {
  hipLaunchKernelGGL(k_sqrt1, dim3(1), dim3(64), 0, st, p);
  return hipGetLastError();
}
}  // namespace qbk
