// Device FFT for lengths known at run time: an in-place mixed-radix
// decimation-in-time pass sequence over columns held in LDS.
//
// Data placement: sample n of a column must be stored at LDS position
// perm[n] (mixed-radix digit reversal, built by make_fft_plan) before the
// passes run; the transform then comes out in natural order.  Every pass
// combines r sub-transforms of length S into one of length S*r in place, so
// no staging buffer is needed and each thread may process any number of
// butterflies.  Radices up to 16 (make_fft_plan picks few, large ones: a pass
// is bound by its LDS round trip and barrier, so a length of 480 takes three
// passes of 10, 8 and 6 rather than five of 4, 4, 2, 3 and 5).
// Twiddles come from the per-pass tables of pass_twiddles.
#pragma once

#include "fft_ct.h"

namespace nsp {

// LDS position of logical element e of NCOL interleaved columns, dense (lanes
// run over the columns).  NCOL = kPadCol: one column with an unused slot per 16
// elements, so that the passes' power-of-two strides land in different banks.
constexpr int kPadCol = 0;
template <int NCOL>
__host__ __device__ __forceinline__ int lds_pos(int e) {
  return NCOL == kPadCol ? e + (e >> 4) : e;
}

// One pass of radix R and sub-length S (mul = ceil(2^32 / S): exact quotients
// of b < 2^16 by S < 2^16 as the high word of a product).
template <typename T, int NCOL, int SIGN, int R>
__device__ __forceinline__ void fft_pass(cpx<T>* buf, int nb, int S, unsigned mul, const cpx<T>* __restrict__ tw,
                                         int tid, int nthr) {
  constexpr int NC = NCOL == kPadCol ? 1 : NCOL;
  const int total = nb * NC;
  for (int b = tid; b < total; b += nthr) {
    const int col = b % NC;
    const int bb = b / NC;
    const int j = S == 1 ? bb : (int)__umulhi((unsigned)bb, mul);
    const int k = bb - j * S;
    const int base = j * (S * R) + k;
    cpx<T> v[R];
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = buf[lds_pos<NCOL>(col + (base + q * S) * NC)];
    if (S > 1) {
#pragma unroll
      for (int q = 1; q < R; ++q) {
        const cpx<T> w = tw[k * (R - 1) + q - 1];
        v[q] = SIGN < 0 ? cx_mul(v[q], w) : cx_mulc(v[q], w);
      }
    }
    DFT<T, R, SIGN>::run(v);
#pragma unroll
    for (int q = 0; q < R; ++q) buf[lds_pos<NCOL>(col + (base + q * S) * NC)] = v[q];
  }
  __syncthreads();
}

// In-place passes over NCOL columns: element n of column c at
// lds_pos(c + n*NCOL).  Caller has placed inputs at digit-reversed positions
// and synchronised.  SIGN -1 forward (e^{-2 pi i nk/L}), +1 inverse.  Ends
// with a barrier.  MAXR bounds the radices (and registers) of the plan.
template <typename T, int NCOL, int SIGN, int MAXR = 16>
__device__ __forceinline__ void fft_passes(cpx<T>* buf, const FftPlan& P, const cpx<T>* __restrict__ tw, int tid,
                                           int nthr) {
  int S = 1;
  for (int p = 0; p < P.nrad; ++p) {
    const int r = P.rad[p], nb = P.L / r;
    const unsigned mul = P.mul[p];
    switch (r) {
#define NSP_PASS(R)                                                                      \
  case R:                                                                                \
    if constexpr (R <= MAXR) fft_pass<T, NCOL, SIGN, R>(buf, nb, S, mul, tw, tid, nthr); \
    break;
      NSP_PASS(2)
      NSP_PASS(3)
      NSP_PASS(4)
      NSP_PASS(5)
      NSP_PASS(6)
      NSP_PASS(8)
      NSP_PASS(9)
      NSP_PASS(10)
      NSP_PASS(12)
      NSP_PASS(15)
      NSP_PASS(16)
#undef NSP_PASS
      default: break;
    }
    tw += S * (r - 1);
    S *= r;
  }
}

}  // namespace nsp
