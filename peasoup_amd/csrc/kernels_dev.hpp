// kernels_dev.hpp - device-side arithmetic shared by the plain per-stage
// kernels and the fused batched kernels.  Each helper reproduces one
// expression of the reference kernels (src/kernels.cu) with the same
// operation order and precision; multiply-adds that nvcc contracts in the
// reference are written as explicit fma, everything else is unfused (the
// library is built with -ffp-contract=off).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace psx {

// device_resampleII (src/kernels.cu:361): (a*tsamp) is a float product,
// widened to double before the divide by 2c.
__host__ __device__ inline double accel_fact(float acc, float tsamp) {
  const float at = acc * tsamp;
  return (double)at / (2 * 299792458.0);
}

// getAcceleratedIndexII (src/kernels.cu:321-324): __double2ull_rn of
// id + id*af*(id - size), contracted to fma(id*af, id - size, id).  For
// |af|*n < 1 the value lies in [0, n]; the clamp only guards the n edge.
__device__ inline uint64_t resample_index(uint64_t i, uint64_t n, double af) {
  const double di = (double)i;
  double v = fma(di * af, di - (double)n, di);
  v = v > 0.0 ? v : 0.0;
  const uint64_t j = (uint64_t)rint(v);
  return j < n ? j : n - 1;
}

// The same index for series shorter than 2^31 samples, in 32-bit integers
// (identical values: every operand is exactly representable either way).
// n >= 1; the n edge clamps with one unsigned min.
__device__ inline uint32_t resample_index32(uint32_t i, uint32_t n, double dn, double af) {
  const double di = (double)i;
  double v = fma(di * af, di - dn, di);
  v = v > 0.0 ? v : 0.0;
  return min((uint32_t)rint(v), n - 1);
}

// bin_interbin_series_kernel (src/kernels.cu:250-257): the 0.5 is a double
// literal; halving in float gives the identical correctly rounded result.
__device__ inline float interbin(float2 x, float2 prev) {
  const float ampsq = fmaf(x.x, x.x, x.y * x.y);
  const float dr = x.x - prev.x;
  const float di = x.y - prev.y;
  const float ampsq_diff = 0.5f * fmaf(dr, dr, di * di);
  return sqrtf(fmaxf(ampsq, ampsq_diff));
}

// Order statistics for median_scrunch5 (src/kernels.cu:902-959).  The median
// is a unique value, so any correct network returns the reference's value.
__device__ inline void cswap(float& a, float& b) {
  const float lo = fminf(a, b);
  const float hi = fmaxf(a, b);
  a = lo;
  b = hi;
}
__device__ inline float median3(float a, float b, float c) {
  cswap(a, b);
  cswap(b, c);
  cswap(a, b);
  return b;
}
__device__ inline float median4(float a, float b, float c, float d) {
  cswap(a, b);
  cswap(c, d);
  cswap(a, c);
  cswap(b, d);
  cswap(b, c);
  return 0.5f * (b + c);
}
// Seven compare-exchanges leave the median of five in c.
__device__ inline float median5(float a, float b, float c, float d, float e) {
  cswap(a, b);
  cswap(d, e);
  cswap(a, d);
  cswap(b, e);
  cswap(b, c);
  cswap(c, d);
  cswap(b, c);
  return c;
}

// linear_stretch_functor::operator() (src/kernels.cu:1018-1023).  x is
// float(i)*step; the neighbour read past the last input (undefined in the
// reference once x rounds above in_count-1) is clamped to the last input.
__device__ inline float stretch_at(const float* __restrict__ in, uint64_t in_count, unsigned i, float step) {
  const float x = (float)i * step;
  unsigned j = (unsigned)x;
  const float fr = x - (float)j;
  const uint64_t last = in_count - 1;
  const float a = in[j < last ? j : last];
  const float b = in[j + 1 < last ? j + 1 : last];
  return (fr > 1e-5f) ? fmaf(fr, b - a, a) : a + 0.f;
}

// Step of the stretch of in_count values to out_count
// (linear_stretch_functor, src/kernels.cu:1015-1016): float / float.
__host__ __device__ inline float stretch_step(uint64_t in_count, uint64_t out_count) {
  return (float)(in_count - 1) / (float)(out_count - 1);
}

// zap_birdies_kernel (src/kernels.cu:1063-1084): bins
// [floor((f-w)/bw), ceil((f+w)/bw)) of a birdie, clamped to [0, nb-1), as
// [lo, hi); false when there are none (NaN included).  Computed in float as
// the reference does and clamped before any integer conversion.
__device__ inline bool zap_range(float f, float w, float bin_width, uint64_t nb, uint64_t& lo, uint64_t& hi) {
  const double lo_f = (double)floorf((f - w) / bin_width);
  const double hi_f = (double)ceilf((f + w) / bin_width);
  if (!(lo_f < (double)nb)) return false;
  lo = lo_f > 0.0 ? (uint64_t)lo_f : 0;
  hi = hi_f >= (double)(nb - 1) ? nb - 1 : (hi_f > 0.0 ? (uint64_t)hi_f : 0);
  return lo < hi;
}

// Scale of fold K's running sum (1-based): times 2^-K/2, computed in double
// for odd K as the reference does (src/kernels.cu:38-98).  Host and device
// round every step alike (IEEE multiply and conversion, nearest even).
template <int K>
__host__ __device__ inline float fold_scale(float val) {
  if constexpr (K == 1) return (float)((double)val * 0.70710678118654752440);
  else if constexpr (K == 2) return val * 0.5f;
  else if constexpr (K == 3) return (float)((double)val * 0.35355339059327376220);
  else if constexpr (K == 4) return val * 0.25f;
  else return (float)((double)val * 0.17677669529663688110);
}

// harmonic_sum_kernel (src/kernels.cu:38-98).  Fold k adds the bins
// (int)(i*j/2^(k+1) + 0.5) for odd j, in the order the reference lists them
// (fold 1 adds 3/4 before 1/4), to one running float sum, and stores the
// running sum times 2^-(k+1)/2 computed in double.
template <int NF>
__device__ inline void harmonic_sums(const float* __restrict__ P, uint64_t i, float (&s)[5]) {
  float val = P[i];
  if (NF > 0) {
    val += P[(i + 1) >> 1];
    s[0] = fold_scale<1>(val);
  }
  if (NF > 1) {
    val += P[(3 * i + 2) >> 2];
    val += P[(i + 2) >> 2];
    s[1] = fold_scale<2>(val);
  }
  if (NF > 2) {
#pragma unroll
    for (uint64_t j = 1; j < 8; j += 2) val += P[(j * i + 4) >> 3];
    s[2] = fold_scale<3>(val);
  }
  if (NF > 3) {
#pragma unroll
    for (uint64_t j = 1; j < 16; j += 2) val += P[(j * i + 8) >> 4];
    s[3] = fold_scale<4>(val);
  }
  if (NF > 4) {
#pragma unroll
    for (uint64_t j = 1; j < 32; j += 2) val += P[(j * i + 16) >> 5];
    s[4] = fold_scale<5>(val);
  }
}

// The same sums with 32-bit bin arithmetic (valid for i < 2^27, where every
// j*i + 2^(m-1) fits in 32 bits).
template <int NF>
__device__ inline void harmonic_sums32(const float* __restrict__ P, uint32_t i, float (&s)[5]) {
  float val = P[i];
  if (NF > 0) {
    val += P[(i + 1) >> 1];
    s[0] = fold_scale<1>(val);
  }
  if (NF > 1) {
    val += P[(3 * i + 2) >> 2];
    val += P[(i + 2) >> 2];
    s[1] = fold_scale<2>(val);
  }
  if (NF > 2) {
#pragma unroll
    for (uint32_t j = 1; j < 8; j += 2) val += P[(j * i + 4) >> 3];
    s[2] = fold_scale<3>(val);
  }
  if (NF > 3) {
#pragma unroll
    for (uint32_t j = 1; j < 16; j += 2) val += P[(j * i + 8) >> 4];
    s[3] = fold_scale<4>(val);
  }
  if (NF > 4) {
#pragma unroll
    for (uint32_t j = 1; j < 32; j += 2) val += P[(j * i + 16) >> 5];
    s[4] = fold_scale<5>(val);
  }
}

// The same sums for D bins per lane: lane l of a wave holds the bins i0 + 64d,
// i0 = base + l.  Fold k's harmonic j of bin i is bin (j*i + 2^(k-1)) >> k, and
// with i = i0 + 64d that is ((j*i0 + 2^(k-1)) >> k) + d*64j/2^k exactly (2^k
// divides 64), so each harmonic costs one index per lane and D loads at
// constant instruction offsets from it: the gathers stay coalesced across
// lanes and the index arithmetic drops out of the loop.  val takes the same
// addends in the same order as harmonic_sums32 (bins below 2^27).
//
// Harmonics at 1/16 of the bin or less (step <= 4) touch only D*step + 1
// consecutive bins per wave, fewer than 64: the wave loads them once (one
// load per lane) and each d takes its value from the owning lane with
// ds_bpermute, instead of D loads of a few distinct floats each (2% faster
// batched harmonic pass).  The values are the same bins, so the sums are unchanged.
template <int K, int J, int D>
__device__ inline void add_harmonic(const PSX_GLOBAL float* p, uint32_t i0, float (&val)[D]) {
  constexpr uint32_t step = (64u * J) >> K;
  constexpr uint32_t c = 1u << (K - 1);
  if constexpr (step <= 4 && D * step + 1 < 64) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t s0 = (J * (i0 - lane) + c) >> K;  // the wave's first bin of this harmonic
    const uint32_t r = ((J * i0 + c) >> K) - s0;     // this lane's offset, <= step
    const float chunk = p[s0 + lane];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int addr = (int)((r + (uint32_t)d * step) << 2);
      val[d] += __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(chunk)));
    }
  } else {
    const PSX_GLOBAL float* q = p + ((J * i0 + c) >> K);
#pragma unroll
    for (int d = 0; d < D; ++d) val[d] += q[d * step];
  }
}
// odd harmonics J, J+2, ... below JEND of fold K, in increasing order
template <int K, int J, int JEND, int D>
__device__ inline void add_harmonics(const PSX_GLOBAL float* p, uint32_t i0, float (&val)[D]) {
  add_harmonic<K, J, D>(p, i0, val);
  if constexpr (J + 2 < JEND) add_harmonics<K, J + 2, JEND, D>(p, i0, val);
}
// Number of set bits of mask in the lanes below the calling lane (wave64).
__device__ inline unsigned mbcnt64(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

}  // namespace psx
