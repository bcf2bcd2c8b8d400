// prologue.hip - fused DM prologues of the batched search (gfx950).
//
// The Worker's prologue (pipeline_multi.cu:170-238) is some 36 small launches
// per DM when each library call is its own kernel, which for the short series
// of segmented searches costs several times their few acceleration trials
// (64 DMs of 2^20 samples: 7.5 of 10.3 ms; in groups of 16 DMs 1.3 of 3.2 ms).
// Here a group of DMs takes twelve:
//   k_base_sum, k_base_step  (twice) the baseline loop's means
//   k_base_apply             series - means, zero padded
//   (R2C passes)             half-length spectra Z of all DMs of the group
//   k_median                 untangle + amplitude + the three scrunches
//   k_deredden               untangle + stretched median + divide + zap +
//                            interbin sums + the C2R's input
//   k_stats                  the sums of each DM
//   (C2R passes)             dereddened series
// Each value is computed with the per-stage kernels' expressions
// (kernels_dev.hpp, fft_plan.hpp), so the series equal the Worker's bit for
// bit; the sums of the interbinned spectrum are taken in double in another
// order and rounded to float as psx_mean_rms does.  All passes stream:
// k_median reads Z twice over (each bin and its mirror), k_deredden once.
#include "prologue.hpp"

#include <algorithm>

#include "common.hpp"
#include "kernels_dev.hpp"

using namespace psx::fft;

namespace psx {
namespace prologue {
namespace {

constexpr unsigned kB = 256;
constexpr unsigned kSumBlocks = 1024;  // as psx_mean_rms's first level: the same order of additions
constexpr unsigned kSpecBlocks = 1024;
constexpr unsigned kPartials = kSumBlocks > kSpecBlocks ? kSumBlocks : kSpecBlocks;

__device__ inline double block_sum(double s, double (&r)[kB]) {
  r[threadIdx.x] = s;
  __syncthreads();
  for (unsigned o = kB / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) r[threadIdx.x] += r[threadIdx.x + o];
    __syncthreads();
  }
  return r[0];
}

// Sum of trial blockIdx.y after the loop's first STEP - 1 subtractions.
template <int STEP>
__global__ void __launch_bounds__(kB) k_base_sum(const float* src, int64_t tstride, uint64_t n,
                                                 const Result* __restrict__ res, double2* __restrict__ partial) {
  const uint32_t d = blockIdx.y;
  float m0 = 0.f;
  if constexpr (STEP > 1) {
    if (res[d].base.done) return;
    m0 = res[d].base.mean[0];
  }
  const float* x = src + (int64_t)d * tstride;
  double s = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * kB;
#pragma unroll 4
  for (uint64_t i = (uint64_t)blockIdx.x * kB + threadIdx.x; i < n; i += stride) {
    float v = x[i];
    if constexpr (STEP > 1) v -= m0;
    s += (double)v;
  }
  __shared__ double r[kB];
  s = block_sum(s, r);
  if (threadIdx.x == 0) partial[(uint64_t)d * kPartials + blockIdx.x].x = s;
}

// do { mean; subtract; if (count++ > 100) break; } while (fabsf(mean) > 5e-7 * (double)n);
template <int STEP>
__global__ void __launch_bounds__(kB) k_base_step(const double2* __restrict__ partial, unsigned np, uint64_t n,
                                                  Result* __restrict__ res) {
  const uint32_t d = blockIdx.x;
  if (STEP > 1 && res[d].base.done) return;
  double s = 0.0;
  for (unsigned i = threadIdx.x; i < np; i += kB) s += partial[(uint64_t)d * kPartials + i].x;
  __shared__ double r[kB];
  s = block_sum(s, r);
  if (threadIdx.x == 0) {
    const float mean = (float)s / (float)(int64_t)n;
    res[d].base.mean[STEP - 1] = mean;
    res[d].base.count = STEP;
    res[d].base.done = (double)fabsf(mean) > 5e-7 * (double)n ? 0 : 1;
  }
}

typedef float psx_f4 __attribute__((ext_vector_type(4), aligned(4)));

// src may be tim (same stride): each thread reads what it writes.
__global__ void __launch_bounds__(kB) k_base_apply(const float* src, int64_t tstride, uint64_t nreal, float* tim,
                                                   uint64_t n, const Result* __restrict__ res) {
  const uint32_t d = blockIdx.y;
  const BaselineState st = res[d].base;
  const float* x = src + (int64_t)d * tstride;
  float* y = tim + (int64_t)d * (int64_t)n;
  const float m0 = st.mean[0], m1 = st.count > 1 ? st.mean[1] : 0.f;
  const uint64_t stride = (uint64_t)gridDim.x * kB;
  // n is even and at least 64; four samples per thread, n - 2 is the last pair
  for (uint64_t q = (uint64_t)blockIdx.x * kB + threadIdx.x; 4 * q < n; q += stride) {
    const uint64_t i = 4 * q;
    if (i + 4 <= nreal) {
      psx_f4 v = *(const PSX_GLOBAL psx_f4*)(x + i);
      v -= m0;
      if (st.count > 1) v -= m1;
      *(PSX_GLOBAL psx_f4*)(y + i) = v;
    } else {
      for (uint64_t j = i; j < i + 4 && j < n; ++j) {
        float v = 0.f;
        if (j < nreal) {
          v = x[j] - m0;
          if (st.count > 1) v -= m1;
        }
        y[j] = v;
      }
    }
  }
}

__global__ void __launch_bounds__(kB) k_mask_clear(uint32_t* __restrict__ mask, uint32_t words) {
  const uint32_t i = blockIdx.x * kB + threadIdx.x;
  if (i < words) mask[i] = 0u;
}

// One block per birdie; k_zap's bins (kernels.hip) as bits.
__global__ void __launch_bounds__(kB) k_mask(uint32_t* __restrict__ mask, const float* __restrict__ freqs,
                                             const float* __restrict__ widths, float bin_width, uint64_t nb) {
  uint64_t lo, hi;
  if (!psx::zap_range(freqs[blockIdx.x], widths[blockIdx.x], bin_width, nb, lo, hi)) return;
  for (uint64_t w = lo / 32 + threadIdx.x; 32 * w < hi; w += kB) {
    const uint64_t a = max(lo, 32 * w), b = min(hi, 32 * w + 32);
    if (a >= b) continue;
    const uint32_t bits = (uint32_t)(((1ull << (b - a)) - 1) << (a - 32 * w));
    atomicOr(&mask[w], bits);
  }
}

// X[k] of the untangled spectrum, k in [0, M], as the untangle pass computes it.
__device__ inline float2 bin_of(const float2* z, uint32_t M, uint32_t k, const RootTable& rt) {
  if (k == M) return untangle_one(ldg2(z, 0), ldg2(z, 0), make_float2(-1.f, 0.f));
  const float2 zk = ldg2(z, k), zm = ldg2(z, k == 0 ? 0 : M - k);
  if (2 * k <= M) return untangle_one(zk, zm, root32(rt, k));
  const float2 w = root32(rt, M - k);
  return untangle_one(zk, zm, make_float2(-w.x, w.y));
}

// Amplitudes (form_power_series way 0, src/kernels.cu:216-234) and the three
// median scrunches (src/kernels.cu:961-972) of kM125 * 125 bins per
// workgroup; the amplitudes live in LDS only.
constexpr uint32_t kM125 = 16;

__global__ void __launch_bounds__(kB) k_median(const float2* __restrict__ Z, uint32_t M, RootTable rt,
                                               float* __restrict__ med, uint64_t med_stride, uint32_t c5, uint32_t c25,
                                               uint32_t c125) {
  __shared__ float a[125 * kM125], s5[25 * kM125], s25[5 * kM125];
  const uint32_t d = blockIdx.y, b = blockIdx.x;
  const float2* z = Z + (uint64_t)d * M;
  float* m5 = med + (uint64_t)d * med_stride;
  float* m25 = m5 + c5;
  float* m125 = m25 + c25;
  const uint32_t k0 = b * 125 * kM125;
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < 125 * kM125; i += kB) {
    float v = 0.f;
    if (k0 + i < 5 * c5) {
      const float2 x = bin_of(z, M, k0 + i, rt);
      v = sqrtf(fmaf(x.x, x.x, x.y * x.y));
    }
    a[i] = v;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < 25 * kM125; i += kB) {
    const float* p = a + 5 * i;
    const float v = psx::median5(p[0], p[1], p[2], p[3], p[4]);
    s5[i] = v;
    if (b * 25 * kM125 + i < c5) m5[b * 25 * kM125 + i] = v;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < 5 * kM125; i += kB) {
    const float* p = s5 + 5 * i;
    const float v = psx::median5(p[0], p[1], p[2], p[3], p[4]);
    s25[i] = v;
    if (b * 5 * kM125 + i < c25) m25[b * 5 * kM125 + i] = v;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kM125; i += kB) {
    const float* p = s25 + 5 * i;
    if (b * kM125 + i < c125) m125[b * kM125 + i] = psx::median5(p[0], p[1], p[2], p[3], p[4]);
  }
}

// The stretched running median (Dereddener::calculate_median,
// dereddener.hpp:41-62): zone [0, z1) from m5, [z1, z2) from m25, the rest
// from m125.
struct Zones {
  uint32_t z1, z2;
  uint32_t c5, c25, c125;
  float step5, step25, step125;
};
__device__ inline float median_at(const float* m5, const Zones& zn, uint32_t i) {
  const float* m = m5;
  uint32_t cnt = zn.c5;
  float step = zn.step5;
  if (i >= zn.z1) {
    m += zn.c5;
    cnt = zn.c25;
    step = zn.step25;
    if (i >= zn.z2) {
      m += zn.c25;
      cnt = zn.c125;
      step = zn.step125;
    }
  }
  return psx::stretch_at(m, cnt, i, step);
}

__device__ inline float2 shfl_f2(float2 v, int src) { return make_float2(__shfl(v.x, src), __shfl(v.y, src)); }

// A wave holds the 64 pairs (k, M-k), k = kw-1 .. kw+62, one per lane, and
// takes the interbin neighbours X[k-1] and X[M-k-1] from the adjacent lanes
// (the layout of the batched search's natural-order spectrum pass); waves
// advance by 63 pairs.  Nothing but W and the sums is written: the dereddened
// spectrum itself is only the C2R's input.
constexpr uint32_t kStep = 63;

template <bool ZAP>
__global__ void __launch_bounds__(kB) k_deredden(const float2* __restrict__ Z, float2* __restrict__ W, uint32_t M,
                                                 RootTable rt, const float* __restrict__ med, uint64_t med_stride,
                                                 Zones zn, const uint32_t* __restrict__ zmask,
                                                 double2* __restrict__ partial) {
  const uint32_t d = blockIdx.y, half = M / 2;
  const float2* z = Z + (uint64_t)d * M;
  float2* w = W + (uint64_t)d * M;
  const float* m5 = med + (uint64_t)d * med_stride;
  const int lane = (int)(threadIdx.x & 63u);
  const uint32_t nchunks = (half + kStep) / kStep;
  auto deredden = [&](float2 x, uint32_t k) {
    if (k < 5) {
      x = make_float2(0.f, 0.f);
    } else {
      const float f = median_at(m5, zn, k);
      x.x = x.x / f;
      x.y = x.y / f;
    }
    if constexpr (ZAP)
      if ((zmask[k >> 5] >> (k & 31u)) & 1u) x = make_float2(1.f, 0.f);
    return x;
  };
  double s1 = 0.0, s2 = 0.0;
  for (uint32_t c = blockIdx.x * (kB / 64) + (threadIdx.x >> 6); c < nchunks; c += gridDim.x * (kB / 64)) {
    const int32_t ks = (int32_t)(c * kStep) + lane - 1;
    const bool valid = ks >= 0 && (uint32_t)ks <= half;
    const uint32_t k = valid ? (uint32_t)ks : 0u;
    float2 xl = make_float2(0.f, 0.f), xu = make_float2(0.f, 0.f), wk = make_float2(0.f, 0.f);
    if (valid) {
      const float2 zk = ldg2(z, k), zm = ldg2(z, k == 0 ? 0 : M - k);
      wk = root32(rt, k);
      xl = deredden(untangle_one(zk, zm, wk), k);
      // the midpoint is its own mirror and keeps the lower formula
      xu = k == half ? xl : deredden(untangle_one(zm, zk, make_float2(-wk.x, wk.y)), M - k);
    }
    const float2 xl_prev = shfl_f2(xl, lane > 0 ? lane - 1 : 0);
    const float2 xu_next = shfl_f2(xu, lane < 63 ? lane + 1 : 63);
    if (valid && lane > 0) {
      const float v = psx::interbin(xl, xl_prev);
      const float sq = v * v;
      s1 += (double)v;
      s2 += (double)sq;
      stg2(w, k, tangle_one(xl, xu, wk));
    }
    if (valid && lane < 63 && k < half) {
      const float v = psx::interbin(xu, xu_next);
      const float sq = v * v;
      s1 += (double)v;
      s2 += (double)sq;
      if (k > 0) stg2(w, M - k, tangle_one(xu, xl, root32(rt, M - k)));
    }
  }
  __shared__ double r[kB];
  s1 = block_sum(s1, r);
  __syncthreads();
  s2 = block_sum(s2, r);
  if (threadIdx.x == 0) partial[(uint64_t)d * kPartials + blockIdx.x] = make_double2(s1, s2);
}

__global__ void __launch_bounds__(kB) k_stats(const double2* __restrict__ partial, unsigned np,
                                              Result* __restrict__ res) {
  const uint32_t d = blockIdx.x;
  double s1 = 0.0, s2 = 0.0;
  for (unsigned i = threadIdx.x; i < np; i += kB) {
    const double2 p = partial[(uint64_t)d * kPartials + i];
    s1 += p.x;
    s2 += p.y;
  }
  __shared__ double r[kB];
  s1 = block_sum(s1, r);
  __syncthreads();
  s2 = block_sum(s2, r);
  if (threadIdx.x == 0) res[d].sums = make_double2(s1, s2);
}

}  // namespace

uint64_t work_bytes(uint64_t n, uint32_t G) {
  const uint64_t nb = n / 2 + 1, c5 = nb / 5;
  return G * ((c5 + c5 / 5 + c5 / 25) * sizeof(float) + kPartials * sizeof(double2) + sizeof(Result)) + nb / 8 + 1024;
}

int work_create(uint64_t n, uint32_t G, Work& w) {
  w = Work();
  w.n = n;
  w.M = n / 2;
  w.G = G;
  const uint64_t nb = n / 2 + 1;
  w.c5 = nb / 5;
  w.c25 = w.c5 / 5;
  w.c125 = w.c25 / 5;
  w.med_stride = w.c5 + w.c25 + w.c125;
  PSX_CHECK_HIP(psx::device_malloc((void**)&w.med, std::max<uint64_t>(1, G * w.med_stride) * sizeof(float)));
  PSX_CHECK_HIP(psx::device_malloc((void**)&w.partial, (uint64_t)G * kPartials * sizeof(double2)));
  PSX_CHECK_HIP(psx::device_malloc((void**)&w.res, G * sizeof(Result)));
  PSX_CHECK_HIP(psx::device_malloc((void**)&w.zmask, (nb / 32 + 1) * sizeof(uint32_t)));
  return PSX_OK;
}

void work_destroy(Work& w) {
  (void)hipFree(w.med);
  (void)hipFree(w.partial);
  (void)hipFree(w.res);
  (void)hipFree(w.zmask);
  w = Work();
}

int baseline(const Work& w, const float* src, int64_t stride, uint64_t nreal, float* tim, uint32_t ndm,
             hipStream_t s) {
  PSX_REQUIRE(src && tim && nreal > 0 && nreal <= w.n && ndm >= 1 && ndm <= w.G, "prologue: bad baseline arguments");
  const unsigned g = psx::grid_for(nreal, kB, kSumBlocks);
  k_base_sum<1><<<dim3(g, ndm), kB, 0, s>>>(src, stride, nreal, w.res, w.partial);
  PSX_CHECK_LAUNCH("k_base_sum");
  k_base_step<1><<<ndm, kB, 0, s>>>(w.partial, g, nreal, w.res);
  PSX_CHECK_LAUNCH("k_base_step");
  static_assert(kBaselineSteps == 2, "the launches below");
  k_base_sum<2><<<dim3(g, ndm), kB, 0, s>>>(src, stride, nreal, w.res, w.partial);
  PSX_CHECK_LAUNCH("k_base_sum");
  k_base_step<2><<<ndm, kB, 0, s>>>(w.partial, g, nreal, w.res);
  PSX_CHECK_LAUNCH("k_base_step");
  k_base_apply<<<dim3(psx::grid_for(w.n / 4, kB, 2048), ndm), kB, 0, s>>>(src, stride, nreal, tim, w.n, w.res);
  PSX_CHECK_LAUNCH("k_base_apply");
  return PSX_OK;
}

int zap_mask(const Work& w, const float* d_freqs, const float* d_widths, uint32_t nbirdies, float bin_width,
             hipStream_t s) {
  PSX_REQUIRE(d_freqs && d_widths && nbirdies >= 1 && nbirdies <= 0x7FFFFFFFu && bin_width > 0,
              "prologue: bad zap list");
  const uint64_t nb = w.M + 1;
  const uint32_t words = (uint32_t)(nb / 32 + 1);
  k_mask_clear<<<(words + kB - 1) / kB, kB, 0, s>>>(w.zmask, words);
  PSX_CHECK_LAUNCH("k_mask_clear");
  k_mask<<<nbirdies, kB, 0, s>>>(w.zmask, d_freqs, d_widths, bin_width, nb);
  PSX_CHECK_LAUNCH("k_mask");
  return PSX_OK;
}

int spectra(const Work& w, const float2* Z, float2* W, const RootTable& rt, double bin_width, float b5, float b25,
            bool zap, uint32_t ndm, hipStream_t s) {
  PSX_REQUIRE(Z && W && bin_width > 0 && ndm >= 1 && ndm <= w.G, "prologue: bad spectrum arguments");
  const uint64_t nb = w.M + 1;
  PSX_REQUIRE(w.c125 >= 1 && w.M % 2 == 0 && w.M < (1ull << 28), "psx_deredden_median: nb too small (%llu)",
              (unsigned long long)nb);
  const uint32_t M = (uint32_t)w.M;
  const unsigned mblocks = (unsigned)((w.c5 + 25 * kM125 - 1) / (25 * kM125));
  k_median<<<dim3(mblocks, ndm), kB, 0, s>>>(Z, M, rt, w.med, w.med_stride, (uint32_t)w.c5, (uint32_t)w.c25,
                                             (uint32_t)w.c125);
  PSX_CHECK_LAUNCH("k_median");
  auto clampz = [&](float b) -> uint32_t {
    const int64_t v = (int64_t)(int)((double)b / bin_width);
    return (uint32_t)(v < 0 ? 0 : (v > (int64_t)nb ? nb : (uint64_t)v));
  };
  Zones zn;
  zn.z1 = clampz(b5);
  zn.z2 = std::max(zn.z1, clampz(b25));
  zn.c5 = (uint32_t)w.c5;
  zn.c25 = (uint32_t)w.c25;
  zn.c125 = (uint32_t)w.c125;
  zn.step5 = psx::stretch_step(w.c5, nb);
  zn.step25 = psx::stretch_step(w.c25, nb);
  zn.step125 = psx::stretch_step(w.c125, nb);
  const uint64_t chunks = (w.M / 2 + kStep) / kStep;
  const unsigned g = psx::grid_for(chunks, kB / 64, kSpecBlocks);
  if (zap)
    k_deredden<true><<<dim3(g, ndm), kB, 0, s>>>(Z, W, M, rt, w.med, w.med_stride, zn, w.zmask, w.partial);
  else
    k_deredden<false><<<dim3(g, ndm), kB, 0, s>>>(Z, W, M, rt, w.med, w.med_stride, zn, w.zmask, w.partial);
  PSX_CHECK_LAUNCH("k_deredden");
  k_stats<<<ndm, kB, 0, s>>>(w.partial, g, w.res);
  PSX_CHECK_LAUNCH("k_stats");
  return PSX_OK;
}

}  // namespace prologue
}  // namespace psx
