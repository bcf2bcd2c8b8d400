// kernels.hip - per-stage kernels of the acceleration-search core for gfx950.
//
// One entry point per function of the reference's kernel layer
// (include/kernels/kernels.h); each kernel cites the reference kernel whose
// arithmetic it reproduces.  All elementwise stages are HBM-bound: they use
// 16-byte vector accesses where the layout allows and grid-stride loops sized
// to keep every CU busy.  Device code is compiled with -ffp-contract=off; the
// multiply-adds that the reference's nvcc build contracts are written as
// explicit fma so that results match the CPU restatement bit for bit.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "common.hpp"
#include "kernels_dev.hpp"
#include "trace.hpp"

using psx::as_stream;

namespace {

constexpr unsigned kBlock = 256;

// ---------------------------------------------------------------- resample
// resample_kernelII (src/kernels.cu:342-353): out[i] = in[rn(fma(i*af, i-n, i))].
__global__ void __launch_bounds__(kBlock) k_resample2(const float* __restrict__ in, float* __restrict__ out,
                                                      uint64_t n, double af) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t n4 = n / 4;
  for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n4; q += stride) {
    float4 r;
    r.x = in[psx::resample_index(4 * q + 0, n, af)];
    r.y = in[psx::resample_index(4 * q + 1, n, af)];
    r.z = in[psx::resample_index(4 * q + 2, n, af)];
    r.w = in[psx::resample_index(4 * q + 3, n, af)];
    reinterpret_cast<float4*>(out)[q] = r;
  }
  for (uint64_t i = 4 * n4 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = in[psx::resample_index(i, n, af)];
}

// resample_kernel (src/kernels.cu:327-339): id + af*((id-n/2)^2 - (n/2)^2),
// contracted as fma(af, fma(t, t, -(h*h)), id).
__global__ void __launch_bounds__(kBlock) k_resample1(const float* __restrict__ in, float* __restrict__ out,
                                                      uint64_t n, double af) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const double h = (double)n / 2.0;
  const double hh = h * h;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const double di = (double)i;
    const double t = di - h;
    const double q = fma(t, t, -hh);
    uint64_t j = (uint64_t)rint(fma(af, q, di));
    j = j < n ? j : n - 1;
    out[i] = in[j];
  }
}

// ---------------------------------------------------------- spectrum forming
// power_series_kernel (src/kernels.cu:216-234): |X|, 0 where |X|^2 == 0.
__global__ void __launch_bounds__(kBlock) k_amplitude(const float2* __restrict__ X, float* __restrict__ A,
                                                      uint64_t nb) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nb; i += stride) {
    const float2 x = X[i];
    const float z = fmaf(x.x, x.x, x.y * x.y);
    A[i] = (z == 0.0f) ? 0.0f : sqrtf(z);
  }
}

// bin_interbin_series_kernel (src/kernels.cu:238-259): two bins per thread,
// one 16-byte load for the pair plus the preceding bin.
__global__ void __launch_bounds__(kBlock) k_interbin(const float2* __restrict__ X, float* __restrict__ A,
                                                     uint64_t nb) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t npair = nb / 2;
  for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q < npair; q += stride) {
    const float4 cur = reinterpret_cast<const float4*>(X)[q];
    const float2 prev = q > 0 ? X[2 * q - 1] : make_float2(0.f, 0.f);
    float2 o;
    o.x = psx::interbin(make_float2(cur.x, cur.y), prev);
    o.y = psx::interbin(make_float2(cur.z, cur.w), make_float2(cur.x, cur.y));
    reinterpret_cast<float2*>(A)[q] = o;
  }
  if (nb & 1) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      const uint64_t k = nb - 1;
      A[k] = psx::interbin(X[k], k > 0 ? X[k - 1] : make_float2(0.f, 0.f));
    }
  }
}

// ------------------------------------------------------------- dereddening
// median_scrunch5_kernel (src/kernels.cu:961-972).
__global__ void __launch_bounds__(kBlock) k_scrunch5(const float* __restrict__ in, float* __restrict__ out,
                                                     uint64_t oc) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < oc; i += stride) {
    const float* p = in + 5 * i;
    out[i] = psx::median5(p[0], p[1], p[2], p[3], p[4]);
  }
}

// median_scrunch5 special cases count = 1..4 (src/kernels.cu:981-997).
__global__ void k_scrunch_small(const float* __restrict__ in, float* __restrict__ out, int count) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  if (count == 1) out[0] = in[0];
  else if (count == 2) out[0] = 0.5f * (in[0] + in[1]);
  else if (count == 3) out[0] = psx::median3(in[0], in[1], in[2]);
  else out[0] = psx::median4(in[0], in[1], in[2], in[3]);
}

// linear_stretch_functor (src/kernels.cu:1010-1024).  step is computed on
// the host in float as the reference does.
__global__ void __launch_bounds__(kBlock) k_stretch(const float* __restrict__ in, uint64_t in_count,
                                                    float* __restrict__ out, uint64_t out_count, float step) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < out_count; i += stride)
    out[i] = psx::stretch_at(in, in_count, (unsigned)i, step);
}

// The three scrunches of Dereddener::calculate_median (dereddener.hpp:41-52)
// in one launch: a workgroup stages 125 * kM125 bins in LDS and scrunches them
// to 5, 25 and 125 bins (2^21 bins: 5.8 us, three launches 8.3 us and their
// gaps).
constexpr uint32_t kM125 = 16;

__global__ void __launch_bounds__(kBlock) k_scrunch125(const float* __restrict__ in, float* __restrict__ m5,
                                                       float* __restrict__ m25, float* __restrict__ m125, uint64_t c5,
                                                       uint64_t c25, uint64_t c125) {
  __shared__ float a[125 * kM125], s5[25 * kM125], s25[5 * kM125];
  const uint64_t b = blockIdx.x;
  const float* p = in + b * 125 * kM125;
  const uint64_t left = 5 * c5 - b * 125 * kM125;
#pragma unroll
  for (uint32_t i = threadIdx.x; i < 125 * kM125; i += kBlock) a[i] = i < left ? p[i] : 0.f;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < 25 * kM125; i += kBlock) {
    const float* q = a + 5 * i;
    s5[i] = psx::median5(q[0], q[1], q[2], q[3], q[4]);
    if (b * 25 * kM125 + i < c5) m5[b * 25 * kM125 + i] = s5[i];
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < 5 * kM125; i += kBlock) {
    const float* q = s5 + 5 * i;
    s25[i] = psx::median5(q[0], q[1], q[2], q[3], q[4]);
    if (b * 5 * kM125 + i < c25) m25[b * 5 * kM125 + i] = s25[i];
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kM125; i += kBlock) {
    const float* q = s25 + 5 * i;
    if (b * kM125 + i < c125) m125[b * kM125 + i] = psx::median5(q[0], q[1], q[2], q[3], q[4]);
  }
}

// Dereddener::calculate_median zone copies (dereddener.hpp:53-61) in one
// launch: the third zone, from z2, overwrites the others, the first ends at
// z1, the second at hi; bins of no zone are left as they are.
struct Stretch {
  const float* in;
  uint64_t count;
  float step;
};
__global__ void __launch_bounds__(kBlock) k_stretch_zones(Stretch s5, Stretch s25, Stretch s125, uint64_t z1,
                                                          uint64_t hi, uint64_t z2, float* __restrict__ out,
                                                          uint64_t nb) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nb; i += stride) {
    const Stretch& s = i >= z2 ? s125 : (i < z1 ? s5 : s25);
    if (i < z2 && i >= z1 && i >= hi) continue;
    out[i] = psx::stretch_at(s.in, s.count, (unsigned)i, s.step);
  }
}

// divide_c_by_f_kernel (src/kernels.cu:1040-1049).
__global__ void __launch_bounds__(kBlock) k_divide(float2* __restrict__ X, const float* __restrict__ f,
                                                   uint64_t nb) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nb; i += stride) {
    float2 x = X[i];
    if (i < 5) {
      x = make_float2(0.f, 0.f);
    } else {
      const float d = f[i];
      x.x = x.x / d;
      x.y = x.y / d;
    }
    X[i] = x;
  }
}

// zap_birdies_kernel (src/kernels.cu:1063-1084): each birdie's bins
// (zap_range) become 1+0i.  One block per birdie.
__global__ void __launch_bounds__(kBlock) k_zap(float2* __restrict__ X, const float* __restrict__ freqs,
                                                const float* __restrict__ widths, float bin_width, uint64_t nb) {
  uint64_t lo, hi;
  if (!psx::zap_range(freqs[blockIdx.x], widths[blockIdx.x], bin_width, nb, lo, hi)) return;
  for (uint64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) X[i] = make_float2(1.0f, 0.0f);
}

// --------------------------------------------------------------- reductions
// Deterministic two-level sum of x and of float(x*x) in double (GPU_mean /
// GPU_rms, src/kernels.cu:433-461, accumulate float terms in float).
constexpr unsigned kReduceBlocks = 1024;

// The workgroup's sums in thread 0: halving tree, its first two levels
// through LDS and the rest inside wave 0.
__device__ inline double2 block_sum2(double s1, double s2) {
  __shared__ double r1[kBlock], r2[kBlock];
  const unsigned t = threadIdx.x;
  r1[t] = s1;
  r2[t] = s2;
  __syncthreads();
  if (t < 64) {
    static_assert(kBlock == 256, "two LDS levels");
    s1 = (r1[t] + r1[t + 128]) + (r1[t + 64] + r1[t + 192]);
    s2 = (r2[t] + r2[t + 128]) + (r2[t + 64] + r2[t + 192]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      s1 += __shfl_down(s1, o);
      s2 += __shfl_down(s2, o);
    }
  }
  return make_double2(s1, s2);
}

__global__ void __launch_bounds__(kBlock) k_sum_sq(const float* __restrict__ x, uint64_t first, uint64_t n,
                                                   double2* __restrict__ partial) {
  double s1 = 0.0, s2 = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
#pragma unroll 8
  for (uint64_t i = first + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float v = x[i];
    const float sq = v * v;
    s1 += (double)v;
    s2 += (double)sq;
  }
  const double2 s = block_sum2(s1, s2);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// The partial sums' total, in thread 0 of the calling workgroup.
__device__ inline double2 sum_partials(const double2* __restrict__ partial, unsigned np) {
  double s1 = 0.0, s2 = 0.0;
#pragma unroll 4
  for (unsigned i = threadIdx.x; i < np; i += kBlock) {
    s1 += partial[i].x;
    s2 += partial[i].y;
  }
  return block_sum2(s1, s2);
}

__global__ void __launch_bounds__(kBlock) k_sum_final(const double2* __restrict__ partial, unsigned np,
                                                      double2* __restrict__ out) {
  const double2 s = sum_partials(partial, np);
  if (threadIdx.x == 0) out[0] = s;
}

// normalisation_kernel (src/kernels.cu:496-507).
__global__ void __launch_bounds__(kBlock) k_normalise(float* __restrict__ p, uint64_t n, float mean, float sigma) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t n4 = n / 4;
  for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n4; q += stride) {
    float4 v = reinterpret_cast<float4*>(p)[q];
    v.x = (v.x - mean) / sigma;
    v.y = (v.y - mean) / sigma;
    v.z = (v.z - mean) / sigma;
    v.w = (v.w - mean) / sigma;
    reinterpret_cast<float4*>(p)[q] = v;
  }
  for (uint64_t i = 4 * n4 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    p[i] = (p[i] - mean) / sigma;
}

// GPU_remove_baseline (src/kernels.cu:463-479) without a host round trip per
// iteration:
//   do { mean; x -= mean; if (count++ > 100) break; } while (fabsf(mean) > 5e-7 * (double)n);
// k_base_sum's partial sums are totalled by every workgroup of k_base_sub,
// which subtracts; its first one keeps the loop's state.  Once the loop has
// stopped, later iterations do nothing.  FIRST: the state is not read.
struct BaselineState {
  int32_t count;
  int32_t done;
};
template <bool FIRST>
__global__ void __launch_bounds__(kBlock) k_base_sum(const float* __restrict__ x, uint64_t n,
                                                     double2* __restrict__ partial,
                                                     const BaselineState* __restrict__ st) {
  if (!FIRST && st->done) return;
  double s = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
#pragma unroll 8
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) s += (double)x[i];
  s = block_sum2(s, 0.0).x;
  if (threadIdx.x == 0) partial[blockIdx.x].x = s;
}
// prev, next: the state before and after this iteration, in different places
// (workgroups that start late still read the one before).
template <bool FIRST>
__global__ void __launch_bounds__(kBlock) k_base_sub(float* __restrict__ x, uint64_t n,
                                                     const double2* __restrict__ partial, unsigned np,
                                                     const BaselineState* __restrict__ prev,
                                                     BaselineState* __restrict__ next) {
  BaselineState st{0, 0};
  if constexpr (!FIRST) {
    st = *prev;
    if (st.done) {
      if (blockIdx.x == 0 && threadIdx.x == 0) *next = st;
      return;
    }
  }
  __shared__ float shared_mean;
  const double s = sum_partials(partial, np).x;
  if (threadIdx.x == 0) {
    const float mean = (float)s / (float)(int64_t)n;
    shared_mean = mean;
    if (blockIdx.x == 0)
      *next = BaselineState{st.count + 1, (st.count > 100 || !((double)fabsf(mean) > 5e-7 * (double)n)) ? 1 : 0};
  }
  __syncthreads();
  const float mean = shared_mean;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
#pragma unroll 4
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) x[i] -= mean;
}

// GPU_fill (src/kernels.cu:482-488).
__global__ void __launch_bounds__(kBlock) k_fill(float* __restrict__ x, uint64_t start, uint64_t end, float v) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = start + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < end; i += stride) x[i] = v;
}

// conversion_kernel (src/kernels.cu:1171-1180).
template <class T>
__global__ void __launch_bounds__(kBlock) k_convert(const T* __restrict__ in, float* __restrict__ out, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = (float)in[i];
}

// ---------------------------------------------------------- harmonic summing
// harmonic_sum_kernel (src/kernels.cu:34-100): fold pointers are passed by
// value, so no pointer table crosses PCIe per call.
struct FoldPtrs {
  float* f[5];
};

// Stores fold K of the lane's bins.
template <int K, int D>
__device__ inline void store_fold(float* __restrict__ f, uint32_t i0, const float (&val)[D]) {
  PSX_GLOBAL float* q = (PSX_GLOBAL float*)f + i0;
#pragma unroll
  for (int d = 0; d < D; ++d) q[64 * d] = psx::fold_scale<K>(val[d]);
}

// A wave takes 64 * D consecutive bins through add_harmonic (nb <= 2^27);
// the last, partial stretch goes bin by bin.  Bound by the traffic behind the
// L2s: the folds' spans re-read the spectrum 8.5 times for four folds (each
// XCD's 4 MB L2 holds a quarter of 2^22 + 1 bins) beside the 67 MB written.
// 2^22 + 1 bins, four folds: 30.3 us with one bin per thread (64-bit indices),
// 25.7 us here with 2, 4 or 8 bins per lane; 2^19 + 1 bins, 5.6 us and 3.9
// (4.3 with 8 per lane).
constexpr int kHarmD = 4;
template <int NF>
__global__ void __launch_bounds__(kBlock) k_harmonic(const float* __restrict__ P, FoldPtrs folds, uint32_t nb) {
  constexpr uint32_t kWave = 64 * kHarmD;
  const PSX_GLOBAL float* p = (const PSX_GLOBAL float*)P;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t base = (blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * kWave;
  if (base >= nb) return;
  const uint32_t i0 = base + lane;
  if (base + kWave > nb) {
    for (uint32_t i = i0; i < nb; i += 64) {
      float s[5];
      psx::harmonic_sums32<NF>(P, i, s);
#pragma unroll
      for (int k = 0; k < NF; ++k) folds.f[k][i] = s[k];
    }
    return;
  }
  float val[kHarmD];
#pragma unroll
  for (int d = 0; d < kHarmD; ++d) val[d] = p[i0 + 64 * d];
  psx::add_harmonic<1, 1, kHarmD>(p, i0, val);
  store_fold<1>(folds.f[0], i0, val);
  if constexpr (NF > 1) {
    psx::add_harmonic<2, 3, kHarmD>(p, i0, val);  // 3/4 before 1/4, as the reference
    psx::add_harmonic<2, 1, kHarmD>(p, i0, val);
    store_fold<2>(folds.f[1], i0, val);
  }
  if constexpr (NF > 2) {
    psx::add_harmonics<3, 1, 8, kHarmD>(p, i0, val);
    store_fold<3>(folds.f[2], i0, val);
  }
  if constexpr (NF > 3) {
    psx::add_harmonics<4, 1, 16, kHarmD>(p, i0, val);
    store_fold<4>(folds.f[3], i0, val);
  }
  if constexpr (NF > 4) {
    psx::add_harmonics<5, 1, 32, kHarmD>(p, i0, val);
    store_fold<5>(folds.f[4], i0, val);
  }
}

// Spectra of more than 2^27 bins: 64-bit indices, one bin per thread.
template <int NF>
__global__ void __launch_bounds__(kBlock) k_harmonic_long(const float* __restrict__ P, FoldPtrs folds, uint64_t nb) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nb; i += stride) {
    float s[5];
    psx::harmonic_sums<NF>(P, i, s);
#pragma unroll
    for (int k = 0; k < NF; ++k) folds.f[k][i] = s[k];
  }
}

template <int NF>
void launch_harmonic(const float* P, const FoldPtrs& fp, uint64_t nb, hipStream_t s) {
  if (nb <= (1ull << 27)) {
    const uint64_t per = 64 * kHarmD * (kBlock / 64);
    k_harmonic<NF><<<(unsigned)((nb + per - 1) / per), kBlock, 0, s>>>(P, fp, (uint32_t)nb);
  } else {
    k_harmonic_long<NF><<<psx::grid_for(nb, kBlock), kBlock, 0, s>>>(P, fp, nb);
  }
}

// ------------------------------------------------------------- peak finding
// device_find_peaks (src/kernels.cu:391-423) as a two-kernel ordered
// compaction: per-tile counts, then each tile with survivors sums the counts
// of the tiles before it and writes them in index order (the last tile does
// so for the total).  Survivors are rare: the counting pass streams (16 bins
// per thread, all four loads in flight), and almost every workgroup of the
// writing pass ends at its count.  4.2 M bins: 7.1 + 8.3 us (one bin per load,
// every workgroup summing counts) -> 4.8 + 4.1 us.  A trial's five spectra go
// through one pair of launches (blockIdx.y: the spectrum): at 2^20 samples
// 5 x (3.4 + 2.7) us -> 4.1 + 3.7 us, and their counts and first pairs come
// back in one copy instead of up to three per spectrum.
constexpr unsigned kPeakTile = kBlock * 16;
typedef float psx_f4u __attribute__((ext_vector_type(4), aligned(4)));

// Bins 4*(thread + kBlock*r) .. + 3 of a tile that ends at bin n (< 4: some).
__device__ inline void peak_load(const float* tile, int64_t n, unsigned r, float thr, float (&v)[4], bool (&hit)[4]) {
  const int64_t at = 4 * (int64_t)(threadIdx.x + kBlock * r);
  if (at + 4 <= n) {
    const psx_f4u x = *(const PSX_GLOBAL psx_f4u*)((const PSX_GLOBAL float*)tile + at);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = x[j];
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = at + j < n ? tile[at + j] : thr;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) hit[j] = at + j < n && v[j] > thr;
}

// One spectrum alone has kernels of its own (NS = 1): with the arguments and
// the head of several, its pair of launches took 0.8 us more at 2^23 samples.
constexpr unsigned kPeakSpectra = PSX_PEAK_SPECTRA;
template <unsigned NS>
struct PeakJobs {
  const float* p[NS];
  int64_t start[NS], end[NS];
  uint32_t tiles[NS];
  uint32_t first[NS];  // first tile's place in the counts
};
// Pair i of spectrum y: lists idx and snr at y*cap + i (i < cap) and, where
// asked for, hidx and hsnr at y*nhead + i (i < nhead).
struct PeakOut {
  int32_t* idx;
  float* snr;
  uint32_t cap;
  uint32_t* total;
  int32_t* hidx;
  float* hsnr;
  uint32_t nhead;
};

template <unsigned NS>
__global__ void __launch_bounds__(kBlock) k_peak_count(const PeakJobs<NS> jobs, float thr,
                                                       uint32_t* __restrict__ all) {
  const unsigned y = NS == 1 ? 0 : blockIdx.y;
  if (blockIdx.x >= jobs.tiles[y]) return;
  const float* __restrict__ p = jobs.p[y];
  const int64_t start = jobs.start[y], end = jobs.end[y];
  uint32_t* __restrict__ counts = all + jobs.first[y];
  const int64_t base = start + (int64_t)blockIdx.x * kPeakTile;
  const int64_t n = min(end - base, (int64_t)kPeakTile);
  unsigned c = 0;
#pragma unroll
  for (unsigned r = 0; r < kPeakTile / (4 * kBlock); ++r) {
    float v[4];
    bool hit[4];
    peak_load(p + base, n, r, thr, v, hit);
#pragma unroll
    for (int j = 0; j < 4; ++j) c += (unsigned)__popcll(__ballot(hit[j]));
  }
  __shared__ unsigned wave_cnt[kBlock / 64];
  if ((threadIdx.x & 63u) == 0) wave_cnt[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned sum = 0;
#pragma unroll
    for (unsigned w = 0; w < kBlock / 64; ++w) sum += wave_cnt[w];
    counts[blockIdx.x] = sum;
  }
}

template <unsigned NS>
__global__ void __launch_bounds__(kBlock) k_peak_write(const PeakJobs<NS> jobs, float thr,
                                                       const uint32_t* __restrict__ all, const PeakOut out) {
  const unsigned y = NS == 1 ? 0 : blockIdx.y;
  const unsigned ntiles = jobs.tiles[y];
  if (blockIdx.x >= ntiles) {
    if (ntiles == 0 && blockIdx.x == 0 && threadIdx.x == 0) out.total[y] = 0;
    return;
  }
  const uint32_t* __restrict__ counts = all + jobs.first[y];
  const unsigned mine = counts[blockIdx.x];
  const bool last = blockIdx.x == ntiles - 1;
  if (mine == 0 && !last) return;
  __shared__ unsigned wave_cnt[kBlock / 64];
  const unsigned lane = threadIdx.x & 63u;
  const unsigned wave = threadIdx.x >> 6;
  // survivors of the tiles before this one
  unsigned pre = 0;
  for (unsigned t = threadIdx.x; t < blockIdx.x; t += kBlock) pre += counts[t];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) pre += __shfl_down(pre, o);
  if (lane == 0) wave_cnt[wave] = pre;
  __syncthreads();
  unsigned offset = 0;
#pragma unroll
  for (unsigned w = 0; w < kBlock / 64; ++w) offset += wave_cnt[w];
  if (last && threadIdx.x == 0) out.total[y] = offset + mine;
  if (mine == 0) return;
  const float* __restrict__ p = jobs.p[y];
  const int64_t start = jobs.start[y], end = jobs.end[y];
  const int64_t base = start + (int64_t)blockIdx.x * kPeakTile;
  const int64_t n = min(end - base, (int64_t)kPeakTile);
  for (unsigned r = 0; r < kPeakTile / (4 * kBlock); ++r) {
    float v[4];
    bool hit[4];
    peak_load(p + base, n, r, thr, v, hit);
    uint64_t mask[4];
    unsigned before = 0, wave_n = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      mask[j] = __ballot(hit[j]);
      before += psx::mbcnt64(mask[j]);  // the lower lanes' survivors
      wave_n += (unsigned)__popcll(mask[j]);
    }
    __syncthreads();
    if (lane == 0) wave_cnt[wave] = wave_n;
    __syncthreads();
    unsigned pos = offset + before;
#pragma unroll
    for (unsigned w = 0; w < kBlock / 64; ++w) {
      if (w < wave) pos += wave_cnt[w];
      offset += wave_cnt[w];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (hit[j]) {
        const int32_t idx = (int32_t)(base + 4 * (int64_t)(threadIdx.x + kBlock * r) + j);
        if (pos < out.cap) {
          out.idx[(uint64_t)y * out.cap + pos] = idx;
          out.snr[(uint64_t)y * out.cap + pos] = v[j];
        }
        if (NS > 1 && pos < out.nhead) {
          out.hidx[y * out.nhead + pos] = idx;
          out.hsnr[y * out.nhead + pos] = v[j];
        }
        ++pos;
      }
  }
}

}  // namespace

// ============================================================ C ABI
extern "C" int psx_resample(const float* in, float* out, uint64_t n, float acc, float tsamp, psx_stream s) {
  PSX_REQUIRE(in && out && n > 0, "psx_resample: bad arguments");
  PSX_REQUIRE(in != out, "psx_resample: in and out may not alias");
  PSX_REQUIRE(((uintptr_t)out & 15) == 0, "psx_resample: out must be 16-byte aligned");
  const double af = psx::accel_fact(acc, tsamp);
  PSX_REQUIRE(fabs(af) * (double)n < 1.0, "psx_resample: |a*tsamp/2c| * n must be < 1 (got %g)",
              fabs(af) * (double)n);
  k_resample2<<<psx::grid_for(n / 4 + 1, kBlock), kBlock, 0, as_stream(s)>>>(in, out, n, af);
  PSX_CHECK_LAUNCH("k_resample2");
  return psx::ok();
}

extern "C" int psx_resample_v1(const float* in, float* out, uint64_t n, float acc, float tsamp, psx_stream s) {
  PSX_REQUIRE(in && out && n > 0, "psx_resample_v1: bad arguments");
  PSX_REQUIRE(in != out, "psx_resample_v1: in and out may not alias");
  const double af = psx::accel_fact(acc, tsamp);
  PSX_REQUIRE(fabs(af) * (double)n < 1.0, "psx_resample_v1: |a*tsamp/2c| * n must be < 1");
  k_resample1<<<psx::grid_for(n, kBlock), kBlock, 0, as_stream(s)>>>(in, out, n, af);
  PSX_CHECK_LAUNCH("k_resample1");
  return psx::ok();
}

extern "C" int psx_form_amplitude(const psx_c32* X, float* A, uint64_t nb, psx_stream s) {
  PSX_REQUIRE(X && A, "psx_form_amplitude: null pointer");
  if (!nb) return psx::ok();
  k_amplitude<<<psx::grid_for(nb, kBlock), kBlock, 0, as_stream(s)>>>((const float2*)X, A, nb);
  PSX_CHECK_LAUNCH("k_amplitude");
  return psx::ok();
}

extern "C" int psx_form_interbin(const psx_c32* X, float* A, uint64_t nb, psx_stream s) {
  PSX_REQUIRE(X && A, "psx_form_interbin: null pointer");
  PSX_REQUIRE(((uintptr_t)X & 15) == 0 && ((uintptr_t)A & 7) == 0, "psx_form_interbin: misaligned buffers");
  if (!nb) return psx::ok();
  k_interbin<<<psx::grid_for(nb / 2 + 1, kBlock), kBlock, 0, as_stream(s)>>>((const float2*)X, A, nb);
  PSX_CHECK_LAUNCH("k_interbin");
  return psx::ok();
}

extern "C" int psx_median_scrunch5(const float* in, uint64_t count, float* out, psx_stream s) {
  PSX_REQUIRE(in && out && count > 0, "psx_median_scrunch5: bad arguments");
  if (count < 5) {
    k_scrunch_small<<<1, 64, 0, as_stream(s)>>>(in, out, (int)count);
    PSX_CHECK_LAUNCH("k_scrunch_small");
    return psx::ok();
  }
  const uint64_t oc = count / 5;
  k_scrunch5<<<psx::grid_for(oc, kBlock), kBlock, 0, as_stream(s)>>>(in, out, oc);
  PSX_CHECK_LAUNCH("k_scrunch5");
  return psx::ok();
}

extern "C" int psx_linear_stretch(const float* in, uint64_t in_count, float* out, uint64_t out_count,
                                  psx_stream s) {
  PSX_REQUIRE(in && out && in_count > 0 && out_count > 1, "psx_linear_stretch: bad arguments");
  PSX_REQUIRE(out_count <= 0xFFFFFFFFull, "psx_linear_stretch: out_count exceeds 32-bit index");
  k_stretch<<<psx::grid_for(out_count, kBlock), kBlock, 0, as_stream(s)>>>(in, in_count, out, out_count,
                                                                           psx::stretch_step(in_count, out_count));
  PSX_CHECK_LAUNCH("k_stretch");
  return psx::ok();
}

extern "C" int psx_divide_c_by_f(psx_c32* X, const float* f, uint64_t nb, psx_stream s) {
  PSX_REQUIRE(X && f, "psx_divide_c_by_f: null pointer");
  if (!nb) return psx::ok();
  k_divide<<<psx::grid_for(nb, kBlock), kBlock, 0, as_stream(s)>>>((float2*)X, f, nb);
  PSX_CHECK_LAUNCH("k_divide");
  return psx::ok();
}

extern "C" int psx_zap_birdies(psx_c32* X, const float* freqs, const float* widths, uint32_t nbirdies,
                               float bin_width, uint64_t nb, psx_stream s) {
  if (!nbirdies || !nb) return psx::ok();
  PSX_REQUIRE(X && freqs && widths && bin_width > 0, "psx_zap_birdies: bad arguments");
  PSX_REQUIRE(nbirdies <= 0x7FFFFFFFu, "psx_zap_birdies: too many birdies");
  k_zap<<<nbirdies, kBlock, 0, as_stream(s)>>>((float2*)X, freqs, widths, bin_width, nb);
  PSX_CHECK_LAUNCH("k_zap");
  return psx::ok();
}

extern "C" uint64_t psx_deredden_work_floats(uint64_t nb) { return nb / 5 + nb / 25 + nb / 125 + 3; }

// Dereddener::calculate_median (dereddener.hpp:41-62).  The three stretched
// medians are written straight into their zones of `median`, which equals
// the reference's copy sequence (the second copy's overrun past pos25 is
// overwritten by the third).
extern "C" int psx_deredden_median(const float* A, uint64_t nb, double bin_width, float b5, float b25,
                                   float* median, float* work, psx_stream s) {
  PSX_REQUIRE(A && median && work && nb >= 5 && bin_width > 0, "psx_deredden_median: bad arguments");
  const uint64_t c5 = nb / 5, c25 = nb / 5 / 5, c125 = nb / 5 / 5 / 5;
  PSX_REQUIRE(c125 >= 1, "psx_deredden_median: nb too small (%llu)", (unsigned long long)nb);
  float* m5 = work;
  float* m25 = m5 + c5 + 1;
  float* m125 = m25 + c25 + 1;
  const hipStream_t hs = as_stream(s);
  k_scrunch125<<<(unsigned)((c5 + 25 * kM125 - 1) / (25 * kM125)), kBlock, 0, hs>>>(A, m5, m25, m125, c5, c25, c125);
  PSX_CHECK_LAUNCH("k_scrunch125");
  const int64_t pos5 = (int64_t)(int)((double)b5 / bin_width);
  const int64_t pos25 = (int64_t)(int)((double)b25 / bin_width);
  auto clampz = [&](int64_t v) -> uint64_t { return v < 0 ? 0 : (v > (int64_t)nb ? nb : (uint64_t)v); };
  // zone [0, pos5) <- m5, zone [pos5, pos25) <- m25 (the reference copies
  // pos25 elements from pos5; everything from pos25 on is rewritten by the
  // third zone), zone [pos25, nb) <- m125
  const uint64_t z1 = clampz(pos5), z2 = clampz(pos25);
  const uint64_t hi = std::min(clampz(pos5 + pos25), std::max(z1, z2));
  k_stretch_zones<<<psx::grid_for(nb, kBlock), kBlock, 0, hs>>>(
      Stretch{m5, c5, psx::stretch_step(c5, nb)}, Stretch{m25, c25, psx::stretch_step(c25, nb)},
      Stretch{m125, c125, psx::stretch_step(c125, nb)}, z1, hi, z2, median, nb);
  PSX_CHECK_LAUNCH("k_stretch_zones");
  return psx::ok();
}

// ------------------------------------------------ running median, no allocation
// psx_deredden_median_noalloc: the same kernels, with the three scrunched
// medians kept in a file-scope device array instead of a caller workspace.
// The array's name is only a host-side handle: kernels get its device
// address, looked up once per device with hipGetSymbolAddress.  Every call on
// a device shares that device's array (calls that overlap on one device
// race); every element a call reads is written earlier in the same call, so
// nothing needs clearing.
namespace {
constexpr uint64_t kNoAllocMaxBins = (1ull << 25) + 1;  // 2^26-sample series
constexpr uint64_t kNoAllocScratchFloats = kNoAllocMaxBins / 5 + kNoAllocMaxBins / 25 + kNoAllocMaxBins / 125 + 3;
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

static __device__ __align__(256) float scratch[kNoAllocScratchFloats];

static int scratch_on_current_device(float** out) {
  int dev = 0;
  PSX_CHECK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return psx::fail(PSX_ERR_UNSUPPORTED, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return psx::fail(PSX_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = (float*)p;
  }
  *out = g_scratch_ptr[dev];
  return PSX_OK;
}

extern "C" uint64_t psx_deredden_noalloc_max_bins(void) { return kNoAllocMaxBins; }

extern "C" int psx_deredden_median_noalloc(const float* A, uint64_t nb, double bin_width, float b5, float b25,
                                           float* median, psx_stream s) {
  PSX_REQUIRE(nb <= kNoAllocMaxBins,
              "psx_deredden_median_noalloc: %llu bins exceed the static scratch (at most %llu bins)",
              (unsigned long long)nb, (unsigned long long)kNoAllocMaxBins);
  float* work = nullptr;
  const int rc = scratch_on_current_device(&work);
  if (rc) return rc;
  return psx_deredden_median(A, nb, bin_width, b5, b25, median, work, s);
}

extern "C" uint64_t psx_reduce_work_bytes(void) { return (kReduceBlocks + 1) * sizeof(double2); }

static int sum_sq(const float* x, uint64_t first, uint64_t n, void* work, psx_stream s, double* s1, double* s2) {
  double2* partial = (double2*)work;
  double2* out = partial + kReduceBlocks;
  const unsigned g = psx::grid_for(n - first, kBlock, kReduceBlocks);
  k_sum_sq<<<g, kBlock, 0, as_stream(s)>>>(x, first, n, partial);
  PSX_CHECK_LAUNCH("k_sum_sq");
  k_sum_final<<<1, kBlock, 0, as_stream(s)>>>(partial, g, out);
  PSX_CHECK_LAUNCH("k_sum_final");
  double2 h;
  PSX_CHECK_HIP(hipMemcpyAsync(&h, out, sizeof(h), hipMemcpyDeviceToHost, as_stream(s)));
  PSX_CHECK_HIP(hipStreamSynchronize(as_stream(s)));
  *s1 = h.x;
  *s2 = h.y;
  return PSX_OK;
}

// stats: GPU_rms then GPU_mean (src/kernels.cu:433-461): float(sum)/float(n).
extern "C" int psx_mean_rms(const float* x, uint64_t n, uint64_t first, float* mean, float* rms, void* work,
                            psx_stream s) {
  PSX_REQUIRE(x && work && n > first, "psx_mean_rms: bad arguments");
  double s1, s2;
  int rc = sum_sq(x, first, n, work, s, &s1, &s2);
  if (rc) return rc;
  const float cnt = (float)(int64_t)(n - first);
  if (mean) *mean = (float)s1 / cnt;
  if (rms) *rms = sqrtf((float)s2 / cnt);
  return psx::ok();
}

extern "C" int psx_normalise(float* p, float mean, float sigma, uint64_t n, psx_stream s) {
  PSX_REQUIRE(p, "psx_normalise: null pointer");
  PSX_REQUIRE(((uintptr_t)p & 15) == 0, "psx_normalise: buffer must be 16-byte aligned");
  if (!n) return psx::ok();
  k_normalise<<<psx::grid_for(n / 4 + 1, kBlock), kBlock, 0, as_stream(s)>>>(p, n, mean, sigma);
  PSX_CHECK_LAUNCH("k_normalise");
  return psx::ok();
}

// GPU_remove_baseline (src/kernels.cu:463-479): two iterations per look at
// the loop's state (series need one or two).
extern "C" int psx_remove_baseline(float* x, uint64_t n, void* work, psx_stream s) {
  PSX_REQUIRE(x && work && n > 0, "psx_remove_baseline: bad arguments");
  const hipStream_t hs = as_stream(s);
  double2* partial = (double2*)work;
  BaselineState* st = (BaselineState*)(partial + kReduceBlocks);  // two states
  static_assert(2 * sizeof(BaselineState) <= sizeof(double2), "states in the total's place");
  const unsigned g = psx::grid_for(n, kBlock, kReduceBlocks);
  bool first = true;
  BaselineState h;
  do {
    for (int i = 0; i < 2; ++i) {
      if (first) {
        k_base_sum<true><<<g, kBlock, 0, hs>>>(x, n, partial, nullptr);
        PSX_CHECK_LAUNCH("k_base_sum");
        k_base_sub<true><<<g, kBlock, 0, hs>>>(x, n, partial, g, nullptr, st);
      } else {
        k_base_sum<false><<<g, kBlock, 0, hs>>>(x, n, partial, st + (i ^ 1));
        PSX_CHECK_LAUNCH("k_base_sum");
        k_base_sub<false><<<g, kBlock, 0, hs>>>(x, n, partial, g, st + (i ^ 1), st + i);
      }
      PSX_CHECK_LAUNCH("k_base_sub");
      first = false;
    }
    PSX_CHECK_HIP(hipMemcpyAsync(&h, st + 1, sizeof(h), hipMemcpyDeviceToHost, hs));
    PSX_CHECK_HIP(hipStreamSynchronize(hs));
  } while (!h.done);
  return psx::ok();
}

extern "C" int psx_fill(float* x, uint64_t start, uint64_t end, float value, psx_stream s) {
  PSX_REQUIRE(x, "psx_fill: null pointer");
  if (end <= start) return psx::ok();
  k_fill<<<psx::grid_for(end - start, kBlock), kBlock, 0, as_stream(s)>>>(x, start, end, value);
  PSX_CHECK_LAUNCH("k_fill");
  return psx::ok();
}

extern "C" int psx_convert_to_f32(const void* in, int in_type, float* out, uint64_t n, psx_stream s) {
  PSX_REQUIRE(in && out, "psx_convert_to_f32: null pointer");
  if (!n) return psx::ok();
  const unsigned g = psx::grid_for(n, kBlock);
  const hipStream_t hs = as_stream(s);
  switch (in_type) {
    case PSX_U8: k_convert<uint8_t><<<g, kBlock, 0, hs>>>((const uint8_t*)in, out, n); break;
    case PSX_I8: k_convert<int8_t><<<g, kBlock, 0, hs>>>((const int8_t*)in, out, n); break;
    case PSX_U32: k_convert<uint32_t><<<g, kBlock, 0, hs>>>((const uint32_t*)in, out, n); break;
    case PSX_F32: k_convert<float><<<g, kBlock, 0, hs>>>((const float*)in, out, n); break;
    default: return psx::fail(PSX_ERR_ARG, "psx_convert_to_f32: unknown input type %d", in_type);
  }
  PSX_CHECK_LAUNCH("k_convert");
  return psx::ok();
}

extern "C" int psx_harmonic_sum(const float* P, float* const* folds, uint32_t nfolds, uint64_t nb, psx_stream s) {
  PSX_REQUIRE(P && folds, "psx_harmonic_sum: null pointer");
  PSX_REQUIRE(nfolds >= 1 && nfolds <= 5, "psx_harmonic_sum: nfolds must be 1..5 (got %u)", nfolds);
  FoldPtrs fp = {};
  for (uint32_t k = 0; k < nfolds; ++k) {
    PSX_REQUIRE(folds[k], "psx_harmonic_sum: null fold pointer %u", k);
    fp.f[k] = folds[k];
  }
  if (!nb) return psx::ok();
  psx::TraceRange range("Harmonic summing");
  const hipStream_t hs = as_stream(s);
  switch (nfolds) {
    case 1: launch_harmonic<1>(P, fp, nb, hs); break;
    case 2: launch_harmonic<2>(P, fp, nb, hs); break;
    case 3: launch_harmonic<3>(P, fp, nb, hs); break;
    case 4: launch_harmonic<4>(P, fp, nb, hs); break;
    default: launch_harmonic<5>(P, fp, nb, hs); break;
  }
  PSX_CHECK_LAUNCH("k_harmonic");
  return psx::ok();
}

extern "C" uint64_t psx_find_peaks_work_bytes(uint64_t n) {
  return ((n + kPeakTile - 1) / kPeakTile + 1) * sizeof(uint32_t);
}

namespace {
template <unsigned NS>
int find_peaks(const float* const* p, const int64_t* start, const int64_t* end, uint32_t nspec, float thr,
               const PeakOut& out, void* work, hipStream_t hs) {
  PeakJobs<NS> jobs{};
  uint32_t most = 1, sum = 0;
  for (uint32_t y = 0; y < nspec; ++y) {
    const int64_t a = std::max<int64_t>(start[y], 0);
    const uint64_t n = end[y] > a ? (uint64_t)(end[y] - a) : 0;
    PSX_REQUIRE(n < (1ull << 31), "psx_find_peaks: range exceeds 2^31 bins");
    jobs.p[y] = p[y];
    jobs.start[y] = a;
    jobs.end[y] = a + (int64_t)n;
    jobs.tiles[y] = (uint32_t)((n + kPeakTile - 1) / kPeakTile);
    jobs.first[y] = sum;
    sum += jobs.tiles[y];
    most = std::max(most, jobs.tiles[y]);
  }
  uint32_t* counts = (uint32_t*)work;
  if (sum) {
    k_peak_count<NS><<<dim3(most, nspec), kBlock, 0, hs>>>(jobs, thr, counts);
    PSX_CHECK_LAUNCH("k_peak_count");
  }
  k_peak_write<NS><<<dim3(most, nspec), kBlock, 0, hs>>>(jobs, thr, counts, out);
  PSX_CHECK_LAUNCH("k_peak_write");
  return psx::ok();
}
}  // namespace

extern "C" int psx_find_peaks(const float* p, int64_t start, int64_t end, float thr, int32_t* d_idx,
                              float* d_snr, uint32_t cap, uint32_t* d_count, void* work, psx_stream s) {
  PSX_REQUIRE(p && d_count && work, "psx_find_peaks: null pointer");
  PSX_REQUIRE(cap == 0 || (d_idx && d_snr), "psx_find_peaks: null output arrays");
  return find_peaks<1>(&p, &start, &end, 1, thr, PeakOut{d_idx, d_snr, cap, d_count, nullptr, nullptr, 0}, work,
                       as_stream(s));
}

extern "C" int psx_find_peaks_spectra(const float* const* spectra, const int64_t* start, const int64_t* end,
                                      uint32_t nspec, float thr, int32_t* d_idx, float* d_snr, uint32_t cap,
                                      void* d_head, uint32_t nhead, void* work, psx_stream s) {
  PSX_REQUIRE(spectra && start && end && d_head && work, "psx_find_peaks_spectra: null pointer");
  PSX_REQUIRE(nspec >= 1 && nspec <= kPeakSpectra, "psx_find_peaks_spectra: 1..%u spectra", kPeakSpectra);
  PSX_REQUIRE(cap == 0 || (d_idx && d_snr), "psx_find_peaks_spectra: null output arrays");
  PSX_REQUIRE(nhead <= (1u << 20), "psx_find_peaks_spectra: nhead too large");
  for (uint32_t y = 0; y < nspec; ++y) PSX_REQUIRE(spectra[y], "psx_find_peaks_spectra: null spectrum");
  uint32_t* head = (uint32_t*)d_head;
  return find_peaks<kPeakSpectra>(spectra, start, end, nspec, thr,
                                  PeakOut{d_idx, d_snr, cap, head, (int32_t*)(head + nspec),
                                          (float*)(head + nspec + nspec * nhead), nhead},
                                  work, as_stream(s));
}
