// batch.hip - fused kernels of the batched acceleration search (gfx950).
//
// One batch = up to B acceleration trials of the same FFT length.  Per batch:
//   k_fft_pass (resample fused into the first pass) ... FFT passes -> Z
//   k_spec_post   untangle + interbin + normalise          Z -> P
//   k_pool_peaks  fundamental threshold + bound spectrum   P -> Q, candidates
//   k_harm_bound  2..2^F harmonic sums over Q (upper bounds of the fold
//                 sums, two bins at a time); exact sums of P
//                 where a bound crosses the threshold      Q, P -> candidates
// (k_harm_peaks, the exact sums of every bin, is the alternative harmonic
// pass: same candidates, more memory traffic.)
// The per-trial arithmetic is the plain path's, operation for operation
// (untangled_bin, interbin, (v-mean)/std, harmonic_sums), so every value the
// batched path thresholds equals the plain path's bit for bit; only the
// intermediate HBM round trips (X, the interbinned spectrum before
// normalisation, the F fold spectra) disappear.
#include "batch.hpp"

#include <cmath>
#include <cstring>

#include "common.hpp"
#include "kernels_dev.hpp"

using namespace psx::fft;

namespace psx {
namespace batch {
namespace {

constexpr unsigned kB = 256;

// untangle + form_interpolated + normalise (src/kernels.cu:238-259,496-507).
// The half-length spectrum pair (Z[k], Z[M-k]), k <= M/2, untangles into both
// X[k] and X[M-k] (the two halves of the plain untangle pass, same
// arithmetic).  Interbinning needs X[k-1] beside X[k], and X[M-k-1] (the
// upper half of pair k+1) beside X[M-k].  A wave holds 64 consecutive pairs
// k = kw-1 .. kw+62 (one lane per pair, both loads coalesced, the mirror row
// descending) and takes every neighbour from the adjacent lane by a shuffle:
// lanes 1..63 write P[k], lanes 0..62 write P[M-k], and consecutive waves
// advance by 63 pairs, so no lane ever loads a neighbour itself.
__device__ inline float normalised(float2 x, float2 prev, float mean_n, float std_n) {
  float v = psx::interbin(x, prev);
  v -= mean_n;
  v /= std_n;
  return v;
}

// An upper bound of normalised(x, prev, mean_n, std_n) (std_n > 0) from the
// hardware's approximate square root and reciprocal (each within 1 ulp):
// the interbin square root is raised by 2^-20 of itself (8 ulp, more than
// the approximation's error), the mean subtracted as the reference does
// (rounding is monotone), and the quotient taken as a product with the
// approximate reciprocal and raised by 2^-20 of its magnitude (its error is
// under 2 ulp of the quotient, plus the half ulp of correct rounding).
// About a third of normalised's instructions: the bound-form spectrum pass
// needs the exact value only where this one exceeds the threshold.
__device__ inline float normalised_up(float2 x, float2 prev, float mean_n, float std_n) {
  const float ampsq = fmaf(x.x, x.x, x.y * x.y);
  const float dr = x.x - prev.x;
  const float di = x.y - prev.y;
  const float ampsq_diff = 0.5f * fmaf(dr, dr, di * di);
  const float a = __builtin_amdgcn_sqrtf(fmaxf(ampsq, ampsq_diff));
  const float v = fmaf(a, 0x1p-20f, a) - mean_n;
  const float q = v * __builtin_amdgcn_rcpf(std_n);
  return fmaf(fabsf(q), 0x1p-20f, q);
}

__device__ inline float2 shfl_f2(float2 v, int src) {
  return make_float2(__shfl(v.x, src), __shfl(v.y, src));
}

constexpr uint32_t kStep = 63;  // pairs written per wave

// bfloat16 bits (the top half of the float) of the smallest bfloat16 >= x:
// a positive float with any of its low 16 bits set rounds its top half up
// (a carry into the exponent is the next binade, and past the largest
// finite value +inf); a negative one truncates toward zero, which is up.
__device__ inline uint16_t bf16_up(float x) {
  const uint32_t u = __float_as_uint(x);
  return (uint16_t)(((int32_t)u < 0 ? u : u + 0xFFFFu) >> 16);
}
__device__ inline float bf16_value(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// Reads the kBoundD LDS entries e[0], e[STRIDE], ... into the high halves of
// t[0..kBoundD), whose low halves the caller keeps at zero: ds_read_u16_d16_hi
// writes only the high half, so t[d] is the entry's float value with no
// conversion instruction.  The reads and their wait are one asm statement.
template <int STRIDE>
__device__ inline void lds_bf16x8(const uint16_t* e, float (&t)[8]) {
  const uint32_t a = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)e;
  asm volatile(
      "ds_read_u16_d16_hi %0, %8\n\t"
      "ds_read_u16_d16_hi %1, %8 offset:%9\n\t"
      "ds_read_u16_d16_hi %2, %8 offset:%10\n\t"
      "ds_read_u16_d16_hi %3, %8 offset:%11\n\t"
      "ds_read_u16_d16_hi %4, %8 offset:%12\n\t"
      "ds_read_u16_d16_hi %5, %8 offset:%13\n\t"
      "ds_read_u16_d16_hi %6, %8 offset:%14\n\t"
      "ds_read_u16_d16_hi %7, %8 offset:%15\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]), "+v"(t[4]), "+v"(t[5]), "+v"(t[6]), "+v"(t[7])
      : "v"(a), "i"(2 * STRIDE), "i"(4 * STRIDE), "i"(6 * STRIDE), "i"(8 * STRIDE), "i"(10 * STRIDE),
        "i"(12 * STRIDE), "i"(14 * STRIDE));
}

// The same for two runs of entries under one wait.
template <int S1, int S2>
__device__ inline void lds_bf16x16(const uint16_t* e, const uint16_t* e2, float (&t)[8], float (&u)[8]) {
  const uint32_t a = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)e;
  const uint32_t b = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)e2;
  asm volatile(
      "ds_read_u16_d16_hi %0, %16\n\t"
      "ds_read_u16_d16_hi %1, %16 offset:1*%18\n\t"
      "ds_read_u16_d16_hi %2, %16 offset:2*%18\n\t"
      "ds_read_u16_d16_hi %3, %16 offset:3*%18\n\t"
      "ds_read_u16_d16_hi %4, %16 offset:4*%18\n\t"
      "ds_read_u16_d16_hi %5, %16 offset:5*%18\n\t"
      "ds_read_u16_d16_hi %6, %16 offset:6*%18\n\t"
      "ds_read_u16_d16_hi %7, %16 offset:7*%18\n\t"
      "ds_read_u16_d16_hi %8, %17\n\t"
      "ds_read_u16_d16_hi %9, %17 offset:1*%19\n\t"
      "ds_read_u16_d16_hi %10, %17 offset:2*%19\n\t"
      "ds_read_u16_d16_hi %11, %17 offset:3*%19\n\t"
      "ds_read_u16_d16_hi %12, %17 offset:4*%19\n\t"
      "ds_read_u16_d16_hi %13, %17 offset:5*%19\n\t"
      "ds_read_u16_d16_hi %14, %17 offset:6*%19\n\t"
      "ds_read_u16_d16_hi %15, %17 offset:7*%19\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]), "+v"(t[4]), "+v"(t[5]), "+v"(t[6]), "+v"(t[7]),
        "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]), "+v"(u[4]), "+v"(u[5]), "+v"(u[6]), "+v"(u[7])
      : "v"(a), "v"(b), "i"(2 * S1), "i"(2 * S2));
}

// Outputs of the spectrum pass for the bound-filtered harmonic pass: the
// bound spectrum (one bfloat16 upper bound of the bins 2u-1, 2u, 2u+1) and
// the fundamental's above-threshold bins (device_find_peaks over
// PeakFinder's nh = 0 window, src/kernels.cu:391-423, peakfinder.hpp:78-83).
struct BoundOut {
  uint16_t* Q;
  int64_t qstride;
  int32_t start0, end0;
  float thr;
  Cand16* out;
  uint32_t cap;
  uint32_t* count;
};

// Appends the calling lanes' hits (bin k, value v) as fundamental
// candidates of slot; every lane of the wave calls it, lane 0 included.
__device__ inline void append_fundamental(bool hit, uint32_t slot, uint32_t k, float v, const BoundOut& bo) {
  const uint64_t mask = __ballot(hit);
  if (mask == 0) return;
  uint32_t b = 0;
  if ((threadIdx.x & 63u) == 0) b = atomicAdd(bo.count, (uint32_t)__popcll(mask));
  b = __shfl(b, 0);
  if (hit) {
    const uint32_t pos = b + psx::mbcnt64(mask);
    if (pos < bo.cap) bo.out[pos] = Cand16{slot, 0u, (int32_t)k, v};
  }
}
__device__ inline bool fundamental_hit(float v, uint32_t k, const BoundOut& bo) {
  return v > bo.thr && (int32_t)k >= bo.start0 && (int32_t)k < bo.end0;
}

template <int Q>
__global__ void __launch_bounds__(kB) k_spec_post(const float2* __restrict__ Z, float* __restrict__ P, uint64_t M,
                                                  int64_t pstride, RootTable rt, const TrialDesc* __restrict__ descs) {
  const uint32_t tr = blockIdx.y;
  const float2* z = Z + (int64_t)tr * (int64_t)M;
  float* p = P + (int64_t)tr * pstride;
  const float mean_n = descs[tr].mean_n;
  const float std_n = descs[tr].std_n;
  const uint32_t m = (uint32_t)M, half = m / 2;
  const int lane = (int)(threadIdx.x & 63u);
  const uint32_t waves = gridDim.x * (kB / 64);
  const uint32_t wave0 = blockIdx.x * (kB / 64) + (threadIdx.x >> 6);
  const uint32_t nwchunks = (half + 1 + kStep - 1) / kStep;  // waves of 63 lower outputs cover 0..half
  for (uint32_t c = wave0; c < nwchunks; c += waves * Q) {
    float2 zk[Q], zm[Q];
    int32_t kq[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const uint32_t cw = c + (uint32_t)q * waves;
      const int32_t k = (int32_t)(cw * kStep) + lane - 1;
      kq[q] = k;
      zk[q] = zm[q] = make_float2(0.f, 0.f);
      if (cw < nwchunks && k >= 0 && (uint32_t)k <= half) {
        zk[q] = z[k];
        zm[q] = z[k == 0 ? 0 : m - (uint32_t)k];
      }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int32_t k = kq[q];
      const bool valid = (c + (uint32_t)q * waves) < nwchunks && k >= 0 && (uint32_t)k <= half;
      float2 xl = make_float2(0.f, 0.f), xu = make_float2(0.f, 0.f);
      if (valid) {
        const float2 w = root(rt, (uint64_t)k);
        xl = untangle_one(zk[q], zm[q], w);
        // W_n^(M-k) = -conj(W_n^k); the midpoint is its own mirror and keeps
        // the lower formula, as the plain pass writes it
        xu = ((uint32_t)k == half) ? xl : untangle_one(zm[q], zk[q], make_float2(-w.x, w.y));
      }
      // X[k-1] from the lane below (zero below bin 0), X[M-k-1] from above
      const float2 xl_prev = shfl_f2(xl, lane > 0 ? lane - 1 : 0);
      const float2 xu_next = shfl_f2(xu, lane < 63 ? lane + 1 : 63);
      if (valid) {
        if (lane > 0) p[k] = normalised(xl, xl_prev, mean_n, std_n);
        if (lane < 63 && (uint32_t)k < half) p[m - (uint32_t)k] = normalised(xu, xu_next, mean_n, std_n);
      }
    }
  }
}

// The same spectrum pass over the transposed half-length spectrum that a
// last FFT pass writing contiguous rows leaves: row r (R rows of L
// elements) holds Z(r, e) = Z[r + R*e].  Bin k = r + R*e pairs with M - k,
// which is (R - r, L-1-e) for r >= 1 and, for r = 0, (0, L-e), i.e. the
// virtual row R = row 0 shifted by one column (Z[M] = Z[0]).  Interbinning
// takes X[k-1] = X(r-1, e) from the row below, in the same column.
//
// A workgroup owns lower rows [ra, ra+64) (1 <= r < R/2) and their mirror
// rows R - r, over 64 columns.  Wave w sweeps pair rows q = r0-1 .. r0+16
// (r0 = ra + 16w), one column per lane: it loads Z(q, e) (row contiguous)
// and the mirror Z(R-q, L-1-e) (row descending), untangles both bins with
// the plain pass's arithmetic, and keeps the previous pair row in registers
// for the interbin neighbours: P(q, e) uses X(q-1, e), and P(R-q', L-1-e)
// uses X(R-q'-1, L-1-e), the mirror of pair row q'+1.  Results are
// transposed through LDS and written as 64-bin runs of P (natural order).
// Rows 0 and R/2 and bin M pair within their own row: the grid's last row
// of workgroups computes them (spec_edge_bin), beside the tiles.
constexpr int kRowTile = 64;  // lower rows per workgroup (16 per wave)
constexpr int kColTile = 64;  // columns per workgroup (one per lane)
// the write-out gives each lane one row of the tile
static_assert(kRowTile == 64 && kColTile == 64, "k_spec_rows writes one tile row per lane");

// X[k] of the pair (Z[k], Z[M-k]) exactly as untangled_bin computes it:
// the root of min(k, M-k), mirrored for the upper bin.
// hi (optional): the root table's high factor of this root, when the
// caller already holds it; the product is the same cmul either way.
__device__ inline void untangle_pair(float2 zk, float2 zm, uint32_t k, uint32_t M, const RootTable& rt, float2& xk,
                                     float2& xm, const float2* hi = nullptr) {
  const bool upper = 2 * k > M;
  const uint32_t ri = upper ? M - k : k;
  const float2 w = hi ? cmul(*hi, ldg2(rt.lo, ri & rt.mask)) : root32(rt, ri);
  const float2 wm = make_float2(-w.x, w.y);
  xk = untangle_one(zk, zm, upper ? wm : w);
  xm = untangle_one(zm, zk, upper ? w : wm);
}

// Bins of rows 0 and R/2 (k = R*e and R/2 + R*e) and the Nyquist bin M of
// the transposed layout, one thread each, through the natural-index view.
// rshift: log2(R) when R is a power of two (the row and column of j by a
// mask and a shift), else 32 (by division).
__device__ inline float2 z_rows(const float2* y, uint32_t R, uint32_t L, uint32_t j, uint32_t rshift = 32) {
  const uint32_t M = R * L;
  if (j >= M) j -= M;
  return rshift < 32 ? y[(j & (R - 1)) * L + (j >> rshift)] : y[(j % R) * L + j / R];
}
__device__ inline float2 x_rows(const float2* y, uint32_t R, uint32_t L, uint32_t k, const RootTable& rt,
                                uint32_t rshift = 32) {
  const uint32_t M = R * L;
  float2 xk, xm;
  untangle_pair(z_rows(y, R, L, k, rshift), z_rows(y, R, L, M - k, rshift), k, M, rt, xk, xm);
  return xk;
}
// t < L: row 0; t < 2L: row R/2; t == 2L: bin M.  Returns the bin and its
// value; with BOUND, also the bound of the bins k-1, k, k+1 (k is even), whose
// outer ones (other rows' bins) are recomputed here through the same untangle
// and interbin arithmetic.
template <bool BOUND>
__device__ inline float spec_edge_bin(const float2* y, float* p, uint32_t R, uint32_t L, uint32_t t,
                                      const RootTable& rt, float mean_n, float std_n, uint16_t* q, uint32_t& k) {
  const uint32_t M = R * L;
  k = t < L ? R * t : (t < 2 * L ? R / 2 + R * (t - L) : M);
  float2 x, prev = make_float2(0.f, 0.f);
  if (k == M) {
    // X[M] is the upper bin of pair 0
    float2 x0;
    untangle_pair(y[0], y[0], 0, M, rt, x0, x);
  } else {
    x = x_rows(y, R, L, k, rt);
  }
  if (k > 0) prev = x_rows(y, R, L, k - 1, rt);
  const float v = normalised(x, prev, mean_n, std_n);
  if constexpr (!BOUND) p[k] = v;
  if constexpr (BOUND) {
    float m = v;
    if (k > 0) {
      const float2 prev2 = k > 1 ? x_rows(y, R, L, k - 2, rt) : make_float2(0.f, 0.f);
      m = fmaxf(m, normalised(prev, prev2, mean_n, std_n));
    }
    // bin M is the last
    if (k < M) m = fmaxf(m, normalised(x_rows(y, R, L, k + 1, rt), x, mean_n, std_n));
    q[k / 2] = bf16_up(m);
  }
  return v;
}

// BOUND: the bound spectrum and the fundamental's candidates instead of the
// spectra (the bound-filtered harmonic pass recomputes the few bins it sums
// exactly from Y); the tile's values are then upper bounds (normalised_up),
// and a value above the threshold is recomputed exactly for the fundamental.
template <bool HI_FIXED, bool BOUND>
__global__ void __launch_bounds__(kB) k_spec_rows(const float2* __restrict__ Y, float* __restrict__ P, uint32_t R,
                                                  uint32_t L, int64_t pstride, RootTable rt,
                                                  const TrialDesc* __restrict__ descs, BoundOut bo) {
  __shared__ float lo_t[kColTile][kRowTile + 1];
  __shared__ float up_t[kColTile][kRowTile + 1];
  __shared__ float2 edge_lo[kB / 64][kColTile];  // X of each wave's last lower row
  __shared__ float2 edge_hi[kB / 64][kColTile];  // X of each wave's first upper row
  const uint32_t tr = blockIdx.z;
  const uint32_t M = R * L, half_rows = R / 2;
  const float2* y = Y + (uint64_t)tr * M;
  float* p = P + (int64_t)tr * pstride;
  const float mean_n = descs[tr].mean_n, std_n = descs[tr].std_n;
  uint16_t* q = BOUND ? bo.Q + (int64_t)tr * bo.qstride : nullptr;
  auto tile_value = [&](float2 xv, float2 pv) {
    if constexpr (BOUND)
      return normalised_up(xv, pv, mean_n, std_n);
    else
      return normalised(xv, pv, mean_n, std_n);
  };
  if (blockIdx.y == gridDim.y - 1) {
    // the edge bins: L/64 workgroups of kB threads cover the 2L+1 of them
    const uint32_t t = blockIdx.x * kB + threadIdx.x;
    const bool valid = t <= 2 * L;
    uint32_t k = 0;
    float v = 0.f;
    if (valid) v = spec_edge_bin<BOUND>(y, p, R, L, t, rt, mean_n, std_n, q, k);
    if constexpr (BOUND) append_fundamental(valid && fundamental_hit(v, k, bo), descs[tr].slot, k, v, bo);
    return;
  }
  const uint32_t ra = 1 + blockIdx.y * kRowTile, ea = blockIdx.x * kColTile;
  const unsigned lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
  const uint32_t e = ea + lane, emir = L - 1 - e;
  constexpr int kWaveRows = kRowTile / (kB / 64);
  const uint32_t r0 = ra + wv * kWaveRows;
  // pair row q -> (X(q, e), X(R-q, L-1-e)); rows past R/2 are never used
  // and load row R/2 instead (in bounds, results discarded)
  auto pair_row = [&](uint32_t qq, float2& xlo, float2& xhi) {
    const uint32_t q = min(qq, half_rows);
    const uint32_t ih = q == 0 ? (e == 0 ? 0 : L - e) : (R - q) * L + emir;
    untangle_pair(ldg2(y, q * L + e), ldg2(y, ih), q + R * e, M, rt, xlo, xhi);
  };
  // HI_FIXED (R a power of two no larger than the root table's low span
  // 2^shift, checked by the launcher): for rows q in [1, R/2] of one column
  // the root index is q + R*e or its mirror R*(L-e) - q, whose high part
  // (index >> shift) is then the same for all of them, so the sweep loads
  // that factor once per lane.
  float2 hi_e = make_float2(0.f, 0.f);
  if constexpr (HI_FIXED) {
    const uint32_t k0 = min(r0, half_rows) + R * e;
    hi_e = ldg2(rt.hi, (2 * k0 > M ? M - k0 : k0) >> rt.shift);
  }
  auto sweep_row = [&](uint32_t qq, float2& xlo, float2& xhi) {
    const uint32_t q = min(qq, half_rows);  // >= 1 in the sweep
    untangle_pair(ldg2(y, q * L + e), ldg2(y, (R - q) * L + emir), q + R * e, M, rt, xlo, xhi,
                  HI_FIXED ? &hi_e : nullptr);
  };
  // results of rows outside [1, R/2) go to the spare slot kRowTile
  auto slot = [&](uint32_t qq) { return qq < half_rows ? qq - ra : (uint32_t)kRowTile; };
  // Branch-free sweep over the wave's own rows (so the loads of later rows
  // issue early); the interbin neighbours across wave boundaries come from
  // the adjacent waves through LDS, and only the workgroup's outer halo
  // rows (ra-1 below, ra+64 above) are computed twice.
  float2 xlo_prev = make_float2(0.f, 0.f), xhi_prev = make_float2(0.f, 0.f);
  float2 xlo_first = xlo_prev, xhi_last = xhi_prev;
  // With the high root factor fixed, every row's loads (both bins and the
  // low root factor) are issued before any is used: 16 rows of loads in
  // flight per wave (127 VGPRs, the occupancy the LDS tiles allow anyway)
  // instead of the few the compiler keeps when loads and arithmetic
  // interleave.  The arithmetic is sweep_row's.
  float2 zl[kWaveRows], zh[kWaveRows], wl[kWaveRows];
  if constexpr (HI_FIXED) {
#pragma unroll
    for (int i = 0; i < kWaveRows; ++i) {
      const uint32_t q = min(r0 + (uint32_t)i, half_rows);
      const uint32_t k = q + R * e;
      zl[i] = ldg2(y, q * L + e);
      zh[i] = ldg2(y, (R - q) * L + emir);
      wl[i] = ldg2(rt.lo, (2 * k > M ? M - k : k) & rt.mask);
    }
  }
#pragma unroll
  for (int i = 0; i < kWaveRows; ++i) {
    const uint32_t qq = r0 + (uint32_t)i;
    float2 xlo, xhi;
    if constexpr (HI_FIXED) {
      const uint32_t k = min(qq, half_rows) + R * e;
      const bool upper = 2 * k > M;
      const float2 w = cmul(hi_e, wl[i]);
      const float2 wm = make_float2(-w.x, w.y);
      xlo = untangle_one(zl[i], zh[i], upper ? wm : w);
      xhi = untangle_one(zh[i], zl[i], upper ? w : wm);
    } else {
      sweep_row(qq, xlo, xhi);
    }
    if (i == 0) {
      xlo_first = xlo;
      edge_hi[wv][lane] = xhi;
    } else {
      lo_t[lane][slot(qq)] = tile_value(xlo, xlo_prev);       // P(q)
      up_t[lane][slot(qq - 1)] = tile_value(xhi_prev, xhi);   // P(R-(q-1))
    }
    xlo_prev = xlo;
    xhi_prev = xhi;
  }
  edge_lo[wv][lane] = xlo_prev;
  xhi_last = xhi_prev;
  float2 below = make_float2(0.f, 0.f), above = make_float2(0.f, 0.f), above2 = above, next_lo, unused;
  if (wv == 0) pair_row(ra - 1, below, unused);
  if (wv == kB / 64 - 1) {
    pair_row(ra + kRowTile, next_lo, above);
    if constexpr (BOUND) pair_row(ra + kRowTile + 1, unused, above2);
  }
  __syncthreads();
  if (wv > 0) below = edge_lo[wv - 1][lane];
  if (wv < kB / 64 - 1) above = edge_hi[wv + 1][lane];
  lo_t[lane][slot(r0)] = tile_value(xlo_first, below);
  up_t[lane][slot(r0 + kWaveRows - 1)] = tile_value(xhi_last, above);
  if constexpr (BOUND) {
    // The next tile's first rows, lower (ra + 64) and upper (R - ra - 64),
    // which the bounds of this tile's last lower and upper pairs include:
    // their X were loaded for the halo.  Slot kRowTile is free in every tile
    // but the last, which has no such pairs.
    if (wv == kB / 64 - 1 && ra + kRowTile < half_rows) {
      lo_t[lane][kRowTile] = tile_value(next_lo, xlo_prev);
      up_t[lane][kRowTile] = tile_value(above, above2);
    }
  }
  __syncthreads();
  const uint32_t rr = threadIdx.x & 63u;
  const uint32_t r = ra + rr;
  if constexpr (!BOUND) {
    if (r < half_rows) {
#pragma unroll 4
      for (uint32_t j = wv; j < (uint32_t)kColTile; j += kB / 64) {
        stg1(p, r + R * (ea + j), lo_t[j][rr]);
        stg1(p, (R - r) + R * (L - 1 - (ea + j)), up_t[j][rr]);
      }
    }
  } else {
    // Bounds of the bins (2u-1, 2u, 2u+1): those of the even rows 0 and R/2 of
    // every column are the edge workgroups'; a tile's column holds 32 lower
    // ones, around rows ra+2i+1, i < 32 (slot kRowTile for the last one's
    // third row), and 32 upper ones, around rows R-r, r = ra+63-2i (slot
    // kRowTile for the first one's first row).  Lane i < 32 bounds lower
    // triple i, lane 32+i upper triple i: one 16-bit store covers both runs of
    // 32 entries.  Every value written is also tested as a fundamental.
    const bool rv = r < half_rows;
    const bool lower = rr < 32;
    const uint32_t i = rr & 31u;
    const uint32_t s0 = lower ? 2 * i + 1 : 63 - 2 * i;  // slot of the even row; its neighbours' are beside it
    const uint32_t rpair = ra + s0;                      // lower-half row of the even-row slot
    const bool pv = rpair < half_rows;
    bool any = false;
#pragma unroll 4
    for (uint32_t j = wv; j < (uint32_t)kColTile; j += kB / 64) {
      const float vl = lo_t[j][rr], vu = up_t[j][rr];
      if (rv) any |= fmaxf(vl, vu) > bo.thr;
      if (pv) {
        const float* t = lower ? lo_t[j] : up_t[j];
        const float m = fmaxf(fmaxf(t[s0 - 1], t[s0]), t[s0 + 1]);
        const uint32_t k2 = lower ? rpair + R * (ea + j) : (R - rpair) + R * (L - 1 - (ea + j));
        q[k2 / 2] = bf16_up(m);
      }
    }
    // bounds above the threshold are rare: a second sweep over the tile, in
    // the waves that have any, recomputes those bins exactly (the same
    // untangle, interbin and normalisation of the same inputs as the exact
    // pass) and appends the ones above threshold
    if (__ballot(any) != 0) {
      const uint32_t slot_id = descs[tr].slot;
      const uint32_t rshift = HI_FIXED ? (uint32_t)__builtin_ctz(R) : 32u;
      auto exact = [&](uint32_t k) {
        const float2 prev = k > 0 ? x_rows(y, R, L, k - 1, rt, rshift) : make_float2(0.f, 0.f);
        return normalised(x_rows(y, R, L, k, rt, rshift), prev, mean_n, std_n);
      };
      for (uint32_t j = wv; j < (uint32_t)kColTile; j += kB / 64) {
        const uint32_t kl = r + R * (ea + j);
        const uint32_t ku = (R - r) + R * (L - 1 - (ea + j));
        float vl = lo_t[j][rr], vu = up_t[j][rr];
        const bool cl = rv && fundamental_hit(vl, kl, bo);
        const bool cu = rv && fundamental_hit(vu, ku, bo);
        if (cl) vl = exact(kl);
        if (cu) vu = exact(ku);
        append_fundamental(cl && vl > bo.thr, slot_id, kl, vl, bo);
        append_fundamental(cu && vu > bo.thr, slot_id, ku, vu, bo);
      }
    }
  }
}

// harmonic_sum_kernel (src/kernels.cu:34-100) + device_find_peaks
// (src/kernels.cu:391-423) for the fundamental and every fold, each over
// its own PeakFinder window (peakfinder.hpp:78-83).  Survivors are appended
// to `out` with one atomic per bin row of a wave (all folds together); the
// host orders them by bin.
//
// A wave covers kHarmWaveBins consecutive bins, D per lane, through
// add_harmonic (kernels_dev.hpp): the running sums take harmonic_sums32's
// addends in its order, so the thresholded values are bit-identical to it.  The
// loop only decides whether any value of a lane crosses the threshold; a
// wave with a crossing recomputes its bins one by one with harmonic_sums32,
// applies the fold windows and appends.
template <int K, int D>
__device__ inline bool fold_crosses(const float (&val)[D], float thr) {
  bool any = false;
#pragma unroll
  for (int d = 0; d < D; ++d) any |= fold_scale<K>(val[d]) > thr;
  return any;
}

template <int NF>
__global__ void __launch_bounds__(kB) k_harm_peaks(const float* __restrict__ P, int64_t pstride, Windows w,
                                                   const TrialDesc* __restrict__ descs, Cand16* __restrict__ out,
                                                   uint32_t cap, uint32_t* __restrict__ count) {
  constexpr int D = kHarmWaveBins / 64;
  const uint32_t tr = blockIdx.y;
  const float* p = P + (int64_t)tr * pstride;
  const PSX_GLOBAL float* pg = (const PSX_GLOBAL float*)p;
  const unsigned lane = threadIdx.x & 63u;
  const uint32_t hi = (uint32_t)w.hi;
  const uint32_t wstep = gridDim.x * (kB / 64) * kHarmWaveBins;
  for (uint32_t base = (uint32_t)w.lo + (blockIdx.x * (kB / 64) + (threadIdx.x >> 6)) * kHarmWaveBins; base < hi;
       base += wstep) {
    const uint32_t i0 = base + lane;
    float val[D];
    bool any = false;
    {
      const PSX_GLOBAL float* q = pg + i0;
#pragma unroll
      for (int d = 0; d < D; ++d) val[d] = q[64 * d];
#pragma unroll
      for (int d = 0; d < D; ++d) any |= val[d] > w.thr;
    }
    if constexpr (NF > 0) {
      psx::add_harmonic<1, 1, D>(pg, i0, val);
      any |= fold_crosses<1, D>(val, w.thr);
    }
    if constexpr (NF > 1) {
      psx::add_harmonic<2, 3, D>(pg, i0, val);  // 3/4 before 1/4, as the reference
      psx::add_harmonic<2, 1, D>(pg, i0, val);
      any |= fold_crosses<2, D>(val, w.thr);
    }
    if constexpr (NF > 2) {
      psx::add_harmonics<3, 1, 8, D>(pg, i0, val);
      any |= fold_crosses<3, D>(val, w.thr);
    }
    if constexpr (NF > 3) {
      psx::add_harmonics<4, 1, 16, D>(pg, i0, val);
      any |= fold_crosses<4, D>(val, w.thr);
    }
    if constexpr (NF > 4) {
      psx::add_harmonics<5, 1, 32, D>(pg, i0, val);
      any |= fold_crosses<5, D>(val, w.thr);
    }
    // survivors are rare: one ballot decides whether this wave appends at all
    if (__ballot(any) == 0) continue;
    const uint32_t slot = descs[tr].slot;
#pragma unroll 1
    for (int d = 0; d < D; ++d) {
      const uint32_t i = i0 + 64u * (uint32_t)d;
      const bool valid = i < hi;
      float s[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (valid) {
        float f[5];
        psx::harmonic_sums32<NF>(p, i, f);
        s[0] = p[i];
#pragma unroll
        for (int k = 0; k < NF; ++k) s[k + 1] = f[k];
      }
      // one atomic for the wave's hits of all folds at this d
      bool hit[NF + 1];
      uint64_t mask[NF + 1];
      uint32_t total = 0;
#pragma unroll
      for (int nh = 0; nh <= NF; ++nh) {
        hit[nh] = valid && (int32_t)i >= w.start[nh] && (int32_t)i < w.end[nh] && s[nh] > w.thr;
        mask[nh] = __ballot(hit[nh]);
        total += (uint32_t)__popcll(mask[nh]);
      }
      if (total == 0) continue;
      uint32_t b = 0;
      if (lane == 0) b = atomicAdd(count, total);
      b = __shfl(b, 0);
#pragma unroll
      for (int nh = 0; nh <= NF; ++nh) {
        if (hit[nh]) {
          const uint32_t pos = b + psx::mbcnt64(mask[nh]);
          if (pos < cap) out[pos] = Cand16{slot, (uint32_t)nh, (int32_t)i, s[nh]};
        }
        b += (uint32_t)__popcll(mask[nh]);
      }
    }
  }
}


// ------------------------------------------------------------------------
// Bound-filtered harmonic pass.
//
// The gather form above reads each spectrum once per fold span (8.5 spectra
// for four folds) and is bound by the L2-miss path: every XCD's 4 MB L2
// holds a fraction of one 16 MB spectrum, and the miss path moves about
// 7.5 TB/s whether the MALL or HBM serves it.  Candidates are rare, so this
// form first proves most bins empty from a smaller array:
//   Q[u] = max(P[2u-1], P[2u], P[2u+1]) rounded up to bfloat16,
// one 16-bit entry per two bins (a quarter of the spectrum's bytes), and sums
// it for two bins at a time.  Harmonic j/2^k of the bins 2g and 2g+1 takes
// the source bins s0 <= s1 <= s0 + 1, s1 = (j*(2g+1) + 2^(k-1)) >> k: both are
// covered by Q[s1/2].  Float addition, fold_scale and the comparison are
// monotone (round to nearest never reverses an order), so the running sum of
// those entries in the reference's addend order is at least the exact running
// sum of either bin at every fold: where the bound of fold k stays at or
// below the threshold, so do fold k's exact values.  Only the pairs of bins
// whose bound crosses (3e-5 of noise, and every real detection) are
// summed exactly from P with harmonic_sums32's addends in its order,
// thresholded and appended, so the candidates are the gather form's bit for
// bit.  bfloat16 (8 significant bits) loosens the bound no more than half
// precision does at these values (the same rate of crossing noise bins in a
// float64 simulation), and rounds up with two integer operations where half
// precision needs a conversion, a check and a step.
//
// fold_scale<K>(v) > thr is tested as v > T[K], T[K] the largest float
// whose fold_scale is at most thr (found on the host by bisection over the
// float order; fold_scale is monotone), which keeps double arithmetic out
// of the loop.
//
// A wave covers kBoundWavePairs pairs of bins, lane l holding the pairs
// base + l + 64d (d < 8).  Harmonic j/2^k takes its addends from one run of
// at most kBoundWavePairs*j/2^k + 2 entries of Q; the wave copies every run (and the
// fundamental's) into its own LDS area with global_load_lds_dwordx4 (one
// instruction per run, 16 bytes per lane, no registers), waits once, and then
// reads each addend from LDS at a constant offset per d, two harmonics per
// wait.  A workgroup is one wave, so its 9 KB of LDS free up by themselves (16
// waves per CU).  Per 64 trials of 2^23: 0.80 ms the gather form, 0.34-0.36 ms
// with max(P[2u], P[2u+1]) summed for every bin, 0.26 ms for two bins at a
// time in workgroups of four waves, 0.24 ms in workgroups of one with two
// harmonics per wait.  Bound by its some 330 vector instructions per wave and
// the LDS and L2 latencies that four waves per SIMD leave uncovered.

// Harmonic h (0-based, in the reference's addend order, fold 2 taking 3/4
// before 1/4) is j/2^k with k = hK(h), j = hJ(h); fold k ends at h = 2^k - 2.
__host__ __device__ constexpr int hK(int h) { return h < 1 ? 1 : h < 3 ? 2 : h < 7 ? 3 : h < 15 ? 4 : 5; }
__host__ __device__ constexpr int hJ(int h) {
  return h == 0 ? 1 : h == 1 ? 3 : h == 2 ? 1 : h < 7 ? 2 * (h - 3) + 1 : h < 15 ? 2 * (h - 7) + 1 : 2 * (h - 15) + 1;
}
constexpr int kBoundChunk = 8;  // entries per 16-byte chunk
constexpr int kBoundD = kBoundWavePairs / 64;
// chunks of harmonic h's run: W*j/2^k + 2 entries and the chunk alignment
__host__ __device__ constexpr int run_chunks(int h) {
  return (hJ(h) * (int)kBoundWavePairs >> hK(h)) / kBoundChunk + 2;
}
// LDS offset (entries) of run h; the fundamental's run (W entries, aligned)
// comes first, at 0
__host__ __device__ constexpr int run_offset(int h) {
  int r = (int)kBoundWavePairs;
  for (int g = 0; g < h; ++g) r += run_chunks(g) * kBoundChunk;
  return r;
}
static_assert(run_chunks(30) <= 64 && (int)kBoundWavePairs / kBoundChunk <= 64 && kBoundWavePairs % kBoundChunk == 0,
              "one 64-lane instruction per run");

typedef float psx_f4v __attribute__((ext_vector_type(4)));

// The bound spectrum Q of every trial row, and the fundamental's threshold
// test (device_find_peaks over PeakFinder's nh = 0 window,
// src/kernels.cu:391-423, peakfinder.hpp:78-83) on the same read of P.
// Each lane takes four bins (one 16-byte load) and writes two entries.
__global__ void __launch_bounds__(kB) k_pool_peaks(const float* __restrict__ P, int64_t pstride, uint32_t nb,
                                                   Windows w, uint16_t* __restrict__ Q, int64_t qstride,
                                                   const TrialDesc* __restrict__ descs, Cand16* __restrict__ out,
                                                   uint32_t cap, uint32_t* __restrict__ count) {
  const uint32_t tr = blockIdx.y;
  const float* p = P + (int64_t)tr * pstride;
  uint16_t* q = Q + (int64_t)tr * qstride;
  const unsigned lane = threadIdx.x & 63u;
  const uint32_t start = (uint32_t)max(w.start[0], 0), end = (uint32_t)max(w.end[0], 0);
  const uint32_t ngroups = (nb + 3) / 4;
  const uint32_t stride = gridDim.x * kB;
  // whole-wave trip count, so the ballots below see every lane
  for (uint32_t g0 = blockIdx.x * kB + (threadIdx.x & ~63u); g0 < ngroups; g0 += stride) {
    const uint32_t g = g0 + lane;
    const uint32_t k0 = 4 * g;
    float x[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    // the bin before the wave's first (an entry includes the bin below its pair)
    float before = -INFINITY;
    if (lane == 0 && k0 > 0) before = p[k0 - 1];
    if (g < ngroups) {
      // k0 + 3 < pstride: rows are padded to a multiple of 64 bins
      const psx_f4v v = __builtin_nontemporal_load((const PSX_GLOBAL psx_f4v*)(p + k0));
      x[0] = v.x;
      x[1] = k0 + 1 < nb ? v.y : -INFINITY;
      x[2] = k0 + 2 < nb ? v.z : -INFINITY;
      x[3] = k0 + 3 < nb ? v.w : -INFINITY;
    }
    const float last = __shfl_up(x[3], 1);
    if (lane > 0) before = last;
    if (g < ngroups) {
      const uint32_t pair = (uint32_t)bf16_up(fmaxf(fmaxf(before, x[0]), x[1])) |
                            ((uint32_t)bf16_up(fmaxf(fmaxf(x[1], x[2]), x[3])) << 16);
      *(PSX_GLOBAL uint32_t*)(q + 2 * g) = pair;
    }
    bool any = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) any |= x[j] > w.thr;
    if (__ballot(any) == 0) continue;
    const uint32_t slot = descs[tr].slot;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t k = k0 + (uint32_t)j;
      const bool hit = x[j] > w.thr && k >= start && k < end;
      const uint64_t mask = __ballot(hit);
      if (mask == 0) continue;
      uint32_t b = 0;
      if (lane == 0) b = atomicAdd(count, (uint32_t)__popcll(mask));
      b = __shfl(b, 0);
      if (hit) {
        const uint32_t pos = b + psx::mbcnt64(mask);
        if (pos < cap) out[pos] = Cand16{slot, 0u, (int32_t)k, x[j]};
      }
    }
  }
}

struct FoldThr {
  float t[6];  // t[k]: fold k crosses iff its running sum > t[k]
};

// Copies one run of Q (entries s0..s1, rounded out to whole chunks) into
// the wave's LDS at dst; returns the first entry copied.
__device__ inline uint32_t stage_run(const PSX_GLOBAL uint16_t* q, uint32_t s0, uint32_t s1, uint16_t* dst,
                                     unsigned lane) {
  const uint32_t a0 = s0 & ~(uint32_t)(kBoundChunk - 1);
  const uint32_t n = (s1 - a0) / kBoundChunk + 1;
  if (lane < n)
    __builtin_amdgcn_global_load_lds((const PSX_GLOBAL void*)(q + a0 + kBoundChunk * lane),
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
  return a0;
}

// Entry of Q that covers harmonic J/2^K of the pair of bins g.
template <int K, int J>
__device__ inline uint32_t pair_entry(uint32_t g) {
  return ((J * (2 * g + 1) + (1u << (K - 1))) >> K) >> 1;
}

template <int NH, int H>
struct BoundRuns {
  __device__ static void stage(const PSX_GLOBAL uint16_t* q, uint32_t base, uint16_t* my, uint32_t (&a0)[NH],
                               unsigned lane) {
    if constexpr (H < NH) {
      constexpr int K = hK(H), J = hJ(H);
      a0[H] = stage_run(q, pair_entry<K, J>(base), pair_entry<K, J>(base + kBoundWavePairs - 1), my + run_offset(H),
                        lane);
      BoundRuns<NH, H + 1>::stage(q, base, my, a0, lane);
    }
  }
  // adds the bounds of harmonics H and H + 1 (alone: harmonic 0) to every
  // running sum; at a fold's last addend marks the pairs whose bound crosses
  // that fold's threshold
  __device__ static void add(const uint16_t* my, const uint32_t (&a0)[NH], uint32_t g0, const FoldThr& ft,
                             float (&val)[kBoundD], bool (&fail)[kBoundD], float (&t)[kBoundD],
                             float (&u)[kBoundD]) {
    if constexpr (H < NH) {
      constexpr int H2 = H == 0 ? H : H + 1;
      constexpr int K = hK(H), J = hJ(H), K2 = hK(H2), J2 = hJ(H2);
      // entries between a lane's pairs: 128 bins apart, 128J/2^K source bins
      static_assert((64 * J) % (1 << K) == 0 && (64 * J2) % (1 << K2) == 0, "constant LDS offsets per d");
      static_assert(kBoundD == 8, "eight entries per run");
      const uint16_t* b = my + run_offset(H) + (pair_entry<K, J>(g0) - a0[H]);
      if constexpr (H == 0) {
        lds_bf16x8<((64 * J) >> K)>(b, t);
      } else {
        const uint16_t* b2 = my + run_offset(H2) + (pair_entry<K2, J2>(g0) - a0[H2]);
        lds_bf16x16<((64 * J) >> K), ((64 * J2) >> K2)>(b, b2, t, u);
      }
#pragma unroll
      for (int d = 0; d < kBoundD; ++d) val[d] += t[d];
      if constexpr (H > 0) {
#pragma unroll
        for (int d = 0; d < kBoundD; ++d) val[d] += u[d];
      }
      if constexpr (((H2 + 2) & (H2 + 1)) == 0) {  // H2 = 2^K - 2: fold K complete
#pragma unroll
        for (int d = 0; d < kBoundD; ++d) fail[d] |= val[d] > ft.t[K2];
      }
      BoundRuns<NH, H2 + 1>::add(my, a0, g0, ft, val, fail, t, u);
    }
  }
};

// Where the exact sums of the bins whose bound crosses take the spectrum
// from: P, or (rows != nullptr) bin by bin from the row-layout FFT output the
// spectrum pass read, through its untangle, interbin and normalisation
// (x_rows and normalised: for every bin the same operations on the same
// inputs as the spectrum pass, so the same value bit for bit).
struct ExactSrc {
  const float2* rows;  // Y of trial 0 (trial stride R*L), or nullptr: read P
  uint32_t R, L;
  uint32_t rshift;     // log2(R) for a power of two, else 32
  RootTable rt;
};
// First pair of the first wave: the window's, at a whole chunk of entries.
__host__ __device__ inline uint32_t bound_first_pair(int64_t lo) {
  return ((uint32_t)lo / 2) & ~(uint32_t)(kBoundChunk - 1);
}
// harmonic_sums32's sums (the same addends in the same order) with the
// spectrum value of bin x given by f(x), one addend per iteration of a loop
// the compiler keeps rolled: this path runs for the rare bins whose bound
// crosses, and an unrolled recomputation of 2^NF spectrum values would hold
// enough registers to cost the main loop its occupancy.
template <int NF, class F>
__device__ inline void harmonic_sums_rolled(F f, uint32_t i, float (&s)[5]) {
  float val = f(i);
#pragma unroll 1
  for (int h = 0; h < (1 << NF) - 1; ++h) {
    const int K = hK(h), J = hJ(h);
    val += f(((uint32_t)J * i + (1u << (K - 1))) >> K);
    if (h == 0) s[0] = psx::fold_scale<1>(val);
    else if (h == 2) s[1] = psx::fold_scale<2>(val);
    else if (h == 6) s[2] = psx::fold_scale<3>(val);
    else if (h == 14) s[3] = psx::fold_scale<4>(val);
    else if (h == 30) s[4] = psx::fold_scale<5>(val);
  }
}

// The exact folds of the two bins of pair g (the same for all lanes): lane
// h < 2^NF of each half wave takes addend h of bin 2g + half, all of them at
// once, and then sums them in harmonic_sums32's order; lane k < NF of a half
// has fold k + 1.  A crossing pair costs one round of the addends' loads this
// way, where one lane walking through its addends pays their latency 2^NF
// times.
template <int NF, class F>
__device__ inline void pair_folds(F f, uint32_t g, uint32_t hi, uint32_t& i, float& s) {
  const uint32_t lane = threadIdx.x & 63u, h = lane & 31u;
  i = 2 * g + (lane >> 5);
  float v = 0.f;
  if (h < (1u << NF) && i < hi) {
    const int K = hK((int)h - 1), J = hJ((int)h - 1);
    v = f(h == 0 ? i : ((uint32_t)J * i + (1u << (K - 1))) >> K);
  }
  const int first = (int)(lane & 32u);
  float val = __shfl(v, first);
  s = 0.f;
#pragma unroll
  for (int a = 0; a < (1 << NF) - 1; ++a) {
    val += __shfl(v, first + 1 + a);
    if (a == 0 && h == 0) s = psx::fold_scale<1>(val);
    if (a == 2 && h == 1) s = psx::fold_scale<2>(val);
    if (a == 6 && h == 2) s = psx::fold_scale<3>(val);
    if (a == 14 && h == 3) s = psx::fold_scale<4>(val);
    if (a == 30 && h == 4) s = psx::fold_scale<5>(val);
  }
}
// Pairs of one lane row (d) up to which the wave takes them one after the
// other; where more cross (thresholds inside the noise) each lane sums its own,
// first from the bins' own bounds.  (Searches of 2^23 samples, 64 trials, five
// folds at S/N 5.5: 8 pairs and no own bounds 21.7 ms, with them 15.6, 24 pairs
// 12.7; at S/N 5 114, 104, 98.)
template <int NF>
constexpr int kSerialPairs = NF == 5 ? 24 : 8;

template <int NF, bool FROM_ROWS>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(NF <= 4 ? 4 : 2)))
k_harm_bound(const float* __restrict__ P, int64_t pstride, const uint16_t* __restrict__ Q, int64_t qstride, Windows w,
             FoldThr ft, const TrialDesc* __restrict__ descs, const ExactSrc* __restrict__ srcp, uint32_t xcd_order,
             Cand16* __restrict__ out, uint32_t cap, uint32_t* __restrict__ count) {
  constexpr int NH = (1 << NF) - 1;
  constexpr int WE = run_offset(NH);  // LDS entries per wave
  __shared__ __align__(16) uint16_t my[WE];
  uint32_t tr = blockIdx.y, bx = blockIdx.x;
  if (xcd_order) {
    // workgroups reach the 8 XCDs round robin: hardware block b runs on XCD
    // b % 8, so trial t is given to XCD t % 8 whole (its bound spectrum
    // stays in one L2); the launcher asks for this only when 8 divides the
    // trial count
    const uint32_t b = blockIdx.y * gridDim.x + blockIdx.x;
    const uint32_t k = b >> 3;
    tr = (b & 7u) + 8u * (k / gridDim.x);
    bx = k % gridDim.x;
  }
  const float* p = P + (int64_t)tr * pstride;
  const PSX_GLOBAL uint16_t* qg = (const PSX_GLOBAL uint16_t*)(Q + (int64_t)tr * qstride);
  const unsigned lane = threadIdx.x & 63u;
  const uint32_t hi = (uint32_t)w.hi;
  const uint32_t wstep = gridDim.x * kBoundWavePairs;
  // registers the bound entries are read into, high halves only: their low
  // halves stay zero for the whole kernel
  float t[kBoundD], u[kBoundD];
#pragma unroll
  for (int d = 0; d < kBoundD; ++d) t[d] = u[d] = 0.f;
  for (uint32_t base = bound_first_pair(w.lo) + bx * kBoundWavePairs; 2 * base < hi; base += wstep) {
    const uint32_t g0 = base + lane;
    // the previous tile's LDS reads are complete before the area is refilled
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    uint32_t a0[NH];
    stage_run(qg, base, base + kBoundWavePairs - 1, my, lane);
    BoundRuns<NH, 0>::stage(qg, base, my, a0, lane);
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    float val[kBoundD];
    bool fail[kBoundD];
    lds_bf16x8<64>(my + lane, t);
#pragma unroll
    for (int d = 0; d < kBoundD; ++d) {
      val[d] = t[d];
      fail[d] = false;
    }
    BoundRuns<NH, 0>::add(my, a0, g0, ft, val, fail, t, u);
    bool any = false;
#pragma unroll
    for (int d = 0; d < kBoundD; ++d) any |= fail[d];
    if (__ballot(any) == 0) continue;
    // exact folds of the pairs whose bound crossed (the fundamental is the
    // spectrum stage's)
    const uint32_t slot = descs[tr].slot;
    // the spectrum's value: read from P, or recomputed from the FFT output
    // (the source is read from memory here, not held in scalar registers by
    // the loop)
    auto pval = [&](uint32_t x) {
      if constexpr (FROM_ROWS) {
        const ExactSrc src = *srcp;
        const float2* y = src.rows + (uint64_t)tr * (src.R * src.L);
        const float2 xk = x_rows(y, src.R, src.L, x, src.rt, src.rshift);
        const float2 prev = x > 0 ? x_rows(y, src.R, src.L, x - 1, src.rt, src.rshift) : make_float2(0.f, 0.f);
        return normalised(xk, prev, descs[tr].mean_n, descs[tr].std_n);
      } else {
        return p[x];
      }
    };
    // appends the hits (bin i, fold k + 1, value s) of the calling lanes
    auto append = [&](bool hit, uint32_t i, uint32_t k, float s) {
      const uint64_t mask = __ballot(hit);
      if (mask == 0) return;
      uint32_t b = 0;
      if (lane == 0) b = atomicAdd(count, (uint32_t)__popcll(mask));
      b = __shfl(b, 0);
      if (hit) {
        const uint32_t pos = b + psx::mbcnt64(mask);
        if (pos < cap) out[pos] = Cand16{slot, k + 1, (int32_t)i, s};
      }
    };
    auto in_window = [&](uint32_t i, int k) { return (int32_t)i >= w.start[k + 1] && (int32_t)i < w.end[k + 1]; };
    // a bin's own bound: an odd bin lies in two entries
    auto qval = [&](uint32_t x) {
      const float a = __uint_as_float((uint32_t)qg[x / 2] << 16), b = __uint_as_float((uint32_t)qg[(x + 1) / 2] << 16);
      return fminf(a, b);
    };
#pragma unroll
    for (int d = 0; d < kBoundD; ++d) {
      uint64_t crossing = __ballot(fail[d]);
      bool refined = false;
      if (__popcll(crossing) > kSerialPairs<NF>) {
        refined = true;
        // each lane sums its pair again from the bins' own bounds
        bool still = false;
#pragma unroll 1
        for (uint32_t b = 0; b < 2; ++b) {
          const uint32_t i = 2 * (g0 + 64u * (uint32_t)d) + b;
          float s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
          if (fail[d] && i < hi) harmonic_sums_rolled<NF>(qval, i, s);
#pragma unroll
          for (int k = 0; k < NF; ++k) still |= s[k] > w.thr;
        }
        fail[d] = fail[d] && still;
        crossing = __ballot(fail[d]);
      }
      if (__popcll(crossing) <= kSerialPairs<NF>) {
        while (crossing) {
          const uint32_t g = base + 64u * (uint32_t)d + (uint32_t)__builtin_ctzll(crossing);
          crossing &= crossing - 1;
          uint32_t i;
          float s;
          const uint32_t k = lane & 31u;
          if (NF == 5 && !refined) {
            // 32 bounds over three bins each cross for 1.7e-3 of the bins of
            // noise (fold 4: 3e-5): first the sums of the bins' own bounds,
            // which are no less than the exact ones, added in their order
            // (searches of 2^24 samples with five folds 17.3 -> 15.9 ms, of
            // 2^23 5.4 -> 5.0; no difference at four)
            pair_folds<NF>(qval, g, hi, i, s);
            if (__ballot(k < NF && i < hi && s > w.thr) == 0) continue;
          }
          pair_folds<NF>(pval, g, hi, i, s);
          bool in = false;
#pragma unroll
          for (int f = 0; f < NF; ++f) in |= k == (uint32_t)f && in_window(i, f);
          append(in && i < hi && s > w.thr, i, k, s);
        }
      } else {
#pragma unroll 1
        for (uint32_t b = 0; b < 2; ++b) {
          const uint32_t i = 2 * (g0 + 64u * (uint32_t)d) + b;
          const bool valid = fail[d] && i < hi;
          float s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
          if (valid) harmonic_sums_rolled<NF>(pval, i, s);
#pragma unroll
          for (int k = 0; k < NF; ++k) append(valid && in_window(i, k) && s[k] > w.thr, i, (uint32_t)k, s[k]);
        }
      }
    }
  }
}

// Largest float v with fold_scale<K>(v) <= thr, by bisection over the float
// order (fold_scale is monotone non-decreasing).
template <int K>
float fold_threshold(float thr) {
  auto from_order = [](int64_t o) {
    const uint32_t u = o >= 0 ? (uint32_t)o : ((uint32_t)(-o) | 0x80000000u);
    float f;
    std::memcpy(&f, &u, 4);
    return f;
  };
  int64_t lo = -(int64_t)0x7F7FFFFF, hi = 0x7F7FFFFF;  // -FLT_MAX .. FLT_MAX
  if (!(psx::fold_scale<K>(from_order(lo)) <= thr)) return -INFINITY;
  if (psx::fold_scale<K>(from_order(hi)) <= thr) return INFINITY;
  while (hi - lo > 1) {
    const int64_t mid = lo + (hi - lo) / 2;
    if (psx::fold_scale<K>(from_order(mid)) <= thr)
      lo = mid;
    else
      hi = mid;
  }
  return from_order(lo);
}

__global__ void k_zero_u32(uint32_t* p) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *p = 0u;
}

}  // namespace

int launch_spec_post(const float2* Z, float* P, uint64_t M, int64_t pstride, const RootTable& rt,
                     const TrialDesc* d_descs, uint32_t ntr, hipStream_t s) {
  if (M < 8 || M > 0x7FFFFFFFull) return psx::fail(PSX_ERR_ARG, "spec_post: unsupported length");
  constexpr int Q = 4;
  const uint64_t chunks = (M / 2 + 1 + kStep - 1) / kStep;  // one wave each
  const unsigned gx = psx::grid_for(chunks * 64, kB * Q, 2048);
  k_spec_post<Q><<<dim3(gx, ntr), kB, 0, s>>>(Z, P, M, pstride, rt, d_descs);
  PSX_CHECK_LAUNCH("k_spec_post");
  return PSX_OK;
}

int launch_spec_rows(const float2* Y, float* P, uint32_t R, uint32_t L, int64_t pstride, const RootTable& rt,
                     const TrialDesc* d_descs, uint32_t ntr, hipStream_t s, const SpecBound* bound) {
  if (R < 4 || R % 2 || L % kColTile || (uint64_t)R * L > 0x7FFFFFFFull || pstride < (int64_t)R * L + 1)
    return psx::fail(PSX_ERR_ARG, "spec_rows: unsupported layout %u x %u", R, L);
  // a tile's bounds lie around its even rows, and so does row R/2's (R - r is
  // even with r; R/2 is the edge workgroups')
  if (bound && (R % 4 || bound->qstride < bound_stride(pstride)))
    return psx::fail(PSX_ERR_ARG, "spec_rows: unsupported bound layout %u x %u", R, L);
  // row tiles of rows [1, R/2), then one row of workgroups for the edge bins
  const unsigned row_tiles = (R / 2 - 1 + kRowTile - 1) / kRowTile;
  static_assert(kColTile * 2 <= kB, "the edge row needs 2L+1 threads from L/kColTile workgroups");
  const dim3 grid(L / kColTile, row_tiles + 1, ntr);
  BoundOut bo{};
  if (bound)
    bo = BoundOut{bound->Q, bound->qstride, max(bound->w.start[0], 0), max(bound->w.end[0], 0),
                  bound->w.thr, bound->out, bound->cap, bound->count};
  const bool hi_fixed = (R & (R - 1)) == 0 && R <= (1u << rt.shift);
  if (!bound && !P) return psx::fail(PSX_ERR_ARG, "spec_rows: no spectrum buffer");
#define PSX_SPEC_ROWS(HF, BD) k_spec_rows<HF, BD><<<grid, kB, 0, s>>>(Y, P, R, L, pstride, rt, d_descs, bo)
  if (!bound)
    hi_fixed ? PSX_SPEC_ROWS(true, false) : PSX_SPEC_ROWS(false, false);
  else
    hi_fixed ? PSX_SPEC_ROWS(true, true) : PSX_SPEC_ROWS(false, true);
#undef PSX_SPEC_ROWS
  PSX_CHECK_LAUNCH("k_spec_rows");
  return PSX_OK;
}

int launch_harm_peaks(const float* P, int64_t pstride, const Windows& w, uint32_t nfolds, const TrialDesc* d_descs,
                      uint32_t ntr, Cand16* out, uint32_t cap, uint32_t* count, hipStream_t s) {
  if (w.hi <= w.lo) return PSX_OK;
  // 32-bit bin arithmetic: j*i < 32 * 2^27
  if (w.hi > (1ll << 27)) return psx::fail(PSX_ERR_UNSUPPORTED, "harm_peaks: more than 2^27 bins");
  // a wave reads up to kHarmWaveBins - 1 bins past w.hi: the spectrum
  // buffer holds that many floats beyond the last trial's row
  if (w.lo < 0 || w.hi > pstride) return psx::fail(PSX_ERR_ARG, "harm_peaks: window outside the spectrum row");
  const unsigned gx = psx::grid_for((uint64_t)(w.hi - w.lo), (uint64_t)kHarmWaveBins * (kB / 64), 2048);
  const dim3 g(gx, ntr);
  switch (nfolds) {
    case 1: k_harm_peaks<1><<<g, kB, 0, s>>>(P, pstride, w, d_descs, out, cap, count); break;
    case 2: k_harm_peaks<2><<<g, kB, 0, s>>>(P, pstride, w, d_descs, out, cap, count); break;
    case 3: k_harm_peaks<3><<<g, kB, 0, s>>>(P, pstride, w, d_descs, out, cap, count); break;
    case 4: k_harm_peaks<4><<<g, kB, 0, s>>>(P, pstride, w, d_descs, out, cap, count); break;
    case 5: k_harm_peaks<5><<<g, kB, 0, s>>>(P, pstride, w, d_descs, out, cap, count); break;
    default: return psx::fail(PSX_ERR_ARG, "nfolds must be 1..5");
  }
  PSX_CHECK_LAUNCH("k_harm_peaks");
  return PSX_OK;
}


float fold_threshold_of(int k, float thr) {
  switch (k) {
    case 1: return fold_threshold<1>(thr);
    case 2: return fold_threshold<2>(thr);
    case 3: return fold_threshold<3>(thr);
    case 4: return fold_threshold<4>(thr);
    case 5: return fold_threshold<5>(thr);
    default: return INFINITY;
  }
}

int64_t bound_stride(int64_t pstride) {
  // a wave's staging reads up to kBoundWavePairs - 1 entries past the window
  // end, plus a chunk of alignment: per-row slack covers both
  return pstride / 2 + kBoundWavePairs + 64;
}

int launch_pool_peaks(const float* P, int64_t pstride, uint64_t nb, const Windows& w, uint16_t* Q, int64_t qstride,
                      const TrialDesc* d_descs, uint32_t ntr, Cand16* out, uint32_t cap, uint32_t* count,
                      hipStream_t s) {
  if (nb < 1 || nb > (1ull << 27) || (int64_t)nb > pstride || pstride % 4 || qstride < bound_stride(pstride))
    return psx::fail(PSX_ERR_ARG, "pool_peaks: unsupported row layout");
  const unsigned gx = psx::grid_for((nb + 3) / 4, kB, 1024);
  k_pool_peaks<<<dim3(gx, ntr), kB, 0, s>>>(P, pstride, (uint32_t)nb, w, Q, qstride, d_descs, out, cap, count);
  PSX_CHECK_LAUNCH("k_pool_peaks");
  return PSX_OK;
}

int write_rows_source(const RowsSource& rs, void* d_src) {
  static_assert(sizeof(ExactSrc) <= kRowsSourceBytes, "kRowsSourceBytes");
  if (!d_src || !rs.Y || rs.R < 4 || (uint64_t)rs.R * rs.L > 0x7FFFFFFFull)
    return psx::fail(PSX_ERR_ARG, "write_rows_source: bad layout");
  const uint32_t R = rs.R;
  const ExactSrc e{rs.Y, R, rs.L, (R & (R - 1)) == 0 ? (uint32_t)__builtin_ctz(R) : 32u, rs.rt};
  PSX_CHECK_HIP(hipMemcpy(d_src, &e, sizeof(e), hipMemcpyHostToDevice));
  return PSX_OK;
}

int launch_harm_bound(const float* P, int64_t pstride, const uint16_t* Q, int64_t qstride, const Windows& w,
                      uint32_t nfolds, const TrialDesc* d_descs, uint32_t ntr, Cand16* out, uint32_t cap,
                      uint32_t* count, hipStream_t s, const RowsSource* rows, const void* d_rows_src) {
  if (w.hi <= w.lo) return PSX_OK;
  if (w.hi > (1ll << 27)) return psx::fail(PSX_ERR_UNSUPPORTED, "harm_bound: more than 2^27 bins");
  if (w.lo < 0 || w.hi > pstride || qstride < bound_stride(pstride))
    return psx::fail(PSX_ERR_ARG, "harm_bound: window outside the spectrum row");
  if (!rows && !P) return psx::fail(PSX_ERR_ARG, "harm_bound: no spectrum for the exact sums");
  if (rows && (!d_rows_src || w.hi > (int64_t)rows->R * rows->L + 1 ||
               (uint64_t)rows->R * rows->L > 0x7FFFFFFFull))
    return psx::fail(PSX_ERR_ARG, "harm_bound: window outside the row layout");
  const ExactSrc* src = rows ? (const ExactSrc*)d_rows_src : nullptr;
  FoldThr ft{};
  for (int k = 1; k <= 5; ++k) ft.t[k] = fold_threshold_of(k, w.thr);
  const uint64_t pairs = ((uint64_t)w.hi + 1) / 2 - bound_first_pair(w.lo);
  const unsigned gx = psx::grid_for(pairs, kBoundWavePairs, 1u << 16);
  const uint32_t xcd = ntr % 8 == 0 ? 1u : 0u;
  const dim3 g(gx, ntr);
  const uint16_t* q = Q;
#define PSX_HB(NF, FR) \
  k_harm_bound<NF, FR><<<g, 64, 0, s>>>(P, pstride, q, qstride, w, ft, d_descs, src, xcd, out, cap, count)
  const bool fr = rows != nullptr;
  switch (nfolds) {
    case 1: fr ? PSX_HB(1, true) : PSX_HB(1, false); break;
    case 2: fr ? PSX_HB(2, true) : PSX_HB(2, false); break;
    case 3: fr ? PSX_HB(3, true) : PSX_HB(3, false); break;
    case 4: fr ? PSX_HB(4, true) : PSX_HB(4, false); break;
    case 5: fr ? PSX_HB(5, true) : PSX_HB(5, false); break;
    default: return psx::fail(PSX_ERR_ARG, "nfolds must be 1..5");
  }
#undef PSX_HB
  PSX_CHECK_LAUNCH("k_harm_bound");
  return PSX_OK;
}

int launch_zero(uint32_t* p, hipStream_t s) {
  k_zero_u32<<<1, 64, 0, s>>>(p);
  PSX_CHECK_LAUNCH("k_zero_u32");
  return PSX_OK;
}

}  // namespace batch
}  // namespace psx
