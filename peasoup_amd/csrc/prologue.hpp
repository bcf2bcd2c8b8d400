// prologue.hpp - the DM prologue (pipeline_multi.cu:170-238) of a group of
// DM trials in one set of launches.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fft_plan.hpp"

namespace psx {
namespace prologue {

// GPU_remove_baseline's loop (src/kernels.cu:463-479) runs kBaselineSteps
// iterations on the device; done == 0 afterwards means it had not stopped and
// the host finishes the DM (a second iteration is usual for short series with
// an offset, a third needs one of about 8 n).
constexpr int kBaselineSteps = 2;
struct BaselineState {
  int32_t count;
  int32_t done;
  float mean[kBaselineSteps];
};
// Per DM, copied to the host: the loop's state and the sums of the
// interbinned spectrum (sum x, sum x^2 over the nb bins).
struct Result {
  BaselineState base;
  double2 sums;
};

// Work of a group of up to G trials of n samples (n/2 = M), besides the two
// G x M complex buffers the caller passes.
struct Work {
  uint64_t n = 0, M = 0;
  uint32_t G = 0;
  uint64_t c5 = 0, c25 = 0, c125 = 0, med_stride = 0;
  float* med = nullptr;        // G x (c5 + c25 + c125)
  double2* partial = nullptr;  // G x kPartials
  Result* res = nullptr;       // G
  uint32_t* zmask = nullptr;   // one bit per bin: zapped
};
uint64_t work_bytes(uint64_t n, uint32_t G);
int work_create(uint64_t n, uint32_t G, Work& w);
void work_destroy(Work& w);

// Baseline removal, zero padding: src (trial d at src + d*stride, nreal
// samples; may be tim itself with stride n) -> tim (n samples per trial).
int baseline(const Work& w, const float* src, int64_t stride, uint64_t nreal, float* tim, uint32_t ndm, hipStream_t s);
// Bits of the bins that the birdies cover (zap_birdies_kernel,
// src/kernels.cu:1063-1084) into w.zmask.
int zap_mask(const Work& w, const float* d_freqs, const float* d_widths, uint32_t nbirdies, float bin_width,
             hipStream_t s);
// Half-length spectra Z (natural order, stride M) -> running medians, then
// dereddened, zapped (zap) and statistics (w.res), and the C2R input W
// (stride M; conjugated, as the forward passes of the inverse take it).
int spectra(const Work& w, const float2* Z, float2* W, const psx::fft::RootTable& rt, double bin_width, float b5,
            float b25, bool zap, uint32_t ndm, hipStream_t s);

}  // namespace prologue
}  // namespace psx
