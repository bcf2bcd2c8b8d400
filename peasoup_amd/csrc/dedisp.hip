// dedisp.hip - incoherent dedispersion of SIGPROC filterbank data (gfx950).
//
// The reference dedisperses with libdedisp (dedisp_execute through
// Dedisperser, include/transforms/dedisperser.hpp:105-186), a dependency not
// in its tree.  This file restates libdedisp's direct algorithm with its
// published delay table, DM-list recurrence and float output scaling:
//   delay(dm, c) = rn(dm * table[c]),
//   table[c]     = 4.15e3 / tsamp * (1/(f0 + c df)^2 - 1/f0^2)   (float)
//   out[dm][t]   = sum_c v(t + delay(dm, c), c) / ((2^nbits - 1) * nchans)
// Three kernels:
//   k_delays    the (DM, channel) delay table, computed on the device;
//   k_unpack_t  packed time-major samples -> one u8 row per channel
//               (a 16 KB byte tile transposed through LDS);
//   k_dedisp_lds / k_dedisp  the sums, 1,024 samples of four DM trials per
//               wave as packed integers, from rows staged in LDS or directly.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "dedisp_pitch.hpp"
#include "trace.hpp"
#include "psx.h"

namespace {

constexpr unsigned kB = 256;
constexpr uint32_t kMaxChans = 8192;

typedef uint32_t psx_u1 __attribute__((ext_vector_type(1), aligned(1)));
typedef uint32_t psx_u4 __attribute__((ext_vector_type(4), aligned(1)));
typedef float psx_f4 __attribute__((ext_vector_type(4), aligned(4)));

// ------------------------------------------------------------------ delays
// Only the unmasked channels have rows: channel c is row rank(c), the number
// of unmasked channels before it.  The mask and the DM list travel as kernel
// arguments, so the call uploads nothing.
struct ChanMask {
  uint32_t on[kMaxChans / 32];      // bit c set: channel c is summed
  uint16_t before[kMaxChans / 32];  // unmasked channels below 32*w
};
__device__ inline bool chan_on(uint32_t word, uint32_t c) { return (word >> (c & 31u)) & 1u; }
__device__ inline uint32_t chan_rank(uint32_t word, uint32_t before, uint32_t c) {
  return before + __popc(word & ((1u << (c & 31u)) - 1u));
}

// rn(dm * table[c]) of every unmasked channel for up to kDelayDms DM trials;
// table[c] is psx_dedisp_delay_table's expression in the same IEEE operations.
constexpr uint32_t kDelayDms = 512;
struct DelayArgs {
  ChanMask mask;
  float dm[kDelayDms];
};
__host__ __device__ inline float table_entry(uint32_t c, double scale, float f0, float df) {
  const float b = 1.f / f0;
  const float a = 1.f / (f0 + (float)c * df);
  return (float)(scale * (double)(a * a - b * b));
}
__host__ __device__ inline int32_t delay_of(float dm, float tab) { return (int32_t)rintf(dm * tab); }

__global__ void __launch_bounds__(kB) k_delays(int32_t* __restrict__ delays, uint32_t nchans, uint32_t nrows,
                                               double scale, float f0, float df, const DelayArgs a) {
  const uint32_t c = blockIdx.x * kB + threadIdx.x;
  if (c >= nchans) return;
  const uint32_t word = a.mask.on[c >> 5];
  if (!chan_on(word, c)) return;
  delays[(uint64_t)blockIdx.y * nrows + chan_rank(word, a.mask.before[c >> 5], c)] =
      delay_of(a.dm[blockIdx.y], table_entry(c, scale, f0, df));
}

// ------------------------------------------------------------------ unpack
// A workgroup transposes TB input bytes x T samples (16 KB) through LDS:
// dwords in (rows of TB contiguous bytes), then each lane takes 16 samples of
// four byte columns, turns them into four dwords per column with byte
// permutes, splits the K channels of each byte and stores 16 bytes per
// channel.  TB follows the sample's bytes (16..128), so narrow filterbanks
// fill the tile too.  LDS dword (t, g) is at t*PW + g + (t/16)*S with
// S = TB/16: both sides then touch 64 different banks.  Memory bound;
// 513 MiB of 8-bit samples (1,024 channels): 0.82 ms (byte accesses, 64-byte
// tiles) -> 0.35 ms.
template <int NBITS, int TB>
__global__ void __launch_bounds__(kB) k_unpack_t(const uint8_t* __restrict__ in, uint64_t nsamps, uint32_t nchans,
                                                 uint8_t* __restrict__ out, const ChanMask cm) {
  constexpr unsigned K = 8 / NBITS;  // channels per byte
  constexpr uint32_t mask = ((1u << NBITS) - 1u) * 0x01010101u;
  constexpr unsigned PW = TB / 4, T = 16384 / TB, S = TB / 16;
  __shared__ uint32_t tile[T * PW + (T / 16) * S];
  const uint64_t rowbytes = (uint64_t)nchans * NBITS / 8, total = nsamps * rowbytes;
  const uint64_t t0 = (uint64_t)blockIdx.x * T;
  const uint32_t b0 = blockIdx.y * TB;
#pragma unroll
  for (unsigned i = 0; i < T * PW / kB; ++i) {
    const unsigned k = i * kB + threadIdx.x, t = k / PW, g = k % PW;
    const uint64_t at = (t0 + t) * rowbytes + b0 + 4 * g;
    uint32_t v = 0;
    if (t0 + t < nsamps && b0 + 4 * g < rowbytes) {
      if (at + 4 <= total) {
        v = (*(const PSX_GLOBAL psx_u1*)(in + at)).x;
      } else {  // the last bytes of the input
        for (unsigned j = 0; j < 4 && at + j < total; ++j) v |= (uint32_t)in[at + j] << (8 * j);
      }
    }
    tile[t * PW + g + (t / 16) * S] = v;
  }
  __syncthreads();
  const unsigned tq = threadIdx.x % (T / 16), g = threadIdx.x / (T / 16);
  if (t0 + 16 * tq >= nsamps || b0 + 4 * g >= rowbytes) return;
  uint32_t col[4][4];  // [byte column][four samples each]
#pragma unroll
  for (unsigned q = 0; q < 4; ++q) {
    uint32_t r[4];
#pragma unroll
    for (unsigned j = 0; j < 4; ++j) r[j] = tile[(16 * tq + 4 * q + j) * PW + g + tq * S];
    // 4x4 bytes: pairs of rows interleaved, then pairs of pairs
    const uint32_t a0 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u), a1 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
    const uint32_t a2 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u), a3 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
    col[0][q] = __builtin_amdgcn_perm(a2, a0, 0x05040100u);
    col[1][q] = __builtin_amdgcn_perm(a2, a0, 0x07060302u);
    col[2][q] = __builtin_amdgcn_perm(a3, a1, 0x05040100u);
    col[3][q] = __builtin_amdgcn_perm(a3, a1, 0x07060302u);
  }
  // the lane's 4K channels share one mask word
  const uint32_t c0 = (b0 + 4 * g) * K, word = cm.on[c0 >> 5], before = cm.before[c0 >> 5];
  const uint64_t tt = t0 + 16 * tq;
  const bool whole = tt + 16 <= nsamps;
#pragma unroll
  for (unsigned j = 0; j < 4; ++j) {
#pragma unroll
    for (unsigned k = 0; k < K; ++k) {
      const uint32_t c = c0 + j * K + k;
      if (c >= nchans || !chan_on(word, c)) continue;
      uint32_t x[4];
#pragma unroll
      for (unsigned q = 0; q < 4; ++q) x[q] = (col[j][q] >> (k * NBITS)) & mask;
      uint8_t* row = out + (uint64_t)chan_rank(word, before, c) * nsamps + tt;
      if (whole) {
        *(PSX_GLOBAL psx_u4*)row = psx_u4{x[0], x[1], x[2], x[3]};
      } else {
        for (unsigned s = 0; tt + s < nsamps; ++s) row[s] = (uint8_t)(x[s / 4] >> (8 * (s % 4)));
      }
    }
  }
}

// --------------------------------------------------------------------- sum
// out[dm][t] = sum_c row_c[t + delay(dm, c)] / denom over tiles of 1,024
// samples, kDms DM trials per wave.  Samples are added four to a dword.  Up to
// 4 bits a run of channels is added as packed bytes (16 x 15, 84 x 3 and
// 252 x 1 fit), then as pairs; 8-bit samples go to the pairs at once.  Of the
// two pairs of 16-bit sums only the odd bytes' one is kept (hi); beside it the
// plain sum of the dwords mod 2^32 (lo), which is the even bytes' pair plus
// 2^8 times the odd bytes' one.  That takes 4 instructions per 8 samples at 8
// bits (6 with both pairs masked out of each dword) and 2 per 16 up to 4 bits.
// The pairs hold 65535: WIDE sums (channels * the largest sample above that)
// spill them into 32-bit sums every kFlush channels.  All sums are exact
// integers.
constexpr int kDms = 4;             // DM trials per wave
using psx::kTileSamps;              // samples per wave: four dwords per lane

template <int NBITS, bool WIDE>
struct DmSums {
  static constexpr uint32_t kFlush = NBITS == 8 ? 256 : 4096;  // kFlush * (2^NBITS - 1) <= 65535
  // channels per run: as many as four packed bytes hold (a multiple of 4)
  static constexpr uint32_t kRun = NBITS == 8 ? kFlush : 255 / ((1 << NBITS) - 1) / 4 * 4;
  uint32_t lo[4], hi[4];  // packed dwords (mod 2^32); samples 4q+1, 4q+3 as pairs
  uint32_t run[NBITS == 8 ? 1 : 4];
  uint32_t sum[WIDE ? 16 : 1];
  __device__ void clear() {
#pragma unroll
    for (int q = 0; q < 4; ++q) lo[q] = hi[q] = 0u;
    if constexpr (NBITS < 8) {
#pragma unroll
      for (int q = 0; q < 4; ++q) run[q] = 0u;
    }
    if constexpr (WIDE) {
#pragma unroll
      for (int q = 0; q < 16; ++q) sum[q] = 0u;
    }
  }
  __device__ static uint32_t odd(uint32_t x) { return __builtin_amdgcn_perm(0u, x, 0x0C030C01u); }
  // dword q of four channels
  __device__ void add4(int q, uint32_t x0, uint32_t x1, uint32_t x2, uint32_t x3) {
    if constexpr (NBITS < 8) {
      run[q] = run[q] + x0 + x1;
      run[q] = run[q] + x2 + x3;
    } else {
      lo[q] = lo[q] + x0 + x1;
      hi[q] = hi[q] + odd(x0) + odd(x1);
      lo[q] = lo[q] + x2 + x3;
      hi[q] = hi[q] + odd(x2) + odd(x3);
    }
  }
  // after at most kRun channels
  __device__ void end_run() {
    if constexpr (NBITS < 8) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        lo[q] += run[q];
        hi[q] += odd(run[q]);
        run[q] = 0u;
      }
    }
  }
  // samples 4q, 4q+2 as pairs
  __device__ uint32_t even(int q) const { return lo[q] - (hi[q] << 8); }
  // after at most kFlush channels
  __device__ void flush() {
    if constexpr (WIDE) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        sum[4 * q] += even(q) & 0xFFFFu;
        sum[4 * q + 1] += hi[q] & 0xFFFFu;
        sum[4 * q + 2] += even(q) >> 16;
        sum[4 * q + 3] += hi[q] >> 16;
        lo[q] = hi[q] = 0u;
      }
    }
  }
  __device__ uint32_t at(int q, int i) const {
    if constexpr (WIDE) return sum[4 * q + i];
    else return i == 0 ? even(q) & 0xFFFFu : i == 1 ? hi[q] & 0xFFFFu : i == 2 ? even(q) >> 16 : hi[q] >> 16;
  }
  // samples t .. t+3 of dword q to o (the first n of them)
  __device__ void store(int q, float denom, float* o, uint32_t n) const {
    const psx_f4 f = {(float)at(q, 0) / denom, (float)at(q, 1) / denom, (float)at(q, 2) / denom,
                      (float)at(q, 3) / denom};
    if (n >= 4) {
      *(PSX_GLOBAL psx_f4*)o = f;
    } else {
#pragma unroll
      for (uint32_t i = 0; i < 3; ++i)
        if (i < n) o[i] = f[i];
    }
  }
};

// Staged form, for ascending DM lists: a workgroup of NW waves owns 4*NW
// neighbouring DM trials of one tile.  Their reads of a channel cover one
// stretch of its row, [tile + delay of the first DM, + 1024 + spread), which
// the workgroup copies into LDS once for all of them, in four copies shifted
// by 0..3 bytes: the (DM, channel) stretch at any byte delay is then a run of
// whole dwords of one copy, read by consecutive lanes without bank conflicts
// (byte-shifted reads of one copy would need a shift per dword; unaligned
// 16-byte loads straight from the rows take 6.0 ms for 128 DMs x 987 8-bit
// channels x 521k samples, this form 2.2 ms, and one byte per lane and load,
// one DM per workgroup, took 33.5 ms).  Channels are staged four at a time,
// double buffered: the next four are loaded into registers while the current
// ones are summed.  What a stage needs of the delay table comes from LDS too,
// filled for 64 channels at a time by all threads: with 20 scalar loads and
// 160 scalar instructions per wave and stage, and the stage's addresses a
// dependent load away, it took 2.6 ms.  Bound by its instructions and by the
// waits of the stages: the adds are 55% of the vector ones (1.2 ms of issue in
// all), staging four copies costs 0.8 ms of the 2.2, waiting for the rows 0.2.
constexpr int kChunk = 4;             // channels per stage
constexpr uint32_t kSpan = 64;        // channels per table
constexpr uint32_t kMaxPitch = 512;   // dwords per copy, at most: 64 KB of LDS (and 9 of tables), two workgroups per CU
struct SumArgs {
  const uint8_t* rows;
  uint64_t nsamps_in;
  uint32_t nrows;
  const int32_t* delays;
  float denom;
  float* out;
  uint64_t out_stride, nout;
  uint32_t ndm;
  uint32_t pitch;  // staged form: dwords per shifted copy
};

template <int NBITS, int NW, bool WIDE>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4)))
k_dedisp_lds(const SumArgs a, uint32_t ngroups, uint32_t nblocks) {
  using Sums = DmSums<NBITS, WIDE>;
  constexpr int kMaxTasks = (int)kMaxPitch / (64 * NW);
  extern __shared__ uint4 lds4[];
  uint32_t* const lds = reinterpret_cast<uint32_t*>(lds4);  // [2][kChunk][4][pitch], then the tables
  uint32_t* const area = lds + 2 * kChunk * 4 * a.pitch;
  // of the channels of two table spans: byte offset in a stage's copies of
  // every (channel, DM) stretch, and the first DM's delay
  uint2* const offs = reinterpret_cast<uint2*>(area);                             // [2][kSpan/4][4*NW]
  int32_t* const first = reinterpret_cast<int32_t*>(area + 2 * kSpan * 2 * NW);  // [2*kSpan]
  const uint32_t blk = psx::xcd_logical_block(blockIdx.x, nblocks);
  const uint64_t tbase = (uint64_t)(blk / ngroups) * kTileSamps;
  const uint32_t g0 = (blk % ngroups) * (kDms * NW);  // first DM of the group
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t dm0 = g0 + wave * kDms;
  // one thread per DM and four channels; channels past the last one hold
  // zeros at any offset
  static_assert(kSpan / 4 * kDms * NW == 64 * NW, "one table entry per thread");
  auto fill = [&](uint32_t span) {
    const uint32_t q = threadIdx.x % (kSpan / 4), d = threadIdx.x / (kSpan / 4);
    const int32_t* f = a.delays + (uint64_t)g0 * a.nrows;
    const int32_t* dl = a.delays + (uint64_t)min(g0 + d, a.ndm - 1) * a.nrows;
    uint32_t o[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t c = min(span * kSpan + 4 * q + j, a.nrows - 1);
      const uint32_t rel = (uint32_t)(dl[c] - f[c]);
      o[j] = 4u * ((4 * j + (rel & 3u)) * a.pitch + (rel >> 2));
      if (d == 0) first[(span & 1u) * kSpan + 4 * q + j] = f[c];
    }
    offs[((span & 1u) * (kSpan / 4) + q) * (kDms * NW) + d] = make_uint2(o[0] | o[1] << 16, o[2] | o[3] << 16);
  };
  const uint32_t nstep = a.pitch / 4;  // 16-byte steps of a copy
  const uint32_t ntasks = kChunk * nstep;
  uint32_t r[kMaxTasks][5];
  // task: 16 bytes of one channel's stretch and the dword behind them.  A
  // step that starts past its row is never summed and loads nothing; one that
  // starts inside it reads at most 19 bytes past the row, in the next row or
  // (last row) the delay table behind the rows
  auto load = [&](uint32_t c0) {
#pragma unroll
    for (int i = 0; i < kMaxTasks; ++i) {
      const uint32_t task = (uint32_t)i * 64 * NW + threadIdx.x;
      const uint32_t j = task / nstep, st = task % nstep, c = c0 + j;
#pragma unroll
      for (int q = 0; q < 5; ++q) r[i][q] = 0u;
      if (task < ntasks && c < a.nrows) {
        const uint64_t at = tbase + (uint32_t)first[c % (2 * kSpan)] + 16u * st;
        if (at < a.nsamps_in) {
          const PSX_GLOBAL uint8_t* p = (const PSX_GLOBAL uint8_t*)(a.rows + (uint64_t)c * a.nsamps_in + at);
          const psx_u4 x = *(const PSX_GLOBAL psx_u4*)p;
          r[i][0] = x.x;
          r[i][1] = x.y;
          r[i][2] = x.z;
          r[i][3] = x.w;
          r[i][4] = (*(const PSX_GLOBAL psx_u1*)(p + 16)).x;
        }
      }
    }
  };
  auto put = [&](uint32_t buf) {
#pragma unroll
    for (int i = 0; i < kMaxTasks; ++i) {
      const uint32_t task = (uint32_t)i * 64 * NW + threadIdx.x;
      if (task >= ntasks) continue;
      const uint32_t j = task / nstep, st = task % nstep;
      uint32_t* d = lds + ((buf * kChunk + j) * 4) * a.pitch + 4 * st;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        uint4 w;
        w.x = __builtin_amdgcn_alignbyte(r[i][1], r[i][0], s);
        w.y = __builtin_amdgcn_alignbyte(r[i][2], r[i][1], s);
        w.z = __builtin_amdgcn_alignbyte(r[i][3], r[i][2], s);
        w.w = __builtin_amdgcn_alignbyte(r[i][4], r[i][3], s);
        *reinterpret_cast<uint4*>(d + s * a.pitch) = w;
      }
    }
  };
  Sums acc[kDms];
#pragma unroll
  for (int k = 0; k < kDms; ++k) acc[k].clear();
  fill(0);
  __syncthreads();
  load(0);
  put(0);
  __syncthreads();
  uint32_t buf = 0, flushed = 0;
#pragma unroll 1
  for (uint32_t cs = 0; cs < a.nrows; cs += Sums::kRun) {
    const uint32_t ce = min(cs + Sums::kRun, a.nrows);
    if (WIDE && ce - flushed > Sums::kFlush) {
#pragma unroll
      for (int k = 0; k < kDms; ++k) acc[k].flush();
      flushed = cs;
    }
#pragma unroll 1
    for (uint32_t c0 = cs; c0 < ce; c0 += kChunk) {
      // the next span's entries replace those of the previous one, last read
      // before the last barrier
      if (c0 % kSpan == 0) fill(c0 / kSpan + 1);
      const uint4* o4 =
          reinterpret_cast<const uint4*>(offs + c0 % (2 * kSpan) / 4 * (kDms * NW) + wave * kDms);
      const uint4 oa = o4[0], ob = o4[1];
      const uint32_t o[8] = {oa.x, oa.y, oa.z, oa.w, ob.x, ob.y, ob.z, ob.w};
      load(c0 + kChunk);
      const uint32_t base = (buf * (kChunk * 4) * a.pitch + lane) * 4;
#pragma unroll
      for (int k = 0; k < kDms; ++k) {
        uint32_t x[kChunk][4];
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
          const uint32_t w = o[2 * k + j / 2];
          const uint32_t at = base + (j & 1 ? w >> 16 : w & 0xFFFFu);
          const uint32_t* p = reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(lds) + at);
#pragma unroll
          for (int q = 0; q < 4; ++q) x[j][q] = p[64 * q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[k].add4(q, x[0][q], x[1][q], x[2][q], x[3][q]);
      }
      put(buf ^ 1u);
      __syncthreads();
      buf ^= 1u;
    }
#pragma unroll
    for (int k = 0; k < kDms; ++k) acc[k].end_run();
  }
#pragma unroll
  for (int k = 0; k < kDms; ++k) acc[k].flush();
#pragma unroll
  for (int k = 0; k < kDms; ++k) {
    if (dm0 + (uint32_t)k >= a.ndm) continue;
    float* o = a.out + (uint64_t)(dm0 + k) * a.out_stride + tbase;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t t = 4 * (lane + 64 * q);
      if (tbase + t < a.nout) acc[k].store(q, a.denom, o + t, (uint32_t)min(a.nout - tbase - t, (uint64_t)4));
    }
  }
}

// Direct form, for lists whose groups spread further than the staged form's
// LDS holds or that do not ascend: every (DM, channel) stretch straight from
// its row, one unaligned 16-byte load per lane from a scalar base
// (row + delay).
template <int NBITS, int D, bool WIDE>
__global__ void __launch_bounds__(kB) k_dedisp(const SumArgs a, uint32_t ngroups, uint32_t nitems) {
  using Sums = DmSums<NBITS, WIDE>;
  const uint32_t blk = psx::xcd_logical_block(blockIdx.x, gridDim.x);
  const uint32_t item = __builtin_amdgcn_readfirstlane(blk * (kB / 64) + (threadIdx.x >> 6));
  if (item >= nitems) return;
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t tbase = (uint64_t)(item / ngroups) * kTileSamps;
  const uint32_t dm0 = (item % ngroups) * D;
  // lanes past the output read the tile's last used stretch instead: a read
  // ends at most 15 samples past nout + max_delay = nsamps_in, in the next
  // row or (last row) in the delay table behind the rows
  const uint32_t left = (uint32_t)min(a.nout - tbase, (uint64_t)kTileSamps);
  const uint32_t off = min(lane * 16u, (left - 1) & ~15u);
  const int32_t* dl[D];
#pragma unroll
  for (int k = 0; k < D; ++k) dl[k] = a.delays + (uint64_t)min(dm0 + (uint32_t)k, a.ndm - 1) * a.nrows;
  const uint8_t* base = a.rows + tbase;
  auto load = [&](uint32_t c, int32_t d) {
    const PSX_GLOBAL uint8_t* p = (const PSX_GLOBAL uint8_t*)(base + (uint64_t)c * a.nsamps_in + (uint32_t)d);
    return *(const PSX_GLOBAL psx_u4*)(p + off);
  };
  Sums acc[D];
#pragma unroll
  for (int k = 0; k < D; ++k) acc[k].clear();
  uint32_t flushed = 0;
  for (uint32_t cs = 0; cs < a.nrows; cs += Sums::kRun) {
    const uint32_t ce = min(cs + Sums::kRun, a.nrows);
    if (WIDE && ce - flushed > Sums::kFlush) {
#pragma unroll
      for (int k = 0; k < D; ++k) acc[k].flush();
      flushed = cs;
    }
    uint32_t c = cs;
    for (; c + 4 <= ce; c += 4) {
#pragma unroll
      for (int k = 0; k < D; ++k) {
        psx_u4 x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = load(c + j, dl[k][c + j]);
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[k].add4(q, x[0][q], x[1][q], x[2][q], x[3][q]);
      }
    }
#pragma unroll 1
    for (; c < ce; ++c) {
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const psx_u4 x = load(c, dl[k][c]);
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[k].add4(q, x[q], 0u, 0u, 0u);
      }
    }
#pragma unroll
    for (int k = 0; k < D; ++k) acc[k].end_run();
  }
#pragma unroll
  for (int k = 0; k < D; ++k) acc[k].flush();
#pragma unroll
  for (int k = 0; k < D; ++k) {
    if (dm0 + (uint32_t)k >= a.ndm) continue;
    float* o = a.out + (uint64_t)(dm0 + k) * a.out_stride + tbase;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t t = 16 * lane + 4 * q;
      if (t < left) acc[k].store(q, a.denom, o + t, min(left - t, 4u));
    }
  }
}

uint64_t round_up(uint64_t x, uint64_t a) { return (x + a - 1) / a * a; }

template <int NBITS>
void launch_unpack(const uint8_t* in, uint64_t nsamps, uint32_t nchans, uint8_t* rows, const ChanMask& cm,
                   hipStream_t s) {
  const uint64_t rowbytes = (uint64_t)nchans * NBITS / 8;
  const uint64_t tb = rowbytes <= 16 ? 16 : rowbytes <= 32 ? 32 : rowbytes <= 64 ? 64 : 128;
  const dim3 g((unsigned)((nsamps + 16384 / tb - 1) / (16384 / tb)), (unsigned)((rowbytes + tb - 1) / tb));
  if (tb == 16) k_unpack_t<NBITS, 16><<<g, kB, 0, s>>>(in, nsamps, nchans, rows, cm);
  else if (tb == 32) k_unpack_t<NBITS, 32><<<g, kB, 0, s>>>(in, nsamps, nchans, rows, cm);
  else if (tb == 64) k_unpack_t<NBITS, 64><<<g, kB, 0, s>>>(in, nsamps, nchans, rows, cm);
  else k_unpack_t<NBITS, 128><<<g, kB, 0, s>>>(in, nsamps, nchans, rows, cm);
}

template <int NBITS, int D, bool WIDE>
int launch_direct(const SumArgs& a, hipStream_t s) {
  const uint64_t groups = (a.ndm + D - 1) / D, tiles = (a.nout + kTileSamps - 1) / kTileSamps;
  PSX_REQUIRE(groups * tiles < (1ull << 31), "psx_dedisperse: too many DMs x samples");
  const uint32_t items = (uint32_t)(groups * tiles);
  k_dedisp<NBITS, D, WIDE><<<(items + kB / 64 - 1) / (kB / 64), kB, 0, s>>>(a, (uint32_t)groups, items);
  PSX_CHECK_LAUNCH("k_dedisp");
  return PSX_OK;
}
template <int NBITS, int NW, bool WIDE>
int launch_lds(const SumArgs& a, hipStream_t s) {
  const uint64_t groups = (a.ndm + kDms * NW - 1) / (kDms * NW), tiles = (a.nout + kTileSamps - 1) / kTileSamps;
  PSX_REQUIRE(groups * tiles < (1ull << 31), "psx_dedisperse: too many DMs x samples");
  const uint32_t blocks = (uint32_t)(groups * tiles);
  const uint32_t lds = 2 * kChunk * 4 * a.pitch * 4 + 2 * kSpan * 2 * NW * 4 + 2 * kSpan * 4;
  if (lds > 65536)
    PSX_CHECK_HIP(hipFuncSetAttribute((const void*)&k_dedisp_lds<NBITS, NW, WIDE>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  k_dedisp_lds<NBITS, NW, WIDE><<<blocks, 64 * NW, lds, s>>>(a, (uint32_t)groups, blocks);
  PSX_CHECK_LAUNCH("k_dedisp_lds");
  return PSX_OK;
}
template <int NBITS>
int launch_sum(SumArgs a, const float* dm_list, float tmax, hipStream_t s) {
  constexpr uint32_t kMax = (1u << NBITS) - 1u;
  const bool wide = (uint64_t)a.nrows * kMax > 65535u;
  constexpr bool kCanWide = (uint64_t)kMaxChans * kMax > 65535u;
  const uint64_t tiles = (a.nout + kTileSamps - 1) / kTileSamps;
  // eight waves (32 DM trials) share a staged stretch; four where eight would
  // leave less than two workgroups per CU or where their stretch is too long
  // for the LDS (128 DMs of 512 2-bit channels x 400k samples to DM 200:
  // directly 2.43 ms, four waves 1.16).  Two waves hold too many of their
  // stretch's bytes in registers and lose to the direct form (40 DMs of 512
  // 4-bit channels to DM 250: 1.63 ms against 0.41)
  uint32_t nw = a.ndm > 16 && (a.ndm + 31) / 32 * tiles >= 512 ? 8 : 4;
  a.pitch = psx::staged_pitch(dm_list, a.ndm, kDms * nw, tmax);
  if (nw == 8 && a.pitch > kMaxPitch) {
    nw = 4;
    a.pitch = psx::staged_pitch(dm_list, a.ndm, kDms * nw, tmax);
  }
  if (a.nrows > 0 && a.ndm > 2 && a.pitch && a.pitch <= kMaxPitch) {
    if constexpr (kCanWide)
      if (wide) return nw == 8 ? launch_lds<NBITS, 8, true>(a, s) : launch_lds<NBITS, 4, true>(a, s);
    return nw == 8 ? launch_lds<NBITS, 8, false>(a, s) : launch_lds<NBITS, 4, false>(a, s);
  }
  // four DM trials per wave share cache lines; one where four would leave the
  // chip short of waves (fewer than eight per CU)
  const bool four = (uint64_t)((a.ndm + 3) / 4) * tiles >= 2048;
  if constexpr (kCanWide)
    if (wide) return four ? launch_direct<NBITS, 4, true>(a, s) : launch_direct<NBITS, 1, true>(a, s);
  return four ? launch_direct<NBITS, 4, false>(a, s) : launch_direct<NBITS, 1, false>(a, s);
}

}  // namespace

extern "C" int psx_dedisp_delay_table(uint32_t nchans, float tsamp, float f0, float df, float* table) {
  PSX_REQUIRE(table && nchans > 0 && tsamp > 0 && f0 > 0, "psx_dedisp_delay_table: bad arguments");
  const double scale = 4.15e3 / (double)tsamp;
  for (uint32_t c = 0; c < nchans; ++c) table[c] = table_entry(c, scale, f0, df);
  return psx::ok();
}

extern "C" int psx_dedisp_dm_list(float dm_start, float dm_end, float tsamp, float pulse_width_us, float f0,
                                  float df, uint32_t nchans, float tol, float* out, uint32_t cap, uint32_t* count) {
  PSX_REQUIRE(count && tsamp > 0 && nchans > 0 && tol > 1.0f, "psx_dedisp_dm_list: bad arguments");
  // smearing budget: (dt^2 + width^2)(tol^2 - 1) with the intra-channel and
  // across-band smearing terms at the centre frequency (GHz), times in us
  const double dt = (double)tsamp * 1e6;
  const double ti = (double)pulse_width_us;
  const double f_ghz = ((double)f0 + ((double)(nchans / 2) - 0.5) * (double)df) * 1e-3;
  const double tol2 = (double)tol * (double)tol;
  const double a = 8.3 * (double)df / (f_ghz * f_ghz * f_ghz);
  const double a2 = a * a;
  const double b2 = a2 * (double)((double)nchans * (double)nchans / 16.0);
  const double c = (dt * dt + ti * ti) * (tol2 - 1.0);
  std::vector<float> dms(1, dm_start);
  while (dms.back() < dm_end) {
    const double prev = dms.back();
    const double k = c + tol2 * a2 * prev * prev;
    const double next = (b2 * prev + std::sqrt(-a2 * b2 * prev * prev + (a2 + b2) * k)) / (a2 + b2);
    dms.push_back((float)next);
    PSX_REQUIRE(dms.size() < (1u << 24), "psx_dedisp_dm_list: DM list does not converge");
  }
  *count = (uint32_t)dms.size();
  for (uint32_t i = 0; i < *count && out && i < cap; ++i) out[i] = dms[i];
  if (out && *count > cap) return psx::fail(PSX_ERR_OVERFLOW, "DM list holds %u of %u", cap, *count);
  return psx::ok();
}

extern "C" uint64_t psx_dedisp_max_delay(const float* dm_list, uint32_t ndm, const float* table, uint32_t nchans) {
  if (!dm_list || !table || !ndm || !nchans) return 0;
  const int32_t d = delay_of(dm_list[ndm - 1], table[nchans - 1]);
  return d > 0 ? (uint64_t)d : 0;
}

extern "C" uint64_t psx_dedisp_work_bytes(uint64_t nsamps_in, uint32_t nchans, uint32_t ndm) {
  return round_up(nsamps_in * nchans, 256) + round_up((uint64_t)ndm * nchans * sizeof(int32_t), 256);
}

extern "C" int psx_dedisperse(const uint8_t* d_in, uint64_t nsamps_in, uint32_t nchans, uint32_t nbits,
                              const float* dm_list, uint32_t ndm, const int32_t* killmask, float tsamp, float f0,
                              float df, float* d_out, uint64_t out_stride, void* d_work, psx_stream s) {
  PSX_REQUIRE(d_in && dm_list && d_out && d_work && ndm > 0 && nsamps_in > 0, "psx_dedisperse: bad arguments");
  psx::TraceRange range("Dedisperse");
  PSX_REQUIRE(nchans > 0 && nchans <= kMaxChans, "psx_dedisperse: nchans must be 1..%u", kMaxChans);
  PSX_REQUIRE(nbits == 1 || nbits == 2 || nbits == 4 || nbits == 8, "psx_dedisperse: nbits must be 1, 2, 4 or 8");
  PSX_REQUIRE((uint64_t)nchans * nbits % 8 == 0, "psx_dedisperse: a sample must fill whole bytes");
  PSX_REQUIRE(df < 0, "psx_dedisperse: channels must run from high to low frequency (foff < 0)");
  PSX_REQUIRE(ndm <= 0x7FFFFFFFu, "psx_dedisperse: too many DMs");
  std::vector<float> table(nchans);
  int rc = psx_dedisp_delay_table(nchans, tsamp, f0, df, table.data());
  if (rc) return rc;
  const uint64_t max_delay = psx_dedisp_max_delay(dm_list, ndm, table.data(), nchans);
  PSX_REQUIRE(max_delay < nsamps_in, "psx_dedisperse: %llu samples do not cover the %llu-sample delay",
              (unsigned long long)nsamps_in, (unsigned long long)max_delay);
  const uint64_t nout = nsamps_in - max_delay;
  PSX_REQUIRE(out_stride >= nout, "psx_dedisperse: out_stride below the %llu output samples",
              (unsigned long long)nout);
  // every read t + delay with t < nout must stay inside the input: delays
  // grow with the DM in every channel, so the largest DM decides
  float top = dm_list[0];
  for (uint32_t d = 0; d < ndm; ++d) {
    PSX_REQUIRE(dm_list[d] >= 0, "psx_dedisperse: negative DM");
    top = std::max(top, dm_list[d]);
  }
  for (uint32_t c = 0; c < nchans; ++c) {
    const int32_t v = delay_of(top, table[c]);
    PSX_REQUIRE(v >= 0 && (uint64_t)v <= max_delay,
                "psx_dedisperse: DM %g needs a delay beyond the list's last DM (sort the list)", top);
  }
  const uint64_t rowbytes = (uint64_t)nchans * nbits / 8;
  PSX_REQUIRE((nsamps_in + 63) / 64 <= 0x7FFFFFFFull && (rowbytes + 63) / 64 <= 65535,
              "psx_dedisperse: input too large");
  uint8_t* rows = static_cast<uint8_t*>(d_work);
  int32_t* d_delays = reinterpret_cast<int32_t*>(rows + round_up(nsamps_in * nchans, 256));
  hipStream_t st = psx::as_stream(s);
  DelayArgs da;
  uint32_t nrows = 0;
  for (uint32_t w = 0; w < kMaxChans / 32; ++w) {
    da.mask.on[w] = 0u;
    da.mask.before[w] = (uint16_t)nrows;
    for (uint32_t c = 32 * w; c < 32 * w + 32 && c < nchans; ++c)
      if (!killmask || killmask[c] != 0) {
        da.mask.on[w] |= 1u << (c & 31u);
        ++nrows;
      }
  }
  for (uint32_t d = 0; d < ndm; d += kDelayDms) {
    const uint32_t n = std::min(kDelayDms, ndm - d);
    std::copy(dm_list + d, dm_list + d + n, da.dm);
    k_delays<<<dim3((nchans + kB - 1) / kB, n), kB, 0, st>>>(d_delays + (uint64_t)d * nrows, nchans, nrows,
                                                             4.15e3 / (double)tsamp, f0, df, da);
    PSX_CHECK_LAUNCH("k_delays");
  }
  switch (nbits) {
    case 1: launch_unpack<1>(d_in, nsamps_in, nchans, rows, da.mask, st); break;
    case 2: launch_unpack<2>(d_in, nsamps_in, nchans, rows, da.mask, st); break;
    case 4: launch_unpack<4>(d_in, nsamps_in, nchans, rows, da.mask, st); break;
    default: launch_unpack<8>(d_in, nsamps_in, nchans, rows, da.mask, st); break;
  }
  PSX_CHECK_LAUNCH("k_unpack_t");
  const float denom = (float)((1u << nbits) - 1u) * (float)nchans;
  const SumArgs sa{rows, nsamps_in, nrows, d_delays, denom, d_out, out_stride, nout, ndm, 0};
  const float tmax = *std::max_element(table.begin(), table.end());
  switch (nbits) {
    case 1: rc = launch_sum<1>(sa, dm_list, tmax, st); break;
    case 2: rc = launch_sum<2>(sa, dm_list, tmax, st); break;
    case 4: rc = launch_sum<4>(sa, dm_list, tmax, st); break;
    default: rc = launch_sum<8>(sa, dm_list, tmax, st); break;
  }
  if (rc) return rc;
  // the trials are complete when the call returns, whatever stream reads them
  PSX_CHECK_HIP(hipStreamSynchronize(st));
  return psx::ok();
}
