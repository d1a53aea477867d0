// Channelizer at rates made of 2, 3, 5 and 7 (mixed_fft.hip).
#pragma once

#include "common.hh"

namespace bl {

// Whether `rate` (two polarizations) runs on the mixed-radix kernel.
bool mixed_fft_covers(uint64_t rate);

// Build the rate's twiddle table (once per device), so that later launches
// allocate nothing.
int mixed_fft_plan(int C);

// CF32 [n_spec spectra of C samples][2] -> [n_spec / S, C, S, 2], fftshifted.
// `made` is set when the call built the rate's table (and below).
int mixed_fft(int C, const float2* in, float2* out, uint64_t S, uint64_t n_spec, hipStream_t s, bool* made);

// Powers summed over Sg consecutive spectra, `groups` integrations per
// (antenna, channel): F32 [n_groups / groups, C, groups, out_pols].
// flags: 1 adds into out, 2 XY -> LR first.  False if it does not take the
// call (adding to earlier blocks, where LDS has no room for the block's sums, or
// more threads than a launch holds).
bool mixed_fft_detect(int C, const float2* in, float* out, uint64_t Sg, int groups, uint64_t n_groups, int out_pols,
                      int flags, hipStream_t s, int* rc, bool* made);

}  // namespace bl
