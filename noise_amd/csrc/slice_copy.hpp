// Where a wave's 64 one-element copies of a slice read when part of it may lie outside the buffer: lane l wants element
// first + l, clamped into [0, numel). A copy takes a 64-bit base common to the wave and a 32-bit byte offset per lane, and a
// buffer may be longer than 2^32 bytes, so the base itself is the clamped first element and a lane only adds its distance from it.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define NOISE_SLICE_FN __host__ __device__ inline
#else
#define NOISE_SLICE_FN inline
#endif

namespace noise {

NOISE_SLICE_FN int64_t slice_clamp(int64_t e, int64_t numel) { return e < 0 ? 0 : e < numel ? e : numel - 1; }

// the element at the wave's base address
NOISE_SLICE_FN int64_t slice_base(int64_t first, int64_t numel) { return slice_clamp(first, numel); }

// lane's byte offset from it: 0 .. 252
NOISE_SLICE_FN uint32_t slice_lane(int64_t first, int lane, int64_t base, int64_t numel) {
    return (uint32_t)(4 * (slice_clamp(first + lane, numel) - base));
}

}  // namespace noise
