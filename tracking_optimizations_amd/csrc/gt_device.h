// gt_device.h -- device helpers shared by the kernels of the locate path.
#pragma once

#include "gt_internal.h"

// Pointers fetched from the frame table are generic; marking them global
// lets the compiler emit global (not flat) memory instructions, whose waits
// do not also drain the LDS counter.  Only the device pass knows the
// address space.
#if defined(__HIP_DEVICE_COMPILE__)
#define GLOBAL __attribute__((address_space(1)))
#else
#define GLOBAL
#endif

namespace gt {

namespace {

constexpr uint32_t NEG_INF_BITS = 0xff800000u;

__device__ __forceinline__ uint32_t xcd_remap(uint32_t bid, uint32_t n) {
    // Workgroups are dispatched round-robin over the 8 XCDs.  Give each XCD a
    // contiguous range of work items so that vertically and horizontally
    // neighbouring tiles (which share halo rows) hit the same L2.
    const uint32_t X = 8;
    const uint32_t xcd = bid % X, local = bid / X;
    const uint32_t q = n / X, r = n % X;
    return xcd * q + min(xcd, r) + local;
}

// Percentile histogram key of a non-negative float bit pattern.
__device__ __forceinline__ uint32_t pct_key(uint32_t bits) {
    if (bits == 0) return 0;
    const uint32_t k = (bits >> 19) + 1u;
    return k < (uint32_t)HIST_BINS ? k : (uint32_t)(HIST_BINS - 1);
}

template <typename T> struct IsFloat { static constexpr bool v = false; };
template <> struct IsFloat<float> { static constexpr bool v = true; };

__device__ __forceinline__ float raw_px(const void* in, int type, size_t i) {
    if (type == IN_U16) return (float)((const uint16_t*)in)[i];
    if (type == IN_U8) return (float)((const uint8_t*)in)[i];
    return ((const float*)in)[i];
}

__device__ __forceinline__ uint32_t wave_sum_u(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Inclusive prefix sum over the 64 lanes of a wave.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, int lane) {
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

__device__ __forceinline__ uint64_t lanemask_lt(int lane) {
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

}  // namespace

}  // namespace gt
