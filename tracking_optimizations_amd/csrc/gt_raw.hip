// gt_raw.hip -- raw signal extraction (execute_gpu.rs:301-333) on the device.
//
// For every output row of a batch, centred on (round(y), round(x)) (f32
// round, half away from zero), on the raw input frame as float32:
//   raw_mass            sum of the signal-disk pixels (circle_inds,
//                       kernels.rs:149-164), one after the other in tap
//                       order in binary32, taps outside the frame skipped
//                       (fold_axis_skipnan);
//   raw_bg_median       median of the background-annulus pixels inside the
//                       frame (annulus_inds, kernels.rs:166-181), with the
//                       linear interpolation of ndarray-stats 0.5.1
//                       (quantile_axis_skipnan_mut, Linear): q = 0.5 of the
//                       n values in order, index 0.5 (n - 1) in binary64,
//                       a + f32(fract * (b - a)) with a, b the order
//                       statistics at floor and ceil of the index; NaN when
//                       no tap is inside;
//   raw_mass_corrected  raw_mass - raw_bg_median * n_signal_taps (binary32,
//                       no fused multiply-add).
// A wave takes a run of up to 64 rows, lane = row for the positions and the
// results.  The rows' taps are then gathered one row after the other, the
// next row's while the current one is worked on: lane t holds taps t, t + 64,
// ...  The order statistics are found bit by bit from the top (the largest
// prefix with at most `rank` keys below it; a compare and a ballot per 64
// taps and bit), which yields the same values as any selection.  The signal
// sum of integer pixels is exact below 2^24 in any order and is added across
// the lanes; otherwise each lane adds its own row's taps in order.
//
// Bound by issued instructions: three background taps per lane take 3 compares
// and 8 scalar operations for each of a uint16's 16 bits (36 exchange stages
// of four registers each when the row was sorted instead).  40 frames of
// 2048^2 with 12.9 k rows each (sig 3, bg 8, gap 1): the whole call 1745 us
// with a sort per row and lane 0 adding the signal taps, 1070 us so.
#include <math.h>

#include <algorithm>

#include "gt_device.h"

#pragma clang fp contract(off)

namespace gt {

namespace {

constexpr int RAW_MAX_REG = 8;   // background taps per lane held in registers

template <typename T> struct RawKey {   // integer pixels: the value itself
    static constexpr int BITS = 8 * (int)sizeof(T);
    static __device__ __forceinline__ uint32_t key(T v) { return v; }
    static __device__ __forceinline__ float value(uint32_t k) { return (float)k; }
};
template <> struct RawKey<float> {      // order-preserving bit pattern
    static constexpr int BITS = 32;
    static __device__ __forceinline__ uint32_t key(float v) {
        const uint32_t b = __float_as_uint(v);
        return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    }
    static __device__ __forceinline__ float value(uint32_t k) {
        return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
    }
};
// Key of a tap that is outside the frame or NaN: above every other, so that
// it is never below a wanted rank (no finite float has it).
constexpr uint32_t RAW_NONE = 0xffffffffu;

// SUM: the signal disk of integer pixels is summed across the lanes.
// NB: background taps per lane (0: no background; RAW_MAX_REG + 1: any
// number, their keys in LDS).
template <typename T, int NB, bool SUM>
__global__ __launch_bounds__(64) void k_raw(Batch b, const Geom* __restrict__ g) {
    using K = RawKey<T>;
    constexpr bool LDS = NB > RAW_MAX_REG;
    constexpr int NR = LDS ? 1 : (NB > 0 ? NB : 1);
    extern __shared__ uint32_t s_key[];   // LDS only
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const int H = (int)fr.H, W = (int)fr.W;
    const int lane = threadIdx.x;
    const int ns = g->raw_ns, nb = g->raw_nb, nc = g->ncols, col = g->col_raw;
    const int reach = g->raw_reach;
    const int8_t* stap = g->raw_tap;
    const int8_t* btap = stap + 2 * ns;
    const GLOBAL char* in = (const GLOBAL char*)fr.in;
    const uint64_t r0 = b.frame_row_base[f];
    if (r0 >= b.rows_cap) return;
    const uint32_t nrows = (uint32_t)min((uint64_t)b.frame_rows[f], b.rows_cap - r0);
    // rows of one run: as few as give every wave of the frame one
    const uint32_t per = min(64u, max(1u, (nrows + gridDim.y - 1) / gridDim.y));

    // this lane's taps: offsets and, for rows whose taps may lie outside the
    // frame, the position
    int bo[NR], bdy[NR], bdx[NR];   // bo: pixels from the centre
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const int t = min(lane + 64 * k, max(nb - 1, 0));
        bdy[k] = NB && nb ? btap[2 * t] : 0;
        bdx[k] = NB && nb ? btap[2 * t + 1] : 0;
        bo[k] = bdy[k] * W + bdx[k];
    }
    // a frame's bytes are 32-bit offsets (fewer than 2^30 pixels)
    auto pixel = [&](uint32_t at) { return *(const GLOBAL T*)(in + at * (uint32_t)sizeof(T)); };
    auto index = [&](int y, int x) { return (uint32_t)y * (uint32_t)W + (uint32_t)x; };
    auto inside = [&](int y, int x) { return y >= 0 && y < H && x >= 0 && x < W; };
    auto key_of = [&](T v, bool ok) {
        if constexpr (IsFloat<T>::v) ok = ok && !isnan(v);
        return ok ? K::key(v) : RAW_NONE;
    };

    for (uint32_t q0 = blockIdx.y * per; q0 < nrows; q0 += gridDim.y * per) {
        const int n = (int)min(per, nrows - q0);
        const uint64_t row = r0 + q0 + (uint32_t)min(lane, n - 1);
        float* const o = b.rows + row * (uint64_t)nc;
        // A walk over values near the binary32 limit ends at an infinite
        // position (its moment overflows before its mass does).  No tap is
        // more than 127 away, so a centre farther out than that reaches no
        // pixel from wherever it is: clamped, its sums below cannot overflow.
        const int cy = min(max((int)roundf(o[2]), -128), H + 127);
        const int cx = min(max((int)roundf(o[3]), -128), W + 127);
        float sig = 0.f, med = 0.f;
        if constexpr (!SUM) {   // lane = row, taps in order
            const uint32_t at = index(cy, cx);
            for (int t = 0; t < ns; ++t) {
                const int dy = stap[2 * t], dx = stap[2 * t + 1];
                const bool ok = inside(cy + dy, cx + dx);
                const T p = pixel(ok ? at + (uint32_t)(dy * W + dx) : 0u);
                const float v = (float)p;
                if (ok && !isnan(v)) sig = sig + v;
            }
        }
        if constexpr (SUM || NB > 0) {
            // lane q holds tap q of the signal disk (SUM) and its background
            // taps of row i
            auto load = [&](int i, T (&bg)[NR], bool (&bok)[NR], uint32_t& sg) {
                const int y = __builtin_amdgcn_readlane(cy, i), x = __builtin_amdgcn_readlane(cx, i);
                const uint32_t at = index(y, x);
                const bool all = y >= reach && y + reach < H && x >= reach && x + reach < W;
                if constexpr (SUM) {
                    sg = 0;
                    for (int t = lane; t < ns; t += 64) {
                        const int dy = stap[2 * t], dx = stap[2 * t + 1];
                        const bool ok = all || inside(y + dy, x + dx);
                        const T p = pixel(ok ? at + (uint32_t)(dy * W + dx) : 0u);
                        sg += ok ? (uint32_t)p : 0u;
                    }
                }
                if constexpr (NB > 0 && !LDS) {
#pragma unroll
                    for (int k = 0; k < NR; ++k) {
                        bok[k] = lane + 64 * k < nb && (all || inside(y + bdy[k], x + bdx[k]));
                        bg[k] = pixel(bok[k] ? at + (uint32_t)bo[k] : 0u);
                    }
                }
            };
            T bg[NR];
            bool bok[NR];
            uint32_t sg = 0;
            load(0, bg, bok, sg);
            for (int i = 0; i < n; ++i) {
                uint32_t key[NR];
                const uint32_t sum = sg;
                if constexpr (NB > 0 && !LDS) {
#pragma unroll
                    for (int k = 0; k < NR; ++k) key[k] = key_of(bg[k], bok[k]);
                }
                if (i + 1 < n) load(i + 1, bg, bok, sg);
                if constexpr (SUM) {
                    const float v = (float)wave_sum_u(sum);
                    sig = lane == i ? v : sig;
                }
                if constexpr (NB > 0) {
                    if constexpr (LDS) {
                        const int y = __builtin_amdgcn_readlane(cy, i), x = __builtin_amdgcn_readlane(cx, i);
                        __syncthreads();
                        for (int t = lane; t < nb; t += 64) {
                            const int dy = btap[2 * t], dx = btap[2 * t + 1];
                            const bool ok = inside(y + dy, x + dx);
                            s_key[t] = key_of(pixel(ok ? index(y + dy, x + dx) : 0u), ok);
                        }
                        __syncthreads();
                    }
                    // keys below c, and the smallest one above c - 1
                    auto below = [&](uint32_t c) {
                        uint32_t m = 0;
                        if constexpr (LDS) {
                            for (int t = lane; t < nb; t += 64) m += s_key[t] < c ? 1u : 0u;
                            m = wave_sum_u(m);
                        } else {
#pragma unroll
                            for (int k = 0; k < NR; ++k)
                                m += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(key[k] < c));
                        }
                        return m;
                    };
                    const uint32_t m = below(RAW_NONE);   // taps that count
                    float v = __builtin_nanf("");
                    if (m > 0) {
                        const uint32_t lo = (m - 1) / 2, hi = m / 2;   // floor and ceil of 0.5 (m - 1)
                        uint32_t a = 0;
#pragma unroll
                        for (int s = K::BITS - 1; s >= 0; --s) {
                            const uint32_t c = a | (1u << s);
                            a = below(c) <= lo ? c : a;
                        }
                        uint32_t c = a;
                        if (hi != lo && below(a + 1) <= hi) {   // the next key up
                            uint32_t w = RAW_NONE;
                            if constexpr (LDS) {
                                for (int t = lane; t < nb; t += 64) w = s_key[t] > a ? min(w, s_key[t]) : w;
                            } else {
#pragma unroll
                                for (int k = 0; k < NR; ++k) w = key[k] > a ? min(w, key[k]) : w;
                            }
                            for (int d = 32; d > 0; d >>= 1) w = min(w, (uint32_t)__shfl_xor((int)w, d, 64));
                            c = w;
                        }
                        const float fa = K::value(a), fc = K::value(c);
                        const double frac = hi != lo ? 0.5 : 0.0;
                        v = fa + (float)(frac * ((double)fc - (double)fa));
                    }
                    med = lane == i ? v : med;
                }
            }
        }
        if (lane < n) {
            o[col] = sig;
            if constexpr (NB > 0) {
                o[col + 1] = med;
                o[col + 2] = sig - med * (float)ns;
            }
        }
    }
}

template <typename T, bool SUM>
hipError_t launch_raw_t(const Batch& b, const Geom& g, const Geom* d_geom, hipStream_t s) {
    // a few waves per SIMD in all, and enough of them where one frame has
    // all the rows
    const uint32_t per_frame = std::max(64u, std::min(512u, 16384u / std::max(b.nframes, 1u)));
    const dim3 grid(b.nframes, per_frame), block(64);
    const int nbt = g.raw_cols == 3 ? (g.raw_nb + 63) / 64 : 0;
    switch (g.raw_cols == 3 ? std::max(nbt, 1) : 0) {
        case 0: hipLaunchKernelGGL((k_raw<T, 0, SUM>), grid, block, 0, s, b, d_geom); break;
        case 1: hipLaunchKernelGGL((k_raw<T, 1, SUM>), grid, block, 0, s, b, d_geom); break;
        case 2: hipLaunchKernelGGL((k_raw<T, 2, SUM>), grid, block, 0, s, b, d_geom); break;
        case 3: hipLaunchKernelGGL((k_raw<T, 3, SUM>), grid, block, 0, s, b, d_geom); break;
        case 4: hipLaunchKernelGGL((k_raw<T, 4, SUM>), grid, block, 0, s, b, d_geom); break;
        case 5: hipLaunchKernelGGL((k_raw<T, 5, SUM>), grid, block, 0, s, b, d_geom); break;
        case 6: hipLaunchKernelGGL((k_raw<T, 6, SUM>), grid, block, 0, s, b, d_geom); break;
        case 7: hipLaunchKernelGGL((k_raw<T, 7, SUM>), grid, block, 0, s, b, d_geom); break;
        case 8: hipLaunchKernelGGL((k_raw<T, 8, SUM>), grid, block, 0, s, b, d_geom); break;
        default:
            hipLaunchKernelGGL((k_raw<T, RAW_MAX_REG + 1, SUM>), grid, block,
                               (size_t)g.raw_nb * sizeof(uint32_t), s, b, d_geom);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_raw(const Batch& b, const Geom& g, const Geom* d_geom, hipStream_t s) {
    if (b.in_type == IN_F32) return launch_raw_t<float, false>(b, g, d_geom, s);
    if (b.in_type == IN_U8) return launch_raw_t<uint8_t, true>(b, g, d_geom, s);   // 4096 * 255 < 2^24
    if (g.raw_ns <= 256) return launch_raw_t<uint16_t, true>(b, g, d_geom, s);     // 256 * 65535 < 2^24
    return launch_raw_t<uint16_t, false>(b, g, d_geom, s);
}

}  // namespace gt
