// gt_bandpass.h -- the streaming bandpass kernel (K1; preprocess_rows.wgsl +
// preprocess_cols.wgsl), instantiated per input type in gt_bandpass_*.hip.
// Pipeline and arithmetic contract: gt_kernels.hip.
#pragma once

#include <algorithm>
#include <type_traits>

#include "gt_device.h"

#pragma clang fp contract(off)

namespace gt {

// ---------------------------------------------------------------------------
// K1 bandpass, streaming column strips.
//
// A workgroup takes a 256-column strip of `seg` output rows of one frame, its
// two waves 128 columns each.  A wave walks down its columns: every input row
// (reflected at the top and bottom edges) is staged once in LDS, each lane
// computes the row pass of its two columns and keeps the last 2R+1 row
// results in a register ring; once the ring is full the column pass produces
// one output row.  Every lane loads its own two columns and HB lanes load one
// more pair of the halo, so every lane is an output lane.  The waves of a
// workgroup share nothing but the percentile histogram: a wave's LDS
// operations are carried out in order, so a row needs no barrier.
//
// Rows may start at any multiple of the element size and have any width: a
// pair of columns is one load of two elements, wherever it lies.  In strips
// that touch the left or right edge a pair's two columns are the reflected
// ones, taken from the in-frame pair that holds them (lane constants), and
// two copies of the row implement the two boundary rules: out-of-frame
// columns are zero in the Gaussian copy (taps skipped, Q3) and mirrored in
// the boxcar copy (Q4).
//
// Integer input: a row's boxcar sum is an exact integer in binary32
// (33 * 65535 < 2^24), so the horizontal boxcar slides.  The vertical one is
// a running sum: for k <= 15 and for uint8 it never reaches 2^24; for wider
// uint16 filters it is kept as an integer, and where one of the wave's sums
// reaches 2^24 the row sums are added in the shader's order instead (its
// partial sums may round there).  Float input sums tap by tap from +0.
// FAST selects the two-part-reciprocal division by the two per-call divisors
// (host-verified to equal IEEE division).
//
// Bound by issued vector instructions (the units that carry them are 80 %
// busy): 50 per pixel at R = 5 (uint16 with a histogram, halo rows and frame
// edges counted), of which 22 are the Gaussian's FMAs, 6 the three divisions
// and 5.5 the boxcar; 40 frames of 2048^2 in 267 us, 3.8 TB/s of input and
// output; corrected single reciprocals (nine for the divisions) took 278
// (four columns per lane on 240-column strips, where four lanes only carry
// halos: 301 us).  Two columns per lane halve the ring, so four waves share a
// SIMD where three did, and leave room for R up to 16 (24 frames of 1024^2 at
// k = 21: 78 us; two passes through a temporary plane: 1008 us) and for any
// width and alignment (96 float32 frames of 517 x 663 at k = 13: 105 us, 121
// with a division for each quotient; in two passes 1032 us).
// ---------------------------------------------------------------------------
struct K1Params {
    float w[17];   // Gaussian weights of offsets 0 .. R (they are symmetric)
    float gn, rgn, rgn_lo, kk, rkk, rkk_lo;
    int seg;
    int hist;
};

constexpr int K1_WAVES = 2;
constexpr int K1_COLS = K1_STRIP / K1_WAVES;   // columns of a wave
static_assert(K1_COLS == 128, "two columns per lane");

// Two neighbouring elements, at any element address.
template <typename T> struct Pair;
template <> struct Pair<uint16_t> { uint32_t v; };
template <> struct Pair<uint8_t> { uint16_t v; };
template <> struct Pair<float> { float2 v; };

typedef uint32_t u32_a2 __attribute__((aligned(2)));
typedef uint16_t u16_a1 __attribute__((aligned(1)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef f2v f2v_a4 __attribute__((aligned(4)));

// base: the frame, ro: byte offset of the row (both wave-uniform, 32 bits:
// frames hold fewer than 2^30 pixels), off: of this lane's column; the load
// takes base + ro as a scalar
template <typename T>
__device__ __forceinline__ Pair<T> ld_pair(const GLOBAL char* base, uint32_t ro, uint32_t off) {
    // (the compiler would widen `off` once before the row loop and then add
    // 64-bit addresses for every load: it has to see the 32-bit offset here)
    asm volatile("" : "+v"(off));
    const GLOBAL char* p = (base + ro) + off;
    Pair<T> c;
    if constexpr (IsFloat<T>::v) {
        const f2v q = *(const GLOBAL f2v_a4*)p;
        c.v = make_float2(q.x, q.y);
    } else if constexpr (sizeof(T) == 2) {
        c.v = *(const GLOBAL u32_a2*)p;
    } else {
        c.v = *(const GLOBAL u16_a1*)p;
    }
    return c;
}

// The pair's elements i0 and i1 (0 or 1) as floats; SEL false: 0 and 1.
template <typename T, bool SEL>
__device__ __forceinline__ f2v unpack_pair(const Pair<T>& c, int i0, int i1) {
    f2v r;
    if constexpr (IsFloat<T>::v) {
        r.x = SEL && i0 ? c.v.y : c.v.x;
        r.y = SEL && !i1 ? c.v.x : c.v.y;
    } else {
        constexpr int B = 8 * (int)sizeof(T);
        constexpr uint32_t M = (1u << B) - 1u;
        const uint32_t v = c.v;
        r.x = (float)((SEL ? v >> (B * i0) : v) & M);
        r.y = (float)((SEL ? v >> (B * i1) : v >> B) & M);
    }
    return r;
}

// r = x / d, correctly rounded, for a lane's two values.  FAST: by the two-part
// reciprocal hi + lo, which the host has checked to give the rounded quotient
// of every significand; that holds while x * lo is a normal number.  Integer
// pixels (gt_api.hip says why) need no test of it; float pixels divide where a
// lane's is not one (a zero, a value beyond 2^-95, infinities and NaN).
// Two instructions a quotient where the corrected one of a single reciprocal
// takes three and the division eleven.
template <bool FAST, bool CHECK>
__device__ __forceinline__ void div_pair(const float (&x)[2], float d, float hi, float lo,
                                         float (&r)[2]) {
    if constexpr (FAST) {
        const float t0 = x[0] * lo, t1 = x[1] * lo;
        r[0] = __builtin_fmaf(x[0], hi, t0);
        r[1] = __builtin_fmaf(x[1], hi, t1);
        if constexpr (CHECK) {
            constexpr int NORMAL = 0x108;   // either sign
            if (~(__builtin_amdgcn_ballot_w64(__builtin_amdgcn_classf(t0, NORMAL)) &
                  __builtin_amdgcn_ballot_w64(__builtin_amdgcn_classf(t1, NORMAL)))) {
                r[0] = x[0] / d;
                r[1] = x[1] / d;
            }
        }
    } else {
        r[0] = x[0] / d;
        r[1] = x[1] / d;
    }
}

// Order of a wave's own LDS operations: the hardware keeps it, the compiler
// has to.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int R>
struct K1Shape {
    static constexpr int NT = 2 * R + 1;
    static constexpr int HB = (R + 1) / 2 * 2;      // halo columns on each side
    static constexpr int ROW = K1_COLS + 2 * HB;    // floats of a staged row
    static constexpr int BUF = 2 * ROW;             // both copies of a wave's row
};

// Most waves per SIMD that leave the registers of a row ring without spills.
template <int R, bool FLT>
constexpr int k1_waves_per_eu() {
    return FLT ? (R <= 3 ? 5 : R <= 5 ? 4 : R <= 8 ? 3 : 2)
               : (R <= 4 ? 5 : R <= 7 ? 4 : R <= 10 ? 3 : 2);
}

template <int R, typename T, bool FAST>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * K1_WAVES, 64 * K1_WAVES),
                          amdgpu_waves_per_eu(k1_waves_per_eu<R, IsFloat<T>::v>())))
void k_bandpass(Batch b, K1Params kp) {
    using S = K1Shape<R>;
    constexpr int NT = S::NT, HB = S::HB;
    constexpr bool FLT = IsFloat<T>::v;
    constexpr bool WIDE = !FLT && sizeof(T) == 2 && R >= 8;   // vertical sums can reach 2^24
    // percentile only: one word per histogram bin (word i: bin i + 1; zeros
    // are counted apart), at offset 0 so that a bin's address needs no base
    extern __shared__ __attribute__((aligned(16))) uint32_t s_hist[];

    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.k1_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.k1_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int sx = (int)(local % fr.k1_tx), sy = (int)(local / fr.k1_tx);
    const int t = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x0 = sx * K1_STRIP + wave * K1_COLS;
    const int y0 = sy * kp.seg;
    const int y1 = min(y0 + kp.seg, H);
    const GLOBAL char* inb = (const GLOBAL char*)fr.in;
    GLOBAL char* P = (GLOBAL char*)fr.P;

    if (kp.hist) {
        for (int i = threadIdx.x; i < HIST_BINS; i += 64 * K1_WAVES) s_hist[i] = 0;
        __syncthreads();
    }
    uint32_t zc = 0;  // zero outputs of this wave (wave-uniform)

    if (x0 < W) {  // wave-uniform: the second wave of a frame's last strip may have no column
    // some pair of this wave's staged row lies outside the frame
    const bool border = (x0 - HB < 0) || (x0 + K1_COLS + HB > W);
    // where the pair of columns c, c + 1 comes from: the in-frame pair at
    // column `src`, its elements i0 and i1 (columns that no output reaches
    // are clamped); W >= 2
    auto pair_src = [&](int c, int& src, int& i0, int& i1, bool& o0, bool& o1) {
        auto refl = [&](int q) { return q < 0 ? -q - 1 : (q >= W ? 2 * W - q - 1 : q); };
        const int m0 = refl(c), m1 = refl(c + 1);
        src = max(0, min(min(m0, m1), W - 2));
        i0 = max(0, min(m0 - src, 1));
        i1 = max(0, min(m1 - src, 1));
        o0 = c < 0 || c >= W;
        o1 = c + 1 < 0 || c + 1 >= W;
    };
    const int cc = x0 + 2 * t;   // this lane's columns cc, cc + 1
    int msrc, mi0, mi1, hsrc, hi0, hi1;
    bool mo0, mo1, ho0, ho1;
    pair_src(cc, msrc, mi0, mi1, mo0, mo1);
    // halo pairs: lanes 0 .. HB/2 - 1 the left ones, HB/2 .. HB - 1 the right;
    // the other lanes repeat the last one (no branch around its load and store)
    const int hpos = t < HB / 2 ? 2 * t : K1_COLS + 2 * min(t, HB - 1);   // position in the staged row
    pair_src(x0 - HB + hpos, hsrc, hi0, hi1, ho0, ho1);
    const uint32_t moff = (uint32_t)msrc * (uint32_t)sizeof(T);
    const uint32_t hoff = (uint32_t)hsrc * (uint32_t)sizeof(T);
    const uint32_t pcoff = 4u * (uint32_t)cc;
    const bool out0 = cc < W, out1 = cc + 1 < W;
    const uint64_t om0 = __builtin_amdgcn_ballot_w64(out0), om1 = __builtin_amdgcn_ballot_w64(out1);

    float w[R + 1];
#pragma unroll
    for (int i = 0; i <= R; ++i) w[i] = kp.w[i];

    // row results: Gaussian, and the boxcar row sums (as integers where the
    // vertical sum is one)
    using BoxT = std::conditional_t<WIDE, uint32_t, float>;
    float rg[NT][2];
    BoxT rb[NT][2];
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
        for (int q = 0; q < 2; ++q) { rg[s][q] = 0.f; rb[s][q] = 0; }
    BoxT vbox[2] = {0, 0};

    const int vr0 = y0 - R, vr1 = y1 + R;
    // byte offset of row vr, reflected at the top (-vr - 1) and bottom
    // (2H - vr - 1) edges without a branch
    auto row_off = [&](int vr) -> uint32_t {
        const int ar = min(max(vr, -vr - 1), 2 * H - 1 - vr);
        return (uint32_t)__builtin_amdgcn_readfirstlane(ar * W * (int)sizeof(T));
    };

    // prefetch: row vr is loaded PF rows ahead into slot (vr - vr0) % NT, so
    // only PF + 1 slots are live at a time; as many as spill nothing (8 rows
    // ahead against 4: 264 against 272 us, 40 frames of 2048^2)
    constexpr int PFMAX = FLT ? (R == 3 ? 3 : 4) : R == 7 ? 4 : R == 4 ? 5 : R == 6 || R == 10 ? 7 : 8;
    constexpr int PF = NT < PFMAX ? NT : PFMAX;
    Pair<T> pm[NT], ph[NT];
#pragma unroll
    for (int s = 0; s < PF; ++s) {
        const uint32_t ro = row_off(min(vr0 + s, vr1 - 1));
        pm[s] = ld_pair<T>(inb, ro, moff);
        ph[s] = ld_pair<T>(inb, ro, hoff);
    }

    // this wave's staged row: boxcar copy (mirrored), then Gaussian copy
    // (zero outside)
    float* const bb_ = (float*)s_hist + (kp.hist ? HIST_BINS : 0) + wave * S::BUF;
    float* const bg_ = bb_ + S::ROW;
    // the row loop, specialised on whether any column of the wave's row lies
    // outside the frame (mirrored / zeroed staging) or none does
    auto rows = [&](auto border_c) {
        constexpr bool BORDER = decltype(border_c)::value;
        // whole groups of NT rows: the last group runs past vr1 (those rows
        // load row vr1 - 1 and emit nothing) so that no branch surrounds a
        // row; one there makes the compiler wait for every load and store in
        // flight before each row instead of only for the row's own pairs
        for (int base = vr0; base < vr1; base += NT) {
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                const int vr = base + s;
                // rows above and below the frame are zero in the Gaussian copy
                // (skipped taps) and mirrored in the boxcar copy
                const bool row_in = (vr >= 0) && (vr < H);
                {
                    f2v m = unpack_pair<T, BORDER>(pm[s], mi0, mi1);
                    *(f2v*)(bb_ + HB + 2 * t) = m;
                    if constexpr (BORDER) {
                        m.x = mo0 || !row_in ? 0.f : m.x;
                        m.y = mo1 || !row_in ? 0.f : m.y;
                        *(f2v*)(bg_ + HB + 2 * t) = m;
                    }
                    // every pair of an interior strip is its own, so the two
                    // copies agree on rows inside the frame and the Gaussian
                    // copy of a row outside it is zero: one copy is staged
                    f2v h = unpack_pair<T, BORDER>(ph[s], hi0, hi1);
                    *(f2v*)(bb_ + hpos) = h;
                    if constexpr (BORDER) {
                        h.x = ho0 || !row_in ? 0.f : h.x;
                        h.y = ho1 || !row_in ? 0.f : h.y;
                        *(f2v*)(bg_ + hpos) = h;
                    }
                }
                {
                    const uint32_t ro = row_off(min(vr + PF, vr1 - 1));
                    pm[(s + PF) % NT] = ld_pair<T>(inb, ro, moff);
                    ph[(s + PF) % NT] = ld_pair<T>(inb, ro, hoff);
                }
                wave_lds_order();

                // staged columns 2t .. 2t + 2 HB + 1: this lane's column q
                // is element HB + q
                float v[2 * HB + 2];
#pragma unroll
                for (int i = 0; i <= HB; ++i) {
                    const f2v p = *(const f2v*)(bb_ + 2 * t + 2 * i);
                    v[2 * i] = p.x;
                    v[2 * i + 1] = p.y;
                }
                float tb[2];
                if constexpr (FLT) {
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        float bx = 0.f;
#pragma unroll
                        for (int i = -R; i <= R; ++i) bx = bx + v[HB + q + i];
                        tb[q] = bx;
                    }
                } else {
                    // whole numbers below 2^24, in any order: the taps that
                    // the two columns share, then each one's own
                    float bx = v[HB - R + 1];
#pragma unroll
                    for (int i = -R + 2; i <= R; ++i) bx = bx + v[HB + i];
                    tb[0] = bx + v[HB - R];
                    tb[1] = bx + v[HB + 1 + R];
                }
                // Gaussian row pass: zeros outside the frame (skipped taps).
                // A row outside the frame sums to +0 (FMAs of +0 into +0)
                // and so divides to +0: interior strips take that zero.
                // (by a reciprocal of 0: the sums of integer pixels are finite)
                constexpr bool ZERO_BY_HI = FAST && !FLT && !BORDER;
                const float ghi = ZERO_BY_HI && !row_in ? 0.f : kp.rgn;
                const float glo = ZERO_BY_HI && !row_in ? 0.f : kp.rgn_lo;
                auto gauss = [&](const float (&u)[2 * HB + 2], float (&tg)[2]) {
                    float gs[2] = {0.f, 0.f};
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int i = -R; i <= R; ++i)
                            gs[q] = __builtin_fmaf(w[i < 0 ? -i : i], u[HB + q + i], gs[q]);
                    div_pair<FAST, FLT>(gs, kp.gn, ghi, glo, tg);
                };
                float tg[2];
                if constexpr (BORDER) {
                    float u[2 * HB + 2];
#pragma unroll
                    for (int i = 0; i <= HB; ++i) {
                        const f2v p = *(const f2v*)(bg_ + 2 * t + 2 * i);
                        u[2 * i] = p.x;
                        u[2 * i + 1] = p.y;
                    }
                    gauss(u, tg);
                } else {
                    gauss(v, tg);
                    if constexpr (!ZERO_BY_HI) {
                        tg[0] = row_in ? tg[0] : 0.f;
                        tg[1] = row_in ? tg[1] : 0.f;
                    }
                }
                wave_lds_order();   // the next row overwrites the staged one
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    if constexpr (!FLT) vbox[q] = (vbox[q] - rb[s][q]) + (BoxT)tb[q];
                    rg[s][q] = tg[q];
                    rb[s][q] = (BoxT)tb[q];
                }

                if (vr >= y0 + R && vr < vr1) {  // wave-uniform
                    float bsum[2];
                    auto add_rows = [&]() {   // the shader's order, from +0
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            float a = 0.f;
#pragma unroll
                            for (int j = 0; j < NT; ++j) a = a + (float)rb[(s + 1 + j) % NT][q];
                            bsum[q] = a;
                        }
                    };
                    if constexpr (FLT) {
                        add_rows();
                    } else if constexpr (WIDE) {
                        if (__builtin_amdgcn_ballot_w64(max(vbox[0], vbox[1]) >= (1u << 24))) {
                            add_rows();
                        } else {
                            bsum[0] = (float)vbox[0];
                            bsum[1] = (float)vbox[1];
                        }
                    } else {
                        bsum[0] = vbox[0];
                        bsum[1] = vbox[1];
                    }
                    float gsum[2] = {0.f, 0.f};
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            gsum[q] = __builtin_fmaf(w[j < R ? R - j : j - R],
                                                     rg[(s + 1 + j) % NT][q], gsum[q]);
                    float gq[2], bq[2], out[2];
                    div_pair<FAST, FLT>(gsum, kp.gn, kp.rgn, kp.rgn_lo, gq);
                    div_pair<FAST, FLT>(bsum, kp.kk, kp.rkk, kp.rkk_lo, bq);
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const float res = gq[q] - bq[q];
                        if constexpr (FLT) out[q] = res < 0.f ? 0.f : res;   // keeps NaN
                        else out[q] = __builtin_fmaxf(res, 0.f);   // res is finite, never -0
                    }
                    // the row's address is a scalar, so the store adds this
                    // lane's column offset only
                    GLOBAL char* const po =
                        P + (uint32_t)__builtin_amdgcn_readfirstlane(4 * (vr - R) * W);
                    uint32_t pc = pcoff;
                    asm volatile("" : "+v"(pc));   // as in ld_pair
                    if (!BORDER || out1) *(GLOBAL f2v_a4*)(po + pc) = f2v{out[0], out[1]};
                    else if (out0) *(GLOBAL float*)(po + pc) = out[0];
                    if (kp.hist) {  // wave-uniform
                        // bin (bits >> 19) + 1 for positive values (finite and
                        // >= +0, so no clamp is needed); zero pixels (most of
                        // a frame) are counted by a ballot over the output
                        // lanes (one compare serves both) instead of
                        // contending for one word
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            uint32_t bits = __float_as_uint(out[q]);
                            const bool pos = bits != 0u;
                            zc += (uint32_t)__popcll(~__builtin_amdgcn_ballot_w64(pos) & (q ? om1 : om0));
                            // float input can give +inf or NaN: the last bin
                            // takes them (bin 4095: word 4094)
                            if constexpr (FLT) bits = min(bits, 0x7ff7ffffu);
                            // shift, then scale and base in one (the
                            // compiler would mask and add the base apart)
                            uint32_t bin;
                            asm("v_lshrrev_b32_e32 %0, 19, %1" : "=v"(bin) : "v"(bits));
                            if ((!BORDER || (q ? out1 : out0)) && pos) atomicAdd(&s_hist[bin], 1u);
                        }
                    }
                }
            }
        }
    };
    if (border) rows(std::true_type{});
    else rows(std::false_type{});
    }

    if (kp.hist) {
        __syncthreads();
        uint32_t* gh = b.hist1 + (size_t)f * HIST_BINS;
        for (int i = threadIdx.x; i < HIST_BINS - 1; i += 64 * K1_WAVES) {
            const uint32_t c = s_hist[i];
            if (c) atomicAdd(&gh[i + 1], c);
        }
        if (t == 0 && zc) atomicAdd(&gh[0], zc);
    }
}

template <int R, typename T>
hipError_t launch_bp_t(const Batch& b, const K1Params& kp, bool fast, hipStream_t s) {
    const size_t lds = (kp.hist ? HIST_BINS * sizeof(uint32_t) : 0) +
                       K1_WAVES * K1Shape<R>::BUF * sizeof(float);
    const dim3 grid(b.k1_items), block(64 * K1_WAVES);
    if (fast) {
        hipLaunchKernelGGL((k_bandpass<R, T, true>), grid, block, lds, s, b, kp);
        return hipGetLastError();
    }
    hipLaunchKernelGGL((k_bandpass<R, T, false>), grid, block, lds, s, b, kp);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_bandpass_t(int R, const Batch& b, const K1Params& kp, bool fast, hipStream_t s) {
    switch (R) {
        case 1: return launch_bp_t<1, T>(b, kp, fast, s);
        case 2: return launch_bp_t<2, T>(b, kp, fast, s);
        case 3: return launch_bp_t<3, T>(b, kp, fast, s);
        case 4: return launch_bp_t<4, T>(b, kp, fast, s);
        case 5: return launch_bp_t<5, T>(b, kp, fast, s);
        case 6: return launch_bp_t<6, T>(b, kp, fast, s);
        case 7: return launch_bp_t<7, T>(b, kp, fast, s);
        case 8: return launch_bp_t<8, T>(b, kp, fast, s);
        case 9: return launch_bp_t<9, T>(b, kp, fast, s);
        case 10: return launch_bp_t<10, T>(b, kp, fast, s);
        case 11: return launch_bp_t<11, T>(b, kp, fast, s);
        case 12: return launch_bp_t<12, T>(b, kp, fast, s);
        case 13: return launch_bp_t<13, T>(b, kp, fast, s);
        case 14: return launch_bp_t<14, T>(b, kp, fast, s);
        case 15: return launch_bp_t<15, T>(b, kp, fast, s);
        case 16: return launch_bp_t<16, T>(b, kp, fast, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace gt
