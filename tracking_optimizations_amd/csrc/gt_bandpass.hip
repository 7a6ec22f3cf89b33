// gt_bandpass.hip -- gfx950 bandpass of the locate path (K1;
// preprocess_rows.wgsl + preprocess_cols.wgsl).  Pipeline and arithmetic
// contract: gt_kernels.hip.
#include <algorithm>
#include <type_traits>

#include "gt_device.h"

#pragma clang fp contract(off)

namespace gt {

// ---------------------------------------------------------------------------
// K1 bandpass, streaming column strips.
//
// A work item is a 256-column strip of `seg` output rows of one frame.  The
// single wave walks down the strip: every input row (reflected at the top and
// bottom edges) is staged once in LDS, each lane computes the row pass of its
// four columns and keeps the last 2R+1 row results in a register ring; once
// the ring is full the column pass produces one output row.  Input rows are
// fetched 2R+1 rows ahead with 8-byte (u16) / 4-byte (u8) vector loads of
// 4-column chunks.  With W % 4 == 0 no chunk straddles a frame edge, so a
// chunk outside the frame is the mirror image of an in-frame chunk: it is
// loaded from there and reversed when staged.  Two staged copies of the row
// implement the two boundary rules: out-of-frame columns are zero in the
// Gaussian copy (taps skipped, Q3) and mirrored in the boxcar copy (Q4).
//
// Integer input with k <= 15 keeps every boxcar sum an exact integer below
// 2^24 in binary32, so the horizontal boxcar slides and the vertical boxcar is
// a running sum.  FAST selects the corrected-reciprocal division by the two
// per-call divisors (host-verified to equal IEEE division).
// ---------------------------------------------------------------------------
struct K1Params {
    float w[17];
    float gn, rgn, kk, rkk;
    int seg;
    int hist;
};

template <typename T> struct Chunk4;
template <> struct Chunk4<uint16_t> { uint2 v; };
template <> struct Chunk4<uint8_t> { uint32_t v; };
template <> struct Chunk4<float> { float4 v; };

// base: the frame (wave-uniform); off: byte offset, 32-bit (frames hold
// fewer than 2^30 pixels), so the load takes the frame as a scalar base
template <typename T>
__device__ __forceinline__ Chunk4<T> ld_chunk(const GLOBAL char* base, uint32_t off) {
    const GLOBAL char* p = base + off;
    Chunk4<T> c;
    if constexpr (IsFloat<T>::v) c.v = *(const GLOBAL float4*)p;
    else if constexpr (sizeof(T) == 2) c.v = *(const GLOBAL uint2*)p;
    else c.v = *(const GLOBAL uint32_t*)p;
    return c;
}

typedef float f4v __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ f4v unpack_chunk(const Chunk4<T>& c) {
    f4v r;
    if constexpr (IsFloat<T>::v) {
        r.x = c.v.x; r.y = c.v.y; r.z = c.v.z; r.w = c.v.w;
    } else if constexpr (sizeof(T) == 2) {
        r.x = (float)(c.v.x & 0xffffu); r.y = (float)(c.v.x >> 16);
        r.z = (float)(c.v.y & 0xffffu); r.w = (float)(c.v.y >> 16);
    } else {
        r.x = (float)(c.v & 0xffu); r.y = (float)((c.v >> 8) & 0xffu);
        r.z = (float)((c.v >> 16) & 0xffu); r.w = (float)(c.v >> 24);
    }
    return r;
}

// Where the 4-column chunk starting at column c (c % 4 == 0) comes from:
// its own columns, or (outside the frame) the mirrored in-frame chunk, read
// in reverse.  Chunks that no output can reach are clamped into the frame.
__device__ __forceinline__ void chunk_src(int c, int W, int& src, bool& rev, bool& oob) {
    if (c < 0) { src = -c - 4; rev = true; oob = true; }
    else if (c >= W) { src = 2 * W - c - 4; rev = true; oob = true; }
    else { src = c; rev = false; oob = false; }
    src = max(0, min(src, W - 4));
}

__device__ __forceinline__ float cdiv_t(float x, float d, float rd, bool fast) {
    if (fast) {
        const float q = x * rd;
        const float r = __builtin_fmaf(-q, d, x);
        return __builtin_fmaf(r, rd, q);
    }
    return x / d;
}

// Five 16-byte LDS reads kept whole (volatile): otherwise the compiler
// drops unused lanes and splits them into 4-byte reads, which at a 16-byte
// lane stride collide on the LDS banks.
__device__ __forceinline__ void lds_ld20(const float* p, float (&v)[20]) {
    const volatile SHARED f4v* q = (const volatile SHARED f4v*)p;
    const f4v a0 = q[0], a1 = q[1], a2 = q[2], a3 = q[3], a4 = q[4];
    v[0] = a0.x;  v[1] = a0.y;  v[2] = a0.z;  v[3] = a0.w;
    v[4] = a1.x;  v[5] = a1.y;  v[6] = a1.z;  v[7] = a1.w;
    v[8] = a2.x;  v[9] = a2.y;  v[10] = a2.z; v[11] = a2.w;
    v[12] = a3.x; v[13] = a3.y; v[14] = a3.z; v[15] = a3.w;
    v[16] = a4.x; v[17] = a4.y; v[18] = a4.z; v[19] = a4.w;
}

// K1 layout: lane t owns the 4-column chunk at column x0 - 8 + 4t; lanes
// 2..61 produce output (a 240-column strip), lanes 0, 1, 62, 63 only load
// the 8-column halos on either side.
constexpr int K1_LANE0 = 2;
constexpr int K1_LANES = K1_STRIP / 4;
static_assert(K1_LANES + 2 * K1_LANE0 == 64, "strip + halo must fill one wave");
constexpr int K1_ROWBUF = 256;   // floats per staged row

// Three waves per SIMD fit without spills up to R = 5.
template <int R, typename T, bool FAST>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 64),
                          amdgpu_waves_per_eu(R <= 5 ? 3 : 2)))
void k_bandpass(Batch b, K1Params kp) {
    constexpr int NT = 2 * R + 1;
    static_assert(R <= 8, "taps must stay inside the staged halo");
    // float input: the boxcar sums are not exact, so they are formed tap by
    // tap in the shader's order (from +0, as preprocess_*.wgsl do) instead
    // of as running sums, and the clamp keeps NaN as the shader's select does
    constexpr bool FLT = IsFloat<T>::v;
    // per parity: boxcar copy (mirrored) then Gaussian copy (zero outside)
    __shared__ __attribute__((aligned(16))) float buf[2][2][K1_ROWBUF];
    // two 16-bit bins per word (word i: bins 2i + 1 and 2i + 2; zeros are
    // counted apart); a work item adds at most K1_STRIP * seg < 65536 to one
    // bin (checked by the host)
    __shared__ uint32_t s_hist[HIST_BINS / 2];

    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.k1_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.k1_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int sx = (int)(local % fr.k1_tx), sy = (int)(local / fr.k1_tx);
    const int x0 = sx * K1_STRIP;
    const int y0 = sy * kp.seg;
    const int y1 = min(y0 + kp.seg, H);
    const int t = threadIdx.x;
    const GLOBAL T* in = (const GLOBAL T*)fr.in;
    GLOBAL float* P = (GLOBAL float*)fr.P;
    // some chunk of this strip (output or halo) lies outside the frame
    const bool border = (x0 - 8 < 0) || (x0 + K1_STRIP + 8 > W);
    const int cc = x0 - 8 + 4 * t;
    int csrc;
    bool crev, coob;
    chunk_src(cc, W, csrc, crev, coob);
    const bool outl = t >= K1_LANE0 && t < K1_LANE0 + K1_LANES && cc < W;
    const uint32_t cboff = (uint32_t)csrc * (uint32_t)sizeof(T);
    const uint32_t pcoff = 4u * (uint32_t)cc;   // used by output lanes only
    // first staged column this lane reads (halo lanes read in range, unused)
    const int rbase = min(max(4 * t - 8, 0), K1_ROWBUF - 20);

    if (kp.hist) {
        for (int i = t; i < HIST_BINS / 2; i += 64) s_hist[i] = 0;
    }

    float w[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) w[i] = kp.w[i];

    float rg[NT][4], rb[NT][4];
#pragma unroll
    for (int s = 0; s < NT; ++s)
#pragma unroll
        for (int q = 0; q < 4; ++q) { rg[s][q] = 0.f; rb[s][q] = 0.f; }
    float vbox[4] = {0.f, 0.f, 0.f, 0.f};

    const int vr0 = y0 - R, vr1 = y1 + R;
    const GLOBAL char* inb = (const GLOBAL char*)in;
    // byte offset of row vr, reflected at the top and bottom edges
    auto row_off = [&](int vr) -> uint32_t {
        const int ar = vr < 0 ? -vr - 1 : (vr >= H ? 2 * H - vr - 1 : vr);
        return (uint32_t)ar * (uint32_t)W * (uint32_t)sizeof(T);
    };

    // prefetch: row vr is loaded PF rows ahead into slot (vr - vr0) % NT,
    // so only PF + 1 slots are live at a time
    // (float chunks take 4 registers each: 3 rows ahead)
    constexpr int PFMAX = FLT ? 3 : 4;
    constexpr int PF = NT < PFMAX ? NT : PFMAX;
    Chunk4<T> pm[NT];
#pragma unroll
    for (int s = 0; s < PF; ++s) pm[s] = ld_chunk<T>(inb, row_off(min(vr0 + s, vr1 - 1)) + cboff);

    uint32_t zc = 0;  // zero outputs of this work item (wave-uniform)
    const uint64_t outl_m = __builtin_amdgcn_ballot_w64(outl);
    // the row loop, specialised on whether any chunk of the strip lies
    // outside the frame (mirrored / zeroed staging) or none does
    auto rows = [&](auto border_c) {
        constexpr bool BORDER = decltype(border_c)::value;
        int parity = 0;
        // whole groups of NT rows: the last group runs past vr1 (those rows
        // load row vr1 - 1 and emit nothing) so that no branch surrounds a
        // row; one there makes the compiler wait for every load and store in
        // flight before each row instead of only for the row's own chunk
        for (int base = vr0; base < vr1; base += NT) {
#pragma unroll
            for (int s = 0; s < NT; ++s) {
                const int vr = base + s;
                {
                float* bb_ = buf[parity][0];
                float* bg_ = buf[parity][1];
                parity ^= 1;
                // rows above and below the frame are zero in the Gaussian copy
                // (skipped taps) and mirrored in the boxcar copy
                const bool row_in = (vr >= 0) && (vr < H);
                {
                    f4v m = unpack_chunk<T>(pm[s]);
                    if constexpr (BORDER) {
                        if (crev) m = m.wzyx;
                        *(f4v*)(bb_ + 4 * t) = m;
                        if (coob || !row_in) m = f4v{0.f, 0.f, 0.f, 0.f};
                        *(f4v*)(bg_ + 4 * t) = m;
                    } else {
                        // every chunk of an interior strip is its own, so the
                        // two copies agree on rows inside the frame and the
                        // Gaussian copy of a row outside it is zero: one copy
                        // is staged
                        *(f4v*)(bb_ + 4 * t) = m;
                    }
                }
                pm[(s + PF) % NT] = ld_chunk<T>(inb, row_off(min(vr + PF, vr1 - 1)) + cboff);
                __syncthreads();

                // boxcar row pass on the mirrored copy (integer sums: exact)
                float v[20];
                lds_ld20(bb_ + rbase, v);
                float tb[4];
                if constexpr (FLT) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        float bx = 0.f;
#pragma unroll
                        for (int i = -R; i <= R; ++i) bx = bx + v[8 + q + i];
                        tb[q] = bx;
                    }
                } else {
                    float bx = v[8 - R];
#pragma unroll
                    for (int i = -R + 1; i <= R; ++i) bx = bx + v[8 + i];
                    tb[0] = bx;
#pragma unroll
                    for (int q = 1; q < 4; ++q) {
                        bx = (bx + v[8 + q + R]) - v[8 + q - 1 - R];
                        tb[q] = bx;
                    }
                }
                // Gaussian row pass: zeros outside the frame (skipped taps).
                // A row outside the frame sums to +0 (FMAs of +0 into +0)
                // and so divides to +0: interior strips skip it.
                auto gauss = [&](const float (&u)[20], float (&tg)[4]) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        float gs = 0.f;
#pragma unroll
                        for (int i = -R; i <= R; ++i) gs = __builtin_fmaf(w[i + R], u[8 + q + i], gs);
                        tg[q] = cdiv_t(gs, kp.gn, kp.rgn, FAST);
                    }
                };
                float tg[4];
                if constexpr (BORDER) {
                    float u[20];
                    lds_ld20(bg_ + rbase, u);
                    gauss(u, tg);
                } else if (row_in) {  // wave-uniform
                    gauss(v, tg);
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) tg[q] = 0.f;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float gq = tg[q];
                    if constexpr (!FLT) vbox[q] = (vbox[q] - rb[s][q]) + tb[q];
                    rg[s][q] = gq;
                    rb[s][q] = tb[q];
                }

                if (vr >= y0 + R && vr < vr1) {  // wave-uniform
                    const int o = vr - R;
                    float out[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        float gsum = 0.f;
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            gsum = __builtin_fmaf(w[j], rg[(s + 1 + j) % NT][q], gsum);
                        if constexpr (FLT) {
                            float bsum = 0.f;
#pragma unroll
                            for (int j = 0; j < NT; ++j) bsum = bsum + rb[(s + 1 + j) % NT][q];
                            const float res = cdiv_t(gsum, kp.gn, kp.rgn, FAST) -
                                              cdiv_t(bsum, kp.kk, kp.rkk, FAST);
                            out[q] = res < 0.f ? 0.f : res;
                        } else {
                            const float res = cdiv_t(gsum, kp.gn, kp.rgn, FAST) -
                                              cdiv_t(vbox[q], kp.kk, kp.rkk, FAST);
                            out[q] = __builtin_fmaxf(res, 0.f);   // res is finite, never -0
                        }
                    }
                    if (outl) {
                        // the row offset goes through a scalar register, so
                        // each store adds one uniform value to this lane's
                        // column offset
                        const uint32_t ro = (uint32_t)__builtin_amdgcn_readfirstlane(
                            (int)(4u * (uint32_t)o * (uint32_t)W));
                        *(GLOBAL float4*)((GLOBAL char*)P + (ro + pcoff)) =
                            make_float4(out[0], out[1], out[2], out[3]);
                    }
                    if (kp.hist) {  // wave-uniform
                        // bin (bits >> 19) + 1 for positive values (finite and
                        // >= +0, so no clamp is needed): word bits >> 20, half
                        // bit 19; zero pixels (most of a frame) are counted by
                        // a ballot over the output lanes (one compare serves
                        // both) instead of contending for one word
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            uint32_t bits = __float_as_uint(out[q]);
                            const bool pos = bits != 0u;
                            zc += (uint32_t)__popcll(~__builtin_amdgcn_ballot_w64(pos) & outl_m);
                            // float input can give +inf or NaN: the last bin
                            // takes them (bin 4095: word 2047, low half)
                            if constexpr (FLT) bits = min(bits, 0x7ff7ffffu);
                            if (outl && pos)
                                atomicAdd(&s_hist[bits >> 20], 1u << ((bits >> 15) & 16u));
                        }
                    }
                }
                }
            }
        }
    };
    if (border) rows(std::true_type{});
    else rows(std::false_type{});

    if (kp.hist) {
        __syncthreads();
        uint32_t* gh = b.hist1 + (size_t)f * HIST_BINS;
        for (int i = t; i < HIST_BINS / 2; i += 64) {
            const uint32_t c = s_hist[i];
            if (c & 0xffffu) atomicAdd(&gh[2 * i + 1], c & 0xffffu);
            if ((c >> 16) && 2 * i + 2 < HIST_BINS) atomicAdd(&gh[2 * i + 2], c >> 16);
        }
        if (t == 0 && zc) atomicAdd(&gh[0], zc);
    }
}

// Generic bandpass for R > 8 (and rows whose width is not a multiple of 4): two straightforward passes through a global
// temporary, each thread one pixel, taps in the shader's order.
__global__ void k_bandpass_rows_generic(Batch b, const Geom* __restrict__ g) {
    const uint32_t f = blockIdx.y;
    const Frame fr = b.frames[f];
    const int H = (int)fr.H, W = (int)fr.W;
    const int R = g->R;
    float* tg = fr.tmp;
    float* tb = tg + (size_t)H * W;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (size_t)H * W;
         idx += (size_t)gridDim.x * blockDim.x) {
        const int u = (int)(idx / W), v = (int)(idx % W);
        float gs = 0.f, cs = 0.f;
        for (int i = -R; i <= R; ++i) {
            int pv = v + i;
            bool dg = true;
            if (pv < 0) { pv = -pv - 1; dg = false; }
            else if (pv >= W) { pv = 2 * W - pv - 1; dg = false; }
            const float p = raw_px(fr.in, b.in_type, (size_t)u * W + pv);
            if (dg) gs = __builtin_fmaf(g->w[i + R], p, gs);
            cs = cs + p;
        }
        tg[idx] = gs / g->gn;
        tb[idx] = cs;
    }
}

__global__ void k_bandpass_cols_generic(Batch b, const Geom* __restrict__ g, int hist) {
    __shared__ uint32_t s_hist[HIST_BINS];
    const uint32_t f = blockIdx.y;
    const Frame fr = b.frames[f];
    const int H = (int)fr.H, W = (int)fr.W;
    const int R = g->R;
    const float* tg = fr.tmp;
    const float* tb = tg + (size_t)H * W;
    if (hist)
        for (int i = threadIdx.x; i < HIST_BINS; i += blockDim.x) s_hist[i] = 0;
    __syncthreads();
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (size_t)H * W;
         idx += (size_t)gridDim.x * blockDim.x) {
        const int u = (int)(idx / W), v = (int)(idx % W);
        float gs = 0.f, cs = 0.f;
        for (int i = -R; i <= R; ++i) {
            int pu = u + i;
            bool dg = true;
            if (pu < 0) { pu = -pu - 1; dg = false; }
            else if (pu >= H) { pu = 2 * H - pu - 1; dg = false; }
            if (dg) gs = __builtin_fmaf(g->w[i + R], tg[(size_t)pu * W + v], gs);
            cs = cs + tb[(size_t)pu * W + v];
        }
        const float res = gs / g->gn - cs / g->kk;
        const float out = res < 0.f ? 0.f : res;
        fr.P[idx] = out;
        if (hist) atomicAdd(&s_hist[pct_key(__float_as_uint(out))], 1u);
    }
    if (hist) {
        __syncthreads();
        uint32_t* gh = b.hist1 + (size_t)f * HIST_BINS;
        for (int i = threadIdx.x; i < HIST_BINS; i += blockDim.x)
            if (s_hist[i]) atomicAdd(&gh[i], s_hist[i]);
    }
}

template <int R, typename T>
static hipError_t launch_bp_t(const Batch& b, const K1Params& kp, bool fast, hipStream_t s) {
    if (fast) hipLaunchKernelGGL((k_bandpass<R, T, true>), dim3(b.k1_items), dim3(64), 0, s, b, kp);
    else hipLaunchKernelGGL((k_bandpass<R, T, false>), dim3(b.k1_items), dim3(64), 0, s, b, kp);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_bp_r(int R, const Batch& b, const K1Params& kp, bool fast, hipStream_t s) {
    switch (R) {
        case 1: return launch_bp_t<1, T>(b, kp, fast, s);
        case 2: return launch_bp_t<2, T>(b, kp, fast, s);
        case 3: return launch_bp_t<3, T>(b, kp, fast, s);
        case 4: return launch_bp_t<4, T>(b, kp, fast, s);
        case 5: return launch_bp_t<5, T>(b, kp, fast, s);
        case 6: return launch_bp_t<6, T>(b, kp, fast, s);
        case 7: return launch_bp_t<7, T>(b, kp, fast, s);
        case 8: return launch_bp_t<8, T>(b, kp, fast, s);
        default: return hipErrorInvalidValue;
    }
}

bool bandpass_fast_path(const Batch& b, const Geom& g) {
    return g.R >= 1 && g.R <= 8 && b.vec &&
           (b.in_type == IN_U16 || b.in_type == IN_U8 || b.in_type == IN_F32);
}

hipError_t launch_bandpass(const Batch& b, const Geom& g, const Geom* d_geom, int seg_rows,
                           hipStream_t s) {
    (void)d_geom;
    if (!bandpass_fast_path(b, g)) return hipErrorInvalidValue;
    K1Params kp;
    for (int i = 0; i < 17; ++i) kp.w[i] = (i < 2 * g.R + 1) ? g.w[i] : 0.f;
    kp.gn = g.gn; kp.rgn = g.rgn; kp.kk = g.kk; kp.rkk = g.rkk;
    kp.seg = seg_rows;
    kp.hist = b.hist1 != nullptr && g.has_pct;
    // the LDS histogram keeps 16-bit bins
    if (kp.hist && (int64_t)K1_STRIP * seg_rows >= 65536) return hipErrorInvalidValue;
    const bool fast = g.fastdiv_gn && g.fastdiv_kk;
    if (b.in_type == IN_U16) return launch_bp_r<uint16_t>(g.R, b, kp, fast, s);
    if (b.in_type == IN_F32) return launch_bp_r<float>(g.R, b, kp, fast, s);
    return launch_bp_r<uint8_t>(g.R, b, kp, fast, s);
}

hipError_t launch_bandpass_generic(const Batch& b, const Geom* d_geom, uint32_t max_px,
                                   int hist, hipStream_t s) {
    const uint32_t bx = (uint32_t)std::min<uint64_t>((max_px + 255) / 256, 2048);
    hipLaunchKernelGGL(k_bandpass_rows_generic, dim3(bx, b.nframes), dim3(256), 0, s, b, d_geom);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_bandpass_cols_generic, dim3(bx, b.nframes), dim3(256), 0, s, b, d_geom,
                       hist);
    return hipGetLastError();
}

}  // namespace gt
