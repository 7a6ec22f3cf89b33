// gt_detect.hip -- gfx950 local maxima and centroid walk of the locate path
// (K2; max_rows.wgsl + walk_cols.wgsl).  Pipeline and arithmetic contract:
// gt_kernels.hip.
#include <algorithm>
#include <type_traits>

#include "gt_device.h"

#pragma clang fp contract(off)

namespace gt {

// ---------------------------------------------------------------------------
// K2 detect: local maxima of the dilation window (ties kept), candidate
// slots in raster order within each TILE_W x TILE_H tile.
// ---------------------------------------------------------------------------
struct DetParams {
    int a;              // window start offset
    int kd;             // window size (runtime copy for the generic kernel)
    int band;
    int diw;            // disk inside window (zero-valued maxima cannot yield rows)
    int has_pct;
    int walk_ri;        // disk radius of the walk run inside detect (0: none)
    int nans;           // k_detect_wide: NaN values hide no neighbour
    uint32_t maxit;
    float minmass;
    uint64_t slot_cap;
};

// y[i] = max(x[i .. i+K-1]) for i in [0, N) (van Herk / Gil-Werman): the
// input is cut into blocks of K; a window is the suffix maximum of one block
// joined with the prefix maximum of the next.  All indices are compile-time.
//
// The detect kernels run it on float bit patterns as signed integers: their
// values are finite floats >= +0 (bandpass output, never -0) or -inf (outside
// the frame), for which signed integer order is float order and equal values
// have equal bits.  Integer max needs no NaN canonicalisation.
template <int N, int K>
__device__ __forceinline__ void sliding_max(const int32_t (&x)[N + K - 1], int32_t (&y)[N]) {
    constexpr int L = N + K - 1;
    int32_t S[N];   // suffix max to the end of the block, positions 0..N-1
    int32_t Pm[L];  // prefix max from the start of the block
#pragma unroll
    for (int j = N - 1; j >= 0; --j) {
        const int be = ((j / K) + 1) * K - 1 < L - 1 ? ((j / K) + 1) * K - 1 : L - 1;
        if (j == be) {
            S[j] = x[j];
        } else if (j + 1 < N) {
            S[j] = max(x[j], S[j + 1]);
        } else {
            int32_t m = x[j];
#pragma unroll
            for (int q = j + 1; q <= be; ++q) m = max(m, x[q]);
            S[j] = m;
        }
    }
#pragma unroll
    for (int j = 0; j < L; ++j) Pm[j] = (j % K == 0) ? x[j] : max(Pm[j - 1], x[j]);
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = max(S[i], Pm[i + K - 1]);
}

// Centroid walk of the tile's candidates (centers.wgsl:23-109 and the walk
// of walk_cols.wgsl, as in k_refine): candidate k of the tile (raster
// order) walks in lane k % 256 of the workgroup, so a typical tile (a few
// dozen candidates) occupies part of one wave.  Disks inside the staged area
// are summed from LDS with the taps in the shader's order, others from P.
// L: the staged area, LR rows and LC columns of it valid, LS floats a row.
template <int RI>
__device__ __forceinline__ void walk_tile(const Batch& b, const DetParams& dp,
                                          const float* __restrict__ L, const int LR, const int LC,
                                          const int LS,
                                          const GLOBAL uint16_t* __restrict__ slots,
                                          uint32_t total, uint32_t item,
                                          const GLOBAL float* __restrict__ P, int H, int W,
                                          int x0, int y0, int a, int tid) {
    constexpr int BW = 2 * RI + 1;
    const float sthr = 0.6f;
    const int band = dp.band;
    const size_t slot0 = (size_t)item * TILE_PX;
    const uint64_t cap = dp.slot_cap;
    float* rec = b.rec;
    for (uint32_t k = (uint32_t)tid; k < total; k += 256) {
        const uint32_t l = slots[k];  // written by this workgroup before the barrier
        const int lr0 = (int)(l / TILE_W), lc0 = (int)(l % TILE_W);
        int u = y0 + lr0, v = x0 + lc0;
        float m = 0.f, c0 = 0.f, c1 = 0.f;
        for (uint32_t it = 0; it < dp.maxit; ++it) {
            if (u - band < 0 || u + band >= H || v - band < 0 || v + band >= W) {
                m = 0.f; c0 = 0.f; c1 = 0.f;
            } else {
                // top-left corner of the disk's box in the staged area
                const int br = u - y0 + a - RI, bc = v - x0 + a - RI;
                float s0 = 0.f, s1 = 0.f, ms = 0.f;
                // a tap with a zero coefficient leaves its sum unchanged:
                // fma(d, 0, s) = s exactly (d is finite and s never -0,
                // since the sums start at +0), so those FMAs are skipped
                if (br >= 0 && br + BW <= LR && bc >= 0 && bc + BW <= LC) {
                    const float* box = L + br * LS + bc;
#pragma unroll
                    for (int di = -RI; di <= RI; ++di)
#pragma unroll
                        for (int dj = -RI; dj <= RI; ++dj) {
                            if (di * di + dj * dj > RI * RI) continue;
                            const float d = box[(di + RI) * LS + (dj + RI)];
                            if (di != 0) s0 = __builtin_fmaf(d, (float)di, s0);
                            if (dj != 0) s1 = __builtin_fmaf(d, (float)dj, s1);
                            ms = ms + d;
                        }
                } else if constexpr (RI <= 7) {
#pragma unroll
                    for (int di = -RI; di <= RI; ++di) {
                        const GLOBAL float* row = P + (size_t)(u + di) * W + v;
#pragma unroll
                        for (int dj = -RI; dj <= RI; ++dj) {
                            if (di * di + dj * dj > RI * RI) continue;
                            const float d = row[dj];
                            if (di != 0) s0 = __builtin_fmaf(d, (float)di, s0);
                            if (dj != 0) s1 = __builtin_fmaf(d, (float)dj, s1);
                            ms = ms + d;
                        }
                    }
                } else {   // a rare path: not worth the code of 700 taps
                    int hw = 0;   // half width of the disk's row
                    for (int di = -RI; di <= RI; ++di) {
                        while ((hw + 1) * (hw + 1) + di * di <= RI * RI) ++hw;
                        while (hw * hw + di * di > RI * RI) --hw;
                        const GLOBAL float* row = P + (size_t)(u + di) * W + v;
#pragma unroll 4
                        for (int dj = -hw; dj <= hw; ++dj) {
                            const float d = row[dj];
                            s0 = __builtin_fmaf(d, (float)di, s0);
                            s1 = __builtin_fmaf(d, (float)dj, s1);
                            ms = ms + d;
                        }
                    }
                }
                m = ms;
                c0 = s0 / ms;
                c1 = s1 / ms;
            }
            bool changed = false;
            if (c0 > sthr && u < H - 1) { u += 1; changed = true; }
            else if (c0 < -sthr && u > 0) { u -= 1; changed = true; }
            if (c1 > sthr && v < W - 1) { v += 1; changed = true; }
            else if (c1 < -sthr && v > 0) { v -= 1; changed = true; }
            if (!changed) break;
        }
        const bool valid = (m > dp.minmass) && (m != 0.f);
        rec[REC_MASS * cap + slot0 + k] = valid ? m : 0.f;
        rec[REC_Y * cap + slot0 + k] = (float)u + c0;
        rec[REC_X * cap + slot0 + k] = (float)v + c1;
        if (dp.has_pct) rec[REC_CENTER * cap + slot0 + k] = L[(lr0 + a) * LS + (lc0 + a)];
    }
}

// Bit-pattern range [base, base + width) of percentile histogram bin k
// (width 0 for bin 0 and for "no bin"): a value is listed when
// bits - base < width, unsigned.
__device__ __forceinline__ void pct_bin_range(int32_t k, uint32_t& base, uint32_t& width) {
    if (k <= 0) { base = 0; width = 0; return; }
    base = (uint32_t)(k - 1) << 19;
    width = (k >= HIST_BINS - 1) ? 0x80000000u - base : (1u << 19);
}

// The candidate test of a detect kernel: lane A + c of wave kw holds column c
// of the tile (the other lanes none) in the rows kw * 16 .. + 15, `center` and
// `cm` their values and window maxima.  Writes the tile's slots in raster
// order, its percentile list and its counts; returns the tile's candidate
// count, with the slots not yet visible to the other waves.
//
// Bound by vector instructions, so everything that is one per row is scalar:
// the row's lanes are one compare into a scalar mask, counts and first ranks
// are s_bcnt sums, and a store's lanes are the mask itself.  Per wave that is
// four vector instructions a row and, where the row has an entry, six more
// for the store, and one barrier; by per-lane bits, scans and conditional
// stores it was 18 a row and two barriers.  40 frames of 2048 x 2048, window 15
// with the walk: 321 us then, 289 now; 48 of 1024 x 1024: 85 and 74; window 19,
// 96 of 517 x 663: 67 and 57; window 31, 24 of 1024 x 1024: 82 and 67.
// s_cnt: eight counts, each wave's candidates and list entries.
template <int A>
__device__ __forceinline__ uint32_t row_candidates(const Batch& b, const DetParams& dp,
                                                   const int32_t (&center)[16],
                                                   const int32_t (&cm)[16], uint32_t item,
                                                   uint32_t f, int H, int W, int x0, int y0,
                                                   int tid, uint32_t* s_cnt) {
    constexpr int N = 16;
    const int c = tid & 63;
    const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int v = x0 - A + c;
    const uint64_t omask = ((1ull << TILE_W) - 1) << A;   // lanes with a column of the tile
    const uint64_t colmask = omask & __builtin_amdgcn_ballot_w64((v < W) & (v - dp.band >= 0) &
                                                                 (v + dp.band < W));
    // where a disk inside the window cannot give a zero-valued maximum a row,
    // a candidate is a positive value: values in the frame are >= +0
    int32_t least = dp.diw != 0 ? 1 : INT32_MIN;
    // rows m of the wave's run that can hold a candidate: band <= u0 + m <= H - 1 - band
    const int u0 = y0 + kw * N;
    const int rlo = max(dp.band - u0, 0), rhi = min(H - 1 - dp.band - u0, N - 1);
    const uint32_t rowbits = rhi >= rlo ? ((2u << rhi) - (1u << rlo)) : 0u;
    // values in the two histogram bins holding the order statistics go to
    // the tile's list (any order), each pixel from the one tile whose
    // output lanes hold it; out-of-frame centres are -inf and fall
    // outside every range.  The two order statistics have adjacent
    // ranks, so no value lies strictly between their bins: one range
    // from the start of the lower bin to the end of the upper one holds
    // exactly the two bins.
    uint32_t lcnt = 0, base = 0, width = 0;
    if (dp.has_pct) {
        uint32_t lb, lw, hb, hw;
        pct_bin_range(b.selstate[f * 4 + 0], lb, lw);
        pct_bin_range(b.selstate[f * 4 + 2], hb, hw);
        base = lw ? lb : hb;
        width = hw ? (hb + hw - base) : lw;
#pragma unroll
        for (int m = 0; m < N; ++m)
            lcnt += (uint32_t)__popcll(
                omask & __builtin_amdgcn_ballot_w64((uint32_t)center[m] - base < width));
    }
    uint64_t bal[N];
    uint32_t cnt = 0;
#pragma unroll
    for (int m = 0; m < N; ++m) {
        bal[m] = __builtin_amdgcn_ballot_w64(center[m] >= max(cm[m], least)) &
                 ((rowbits >> m) & 1u ? colmask : 0ull);
        cnt += (uint32_t)__popcll(bal[m]);
    }
    if (c == 0) {
        s_cnt[kw] = cnt;
        s_cnt[4 + kw] = lcnt;
    }
    __syncthreads();
    uint32_t slot = 0, total = 0, entry = 0, ltotal = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t n = __builtin_amdgcn_readfirstlane(s_cnt[w]);
        slot += w < kw ? n : 0u;
        total += n;
        const uint32_t l = __builtin_amdgcn_readfirstlane(s_cnt[4 + w]);
        entry += w < kw ? l : 0u;
        ltotal += l;
    }
    if (tid == 0) {
        b.tile_count[item] = total;
        if (dp.has_pct) b.tile_lcount[item] = ltotal;
    }
    GLOBAL char* slots = (GLOBAL char*)(b.slots + (size_t)item * TILE_PX);
#pragma unroll
    for (int m = 0; m < N; ++m) {
        if (bal[m] == 0) continue;  // wave-uniform: most rows hold no candidate
        if (__builtin_amdgcn_inverse_ballot_w64(bal[m])) {
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                (uint32_t)(bal[m] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal[m], slot));
            *(GLOBAL uint16_t*)(slots + (uint32_t)(2u * rank)) =
                (uint16_t)((kw * N + m) * TILE_W + (c - A));
        }
        slot += (uint32_t)__popcll(bal[m]);
    }
    if (dp.has_pct && lcnt) {
        GLOBAL char* list = (GLOBAL char*)(b.list + (size_t)item * TILE_PX);
        // the rows' masks again: kept from the count they would not fit the
        // scalar registers beside the candidates'
        asm volatile("" : "+s"(base));
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const uint64_t in = omask & __builtin_amdgcn_ballot_w64((uint32_t)center[m] - base < width);
            if (in == 0) continue;
            if (__builtin_amdgcn_inverse_ballot_w64(in)) {
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(in >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)in, entry));
                *(GLOBAL uint32_t*)(list + (uint32_t)(4u * rank)) = (uint32_t)center[m];
            }
            entry += (uint32_t)__popcll(in);
        }
    }
    return total;
}

// One workgroup per 48x64 tile (TILE_W x TILE_H).  Lane c of every wave owns
// staged column c, frame column x0 - a + c: the 64 lanes hold the tile's 48
// columns and the dilation window's halo (KD - 1 <= 16 columns), so the
// column maxima come out in the lanes that own the columns, and the row
// window over them is formed by lane shifts (DPP and ds_bpermute).  The
// staged tile ((64 + KD - 1) x 64 floats: 19.5 KB for KD = 15) is never
// overwritten, so the walk reads it as staged; wave w tests output rows
// 16w .. 16w + 15.  With about 20 KB of LDS and 64 VGPRs, eight workgroups
// share a CU.
//
// RI > 0: the centroid walk of every candidate (refine) runs here too, on
// the staged tile: each candidate walks in one lane, reading its disk from
// LDS (from P when the walk leaves the staged area).  Every candidate walks;
// the percentile test on its start value is applied in dedup, which reads
// that value from the REC_CENTER plane.
template <int KD, int RI>
__global__ __launch_bounds__(256) void k_detect(Batch b, DetParams dp) {
    constexpr int N = 16;
    constexpr int A = (KD - 1) / 2;   // window start trunc(KD / 2 - 0.5), as dp.a
    constexpr int LR = TILE_H + KD - 1;
    constexpr int LS = 64;            // staged columns: one per lane
    constexpr int NIN = N + KD - 1;
    // largest power of two <= KD: the span the doubling steps reach
    constexpr int P2 = KD >= 16 ? 16 : KD >= 8 ? 8 : KD >= 4 ? 4 : KD >= 2 ? 2 : 1;
    static_assert(TILE_W + KD - 1 <= LS, "tile and window halo must fit the 64 lanes");
    __shared__ __attribute__((aligned(16))) float L[LR * LS];
    __shared__ uint32_t s_cnt[8];

    const int tid = threadIdx.x;
    const int c = tid & 63;
    const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.tile_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.tile_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int x0 = (int)(local % fr.tx) * TILE_W;
    const int y0 = (int)(local / fr.tx) * TILE_H;
    const int v = x0 - A + c;         // this lane's frame column
    const GLOBAL float* P = (const GLOBAL float*)fr.P;

    // Staging: wave kw fills rows kw, kw + 4, ...; every row is one 256-byte
    // load across the wave.  Tiles whose staged area lies inside the frame
    // (most of them) load with one 32-bit byte offset per lane, advanced by
    // four rows per load (the frame base stays scalar); the others clamp
    // their indices into the frame (every load in bounds) and store -inf
    // outside it.  All loads are issued before any store.
    {
        constexpr int RPW = (LR + 3) / 4;
        constexpr int QF = RPW - 1;
        const GLOBAL char* Pb = (const GLOBAL char*)P;
        const bool inner = (x0 - A >= 0) && (x0 - A + LS <= W) && (y0 - A >= 0) && (y0 - A + LR <= H);
        float fv[RPW];
        if (inner) {  // workgroup-uniform
            // rows kw + 4q, q < QF, always exist; the last group only for the
            // first waves
            const bool last = kw + 4 * QF < LR;  // wave-uniform
            const uint32_t step = 16u * (uint32_t)W;
            const uint32_t o = 4u * (uint32_t)((y0 - A + kw) * W + v);
#pragma unroll
            for (int q = 0; q < QF; ++q) fv[q] = *(const GLOBAL float*)(Pb + (o + (uint32_t)q * step));
            if (last) fv[QF] = *(const GLOBAL float*)(Pb + (o + (uint32_t)QF * step));
            float* d = L + kw * LS + c;
#pragma unroll
            for (int q = 0; q < QF; ++q) d[4 * q * LS] = fv[q];
            if (last) d[4 * QF * LS] = fv[QF];
        } else {
            const uint32_t oc = 4u * (uint32_t)min(max(v, 0), W - 1);
            const bool cin = v >= 0 && v < W;
#pragma unroll
            for (int q = 0; q < RPW; ++q) {
                const int r = min(kw + 4 * q, LR - 1);  // repeated last row: same values
                const int u = y0 - A + r;
                const uint32_t rb = 4u * (uint32_t)(min(max(u, 0), H - 1) * W);
                fv[q] = *(const GLOBAL float*)(Pb + (rb + oc));
            }
#pragma unroll
            for (int q = 0; q < RPW; ++q) {
                const int r = min(kw + 4 * q, LR - 1);
                const int u = y0 - A + r;
                const bool ur = u >= 0 && u < H;  // wave-uniform
                L[r * LS + c] = (ur && cin) ? fv[q] : __uint_as_float(NEG_INF_BITS);
            }
        }
    }
    __syncthreads();

    // Column pass: this lane's column over the wave's 16 output rows and the
    // window's rows below them; the max filter works on the bit patterns
    // (see sliding_max).  x[m + A] is the centre of output row kw * 16 + m.
    const int32_t* Li = (const int32_t*)L;
    int32_t x[NIN];
#pragma unroll
    for (int m = 0; m < NIN; ++m) x[m] = Li[(kw * N + m) * LS + c];
    int32_t wm[N];
    sliding_max<N, KD>(x, wm);
    // Row window by lane shifts: after the doubling steps wm[m] in lane j is
    // the maximum over lanes j .. j + P2 - 1; the window of the output in
    // lane c is lanes c - A .. c - A + KD - 1, the union of the spans that
    // start at c - A and at c - A + KD - P2.  Lanes past 63 wrap around and
    // feed only lanes that hold no output (c <= A + TILE_W - 1 reads at
    // most lane A + TILE_W - 1 - A + KD - 1 <= 63).
    // Shifts by 1 and 2 are DPP wave shifts (lane j reads lane j + 1; lane
    // 63 reads 0, and lanes past the last output's window feed no output),
    // folded into the max; longer shifts go through ds_bpermute (measured:
    // a shift by 4 as four DPP moves is slower).
#pragma unroll
    for (int s2 = 1; s2 < P2; s2 *= 2) {
        if (s2 <= 2) {
#pragma unroll
            for (int m = 0; m < N; ++m) {
                int32_t t = wm[m];
#pragma unroll
                for (int q = 0; q < s2; ++q) t = __builtin_amdgcn_mov_dpp(t, 0x130, 0xf, 0xf, true);
                wm[m] = max(wm[m], t);
            }
        } else {
            const int src = 4 * ((c + s2) & 63);
#pragma unroll
            for (int m = 0; m < N; ++m) wm[m] = max(wm[m], __builtin_amdgcn_ds_bpermute(src, wm[m]));
        }
    }
    {
        constexpr int D0 = -A, D1 = KD - P2 - A;
        const int src0 = 4 * ((c + D0) & 63), src1 = 4 * ((c + D1) & 63);
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const int32_t w0 = D0 == 0 ? wm[m] : __builtin_amdgcn_ds_bpermute(src0, wm[m]);
            const int32_t w1 = D1 == D0 ? w0
                               : D1 == 0 ? wm[m]
                                         : __builtin_amdgcn_ds_bpermute(src1, wm[m]);
            wm[m] = max(w0, w1);
        }
    }

    int32_t center[N];
#pragma unroll
    for (int m = 0; m < N; ++m) center[m] = x[m + A];
    const uint32_t total = row_candidates<A>(b, dp, center, wm, item, f, H, W, x0, y0, tid, s_cnt);

    if constexpr (RI > 0) {
        if (total == 0) return;  // workgroup-uniform
        const GLOBAL uint16_t* slots = (const GLOBAL uint16_t*)b.slots + (size_t)item * TILE_PX;
        __syncthreads();         // slots visible
        walk_tile<RI>(b, dp, L, LR, LS, LS, slots, total, item, P, H, W, x0, y0, A, tid);
    }
}

// Detect for dilation windows too wide for the lanes of k_detect (KD 18 to
// 26, separation 13 to 19), row first: one workgroup per 48x64 tile, the tile
// and its window halo staged in LDS (all loads issued before the first
// store); the row maxima overwrite the staged tile in place, so one tile
// needs (64+KD-1) x (48+KD+3) floats of LDS and six workgroups share a CU.
// Lane c holds output column c (lanes 48..63 hold none in the column pass).
//
// RI > 0: the centroid walk of every candidate (refine) runs here too, on
// the staged tile: after the candidate test the tile's columns are staged
// again from P (the row maxima overwrote them) and each candidate walks in
// one lane, reading its disk from LDS (from P when the walk leaves the
// staged area).  Every candidate walks; the percentile test on its start
// value is applied in dedup, which reads that value from the REC_CENTER
// plane.
template <int KD, int RI>
__global__ __launch_bounds__(256) void k_detect_rows(Batch b, DetParams dp) {
    constexpr int N = 16;
    constexpr int LR = TILE_H + KD - 1;
    constexpr int LC = TILE_W + KD - 1;
    constexpr int LS = ((LC + 3) / 4) * 4 + 4;
    constexpr int NIN = N + KD - 1;
    constexpr int NV4 = (NIN + 3) / 4;
    constexpr int RUNS = TILE_W / N;              // 16-column runs of an output row
    constexpr int NRUN = (LR * RUNS + 255) / 256;
    static_assert(LC - 64 <= 64, "halo wider than one extra column pass");
    static_assert(LC >= 64, "the first staging pass fills 64 columns");
    __shared__ __attribute__((aligned(16))) float L[LR * LS];
    __shared__ uint32_t s_cnt[8];

    const int tid = threadIdx.x;
    const int a = dp.a;
    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.tile_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.tile_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int x0 = (int)(local % fr.tx) * TILE_W;
    const int y0 = (int)(local / fr.tx) * TILE_H;
    const GLOBAL float* P = (const GLOBAL float*)fr.P;

    // Staging: wave w fills rows w, w+4, ...: lane = column (plus a second
    // pass over the KD-1 halo columns).  Indices are clamped into the frame
    // so every load is in bounds; out-of-frame cells become -inf.  All loads
    // are issued before any store.
    // Tiles whose staged area lies inside the frame (most of them) skip the
    // -inf selects.  Byte offsets are 32-bit (frames hold < 2^30 pixels), so
    // the loads take the frame base as a scalar address.
    const bool inner = (x0 - a >= 0) && (x0 - a + LC <= W) && (y0 - a >= 0) && (y0 - a + LR <= H);
    const GLOBAL char* Pb = (const GLOBAL char*)P;
    auto stage_tile = [&](bool halo) {
        constexpr int RPW = (LR + 3) / 4;
        const int lane = tid & 63;
        const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int v1 = x0 - a + lane, v2 = v1 + 64;
        const bool h2 = halo && lane < LC - 64;
        if (inner) {  // workgroup-uniform
            // every staged row lies inside the frame: one byte offset per
            // lane, advanced by four rows per load, and LDS stores at
            // constant offsets from one address (rows wv + 4q, q < RPW - 1,
            // always exist; the last group only for the first waves)
            constexpr int QF = RPW - 1;
            const bool last = wv + 4 * QF < LR;  // wave-uniform
            const uint32_t step = 16u * (uint32_t)W;
            const uint32_t o = 4u * (uint32_t)((y0 - a + wv) * W + v1);
            float f1[RPW], f2[RPW];
#pragma unroll
            for (int q = 0; q < QF; ++q) f1[q] = *(const GLOBAL float*)(Pb + (o + (uint32_t)q * step));
            if (last) f1[QF] = *(const GLOBAL float*)(Pb + (o + (uint32_t)QF * step));
            if (h2) {
#pragma unroll
                for (int q = 0; q < QF; ++q)
                    f2[q] = *(const GLOBAL float*)(Pb + (o + 256u + (uint32_t)q * step));
                if (last) f2[QF] = *(const GLOBAL float*)(Pb + (o + 256u + (uint32_t)QF * step));
            }
            float* d = L + wv * LS + lane;
#pragma unroll
            for (int q = 0; q < QF; ++q) d[4 * q * LS] = f1[q];
            if (last) d[4 * QF * LS] = f1[QF];
            if (h2) {
#pragma unroll
                for (int q = 0; q < QF; ++q) d[4 * q * LS + 64] = f2[q];
                if (last) d[4 * QF * LS + 64] = f2[QF];
            }
            return;
        }
        const uint32_t o1 = 4u * (uint32_t)min(max(v1, 0), W - 1);
        const uint32_t o2 = 4u * (uint32_t)min(max(v2, 0), W - 1);
        float f1[RPW], f2[RPW];
#pragma unroll
        for (int q = 0; q < RPW; ++q) {
            const int r = min(wv + 4 * q, LR - 1);  // repeated last row: same values
            const int u = y0 - a + r;
            const uint32_t rb = 4u * (uint32_t)(min(max(u, 0), H - 1) * W);
            f1[q] = *(const GLOBAL float*)(Pb + (rb + o1));
            if (h2) f2[q] = *(const GLOBAL float*)(Pb + (rb + o2));
        }
        const bool c1 = v1 >= 0 && v1 < W;
        const bool c2 = v2 >= 0 && v2 < W;
#pragma unroll
        for (int q = 0; q < RPW; ++q) {
            const int r = min(wv + 4 * q, LR - 1);
            const int u = y0 - a + r;
            const bool ur = u >= 0 && u < H;  // wave-uniform
            L[r * LS + lane] = (ur && c1) ? f1[q] : __uint_as_float(NEG_INF_BITS);
            if (h2) L[r * LS + 64 + lane] = (ur && c2) ? f2[q] : __uint_as_float(NEG_INF_BITS);
        }
    };
    stage_tile(true);
    __syncthreads();

    // the max filter works on the bit patterns (see sliding_max)
    const int32_t* Li = (const int32_t*)L;
    // centre values of this thread's 16 outputs, read before the overwrite
    // (lanes past the tile read a column inside it; they hold no output)
    const int c = tid & 63;
    const int cc = min(c, TILE_W - 1);
    const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    int32_t center[N];
#pragma unroll
    for (int m = 0; m < N; ++m) center[m] = Li[(kw * N + m + a) * LS + (cc + a)];

    // row pass: RM[r][c] = max(L[r][c .. c+KD-1]), written over L[r][0..47]
    int32_t y[NRUN][N];
#pragma unroll
    for (int k2 = 0; k2 < NRUN; ++k2) {
        const int run = tid + k2 * 256;
        if (run < LR * RUNS) {
            const int r = run / RUNS, c0 = (run % RUNS) * N;
            int32_t x[NIN];
            const int32_t* src = Li + r * LS + c0;
#pragma unroll
            for (int m = 0; m < NV4; ++m) {
                const int4 q = *(const int4*)(src + 4 * m);
                if (4 * m + 0 < NIN) x[4 * m + 0] = q.x;
                if (4 * m + 1 < NIN) x[4 * m + 1] = q.y;
                if (4 * m + 2 < NIN) x[4 * m + 2] = q.z;
                if (4 * m + 3 < NIN) x[4 * m + 3] = q.w;
            }
            sliding_max<N, KD>(x, y[k2]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k2 = 0; k2 < NRUN; ++k2) {
        const int run = tid + k2 * 256;
        if (run < LR * RUNS) {
            const int r = run / RUNS, c0 = (run % RUNS) * N;
            int32_t* dst = (int32_t*)L + r * LS + c0;
#pragma unroll
            for (int m = 0; m < N / 4; ++m)
                *(int4*)(dst + 4 * m) =
                    make_int4(y[k2][4 * m], y[k2][4 * m + 1], y[k2][4 * m + 2], y[k2][4 * m + 3]);
        }
    }
    __syncthreads();

    // column pass + candidate test: lane = column, wave = 16-row run
    int32_t cm[N];
    {
        int32_t x[NIN];
#pragma unroll
        for (int m = 0; m < NIN; ++m) x[m] = Li[(kw * N + m) * LS + cc];
        sliding_max<N, KD>(x, cm);
    }

    // the maxima are finished here, not after the list's branch, where their
    // two operands would be kept instead (146 registers for 77)
#pragma unroll
    for (int m = 0; m < N; ++m) asm volatile("" : "+v"(cm[m]));
    const uint32_t total = row_candidates<0>(b, dp, center, cm, item, f, H, W, x0, y0, tid, s_cnt);

    if constexpr (RI > 0) {
        const GLOBAL uint16_t* slots = (const GLOBAL uint16_t*)b.slots + (size_t)item * TILE_PX;
        if (total == 0) return;  // workgroup-uniform
        __syncthreads();         // column pass done with L; slots visible
        stage_tile(false);       // columns 0..63 again hold P
        __syncthreads();
        walk_tile<RI>(b, dp, L, LR, LC, LS, slots, total, item, P, H, W, x0, y0, a, tid);
    }
}

// Floats of a staged row of k_detect_wide, and bytes of its tile: the last run
// of a row reads up to 16 columns past the tile.
__host__ __device__ constexpr int wide_stride(int kd) { return (TILE_W + kd - 1 + 3) / 4 * 4 + 4; }
constexpr size_t wide_lds(int kd) {
    return sizeof(float) * ((size_t)(TILE_H + kd - 1) * wide_stride(kd) + 64);
}

// Detect for windows without a kernel of their own: any KD from P2 to
// 2 P2 - 1 (P2 = 16 or 32), and walks over disks of radius up to 15.  As
// k_detect_rows, but a window of KD is the union of two windows of P2 that
// start KD - P2 apart, so the maxima over P2 have compile-time indices and
// only the second one's place is a runtime offset: the row pass leaves
// max(L[r][c .. c + P2 - 1]) over the staged tile, the column pass joins the
// two places of a row and of a column.
//
// nans: windows of 28 and more skip NaN (P of float frames whose pixels are
// not all finite), as the shader's compare does and as float maxima do: it is
// staged as -inf for the maxima and is no candidate itself.  (Up to 26 a NaN
// outranks its neighbours here as in the windows' own kernels, so that a call
// may take either.)  The staged tile is gone over once more for it, so that
// integer frames only skip three branches.
//
// Bound by latency and LDS (32 KB at KD = 31, 59 KB at 63: five to two
// workgroups per CU).  24 frames of 1024^2 at diameter 21 (KD = 31): 67 us
// without the walk, where the straightforward window loops took 353 us.
template <int P2, int RI>
__global__ __launch_bounds__(256) void k_detect_wide(Batch b, DetParams dp) {
    constexpr int N = 16, NIN = N + P2 - 1, NV4 = (NIN + 3) / 4;
    constexpr int MAXRUNS = (TILE_W + P2 - 1 + N - 1) / N;            // 16-column runs of a row
    constexpr int NRUN = ((TILE_H + 2 * P2 - 2) * MAXRUNS + 255) / 256;   // of a thread
    extern __shared__ __attribute__((aligned(16))) float L[];
    __shared__ uint32_t s_cnt[8];

    const int tid = threadIdx.x;
    const int a = dp.a, KD = dp.kd, off = KD - P2;
    const int LR = TILE_H + KD - 1, LC = TILE_W + KD - 1, LS = wide_stride(KD);
    const int runs = (TILE_W + off + N - 1) / N;
    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.tile_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.tile_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int x0 = (int)(local % fr.tx) * TILE_W;
    const int y0 = (int)(local / fr.tx) * TILE_H;
    const GLOBAL float* P = (const GLOBAL float*)fr.P;
    const GLOBAL char* Pb = (const GLOBAL char*)P;

    // Staging: wave w fills rows w, w + 4, ...; lane = column, then column
    // 64 + lane.  Indices are clamped into the frame so every load is in
    // bounds; out-of-frame cells become -inf.  Eight rows are loaded before
    // the first is stored.
    auto stage_tile = [&]() {
        const int lane = tid & 63;
        const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int v1 = x0 - a + lane, v2 = v1 + 64;
        const uint32_t o1 = 4u * (uint32_t)min(max(v1, 0), W - 1);
        const uint32_t o2 = 4u * (uint32_t)min(max(v2, 0), W - 1);
        const bool c1 = lane < LC && v1 >= 0 && v1 < W, c2 = v2 >= 0 && v2 < W;
        const bool h1 = lane < LC, h2 = lane + 64 < LC;
        for (int r0 = wv; r0 < LR; r0 += 32) {
            float f1[8], f2[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int u = y0 - a + r0 + 4 * q;
                const uint32_t rb = 4u * (uint32_t)(min(max(u, 0), H - 1) * W);
                f1[q] = *(const GLOBAL float*)(Pb + (rb + o1));
                f2[q] = *(const GLOBAL float*)(Pb + (rb + o2));
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int r = r0 + 4 * q;
                const int u = y0 - a + r;
                const bool ur = u >= 0 && u < H;  // wave-uniform
                if (r < LR) {
                    if (h1) L[r * LS + lane] = (ur && c1) ? f1[q] : __uint_as_float(NEG_INF_BITS);
                    if (h2) L[r * LS + 64 + lane] = (ur && c2) ? f2[q] : __uint_as_float(NEG_INF_BITS);
                }
            }
        }
    };
    stage_tile();
    const int32_t inf = 0x7f800000;
    if (dp.nans) {   // uniform; every thread over the cells it has stored
        int32_t* cells = (int32_t*)L + (tid & 63);
        for (int r = tid >> 6; r < LR; r += 4)
            for (int j = 0; j + (tid & 63) < LC; j += 64)
                if (cells[r * LS + j] > inf) cells[r * LS + j] = (int32_t)NEG_INF_BITS;
    }
    __syncthreads();

    // the max filter works on the bit patterns (see sliding_max)
    const int32_t* Li = (const int32_t*)L;
    const int c = tid & 63;
    const int cc = min(c, TILE_W - 1);   // lanes past the tile hold no output
    const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    int32_t center[N];
#pragma unroll
    for (int m = 0; m < N; ++m) center[m] = Li[(kw * N + m + a) * LS + (cc + a)];
    if (dp.nans) {   // the values themselves, for the percentile list
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const int u = y0 + kw * N + m, v = x0 + cc;
            const uint32_t o = 4u * (uint32_t)(min(u, H - 1) * W + min(v, W - 1));
            // patterns with the sign set (NaNs) count to the last bin
            const uint32_t x = min(*(const GLOBAL uint32_t*)(Pb + o), (uint32_t)INT32_MAX - 1);
            center[m] = u < H && v < W ? (int32_t)x : (int32_t)NEG_INF_BITS;
        }
    }

    // row pass: max(L[r][c .. c + P2 - 1]) for c < TILE_W + off, over L; the
    // last run of a row reads (but never uses) cells past it
    int32_t y[NRUN][N];
#pragma unroll
    for (int k2 = 0; k2 < NRUN; ++k2) {
        const int run = tid + k2 * 256;
        if (run < LR * runs) {
            const int r = run / runs, c0 = (run % runs) * N;
            int32_t x[NIN];
            const int32_t* src = Li + r * LS + c0;
#pragma unroll
            for (int m = 0; m < NV4; ++m) {
                const int4 q = *(const int4*)(src + 4 * m);
                if (4 * m + 0 < NIN) x[4 * m + 0] = q.x;
                if (4 * m + 1 < NIN) x[4 * m + 1] = q.y;
                if (4 * m + 2 < NIN) x[4 * m + 2] = q.z;
                if (4 * m + 3 < NIN) x[4 * m + 3] = q.w;
            }
            sliding_max<N, P2>(x, y[k2]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k2 = 0; k2 < NRUN; ++k2) {
        const int run = tid + k2 * 256;
        if (run < LR * runs) {
            const int r = run / runs, c0 = (run % runs) * N;
            int32_t* dst = (int32_t*)L + r * LS + c0;
#pragma unroll
            for (int m = 0; m < N / 4; ++m)
                *(int4*)(dst + 4 * m) =
                    make_int4(y[k2][4 * m], y[k2][4 * m + 1], y[k2][4 * m + 2], y[k2][4 * m + 3]);
        }
    }
    __syncthreads();

    // column pass: the row window joins two places, the column window too
    int32_t cm[N];
    {
        auto window = [&](int r0, int32_t (&w)[N]) {
            int32_t x[NIN];
#pragma unroll
            for (int m = 0; m < NIN; ++m) {
                const int32_t* p = Li + (r0 + m) * LS + cc;
                x[m] = max(p[0], p[off]);
            }
            sliding_max<N, P2>(x, w);
        };
        int32_t w2[N];
        window(kw * N, cm);
        window(kw * N + off, w2);
#pragma unroll
        for (int m = 0; m < N; ++m) cm[m] = max(cm[m], w2[m]);
        if (dp.nans) {
#pragma unroll
            for (int m = 0; m < N; ++m) cm[m] = center[m] > inf ? INT32_MAX : cm[m];
        }
    }
    // the maxima are finished here, not after the list's branch, where their
    // two operands would be kept instead (146 registers for 77)
#pragma unroll
    for (int m = 0; m < N; ++m) asm volatile("" : "+v"(cm[m]));
    const uint32_t total = row_candidates<0>(b, dp, center, cm, item, f, H, W, x0, y0, tid, s_cnt);

    if constexpr (RI > 0) {
        const GLOBAL uint16_t* slots = (const GLOBAL uint16_t*)b.slots + (size_t)item * TILE_PX;
        if (total == 0) return;  // workgroup-uniform
        __syncthreads();         // column pass done with L; slots visible
        stage_tile();            // P again
        __syncthreads();
        walk_tile<RI>(b, dp, L, LR, LC, LS, slots, total, item, P, H, W, x0, y0, a, tid);
    }
}

// Generic detect for the smallest windows (KD 1 and 2): straightforward window
// loops over the staged tile.
__global__ __launch_bounds__(256) void k_detect_generic(Batch b, DetParams dp) {
    extern __shared__ float dyn[];
    __shared__ uint64_t s_mask[TILE_H];
    __shared__ uint32_t s_off[TILE_H];
    __shared__ uint32_t s_lcnt;
    if (threadIdx.x == 0) s_lcnt = 0;
    const int KD = dp.kd;
    const int LR = TILE_H + max(KD, 1) - 1, LC = TILE_W + max(KD, 1) - 1;
    float* L = dyn;                  // LR * LC
    float* RM = dyn + LR * LC;       // LR * TILE_W
    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.tile_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.tile_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int x0 = (int)(local % fr.tx) * TILE_W;
    const int y0 = (int)(local / fr.tx) * TILE_H;
    const int tid = threadIdx.x;
    const int a = dp.a;
    const float* P = fr.P;
    for (int idx = tid; idx < LR * LC; idx += 256) {
        const int r = idx / LC, j = idx - r * LC;
        const int u = y0 - a + r, v = x0 - a + j;
        float val = __uint_as_float(NEG_INF_BITS);
        if (u >= 0 && u < H && v >= 0 && v < W) val = P[(size_t)u * W + v];
        L[r * LC + j] = val;
    }
    __syncthreads();
    for (int idx = tid; idx < LR * TILE_W; idx += 256) {
        const int r = idx / TILE_W, c = idx % TILE_W;
        float m = __uint_as_float(NEG_INF_BITS);
        for (int j = 0; j < KD; ++j) m = fmaxf(m, L[r * LC + c + j]);
        RM[idx] = m;
    }
    __syncthreads();
    const int c = tid & 63, k = tid >> 6;   // lanes c >= TILE_W hold no output
    const int v = x0 + c;
    int32_t bin_lo = -1, bin_hi = -1;
    if (dp.has_pct) {
        bin_lo = b.selstate[f * 4 + 0];
        bin_hi = b.selstate[f * 4 + 2];
    }
    uint32_t* list = b.list + (size_t)item * TILE_PX;
    uint32_t cbits = 0;
    for (int m = 0; m < 16; ++m) {
        const int r = k * 16 + m;
        const int u = y0 + r;
        const bool inb = (c < TILE_W) && (u < H) && (v < W);
        float cmx = __uint_as_float(NEG_INF_BITS), center = __uint_as_float(NEG_INF_BITS);
        if (c < TILE_W) {
            for (int i = 0; i < KD; ++i) cmx = fmaxf(cmx, RM[(r + i) * TILE_W + c]);
            center = L[(r + a) * LC + (c + a)];
        }
        const bool interior = (u - dp.band >= 0) && (u + dp.band < H) &&
                              (v - dp.band >= 0) && (v + dp.band < W);
        const bool cand = inb && interior && (center >= cmx) && !(dp.diw && center == 0.f);
        const uint64_t msk = __ballot(cand);
        if (c == 0) s_mask[r] = msk;
        cbits |= (cand ? 1u : 0u) << m;
        if (dp.has_pct) {
            const uint32_t bits = __float_as_uint(center);
            const int key = (int)pct_key(bits);
            const bool match = inb && key != 0 && (key == bin_lo || key == bin_hi);
            const uint64_t mm = __ballot(match);
            if (mm) {
                uint32_t basei = 0;
                if (c == 0) basei = atomicAdd(&s_lcnt, (uint32_t)__popcll(mm));
                basei = __shfl(basei, 0, 64);
                if (match) list[basei + __popcll(mm & lanemask_lt(c))] = bits;
            }
        }
    }
    __syncthreads();
    if (tid < 64) {
        const uint32_t cnt = (uint32_t)__popcll(s_mask[tid]);
        const uint32_t inc = wave_incl_scan(cnt, tid);
        s_off[tid] = inc - cnt;
        if (tid == 63) {
            b.tile_count[item] = inc;
            if (dp.has_pct) b.tile_lcount[item] = s_lcnt;
        }
    }
    __syncthreads();
    uint16_t* slots = b.slots + (size_t)item * TILE_PX;
    for (int m = 0; m < 16; ++m) {
        if (cbits & (1u << m)) {
            const int r = k * 16 + m;
            const uint32_t rank = s_off[r] + (uint32_t)__popcll(s_mask[r] & lanemask_lt(c));
            slots[rank] = (uint16_t)(r * TILE_W + c);
        }
    }
}

// Dilation windows too wide for a staged tile (k_detect_wide's reaches 64 KB of
// LDS past kd = 63, i.e. from separation 46 on): the row maxima of max_rows.wgsl are written to a plane
// (the frame's tmp buffer) by one kernel, and the column test of
// walk_cols.wgsl:23-34 reads that plane in a second.  Each output takes kd
// loads (coalesced across the wave, reused through the caches), as the
// shaders do.
__global__ __launch_bounds__(256) void k_dilate_rows(Batch b, int KD, int a) {
    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.tile_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.tile_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int x0 = (int)(local % fr.tx) * TILE_W;
    const int y0 = (int)(local / fr.tx) * TILE_H;
    const int c = threadIdx.x & 63, k = threadIdx.x >> 6;
    const int v = x0 + c;
    if (c >= TILE_W || v >= W) return;
    const float* P = fr.P;
    float* RM = fr.tmp;
    const int j0 = max(0, a - v), j1 = min(KD, W + a - v);   // in-bounds taps v - a + j
    for (int m = 0; m < 16; ++m) {
        const int u = y0 + k * 16 + m;
        if (u >= H) break;
        const float* row = P + (size_t)u * W;
        float mx = __uint_as_float(NEG_INF_BITS);
        for (int j = j0; j < j1; ++j) mx = fmaxf(mx, row[v - a + j]);
        RM[(size_t)u * W + v] = mx;
    }
}

__global__ __launch_bounds__(256) void k_detect_plane(Batch b, DetParams dp) {
    __shared__ uint64_t s_mask[TILE_H];
    __shared__ uint32_t s_off[TILE_H];
    __shared__ uint32_t s_lcnt;
    if (threadIdx.x == 0) s_lcnt = 0;
    __syncthreads();
    const int KD = dp.kd, a = dp.a;
    const uint32_t item = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t f = b.tile_frame[item];
    const Frame fr = b.frames[f];
    const uint32_t local = item - fr.tile_base;
    const int H = (int)fr.H, W = (int)fr.W;
    const int x0 = (int)(local % fr.tx) * TILE_W;
    const int y0 = (int)(local / fr.tx) * TILE_H;
    const int tid = threadIdx.x, c = tid & 63, k = tid >> 6;
    const int v = x0 + c;
    const float* P = fr.P;
    const float* RM = fr.tmp;
    int32_t bin_lo = -1, bin_hi = -1;
    if (dp.has_pct) {
        bin_lo = b.selstate[f * 4 + 0];
        bin_hi = b.selstate[f * 4 + 2];
    }
    uint32_t* list = b.list + (size_t)item * TILE_PX;
    uint32_t cbits = 0;
    for (int m = 0; m < 16; ++m) {
        const int r = k * 16 + m;
        const int u = y0 + r;
        const bool inb = (c < TILE_W) && (u < H) && (v < W);
        float center = 0.f;
        bool cand = false;
        if (inb) {
            center = P[(size_t)u * W + v];
            const int i0 = max(0, a - u), i1 = min(KD, H + a - u);   // in-bounds rows u - a + i
            float cmx = __uint_as_float(NEG_INF_BITS);
            for (int i = i0; i < i1; ++i) cmx = fmaxf(cmx, RM[(size_t)(u - a + i) * W + v]);
            const bool interior = (u - dp.band >= 0) && (u + dp.band < H) &&
                                  (v - dp.band >= 0) && (v + dp.band < W);
            cand = interior && (center >= cmx) && !(dp.diw && center == 0.f);
        }
        const uint64_t msk = __ballot(cand);
        if (c == 0) s_mask[r] = msk;
        cbits |= (cand ? 1u : 0u) << m;
        if (dp.has_pct) {
            const uint32_t bits = __float_as_uint(center);
            const int key = (int)pct_key(bits);
            const bool match = inb && key != 0 && (key == bin_lo || key == bin_hi);
            const uint64_t mm = __ballot(match);
            if (mm) {
                uint32_t basei = 0;
                if (c == 0) basei = atomicAdd(&s_lcnt, (uint32_t)__popcll(mm));
                basei = __shfl(basei, 0, 64);
                if (match) list[basei + __popcll(mm & lanemask_lt(c))] = bits;
            }
        }
    }
    __syncthreads();
    if (tid < 64) {
        const uint32_t cnt = (uint32_t)__popcll(s_mask[tid]);
        const uint32_t inc = wave_incl_scan(cnt, tid);
        s_off[tid] = inc - cnt;
        if (tid == 63) {
            b.tile_count[item] = inc;
            if (dp.has_pct) b.tile_lcount[item] = s_lcnt;
        }
    }
    __syncthreads();
    uint16_t* slots = b.slots + (size_t)item * TILE_PX;
    for (int m = 0; m < 16; ++m) {
        if (cbits & (1u << m)) {
            const int r = k * 16 + m;
            const uint32_t rank = s_off[r] + (uint32_t)__popcll(s_mask[r] & lanemask_lt(c));
            slots[rank] = (uint16_t)(r * TILE_W + c);
        }
    }
}

static size_t detect_generic_lds(int kd) {
    const int kd1 = max(kd, 1);
    return sizeof(float) * ((size_t)(TILE_H + kd1 - 1) * (TILE_W + kd1 - 1) +
                            (size_t)(TILE_H + kd1 - 1) * TILE_W);
}

// Windows of k_detect_wide: its staged tile stays below 64 KB of LDS.
constexpr int WIDE_MIN = 16, WIDE_MAX = 63;

bool detect_needs_plane(const Geom& g) { return g.kd > WIDE_MAX; }

template <int KD>
static hipError_t launch_det_t(const Batch& b, const DetParams& dp, hipStream_t s) {
    if (dp.a != (KD - 1) / 2) return hipErrorInvalidValue;   // the kernel's window start
    switch (dp.walk_ri) {
        case 0: hipLaunchKernelGGL((k_detect<KD, 0>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 1: hipLaunchKernelGGL((k_detect<KD, 1>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 2: hipLaunchKernelGGL((k_detect<KD, 2>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 3: hipLaunchKernelGGL((k_detect<KD, 3>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 4: hipLaunchKernelGGL((k_detect<KD, 4>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 5: hipLaunchKernelGGL((k_detect<KD, 5>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 6: hipLaunchKernelGGL((k_detect<KD, 6>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 7: hipLaunchKernelGGL((k_detect<KD, 7>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int KD>
static hipError_t launch_det_rows_t(const Batch& b, const DetParams& dp, hipStream_t s) {
    switch (dp.walk_ri) {
        case 0: hipLaunchKernelGGL((k_detect_rows<KD, 0>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 1: hipLaunchKernelGGL((k_detect_rows<KD, 1>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 2: hipLaunchKernelGGL((k_detect_rows<KD, 2>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 3: hipLaunchKernelGGL((k_detect_rows<KD, 3>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 4: hipLaunchKernelGGL((k_detect_rows<KD, 4>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 5: hipLaunchKernelGGL((k_detect_rows<KD, 5>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 6: hipLaunchKernelGGL((k_detect_rows<KD, 6>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 7: hipLaunchKernelGGL((k_detect_rows<KD, 7>), dim3(b.tiles), dim3(256), 0, s, b, dp); break;
        case 8:  // disk radius 8 (diameters 17, 18) walks here from window 22 on
            if constexpr (KD >= 22) {
                hipLaunchKernelGGL((k_detect_rows<KD, 8>), dim3(b.tiles), dim3(256), 0, s, b, dp);
                break;
            } else {
                return hipErrorInvalidValue;
            }
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

static bool detect_specialised(int kd) {
    switch (kd) {
        case 4: case 5: case 7: case 8: case 9: case 11: case 12: case 14: case 15: case 16:
        case 18: case 19: case 21: case 22: case 24: case 25: case 26:
            return true;
        default:
            return false;
    }
}

// Largest disk radius that a window's own kernel walks.
static int specialised_radius(int kd) { return kd >= 22 ? 8 : 7; }

bool walk_in_own_detect(const Geom& g) {
    return g.rint >= 1 && g.max_iterations >= 1 && detect_specialised(g.kd) &&
           g.rint <= specialised_radius(g.kd);
}

bool walk_in_detect_supported(const Geom& g) {
    if (g.rint < 1 || g.max_iterations < 1) return false;
    return walk_in_own_detect(g) || (g.kd >= WIDE_MIN && g.kd <= WIDE_MAX && g.rint <= 15);
}

template <int P2>
static hipError_t launch_det_wide_t(const Batch& b, const DetParams& dp, hipStream_t s) {
    const dim3 grid(b.tiles), block(256);
    const size_t lds = wide_lds(dp.kd);
#define GT_WIDE(RI) \
    case RI: hipLaunchKernelGGL((k_detect_wide<P2, RI>), grid, block, lds, s, b, dp); break;
    switch (dp.walk_ri) {
        GT_WIDE(0) GT_WIDE(1) GT_WIDE(2) GT_WIDE(3) GT_WIDE(4) GT_WIDE(5) GT_WIDE(6) GT_WIDE(7)
        GT_WIDE(8) GT_WIDE(9) GT_WIDE(10) GT_WIDE(11) GT_WIDE(12) GT_WIDE(13) GT_WIDE(14) GT_WIDE(15)
        default: return hipErrorInvalidValue;
    }
#undef GT_WIDE
    return hipGetLastError();
}

hipError_t launch_detect(const Batch& b, const Geom& g, const Geom* d_geom, hipStream_t s) {
    (void)d_geom;
    DetParams dp;
    dp.a = g.a;
    dp.kd = g.kd;
    dp.band = g.band;
    dp.diw = g.disk_in_window;
    dp.has_pct = g.has_pct;
    dp.walk_ri = g.walk_in_detect ? g.rint : 0;
    dp.nans = b.in_type == IN_F32 && !detect_specialised(g.kd);
    dp.maxit = g.max_iterations;
    dp.minmass = g.minmass;
    dp.slot_cap = b.slot_cap;
    // windows of 28 to 63 have no kernel of their own; from 16 on, a disk that
    // the window's kernel does not walk goes the same way
    const bool own = detect_specialised(g.kd) && dp.walk_ri <= specialised_radius(g.kd);
    if (!own && g.kd >= WIDE_MIN && g.kd <= WIDE_MAX) {
        // (the kernel's windows start where the others' do)
        return g.kd < 32 ? launch_det_wide_t<16>(b, dp, s) : launch_det_wide_t<32>(b, dp, s);
    }
    switch (g.kd) {
        case 4: return launch_det_t<4>(b, dp, s);
        case 5: return launch_det_t<5>(b, dp, s);
        case 7: return launch_det_t<7>(b, dp, s);
        case 8: return launch_det_t<8>(b, dp, s);
        case 9: return launch_det_t<9>(b, dp, s);
        case 11: return launch_det_t<11>(b, dp, s);
        case 12: return launch_det_t<12>(b, dp, s);
        case 14: return launch_det_t<14>(b, dp, s);
        case 15: return launch_det_t<15>(b, dp, s);
        case 16: return launch_det_t<16>(b, dp, s);
        case 18: return launch_det_rows_t<18>(b, dp, s);
        case 19: return launch_det_rows_t<19>(b, dp, s);
        case 21: return launch_det_rows_t<21>(b, dp, s);
        case 22: return launch_det_rows_t<22>(b, dp, s);
        case 24: return launch_det_rows_t<24>(b, dp, s);
        case 25: return launch_det_rows_t<25>(b, dp, s);
        case 26: return launch_det_rows_t<26>(b, dp, s);
        default: break;
    }
    if (detect_needs_plane(g)) {
        hipLaunchKernelGGL(k_dilate_rows, dim3(b.tiles), dim3(256), 0, s, b, g.kd, g.a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_detect_plane, dim3(b.tiles), dim3(256), 0, s, b, dp);
        return hipGetLastError();
    }
    const size_t shm = detect_generic_lds(g.kd);
    hipLaunchKernelGGL(k_detect_generic, dim3(b.tiles), dim3(256), shm, s, b, dp);
    return hipGetLastError();
}

}  // namespace gt
