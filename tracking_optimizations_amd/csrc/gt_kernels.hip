// gt_kernels.hip -- gfx950 kernels of the per-frame locate path.
//
// Pipeline per batch of frames (every stage is one launch over all frames of
// the batch; work items are (frame, tile) pairs):
//   begin     clear per-frame counters and histograms, expand item tables
//   bandpass  K1: u16/u8/f32 -> P (float32), optional percentile histogram
//             (preprocess_rows.wgsl + preprocess_cols.wgsl)
//   select1   percentile: histogram bin of the two order statistics
//   detect    K2: grey-dilation local maxima (max_rows.wgsl + walk_cols.wgsl
//             is_max) -> per-tile candidate slots; percentile value list
//   select2   percentile: exact order statistics -> threshold
//   refine    K3: walk + disk mass/centroid (centers.wgsl, walk_cols.wgsl
//             walk), minmass; where detect has not walked
//   dedup     K4: separation suppression (execute_gpu.rs:258-284)
//   scan      row offsets
//   emit      K5: rows in column_names order; then the characterisation and
//             raw signal columns (gt_char.hip, gt_raw.hip)
//
// Arithmetic contract (identical to the CPU oracle): every `acc += a*b` of a
// WGSL shader is one fused multiply-add, every other operation one binary32
// operation in the shader's order; nothing else is contracted (this file is
// compiled with contraction off).  Divisions by the two per-call constants
// (gauss_norm, k*k) multiply by a two-part reciprocal only when the host has
// verified, for every significand, that it rounds exactly like IEEE division;
// otherwise they are IEEE divisions.
#include <algorithm>
#include <type_traits>

#include "gt_device.h"

#pragma clang fp contract(off)

namespace gt {

// ---------------------------------------------------------------------------
// begin: the first launch of a batch.  Clears the per-frame counters and
// histograms, and expands the batch's bases into the per-item tables: frame
// blockIdx.y writes the frame index of each of its bandpass items and tiles
// and the top-left tile of each of its dedup blocks (the frame's blocks in
// raster order).  The first batch of a call also clears the running totals
// (`carry`, two pairs).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_begin(Batch b, const uint32_t* __restrict__ dbases,
                                               uint64_t* __restrict__ carry) {
    const uint32_t f = blockIdx.y;
    const uint32_t k1a = b.k1_bases[f], k1n = b.k1_bases[f + 1] - k1a;
    const uint32_t ta = b.tile_bases[f], tn = b.tile_bases[f + 1] - ta;
    const uint32_t da = dbases[f], dn = dbases[f + 1] - da;
    const uint32_t tx = b.frames[f].tx;
    const uint32_t ds = b.dblock_side;
    const uint32_t bx = (tx + ds - 1) / ds;   // dedup blocks per block row
    uint32_t* k1f = (uint32_t*)b.k1_frame;
    uint32_t* tf = (uint32_t*)b.tile_frame;
    uint32_t* dt = (uint32_t*)b.dblock_tile;
    const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
    if (t0 == 0) b.counts[(size_t)f * b.count_stride] = 0;
    if (carry && f == 0 && t0 < 4) carry[t0] = 0;
    if (b.hist1)
        for (uint32_t i = t0; i < (uint32_t)HIST_BINS; i += step) b.hist1[(size_t)f * HIST_BINS + i] = 0;
    for (uint32_t i = t0; i < k1n + tn + dn; i += step) {
        if (i < k1n) {
            k1f[k1a + i] = f;
        } else if (i < k1n + tn) {
            tf[ta + (i - k1n)] = f;
        } else {
            const uint32_t j = i - k1n - tn;
            dt[da + j] = ta + ds * (j / bx) * tx + ds * (j % bx);
        }
    }
}

hipError_t launch_begin(const Batch& b, const uint32_t* dblock_bases, uint32_t max_frame_work,
                        uint64_t* carry, hipStream_t s) {
    const uint32_t work = std::max(max_frame_work, b.hist1 ? (uint32_t)HIST_BINS : 1u);
    const uint32_t bx = std::min<uint32_t>((work + 255) / 256, 64);
    hipLaunchKernelGGL(k_begin, dim3(bx, b.nframes), dim3(256), 0, s, b, dblock_bases, carry);
    return hipGetLastError();
}

// The end of a call: its totals and, where they are few, its rows written
// straight to pinned host memory, so that the host waits once instead of once
// for the totals and again for each copy.  Latency bound (about 5 us): with the
// tables' single upload a 512 x 512 call went from 220 to 127 us.
__global__ __launch_bounds__(256) void k_export(const uint64_t* __restrict__ totals,
                                                const float* __restrict__ rows,
                                                const int64_t* __restrict__ cand, uint32_t ncols,
                                                uint64_t few, uint64_t* __restrict__ h_totals,
                                                float* __restrict__ h_rows,
                                                int64_t* __restrict__ h_cand) {
    const uint64_t n = totals[0];
    const uint64_t t0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    if (t0 < 2) h_totals[t0] = totals[t0];
    if (n > few) return;
    for (uint64_t i = t0; i < n * ncols; i += step) h_rows[i] = rows[i];
    for (uint64_t i = t0; i < n; i += step) h_cand[i] = cand[i];
}

hipError_t launch_export(const uint64_t* totals, const float* rows, const int64_t* cand,
                         uint32_t ncols, uint64_t few, uint64_t* h_totals, float* h_rows,
                         int64_t* h_cand, hipStream_t s) {
    hipLaunchKernelGGL(k_export, dim3(few ? 16 : 1), dim3(256), 0, s, totals, rows, cand, ncols, few,
                       h_totals, h_rows, h_cand);
    return hipGetLastError();
}

// Plain device copy: 16-byte vectors, grid-stride, byte tail.  Also the kernel
// of known traffic (n bytes read, n written) for scaling byte counters.
__global__ void k_copy(uint4* __restrict__ dst, const uint4* __restrict__ src, uint64_t n16,
                       uint8_t* __restrict__ dtail, const uint8_t* __restrict__ stail,
                       uint32_t ntail) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
        dst[i] = src[i];
    if (blockIdx.x == 0 && threadIdx.x < ntail) dtail[threadIdx.x] = stail[threadIdx.x];
}

hipError_t launch_copy(void* dst, const void* src, uint64_t bytes, hipStream_t s) {
    const uint64_t n16 = bytes / 16;
    const uint32_t ntail = (uint32_t)(bytes % 16);
    uint32_t blocks = (uint32_t)std::min<uint64_t>((n16 + 255) / 256, 8192);
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(k_copy, dim3(blocks), dim3(256), 0, s, (uint4*)dst, (const uint4*)src,
                       n16, (uint8_t*)dst + n16 * 16, (const uint8_t*)src + n16 * 16, ntail);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// select1: histogram bins holding the order statistics lo and hi
// ---------------------------------------------------------------------------
__device__ __forceinline__ void pct_ranks(uint64_t n, float percentile, uint64_t& lo,
                                          uint64_t& hi, double& frac) {
    const double q = (double)percentile / 100.0;
    const double h = (double)(n - 1) * q;
    const double fl = floor(h);
    lo = (uint64_t)fl;
    if (lo > n - 1) lo = n - 1;
    hi = (lo + 1 < n) ? lo + 1 : n - 1;
    frac = h - fl;
}

__global__ __launch_bounds__(256) void k_select1(Batch b, float percentile) {
    __shared__ uint32_t s_part[256];
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const uint64_t n = (uint64_t)fr.H * fr.W;
    uint64_t lo, hi;
    double frac;
    pct_ranks(n, percentile, lo, hi, frac);
    const uint32_t* hist = b.hist1 + (size_t)f * HIST_BINS;
    const int t = threadIdx.x;
    constexpr int PER = HIST_BINS / 256;
    uint32_t c[PER];
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) { c[i] = hist[t * PER + i]; sum += c[i]; }
    s_part[t] = sum;
    __syncthreads();
    // exclusive prefix of the 256 partial sums (serial per thread is cheap
    // enough here: 256 adds from LDS)
    uint64_t before = 0;
    for (int i = 0; i < t; ++i) before += s_part[i];
    uint64_t cum = before;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const uint64_t nxt = cum + c[i];
        if (lo >= cum && lo < nxt) {
            b.selstate[f * 4 + 0] = t * PER + i;
            b.selstate[f * 4 + 1] = (int32_t)(lo - cum);
        }
        if (hi >= cum && hi < nxt) {
            b.selstate[f * 4 + 2] = t * PER + i;
            b.selstate[f * 4 + 3] = (int32_t)(hi - cum);
        }
        cum = nxt;
    }
}

hipError_t launch_select1(const Batch& b, const Geom& g, hipStream_t s) {
    hipLaunchKernelGGL(k_select1, dim3(b.nframes), dim3(256), 0, s, b, g.percentile);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// select2: exact order statistics from the value list, then the threshold
// ---------------------------------------------------------------------------
// Exact order statistics lo and hi of one frame by radix selection over the
// per-tile value lists: level A counts bits [18:8] of the values in each
// target bin, level B bits [7:0] of the values sharing the chosen level-A
// digit.  Both targets share every pass.  Bound by the latency of the list
// reads (16 bytes each): a thread per tile where a frame has about as many
// tiles as the workgroup threads (1376 tiles: 14 us for 40 frames; 16 threads
// each: 44 us), up to 16 threads where it has fewer (88 tiles: 9 against 11
// us).
__global__ __launch_bounds__(1024) void k_select2(Batch b, float percentile) {
    __shared__ uint32_t s_ha[2][2048];
    __shared__ uint32_t s_res[2][3];
    __shared__ uint32_t s_wsum[2][16];
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const uint64_t n = (uint64_t)fr.H * fr.W;
    uint64_t lo, hi;
    double frac;
    pct_ranks(n, percentile, lo, hi, frac);
    const int t = threadIdx.x;
    if (t < 6) s_res[t / 3][t % 3] = 0;
    const int bin[2] = {b.selstate[f * 4 + 0], b.selstate[f * 4 + 2]};
    const int rank[2] = {b.selstate[f * 4 + 1], b.selstate[f * 4 + 3]};
    const bool need[2] = {bin[0] != 0, hi != lo && bin[1] != 0};
    const uint32_t ntiles = fr.tx * fr.ty;
    const uint32_t lpt = ntiles > 512 ? 1u : ntiles > 128 ? 4u : 16u;   // threads per tile
    for (int pass = 0; pass < 2; ++pass) {
        const int nb = pass == 0 ? 2048 : 256;
        for (int i = t; i < 2 * 2048; i += 1024) s_ha[i / 2048][i % 2048] = 0;
        __syncthreads();
        const uint32_t sa0 = pass ? s_res[0][0] : 0u, sa1 = pass ? s_res[1][0] : 0u;
        for (uint32_t tl = (uint32_t)t / lpt; tl < ntiles; tl += 1024 / lpt) {
            const uint32_t it = fr.tile_base + tl;
            const uint32_t cnt = b.tile_lcount[it];
            const GLOBAL uint4* lst = (const GLOBAL uint4*)(b.list + (size_t)it * TILE_PX);
            for (uint32_t i4 = (uint32_t)t % lpt; 4 * i4 < cnt; i4 += lpt) {
                const uint4 q = lst[i4];
                const uint32_t vals[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (i4 * 4 + e >= cnt) break;
                    const uint32_t bits = vals[e];
                    const int key = (int)pct_key(bits);
                    const uint32_t da = (bits >> 8) & 2047u;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        if (!need[s] || key != bin[s]) continue;
                        if (pass == 0) atomicAdd(&s_ha[s][da], 1u);
                        else if (da == (s ? sa1 : sa0)) atomicAdd(&s_ha[s][bits & 255u], 1u);
                    }
                }
            }
        }
        __syncthreads();
        // Selection: a workgroup-wide exclusive prefix sum over the bins
        // (thread t holds bins 2t, 2t+1 of 2048, or bin t of 256); the thread
        // whose range holds the wanted rank picks the bin.
        const uint32_t want0 = pass == 0 ? (uint32_t)rank[0] : s_res[0][1];
        const uint32_t want1 = pass == 0 ? (uint32_t)rank[1] : s_res[1][1];
        uint32_t c0a, c0b, c1a, c1b;
        if (nb == 2048) {
            c0a = s_ha[0][2 * t]; c0b = s_ha[0][2 * t + 1];
            c1a = s_ha[1][2 * t]; c1b = s_ha[1][2 * t + 1];
        } else {
            c0a = t < 256 ? s_ha[0][t] : 0u; c0b = 0u;
            c1a = t < 256 ? s_ha[1][t] : 0u; c1b = 0u;
        }
        const int lane = t & 63, wv = t >> 6;
        const uint32_t l0 = c0a + c0b, l1 = c1a + c1b;
        const uint32_t i0 = wave_incl_scan(l0, lane), i1 = wave_incl_scan(l1, lane);
        if (lane == 63) { s_wsum[0][wv] = i0; s_wsum[1][wv] = i1; }
        __syncthreads();
        uint32_t e0 = i0 - l0, e1 = i1 - l1;
        for (int q = 0; q < wv; ++q) { e0 += s_wsum[0][q]; e1 += s_wsum[1][q]; }
        const int per = nb == 2048 ? 2 : 1;
#pragma unroll
        for (int sidx = 0; sidx < 2; ++sidx) {
            const uint32_t want = sidx ? want1 : want0;
            const uint32_t ex = sidx ? e1 : e0, ca = sidx ? c1a : c0a, cb = sidx ? c1b : c0b;
            if (need[sidx] && want >= ex && want < ex + ca + cb) {
                const bool first = want < ex + ca;
                const uint32_t sel = (uint32_t)(per * t) + (first ? 0u : 1u);
                const uint32_t below = first ? ex : ex + ca;
                if (pass == 0) {
                    s_res[sidx][0] = sel;
                    s_res[sidx][1] = want - below;
                } else {
                    s_res[sidx][2] = ((uint32_t)(bin[sidx] - 1) << 19) | (s_res[sidx][0] << 8) | sel;
                }
            }
        }
        __syncthreads();
    }
    if (t == 0) {
        const float vlo = need[0] ? __uint_as_float(s_res[0][2]) : 0.f;
        const float vhi = (hi == lo) ? vlo : (need[1] ? __uint_as_float(s_res[1][2]) : 0.f);
        b.thr[f] = (double)vlo + frac * ((double)vhi - (double)vlo);
    }
}

hipError_t launch_select2(const Batch& b, const Geom& g, hipStream_t s) {
    hipLaunchKernelGGL(k_select2, dim3(b.nframes), dim3(1024), 0, s, b, g.percentile);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// K3 refine: one lane per candidate, one wave per tile.
// ---------------------------------------------------------------------------

// centers.wgsl:23-109 at one pixel (binary32, taps in shader order).
__device__ __forceinline__ void disk_eval(const float* __restrict__ P, int H, int W, int band,
                                          int rint, int u, int v, float& m, float& c0,
                                          float& c1) {
    if (u - band < 0 || u + band >= H || v - band < 0 || v + band >= W) {
        m = 0.f; c0 = 0.f; c1 = 0.f;
        return;
    }
    float s0 = 0.f, s1 = 0.f, ms = 0.f;
    for (int i = -rint; i <= rint; ++i) {
        int hw = 0;
        while ((hw + 1) * (hw + 1) + i * i <= rint * rint) ++hw;
        const float* row = P + (size_t)(u + i) * W + v;
        const float fi = (float)i;
        for (int j = -hw; j <= hw; ++j) {
            const float d = row[j];
            s0 = __builtin_fmaf(d, fi, s0);
            s1 = __builtin_fmaf(d, (float)j, s1);
            ms = ms + d;
        }
    }
    m = ms;
    c0 = s0 / ms;
    c1 = s1 / ms;
}

// Candidates of RT_TILES consecutive tiles are packed over the 256 lanes of a
// workgroup (a tile holds ~16 candidates on average; one wave per tile would
// leave three quarters of the lanes idle while issuing the same number of
// scattered loads).
constexpr int RT_TILES = 16;

struct RefTile {
    const float* P;
    int x0, y0, H, W;
    uint32_t f, cnt, pref;
};

// Lanes of the first wave fill the workgroup's tiles and their first candidates.
__device__ __forceinline__ void load_ref_tiles(const Batch& b, uint32_t item0, int nt, int tid,
                                               RefTile* s_t, uint32_t& s_total) {
    if (tid >= 64) return;
    uint32_t cnt = 0;
    RefTile rt;
    if (tid < nt) {
        const uint32_t item = item0 + tid;
        const uint32_t f = b.tile_frame[item];
        const Frame fr = b.frames[f];
        const uint32_t local = item - fr.tile_base;
        rt.P = fr.P;
        rt.x0 = (int)(local % fr.tx) * TILE_W;
        rt.y0 = (int)(local / fr.tx) * TILE_H;
        rt.H = (int)fr.H;
        rt.W = (int)fr.W;
        rt.f = f;
        cnt = b.tile_count[item];
        rt.cnt = cnt;
    }
    const uint32_t inc = wave_incl_scan(cnt, tid);
    if (tid < nt) {
        rt.pref = inc - cnt;
        s_t[tid] = rt;
    }
    if (tid == 63) s_total = inc;
}

// Refinement of what k_walk does not take: no iterations, disks of radius 0 or
// above 15.
__global__ __launch_bounds__(256) void k_refine(Batch b, const Geom* __restrict__ g) {
    __shared__ RefTile s_t[RT_TILES];
    __shared__ uint32_t s_total;
    const uint32_t item0 = blockIdx.x * RT_TILES;
    const int nt = (int)min<uint32_t>(RT_TILES, b.tiles - item0);
    const int tid = threadIdx.x;
    load_ref_tiles(b, item0, nt, tid, s_t, s_total);
    __syncthreads();
    const uint32_t total = s_total;
    const int band = g->band, rint = g->rint;
    const uint32_t maxit = g->max_iterations;
    const float minmass = g->minmass;
    const float sthr = 0.6f;
    float* rec = b.rec;
    const uint64_t cap = b.slot_cap;

    for (uint32_t gi = tid; gi < total; gi += 256) {
        int j = 0;
#pragma unroll
        for (int q = 1; q < RT_TILES; ++q)
            if (q < nt && s_t[q].pref <= gi) j = q;
        const RefTile& rt = s_t[j];
        const uint32_t i = gi - rt.pref;
        const uint32_t item = item0 + (uint32_t)j;
        const size_t slot0 = (size_t)item * TILE_PX;
        const int H = rt.H, W = rt.W;
        const float* __restrict__ P = rt.P;
        const double thr = g->has_pct ? b.thr[rt.f] : 0.0;
        const int x0 = rt.x0, y0 = rt.y0;
        const uint32_t l = b.slots[slot0 + i];
        const int u0 = y0 + (int)(l / TILE_W), v0 = x0 + (int)(l % TILE_W);
        bool valid = true;
        if (g->has_pct) valid = (double)P[(size_t)u0 * W + v0] > thr;
        float y = 0.f, x = 0.f, mass = 0.f;
        if (valid) {
            int u = u0, v = v0;
            float c0 = 0.f, c1 = 0.f, m = 0.f;
            if (maxit == 0) {
                float t0, t1;
                disk_eval(P, H, W, band, rint, 0, 0, m, t0, t1);
            }
            for (uint32_t it = 0; it < maxit; ++it) {
                disk_eval(P, H, W, band, rint, u, v, m, c0, c1);
                bool changed = false;
                if (c0 > sthr && u < H - 1) { u += 1; changed = true; }
                else if (c0 < -sthr && u > 0) { u -= 1; changed = true; }
                if (c1 > sthr && v < W - 1) { v += 1; changed = true; }
                else if (c1 < -sthr && v > 0) { v -= 1; changed = true; }
                if (!changed) break;
            }
            y = (float)u + c0;
            x = (float)v + c1;
            mass = m;
            valid = (mass > minmass) && (mass != 0.f);
        }
        rec[REC_MASS * cap + slot0 + i] = valid ? mass : 0.f;
        rec[REC_Y * cap + slot0 + i] = y;
        rec[REC_X * cap + slot0 + i] = x;
    }
}

// Refinement with disks of radius 1 to 15 (max_iterations >= 1).  The
// candidates of RT_TILES tiles are dealt out over the four waves of a
// workgroup, lane = candidate, so that a wave's issue slots serve the few
// candidates of several tiles; a disk row is loaded four pixels at a time (a
// load costs the address units one line per lane).  Bound by the latency of
// the disk rows: 24 frames of 1024^2 at diameter 21 (2.5 candidates a tile,
// 317 taps) in 75 us, against 177 us inside detect on the tile staged again
// and 452 us with a serial loop over scalar loads.
typedef float f4v_a4 __attribute__((ext_vector_type(4), aligned(4)));

template <int RI>
__device__ __forceinline__ void disk_sums(const GLOBAL float* c, int W, float& s0, float& s1,
                                          float& ms) {
    s0 = s1 = ms = 0.f;
#pragma unroll
    for (int di = -RI; di <= RI; ++di) {
        int hw = 0;
        while ((hw + 1) * (hw + 1) + di * di <= RI * RI) ++hw;   // a constant once unrolled
        const GLOBAL float* row = c + (ptrdiff_t)di * W;
        float d[2 * RI + 1];
        // whole chunks from the left, the last one ending at the disk's edge
        const int n = 2 * hw + 1;
        if (n < 4) {
#pragma unroll
            for (int k = 0; k < n; ++k) d[k] = row[k - hw];
        } else {
#pragma unroll
            for (int k = 0; k < n; k += 4) {
                const int at = k + 4 <= n ? k : n - 4;
                const f4v_a4 q = *(const GLOBAL f4v_a4*)(row + at - hw);
                d[at] = q.x;
                d[at + 1] = q.y;
                d[at + 2] = q.z;
                d[at + 3] = q.w;
            }
        }
#pragma unroll
        for (int k = 0; k < n; ++k) {
            // a zero coefficient leaves its sum unchanged (see walk_tile)
            if (di != 0) s0 = __builtin_fmaf(d[k], (float)di, s0);
            if (k != hw) s1 = __builtin_fmaf(d[k], (float)(k - hw), s1);
            ms = ms + d[k];
        }
    }
}

template <int RI>
__global__ __launch_bounds__(256) void k_walk(Batch b, const Geom* __restrict__ g) {
    __shared__ RefTile s_t[RT_TILES];
    __shared__ uint32_t s_total;
    const uint32_t item0 = blockIdx.x * RT_TILES;
    const int nt = (int)min<uint32_t>(RT_TILES, b.tiles - item0);
    const int tid = threadIdx.x;
    load_ref_tiles(b, item0, nt, tid, s_t, s_total);
    __syncthreads();
    const uint32_t total = s_total;
    const int band = g->band;
    const uint32_t maxit = g->max_iterations;
    const float minmass = g->minmass;
    const int has_pct = g->has_pct;
    const float sthr = 0.6f;
    const uint64_t cap = b.slot_cap;
    // candidate gi goes to wave gi % 4
    for (uint32_t gi = (uint32_t)(tid >> 6) + 4u * (uint32_t)(tid & 63); gi < total; gi += 256) {
        int j = 0;
#pragma unroll
        for (int q = 1; q < RT_TILES; ++q)
            if (q < nt && s_t[q].pref <= gi) j = q;
        const RefTile& rt = s_t[j];
        const size_t slot = (size_t)(item0 + (uint32_t)j) * TILE_PX + (gi - rt.pref);
        const int H = rt.H, W = rt.W;
        const GLOBAL float* P = (const GLOBAL float*)rt.P;
        const uint32_t l = b.slots[slot];
        int u = rt.y0 + (int)(l / TILE_W), v = rt.x0 + (int)(l % TILE_W);
        float y = 0.f, x = 0.f, m = 0.f;
        if (!has_pct || (double)P[(size_t)u * W + v] > b.thr[rt.f]) {
            float c0 = 0.f, c1 = 0.f;
            for (uint32_t it = 0; it < maxit; ++it) {
                if (u - band < 0 || u + band >= H || v - band < 0 || v + band >= W) {
                    m = 0.f; c0 = 0.f; c1 = 0.f;
                } else {
                    float s0, s1;
                    disk_sums<RI>(P + (size_t)u * W + v, W, s0, s1, m);
                    c0 = s0 / m;
                    c1 = s1 / m;
                }
                bool changed = false;
                if (c0 > sthr && u < H - 1) { u += 1; changed = true; }
                else if (c0 < -sthr && u > 0) { u -= 1; changed = true; }
                if (c1 > sthr && v < W - 1) { v += 1; changed = true; }
                else if (c1 < -sthr && v > 0) { v -= 1; changed = true; }
                if (!changed) break;
            }
            y = (float)u + c0;
            x = (float)v + c1;
            m = (m > minmass) && (m != 0.f) ? m : 0.f;
        }
        b.rec[REC_MASS * cap + slot] = m;
        b.rec[REC_Y * cap + slot] = y;
        b.rec[REC_X * cap + slot] = x;
    }
}

hipError_t launch_refine(const Batch& b, const Geom& g, const Geom* d_geom, hipStream_t s) {
    if (g.walk_in_detect) return hipSuccess;  // done by detect
    const dim3 grid((b.tiles + RT_TILES - 1) / RT_TILES), block(256);
    if (g.max_iterations >= 1) {
#define GT_WALK(RI) \
    case RI: hipLaunchKernelGGL(k_walk<RI>, grid, block, 0, s, b, d_geom); return hipGetLastError();
        switch (g.rint) {
            GT_WALK(1) GT_WALK(2) GT_WALK(3) GT_WALK(4) GT_WALK(5) GT_WALK(6) GT_WALK(7) GT_WALK(8)
            GT_WALK(9) GT_WALK(10) GT_WALK(11) GT_WALK(12) GT_WALK(13) GT_WALK(14) GT_WALK(15)
            default: break;
        }
#undef GT_WALK
    }
    hipLaunchKernelGGL(k_refine, grid, block, 0, s, b, d_geom);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// K4 dedup: one wave per block of 2x2 tiles (the block's tiles share one
// chain of dependent loads and one staged neighbourhood), or per tile where a
// batch has few (dblock_side).  The valid records
// (mass != 0) of the tiles that can hold a neighbour, and that lie within
// `separation` of the bounding box of the block's own valid positions, are
// staged in LDS as 16-byte entries.  Each lane then tests its own candidate
// against every staged record (execute_gpu.rs:258-284: drop when a record
// strictly within `separation` has a larger mass, or an equal mass and a
// lower raster index).  Neighbourhoods larger than the staging area are
// staged and tested in rounds.  Outputs stay per tile: keep flags, kept
// count and kept rows per pixel row.
// ---------------------------------------------------------------------------
constexpr int DD_CAP = 256;   // staged records per wave and round
constexpr int DD_CELLS_1D = 16;
constexpr int DD_CELLS = DD_CELLS_1D * DD_CELLS_1D;   // cells of a staged neighbourhood

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6)))
void k_dedup(Batch b, const Geom* __restrict__ g) {
    // staged records, one 16-byte entry each: mass, y, x, raster index (bits)
    __shared__ float4 s_rec[4][DD_CAP];
    __shared__ uint32_t s_kr[4][4][TILE_H];   // kept rows per block tile and pixel row
    // staged records are ordered by square cells (row-major, at most 16 x
    // 16): s_perm lists them cell by cell, cell c starting at s_cell[wave][c]
    // (s_cell[wave][DD_CELLS] = staged count)
    __shared__ uint16_t s_cell[4][DD_CELLS + 1];
    __shared__ uint32_t s_ccur[4][DD_CELLS / 2];   // 16-bit counts, then fill cursors
    __shared__ uint8_t s_perm[4][DD_CAP];
    static_assert(DD_CAP <= 256, "record numbers are bytes");
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t item = blockIdx.x * 4 + wave;
    if (item >= b.dblocks) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) s_kr[wave][q][lane] = 0;
    const uint64_t cap = b.slot_cap;
    const GLOBAL float* rmass = (const GLOBAL float*)(b.rec + REC_MASS * cap);
    const GLOBAL float* ry = (const GLOBAL float*)(b.rec + REC_Y * cap);
    const GLOBAL float* rx = (const GLOBAL float*)(b.rec + REC_X * cap);
    const GLOBAL uint16_t* slots = (const GLOBAL uint16_t*)b.slots;
    const float rad = g->sep;
    const float r2 = rad * rad;
    const int rty = g->dedup_rty, rtx = g->dedup_rtx;

    const uint32_t top = b.dblock_tile[item];   // the block's top-left tile
    const uint32_t f = b.tile_frame[top];
    const Frame fr = b.frames[f];
    const uint32_t local = top - fr.tile_base;
    const int W = (int)fr.W;
    const int tx = (int)(local % fr.tx), ty = (int)(local / fr.tx);
    const int last = (int)b.dblock_side - 1;   // the block's last tile row and column
    const bool hx = last && tx + 1 < (int)fr.tx, hy = last && ty + 1 < (int)fr.ty;
    // tile q = 2 dy + dx of the block (absent ones hold no candidate)
    const bool has[4] = {true, hx, hy, hx && hy};
    uint32_t tq[4], cq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        tq[q] = top + (uint32_t)((q >> 1) * (int)fr.tx + (q & 1));
        cq[q] = has[q] ? b.tile_count[tq[q]] : 0u;
    }
    const uint32_t e1 = cq[0], e2 = e1 + cq[1], e3 = e2 + cq[2], own_n = e3 + cq[3];
    // own record j of the block: its tile q and slot
    auto own_q = [&](uint32_t j) { return j < e1 ? 0 : (j < e2 ? 1 : (j < e3 ? 2 : 3)); };
    auto own_slot = [&](uint32_t j, int q) {
        const uint32_t first = q == 0 ? 0u : (q == 1 ? e1 : (q == 2 ? e2 : e3));
        return (size_t)tq[q] * TILE_PX + (j - first);
    };
    // when the walk ran in detect, every candidate walked and the percentile
    // test on its start value (refine's `P > thr`) is applied here
    const bool use_thr = g->walk_in_detect && g->has_pct;
    const double thr = use_thr ? b.thr[f] : 0.0;
    const GLOBAL float* rcen = (const GLOBAL float*)(b.rec + REC_CENTER * cap);
    // a record's start value (percentile test), loaded beside its other
    // fields so that a record costs one round trip to memory
    auto cen_of = [&](size_t s) { return use_thr ? rcen[s] : 0.f; };
    auto ok = [&](float mass, float cen) {
        return (mass != 0.f) & (!use_thr | ((double)cen > thr));
    };
    const int y_lo = max(0, ty - rty), y_hi = min((int)fr.ty - 1, ty + last + rty);
    const int x_lo = max(0, tx - rtx), x_hi = min((int)fr.tx - 1, tx + last + rtx);
    const int nxr = x_hi - x_lo + 1;
    const int ntl = (y_hi - y_lo + 1) * nxr;

    // bounding box of the block's own valid positions (a NaN, which a mass
    // beyond binary32 gives, widens none: such a record is near no other, and
    // an axis that has only those keeps an empty box, which takes no record)
    bool some = false;
    float bymin = INFINITY, bymax = -INFINITY, bxmin = INFINITY, bxmax = -INFINITY;
    for (uint32_t j = lane; j < own_n; j += 64) {
        const size_t sl = own_slot(j, own_q(j));
        const float m0 = rmass[sl], c0 = cen_of(sl), y = ry[sl], x = rx[sl];
        if (ok(m0, c0)) {
            some = true;
            bymin = fminf(bymin, y); bymax = fmaxf(bymax, y);
            bxmin = fminf(bxmin, x); bxmax = fmaxf(bxmax, x);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        bymin = fminf(bymin, __shfl_xor(bymin, o, 64));
        bymax = fmaxf(bymax, __shfl_xor(bymax, o, 64));
        bxmin = fminf(bxmin, __shfl_xor(bxmin, o, 64));
        bxmax = fmaxf(bxmax, __shfl_xor(bxmax, o, 64));
    }
    // rows (low half) and candidates of the frame; nothing waits for the add
    auto count = [&](uint32_t kept_n) {
        if (lane == 0)
            atomicAdd((unsigned long long*)&b.counts[(size_t)f * b.count_stride],
                      (unsigned long long)kept_n | ((unsigned long long)own_n << 32));
    };
    if (!__ballot(some)) {  // no valid own record
        count(0);
        for (uint32_t j = lane; j < own_n; j += 64) b.keep[own_slot(j, own_q(j))] = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!has[q]) continue;
            if (lane == 0) b.tile_keep[tq[q]] = 0;
            b.rowk[(size_t)tq[q] * TILE_H + lane] = 0;
        }
        return;
    }
    // wave-uniform from here on: keep them in scalar registers
    auto uni = [](float v) {
        return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
    };
    const float margin = rad + 1.0f;
    bymin = uni(bymin - margin); bymax = uni(bymax + margin);
    bxmin = uni(bxmin - margin); bxmax = uni(bxmax + margin);
    // cells at least rad + 1 wide: a record strictly within `separation` of
    // a position lies in that position's cell or one of its eight neighbours
    // (cell coordinates are monotone; their rounding is far below one cell)
    const float ch = fmaxf(rad + 1.0f, fmaxf(bymax - bymin, bxmax - bxmin) * (1.0f / 15.0f));
    const float cinv = uni(1.0f / ch);
    const int ncy = max(1, min(DD_CELLS_1D, (int)((bymax - bymin) * cinv) + 1));
    const int ncx = max(1, min(DD_CELLS_1D, (int)((bxmax - bxmin) * cinv) + 1));
    auto cell_y = [&](float yy) { return min(ncy - 1, max(0, (int)((yy - bymin) * cinv))); };
    auto cell_x = [&](float xx) { return min(ncx - 1, max(0, (int)((xx - bxmin) * cinv))); };

    // The neighbourhood is staged in rounds of at most DD_CAP records: the
    // neighbour tiles are taken 64 at a time (lane q holds tile q's count),
    // their records enumerated 64 at a time (the loads of a round are
    // independent) and filtered by the bounding box; when the next 64 could
    // overflow the staging area, the own candidates are tested against what
    // is staged and staging resumes.  When the whole neighbourhood fits in
    // one round it is staged once and serves every batch of own candidates.
    uint32_t S = 0;
    bool resident = false;
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    uint32_t kept[4] = {0, 0, 0, 0};
    for (uint32_t ib = 0; ib < own_n; ib += 64) {
        const uint32_t j = ib + lane;
        const bool own = j < own_n;
        const int q = own ? own_q(j) : 0;
        float m = 0.f, y = 0.f, x = 0.f;
        int32_t idx = -1;
        size_t sl = 0;
        float cen = 0.f;
        if (own) {
            sl = own_slot(j, q);
            m = rmass[sl];
            y = ry[sl];
            x = rx[sl];
            cen = cen_of(sl);
            const uint32_t l = slots[sl];
            idx = ((ty + (q >> 1)) * TILE_H + (int)(l / TILE_W)) * W +
                  ((tx + (q & 1)) * TILE_W + (int)(l % TILE_W));
        }
        const bool valid = own && ok(m, cen);
        bool drop = false;
        // Counting sort of the n staged records by cell into s_perm: count,
        // scan (lane l owns cells 4l .. 4l + 3), then place through per-cell
        // cursors (the cell is recomputed from the staged position, so
        // nothing is held across the passes).
        auto cell_of = [&](uint32_t k) {
            const float4 rr = s_rec[wave][k];
            return cell_y(rr.y) * ncx + cell_x(rr.z);
        };
        // Counts and cursors are 16-bit halves of 32-bit words (at most
        // DD_CAP records).
        auto cell_add = [&](int c) {
            const uint32_t sh = 16u * (uint32_t)(c & 1);
            return (atomicAdd(&s_ccur[wave][c >> 1], 1u << sh) >> sh) & 0xffffu;
        };
        auto cell_sort = [&](uint32_t n) {
            constexpr int PC = DD_CELLS / 64;   // cells per lane in the scan
            static_assert(PC % 2 == 0, "a lane's cells fill whole words");
#pragma unroll
            for (int i = 0; i < PC / 2; ++i) s_ccur[wave][(PC / 2) * lane + i] = 0;
            wave_sync();
            for (uint32_t k = lane; k < n; k += 64) cell_add(cell_of(k));
            wave_sync();
            uint32_t c[PC], tot = 0;
#pragma unroll
            for (int i = 0; i < PC / 2; ++i) {
                const uint32_t w2 = s_ccur[wave][(PC / 2) * lane + i];
                c[2 * i] = w2 & 0xffffu;
                c[2 * i + 1] = w2 >> 16;
                tot += c[2 * i] + c[2 * i + 1];
            }
            uint32_t run = wave_incl_scan(tot, lane) - tot;
#pragma unroll
            for (int i = 0; i < PC / 2; ++i) {
                const uint32_t r0 = run, r1 = run + c[2 * i];
                s_cell[wave][PC * lane + 2 * i] = (uint16_t)r0;
                s_cell[wave][PC * lane + 2 * i + 1] = (uint16_t)r1;
                s_ccur[wave][(PC / 2) * lane + i] = r0 | (r1 << 16);
                run = r1 + c[2 * i + 1];
            }
            if (lane == 63) s_cell[wave][DD_CELLS] = (uint16_t)run;
            wave_sync();
            for (uint32_t k = lane; k < n; k += 64) s_perm[wave][cell_add(cell_of(k))] = (uint8_t)k;
            wave_sync();
        };
        // every lane tests its own candidate against the records of its cell
        // and the eight neighbouring cells, one contiguous run of cells per
        // cell row (execute_gpu.rs:258-284).  A lane's own record never
        // drops it (equal mass, equal raster index), and distinct candidates
        // have distinct raster indices, so no self test is needed.
        auto test_cells = [&]() {
            if (!valid) return;
            const int cy0 = cell_y(y), cx0 = cell_x(x);
            const int cxa = max(cx0 - 1, 0), cxb = min(cx0 + 1, ncx - 1);
            for (int cy = max(cy0 - 1, 0); cy <= min(cy0 + 1, ncy - 1); ++cy) {
                const uint32_t lo = s_cell[wave][cy * ncx + cxa];
                const uint32_t hi = s_cell[wave][cy * ncx + cxb + 1];
                for (uint32_t k = lo; k < hi; ++k) {
                    const float4 rr = s_rec[wave][s_perm[wave][k]];
                    const float dy = rr.y - y, dx = rr.z - x;
                    float d = dy * dy;
                    d = d + dx * dx;
                    const int32_t nidx = __float_as_int(rr.w);
                    drop |= d < r2 && (m < rr.x || (m == rr.x && idx > nidx));
                }
            }
        };
        if (__ballot(valid)) {  // wave-uniform
            if (resident) {
                test_cells();
            } else {
                bool single = true;   // one round held the whole neighbourhood
                for (int g0 = 0; g0 < ntl; g0 += 64) {
                    const int ng = min(64, ntl - g0);
                    uint32_t myc = 0, myit = 0;
                    if (lane < ng) {
                        const int qq = g0 + lane;
                        const int ny = y_lo + qq / nxr, nx = x_lo + qq % nxr;
                        myit = fr.tile_base + (uint32_t)(ny * (int)fr.tx + nx);
                        myc = b.tile_count[myit];
                    }
                    const uint32_t inc = wave_incl_scan(myc, lane);
                    const uint32_t exq = inc - myc;
                    const uint32_t T = __shfl(inc, 63, 64);
                    uint32_t jb = 0;
                    do {
                        S = 0;
                        for (; jb < T; jb += 64) {
                            const uint32_t jj = jb + lane;
                            // tile of record jj: the last qq whose first record is <= jj
                            int qt = 0;
                            for (int qq = 1; qq < ng; ++qq)  // wave-uniform: scalar read of lane qq
                                if ((uint32_t)__builtin_amdgcn_readlane((int)exq, qq) <= jj) qt = qq;
                            const uint32_t it2 = __shfl(myit, qt, 64);
                            const uint32_t i2 = jj - __shfl(exq, qt, 64);
                            const size_t s2 = (size_t)it2 * TILE_PX + i2;
                            bool take = false;
                            float nm = 0.f, yy = 0.f, xx = 0.f, cn = 0.f;
                            uint32_t l2 = 0;
                            if (jj < T) {   // every field of the record in one round trip
                                nm = rmass[s2];
                                yy = ry[s2];
                                xx = rx[s2];
                                cn = cen_of(s2);
                                l2 = slots[s2];
                                take = ok(nm, cn) & (yy >= bymin) & (yy <= bymax) & (xx >= bxmin) &
                                       (xx <= bxmax);
                            }
                            const uint64_t tm = __ballot(take);
                            const uint32_t nt = (uint32_t)__popcll(tm);
                            if (S + nt > (uint32_t)DD_CAP) break;   // test, then resume at jb
                            if (take) {
                                const uint32_t r = S + (uint32_t)__popcll(tm & lanemask_lt(lane));
                                const int qg = g0 + qt;
                                const int ny = y_lo + qg / nxr, nx = x_lo + qg % nxr;
                                const int32_t ri = (ny * TILE_H + (int)(l2 / TILE_W)) * W +
                                                   (nx * TILE_W + (int)(l2 % TILE_W));
                                s_rec[wave][r] = make_float4(nm, yy, xx, __int_as_float(ri));
                            }
                            S += nt;
                        }
                        wave_sync();
                        cell_sort(S);
                        test_cells();
                        if (jb < T || g0 + 64 < ntl) single = false;
                        wave_sync();   // every lane's reads done before the next round's writes
                    } while (jb < T);
                }
                resident = single;
            }
        }
        const bool keep = valid && !drop;
        if (own) b.keep[sl] = keep ? 1 : 0;
        if (keep) {
            const int row = idx / W - (ty + (q >> 1)) * TILE_H;
            atomicAdd(&s_kr[wave][q][row], 1u);
        }
#pragma unroll
        for (int qq = 0; qq < 4; ++qq) kept[qq] += (uint32_t)__popcll(__ballot(keep && q == qq));
    }
    count(kept[0] + kept[1] + kept[2] + kept[3]);
    // kept rows of each tile in pixel rows <= r (the emit order is raster)
    wave_sync();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (!has[q]) continue;
        if (lane == 0) b.tile_keep[tq[q]] = kept[q];
        b.rowk[(size_t)tq[q] * TILE_H + lane] = wave_incl_scan(s_kr[wave][q][lane], lane);
    }
}

hipError_t launch_dedup(const Batch& b, const Geom& g, const Geom* d_geom, hipStream_t s) {
    (void)g;
    hipLaunchKernelGGL(k_dedup, dim3((b.dblocks + 3) / 4), dim3(256), 0, s, b, d_geom);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// scan: row offsets.  One launch of (frame, four tile rows); every wave adds
// up what precedes its own tile row, so nothing waits for another workgroup.
//
// Raster order within a frame (get_work scans masses in raster order,
// execute_gpu.rs:108-195): a kept row at pixel row r of tile t in tile row tr
// comes after every kept row of the earlier tile rows, of tiles left of t in
// pixel rows <= r and of tiles right of t in pixel rows < r; the rows of tile
// t itself are in raster order already.  With K[t][r] = kept rows of tile t
// in pixel rows <= r (from dedup):
//   rowoff[t][r] = base(tr) + sum_{t' < t} K[t'][r] + sum_{t' > t} K[t'][r - 1].
// One wave per tile row, lane = pixel row.  Tile rows of up to 48 tiles
// (frames up to 2304 columns) load every K once, in one round, and take
// K[t][r - 1] from the lane below; wider ones load in chunks of 32 tiles.
//
// The first workgroup of a frame also writes the frame's rows (counted by
// dedup) and their base (the rows of the batches before, `carry_in`, and of the
// frames before), that of the last frame the running totals (`carry_out`).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_scan(Batch b) {
    constexpr int CH = 32;
    constexpr int C1 = 48;
    __shared__ uint64_t s_rows[4], s_cands[4];
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.y == 0) {
        const bool last = f + 1 == b.nframes;
        uint64_t rows = 0, cands = 0;
        for (uint32_t i = threadIdx.x; i < f + (last ? 1u : 0u); i += 256) {
            const uint64_t n = b.counts[(size_t)i * b.count_stride];
            rows += i < f ? n & 0xffffffffu : 0u;
            cands += n >> 32;
        }
        for (int d = 32; d > 0; d >>= 1) {
            rows += __shfl_xor(rows, d, 64);
            cands += __shfl_xor(cands, d, 64);
        }
        if (lane == 0) { s_rows[wave] = rows; s_cands[wave] = cands; }
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint64_t base = b.carry_in[0] + s_rows[0] + s_rows[1] + s_rows[2] + s_rows[3];
            const uint32_t own = (uint32_t)b.counts[(size_t)f * b.count_stride];
            b.frame_row_base[f] = base;
            b.frame_rows[f] = own;
            if (last) {
                b.carry_out[0] = base + own;
                b.carry_out[1] = b.carry_in[1] + s_cands[0] + s_cands[1] + s_cands[2] + s_cands[3];
            }
        }
    }
    const uint32_t tr = blockIdx.y * 4 + (uint32_t)wave;
    if (tr >= fr.ty) return;
    const uint32_t t0 = fr.tile_base + tr * fr.tx;
    uint32_t base = 0;   // kept rows of the tile rows above
    for (uint32_t i = (uint32_t)lane; i < tr * fr.tx; i += 64) base += b.tile_keep[fr.tile_base + i];
    base = wave_sum_u(base);
    const uint32_t* K = b.rowk + (size_t)t0 * TILE_H + lane;
    if (fr.tx <= C1) {  // wave-uniform
        uint32_t kle[C1], klt[C1];
#pragma unroll
        for (int j = 0; j < C1; ++j) kle[j] = (uint32_t)j < fr.tx ? K[(size_t)j * TILE_H] : 0u;
        uint32_t total = 0;
#pragma unroll
        for (int j = 0; j < C1; ++j) {
            const uint32_t up = __shfl_up(kle[j], 1, 64);
            klt[j] = lane > 0 ? up : 0u;
            total += klt[j];
        }
        uint32_t pre = 0, cum = 0;
#pragma unroll
        for (int j = 0; j < C1; ++j) {
            if ((uint32_t)j < fr.tx) {
                cum += klt[j];
                b.rowoff[(size_t)(t0 + j) * TILE_H + lane] = base + pre + (total - cum);
                pre += kle[j];
            }
        }
        return;
    }
    uint32_t total_lt = 0;
    for (uint32_t q0 = 0; q0 < fr.tx; q0 += CH) {
        uint32_t v[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j)
            v[j] = (q0 + j < fr.tx && lane > 0) ? K[(size_t)(q0 + j) * TILE_H - 1] : 0u;
#pragma unroll
        for (int j = 0; j < CH; ++j) total_lt += v[j];
    }
    uint32_t pre_le = 0, cum_lt = 0;
    for (uint32_t q0 = 0; q0 < fr.tx; q0 += CH) {
        uint32_t kle[CH], klt[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const bool in = q0 + j < fr.tx;
            kle[j] = in ? K[(size_t)(q0 + j) * TILE_H] : 0u;
            klt[j] = (in && lane > 0) ? K[(size_t)(q0 + j) * TILE_H - 1] : 0u;
        }
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            if (q0 + j < fr.tx) {
                cum_lt += klt[j];
                b.rowoff[(size_t)(t0 + q0 + j) * TILE_H + lane] = base + pre_le + (total_lt - cum_lt);
                pre_le += kle[j];
            }
        }
    }
}

hipError_t launch_scan(const Batch& b, uint32_t max_ty, hipStream_t s) {
    hipLaunchKernelGGL(k_scan, dim3(b.nframes, (max_ty + 3) / 4), dim3(256), 0, s, b);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// K5 emit: rows [frame, mass, y, x, ...] in frame order, raster order of the
// candidate pixel within a frame (row positions from k_scan).  The columns
// after x (characterisation, raw signal) are left for k_char and k_raw.
// ---------------------------------------------------------------------------
// EMIT_TPW tiles per wave, EMIT_LPT lanes each: a tile holds about a dozen
// candidates, and a wave's time is mostly its chain of dependent loads, so
// fewer, fuller waves finish sooner.
constexpr int EMIT_TPW = 4;
constexpr int EMIT_LPT = 64 / EMIT_TPW;
__global__ __launch_bounds__(256) void k_emit(Batch b, const Geom* __restrict__ g) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int part = lane / EMIT_LPT, hl = lane % EMIT_LPT;
    const uint64_t hmask = (~0ull >> (64 - EMIT_LPT)) << (part * EMIT_LPT);
    const uint32_t item = (blockIdx.x * 4 + wave) * EMIT_TPW + part;
    if (__ballot(item < b.tiles) == 0) return;  // wave-uniform
    const bool tile_in = item < b.tiles;
    const uint32_t it = tile_in ? item : 0u;   // loads stay in bounds
    const uint32_t f = b.tile_frame[it];
    const Frame fr = b.frames[f];
    const uint32_t local = it - fr.tile_base;
    const int W = (int)fr.W;
    const int tx = (int)(local % fr.tx), ty = (int)(local / fr.tx);
    const uint32_t cnt = tile_in ? b.tile_count[it] : 0u;
    const size_t slot0 = (size_t)it * TILE_PX;
    const uint64_t cap = b.slot_cap;
    const int nc = g->ncols;
    const uint64_t fbase = b.frame_row_base[f];
    uint32_t before = 0;  // kept rows of this tile before the chunk
    for (uint32_t ib = 0; ib < cnt; ib += EMIT_LPT) {
        const uint32_t i = ib + (uint32_t)hl;
        // the keep flag, the slot and the position record of every candidate
        // of the chunk are loaded together (all in bounds for i < cnt); only
        // the row offset waits for the slot
        const bool in = i < cnt;
        const size_t s = slot0 + (in ? i : 0u);
        const bool kf = b.keep[s];
        const uint32_t l = b.slots[s];
        const float rm = b.rec[REC_MASS * cap + s];
        const float ryv = b.rec[REC_Y * cap + s];
        const float rxv = b.rec[REC_X * cap + s];
        const bool k = in && kf;
        const uint64_t msk = __ballot(k) & hmask;
        if (k) {
            const uint64_t r = fbase + b.rowoff[(size_t)it * TILE_H + l / TILE_W] + before +
                               (uint64_t)__popcll(msk & lanemask_lt(lane));
            if (r < b.rows_cap) {
                float* o = b.rows + r * (uint64_t)nc;
                o[0] = (float)fr.frame_index;
                o[1] = rm;
                o[2] = ryv;
                o[3] = rxv;
                b.rows_cand[r] = (int64_t)(ty * TILE_H + (int)(l / TILE_W)) * W +
                                 (tx * TILE_W + (int)(l % TILE_W));
            }
        }
        before += (uint32_t)__popcll(msk);
    }
}

hipError_t launch_emit(const Batch& b, const Geom& g, const Geom* d_geom, hipStream_t s) {
    (void)g;
    hipLaunchKernelGGL(k_emit, dim3((b.tiles + 4 * EMIT_TPW - 1) / (4 * EMIT_TPW)), dim3(256), 0, s,
                       b, d_geom);
    return hipGetLastError();
}

}  // namespace gt
