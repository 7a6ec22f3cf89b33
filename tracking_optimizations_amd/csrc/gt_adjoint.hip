// gt_adjoint.hip -- gfx950 adjoint of the locate path (refine + bandpass).
//
// For every output row the particle's forward state is recomputed from the
// batch's bandpass output P with the forward's own arithmetic: the walk from
// the row's candidate pixel gives the last evaluated disk (u_e, v_e), its
// mass m and offsets c = s / m.  With the walk decisions held fixed,
//   y = u_final + c0,  x = v_final + c1,  mass = m,
// so on the disk pixels q
//   dy/dP[q] = (i_q - c0) / m,  dx/dP[q] = (j_q - c1) / m,  dmass/dP[q] = 1,
// zero where the bandpass clamp is active (P[q] == 0).  The bandpass
//   P[q] = max(0, G[q] / gn^2 - B[q] / k^2)
// is linear in the input where P > 0: G is the separable Gaussian with taps
// outside the frame skipped (weight w_i w_j at offset (j, i)), B the boxcar
// over the (2R+1)^2 window with one mirror reflection (a pixel reached twice
// by reflection counts twice).  The Jacobian of (y, x, mass) with respect to
// the input pixels is therefore the disk adjoint pulled back through the
// transposed filters; its support is the S x S patch, S = 2 (rint + R) + 1,
// centred on (u_e, v_e).  The Poisson localisation error of each output is
//   sigma^2 = sum_r J[r]^2 * lambda[r],  lambda[r] = max(I[r], 0).
//
// The vector-Jacobian product used by the Python autograd wrapper adds the
// patches of a frame's rows in row order, one wave per tile of the frame, so
// the gradient is deterministic.
#include <algorithm>
#include <type_traits>

#include "gt_device.h"

#pragma clang fp contract(off)

namespace gt {

namespace {

__device__ __forceinline__ float in_px(const void* in, int type, size_t i) {
    if (type == IN_U16) return (float)((const uint16_t*)in)[i];
    if (type == IN_U8) return (float)((const uint8_t*)in)[i];
    return ((const float*)in)[i];
}

// Boxcar multiplicity: how many offsets d in [-R, R] map input row (or
// column) q + d onto r under the single mirror reflection -i-1 / 2n-i-1.
__device__ __forceinline__ float box_count(int q, int r, int R, int n) {
    float c = 0.f;
    if (abs(r - q) <= R) c += 1.f;           // direct
    if (abs(-r - 1 - q) <= R) c += 1.f;      // reflected at the low edge
    if (abs(2 * n - r - 1 - q) <= R) c += 1.f;  // reflected at the high edge
    return c;
}

constexpr int ADJ_TAPS = 1024;  // disk taps ((2 rint + 1)^2 <= 1024: rint <= 15)

__global__ __launch_bounds__(64) void k_adjoint(Batch b, const Geom* __restrict__ g, AdjOut ao,
                                               uint32_t frame_pos0) {
    __shared__ float s_a[3][ADJ_TAPS];
    __shared__ int16_t s_ti[ADJ_TAPS], s_tj[ADJ_TAPS];
    __shared__ float s_w[33];
    const int lane = threadIdx.x;
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const int H = (int)fr.H, W = (int)fr.W;
    const float* __restrict__ P = fr.P;
    const int band = g->band, rint = g->rint, R = g->R;
    const uint32_t maxit = g->max_iterations;
    const float gn2 = g->gn * g->gn, kk = g->kk;
    const int S = 2 * (rint + R) + 1;
    const uint64_t base = b.frame_row_base[f];
    const uint32_t nrows = b.frame_rows[f];
    const float sthr = 0.6f;

    if (lane < 2 * R + 1) s_w[lane] = g->w[lane];
    // disk tap offsets in the shader's order
    int ntap = 0;
    for (int i = -rint; i <= rint; ++i)
        for (int j = -rint; j <= rint; ++j) {
            if (i * i + j * j > rint * rint) continue;
            if (ntap % 64 == lane) { s_ti[ntap] = (int16_t)i; s_tj[ntap] = (int16_t)j; }
            ++ntap;
        }
    __syncthreads();

    for (uint32_t rl = blockIdx.y; rl < nrows; rl += gridDim.y) {
        const uint64_t row = base + rl;
        if (row >= b.rows_cap) break;
        const int64_t pix = b.rows_cand[row];
        const int u0 = (int)(pix / W), v0 = (int)(pix % W);
        // forward walk, identical arithmetic to the refine stage
        int u = u0, v = v0, ue = u0, ve = v0;
        float m = 0.f, c0 = 0.f, c1 = 0.f;
        for (uint32_t it = 0; it < maxit; ++it) {
            ue = u;
            ve = v;
            if (u - band < 0 || u + band >= H || v - band < 0 || v + band >= W) {
                m = 0.f; c0 = 0.f; c1 = 0.f;
            } else {
                float s0 = 0.f, s1 = 0.f, ms = 0.f;
                for (int t = 0; t < ntap; ++t) {
                    const int i = s_ti[t], j = s_tj[t];
                    const float d = P[(size_t)(u + i) * W + (v + j)];
                    s0 = __builtin_fmaf(d, (float)i, s0);
                    s1 = __builtin_fmaf(d, (float)j, s1);
                    ms = ms + d;
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
        const int py0 = ue - rint - R, px0 = ve - rint - R;
        if (m == 0.f || ue - band < 0 || ue + band >= H || ve - band < 0 || ve + band >= W) {
            // not an output row of the forward (mass 0): nothing to pull back
            if (lane == 0) {
                for (int o = 0; o < 3; ++o) ao.sigma[row * 3 + o] = 0.f;
                ao.origin[row * 2 + 0] = py0;
                ao.origin[row * 2 + 1] = px0;
                ao.rowpos[row] = (int32_t)(frame_pos0 + f);
            }
            if (ao.jac)
                for (int p = lane; p < 3 * S * S; p += 64) ao.jac[(size_t)row * 3 * S * S + p] = 0.f;
            continue;
        }
        // disk adjoint (zero where the clamp is active)
        __syncthreads();
        const float rm = 1.f / m;
        for (int t = lane; t < ntap; t += 64) {
            const int i = s_ti[t], j = s_tj[t];
            const float on = P[(size_t)(ue + i) * W + (ve + j)] > 0.f ? 1.f : 0.f;
            s_a[0][t] = on * (((float)i - c0) * rm);
            s_a[1][t] = on * (((float)j - c1) * rm);
            s_a[2][t] = on;
        }
        __syncthreads();
        // pull back through the transposed bandpass, one patch pixel per lane
        double var[3] = {0.0, 0.0, 0.0};
        for (int p = lane; p < S * S; p += 64) {
            const int ry = py0 + p / S, rx = px0 + p % S;
            float jo[3] = {0.f, 0.f, 0.f};
            if (ry >= 0 && ry < H && rx >= 0 && rx < W) {
                for (int t = 0; t < ntap; ++t) {
                    const int qy = ue + s_ti[t], qx = ve + s_tj[t];
                    const int dy = ry - qy, dx = rx - qx;
                    const float wg = (abs(dy) <= R && abs(dx) <= R)
                                         ? s_w[dy + R] * s_w[dx + R] / gn2 : 0.f;
                    const float wb = box_count(qy, ry, R, H) * box_count(qx, rx, R, W) / kk;
                    const float kq = wg - wb;
#pragma unroll
                    for (int o = 0; o < 3; ++o) jo[o] = __builtin_fmaf(s_a[o][t], kq, jo[o]);
                }
                const double lam = (double)fmaxf(in_px(fr.in, b.in_type, (size_t)ry * W + rx), 0.f);
#pragma unroll
                for (int o = 0; o < 3; ++o) var[o] += (double)jo[o] * (double)jo[o] * lam;
            }
            if (ao.jac) {
#pragma unroll
                for (int o = 0; o < 3; ++o)
                    ao.jac[((size_t)row * 3 + o) * (size_t)(S * S) + p] = jo[o];
            }
        }
#pragma unroll
        for (int o = 0; o < 3; ++o)
            for (int s = 32; s > 0; s >>= 1) var[o] += __shfl_xor(var[o], s, 64);
        if (lane == 0) {
            // output order: y, x, mass
            ao.sigma[row * 3 + 0] = (float)sqrt(var[0]);
            ao.sigma[row * 3 + 1] = (float)sqrt(var[1]);
            ao.sigma[row * 3 + 2] = (float)sqrt(var[2]);
            ao.origin[row * 2 + 0] = py0;
            ao.origin[row * 2 + 1] = px0;
            ao.rowpos[row] = (int32_t)(frame_pos0 + f);
        }
    }
}

// The same adjoint with the filters applied separably.  One wave per row:
//  * the walk is replayed with the forward's own arithmetic (taps summed in
//    the shader's order by every lane), the disk's D x D box of P staged in
//    LDS by all lanes first (D = 2 rint + 1);
//  * the disk adjoint A_o (o = y, x, mass) lives on that box (0 off the
//    disk and where the clamp is active);
//  * the Gaussian part of the pullback, sum_q A(q) w[ry - qy] w[rx - qx] /
//    gn^2, is a column pass T[i][c] = sum_j w[c - j] A[i][j] then a row pass
//    sum_i w[r - i] T[i][c]; the boxcar part the same with the mirror
//    multiplicities box_count (a table per patch row and column).
// Sums are reassociated against the per-pair form of k_adjoint (results
// agree to binary32 rounding).  Dynamic LDS, sized from the geometry.
__global__ __launch_bounds__(64) void k_adjoint_sep(Batch b, const Geom* __restrict__ g,
                                                   AdjOut ao, uint32_t frame_pos0) {
    extern __shared__ float sh[];
    const int lane = threadIdx.x;
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const int H = (int)fr.H, W = (int)fr.W;
    const float* __restrict__ P = fr.P;
    const int band = g->band, rint = g->rint, R = g->R;
    const uint32_t maxit = g->max_iterations;
    const float gn2 = g->gn * g->gn, kk = g->kk;
    const int D = 2 * rint + 1, S = 2 * (rint + R) + 1, NW = 2 * R + 1;
    const uint64_t base = b.frame_row_base[f];
    const uint32_t nrows = b.frame_rows[f];
    const float sthr = 0.6f;
    // LDS: box[D*D] A[3][D*D] TG[3][D*S] TB[3][D*S] BX[S*D] BY[S*D] w[NW]
    float* box = sh;
    float* A = box + D * D;
    float* TG = A + 3 * D * D;
    float* TB = TG + 3 * D * S;
    float* BX = TB + 3 * D * S;
    float* BY = BX + S * D;
    float* w = BY + S * D;
    for (int k = lane; k < NW; k += 64) w[k] = g->w[k];
    __syncthreads();

    for (uint32_t rl = blockIdx.y; rl < nrows; rl += gridDim.y) {
        const uint64_t row = base + rl;
        if (row >= b.rows_cap) break;
        const int64_t pix = b.rows_cand[row];
        const int u0 = (int)(pix / W), v0 = (int)(pix % W);
        // forward walk (refine's arithmetic, every lane alike)
        int u = u0, v = v0, ue = u0, ve = v0;
        float m = 0.f, c0 = 0.f, c1 = 0.f;
        bool staged = false;   // box holds P around (ue, ve)
        for (uint32_t it = 0; it < maxit; ++it) {
            ue = u;
            ve = v;
            if (u - band < 0 || u + band >= H || v - band < 0 || v + band >= W) {
                m = 0.f; c0 = 0.f; c1 = 0.f;
                staged = false;
            } else {
                __syncthreads();
                for (int e = lane; e < D * D; e += 64)
                    box[e] = P[(size_t)(u + e / D - rint) * W + (v + e % D - rint)];
                __syncthreads();
                staged = true;
                float s0 = 0.f, s1 = 0.f, ms = 0.f;
                for (int i = -rint; i <= rint; ++i)
                    for (int j = -rint; j <= rint; ++j) {
                        if (i * i + j * j > rint * rint) continue;
                        const float d = box[(i + rint) * D + (j + rint)];
                        s0 = __builtin_fmaf(d, (float)i, s0);
                        s1 = __builtin_fmaf(d, (float)j, s1);
                        ms = ms + d;
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
        const int py0 = ue - rint - R, px0 = ve - rint - R;
        if (m == 0.f || !staged) {
            // not an output row of the forward (mass 0): nothing to pull back
            if (lane == 0) {
                for (int o = 0; o < 3; ++o) ao.sigma[row * 3 + o] = 0.f;
                ao.origin[row * 2 + 0] = py0;
                ao.origin[row * 2 + 1] = px0;
                ao.rowpos[row] = (int32_t)(frame_pos0 + f);
            }
            if (ao.jac)
                for (int p = lane; p < 3 * S * S; p += 64) ao.jac[(size_t)row * 3 * S * S + p] = 0.f;
            continue;
        }
        // disk adjoint on the box; boxcar multiplicity tables
        const float rm = 1.f / m;
        for (int e = lane; e < D * D; e += 64) {
            const int i = e / D - rint, j = e % D - rint;
            float a0 = 0.f, a1 = 0.f, a2 = 0.f;
            if (i * i + j * j <= rint * rint) {
                const float on = box[e] > 0.f ? 1.f : 0.f;
                a0 = on * (((float)i - c0) * rm);
                a1 = on * (((float)j - c1) * rm);
                a2 = on;
            }
            A[e] = a0;
            A[D * D + e] = a1;
            A[2 * D * D + e] = a2;
        }
        for (int e = lane; e < S * D; e += 64) {
            const int c = e / D, j = e % D;
            BX[e] = box_count(ve + j - rint, px0 + c, R, W);
            BY[e] = box_count(ue + j - rint, py0 + c, R, H);
        }
        __syncthreads();
        // column pass: TG_o[i][c] = sum_j w[c - j] A_o[i][j], TB_o with BX
        for (int e = lane; e < D * S; e += 64) {
            const int i = e / S, c = e % S;
            float tg[3] = {0.f, 0.f, 0.f}, tb[3] = {0.f, 0.f, 0.f};
            for (int j = 0; j < D; ++j) {
                const int k = c - j;
                const float wg = (k >= 0 && k < NW) ? w[k] : 0.f;
                const float wb = BX[c * D + j];
#pragma unroll
                for (int o = 0; o < 3; ++o) {
                    const float a = A[o * D * D + i * D + j];
                    tg[o] = __builtin_fmaf(wg, a, tg[o]);
                    tb[o] = __builtin_fmaf(wb, a, tb[o]);
                }
            }
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                TG[o * D * S + e] = tg[o];
                TB[o * D * S + e] = tb[o];
            }
        }
        __syncthreads();
        // row pass and the Poisson variance, one patch pixel per lane
        double var[3] = {0.0, 0.0, 0.0};
        for (int p = lane; p < S * S; p += 64) {
            const int r = p / S, c = p % S;
            const int ry = py0 + r, rx = px0 + c;
            float jo[3] = {0.f, 0.f, 0.f};
            if (ry >= 0 && ry < H && rx >= 0 && rx < W) {
                float sg[3] = {0.f, 0.f, 0.f}, sb[3] = {0.f, 0.f, 0.f};
                for (int i = 0; i < D; ++i) {
                    const int k = r - i;
                    const float wg = (k >= 0 && k < NW) ? w[k] : 0.f;
                    const float wb = BY[r * D + i];
#pragma unroll
                    for (int o = 0; o < 3; ++o) {
                        sg[o] = __builtin_fmaf(wg, TG[o * D * S + i * S + c], sg[o]);
                        sb[o] = __builtin_fmaf(wb, TB[o * D * S + i * S + c], sb[o]);
                    }
                }
#pragma unroll
                for (int o = 0; o < 3; ++o) jo[o] = sg[o] / gn2 - sb[o] / kk;
                const double lam = (double)fmaxf(in_px(fr.in, b.in_type, (size_t)ry * W + rx), 0.f);
#pragma unroll
                for (int o = 0; o < 3; ++o) var[o] += (double)jo[o] * (double)jo[o] * lam;
            }
            if (ao.jac) {
#pragma unroll
                for (int o = 0; o < 3; ++o)
                    ao.jac[((size_t)row * 3 + o) * (size_t)(S * S) + p] = jo[o];
            }
        }
#pragma unroll
        for (int o = 0; o < 3; ++o)
            for (int sft = 32; sft > 0; sft >>= 1) var[o] += __shfl_xor(var[o], sft, 64);
        if (lane == 0) {
            ao.sigma[row * 3 + 0] = (float)sqrt(var[0]);
            ao.sigma[row * 3 + 1] = (float)sqrt(var[1]);
            ao.sigma[row * 3 + 2] = (float)sqrt(var[2]);
            ao.origin[row * 2 + 0] = py0;
            ao.origin[row * 2 + 1] = px0;
            ao.rowpos[row] = (int32_t)(frame_pos0 + f);
        }
        __syncthreads();   // the next row overwrites the tables
    }
}

// The separable adjoint with everything in registers, for the usual filters
// (smoothing size equal to the diameter: R = RINT, or RINT + 1 for even
// ones).  A lane holds one column of a row's S x S patch and G = 64 / S rows
// share a wave, so the inner sums run over registers with constant indices.
//  * A wave takes a run of rows; lane = row replays the walks (the forward's
//    own arithmetic).
//  * The disk adjoint A_o(i, j) = on(i, j) f_o with f_y = (i - c0) / m,
//    f_x = (j - c1) / m, f_mass = 1, so two column passes serve the three
//    outputs: S_i(c) = sum_j w[c - j] on(i, j) and U_i(c) with f_x; y and
//    mass share S_i.  The boxcar's passes are the same with unit weights.
//  * The row pass is Gaussian FMAs over i; the boxcar's window over i is a
//    prefix or a suffix of the D rows (D <= 2R + 1), a running sum from
//    either end.  Patches that leave the frame take the mirror
//    multiplicities (box_count) instead.
// The two norms multiply as reciprocals of two parts, so no output divides.
//
// Bound by issued instructions, about 400 per row at d = 9: 64 frames of
// 512^2 (80 k rows) in 97 us, against 605 us for the form above with its
// tables in LDS (5 LDS reads per 6 FMAs, six divisions per patch pixel).
//
// Waves per SIMD (adj_waves): the most whose registers hold all, or all but
// four.  Four spilled ones cost less than a wave (64 frames of 512^2: RINT 2,
// R 3 58.5 us at four waves, 61.1 at three without spills; RINT 3, R 4 63.9 at
// three, 71.0 at two), 37 and 45 of them more (RINT 4 at three waves: R 4 117
// against 97 us at two, R 5 104 against 83).
constexpr int adj_waves(int rint) { return rint <= 2 ? 4 : rint <= 3 ? 3 : rint <= 5 ? 2 : 1; }

template <int RINT, int R, typename T>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(adj_waves(RINT))))
void k_adjoint_reg(Batch b, const Geom* __restrict__ g, AdjOut ao, uint32_t frame_pos0) {
    constexpr int D = 2 * RINT + 1, NT = 2 * R + 1, S = 2 * (RINT + R) + 1;
    constexpr int G = 64 / S;
    static_assert(S <= 64 && D <= NT, "a patch column per lane; prefix and suffix windows");
    const int lane = threadIdx.x;
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const int H = (int)fr.H, W = (int)fr.W;
    const GLOBAL float* P = (const GLOBAL float*)fr.P;
    const int band = g->band;
    const uint32_t maxit = g->max_iterations;
    const GLOBAL T* I = (const GLOBAL T*)fr.in;
    // 1 / k^2 and 1 / gauss_norm^2 in two parts each (their rounding would be
    // the same error everywhere)
    const double dkk = 1.0 / (double)g->kk, dgn = 1.0 / ((double)g->gn * (double)g->gn);
    const float rkk = (float)dkk, rkk_lo = (float)(dkk - (double)rkk);
    const float rgg = (float)dgn, rgg_lo = (float)(dgn - (double)rgg);
    const float sthr = 0.6f;
    const uint64_t base = b.frame_row_base[f];
    if (base >= b.rows_cap) return;
    const uint32_t nrows = (uint32_t)min((uint64_t)b.frame_rows[f], b.rows_cap - base);
    // rows of one run: whole groups, as few as give every wave of the frame one
    const uint32_t want = (nrows + gridDim.y - 1) / gridDim.y;
    const uint32_t per = min((uint32_t)(64 / G * G), max(1u, (want + G - 1) / G) * G);
    const int grp = min(lane / S, G - 1);
    const bool lane_in = lane < G * S;
    const int c = lane_in ? lane % S : 0;

    float wd[R + 1];   // weights by distance
#pragma unroll
    for (int k = 0; k <= R; ++k) wd[k] = g->w[R + k];
    float wl[D];       // this lane's column weights w[c - j]
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const int k = c - j - R;   // offset of the tap
        wl[j] = abs(k) <= R ? g->w[R + k] : 0.f;
    }

    for (uint32_t q0 = blockIdx.y * per; q0 < nrows; q0 += gridDim.y * per) {
        const int n = (int)min(per, nrows - q0);
        // forward walk (refine's arithmetic), lane = row
        const int64_t pix = b.rows_cand[base + q0 + (uint32_t)min(lane, n - 1)];
        int u = (int)(pix / W), v = (int)(pix % W);
        int ue = u, ve = v, live = 0;   // live: the last disk lay inside the frame
        float m = 0.f, c0 = 0.f, c1 = 0.f;
        if (lane < n) {
            for (uint32_t it = 0; it < maxit; ++it) {
                ue = u;
                ve = v;
                if (u - band < 0 || u + band >= H || v - band < 0 || v + band >= W) {
                    m = 0.f; c0 = 0.f; c1 = 0.f;
                    live = 0;
                } else {
                    const GLOBAL float* p = P + (size_t)u * W + v;
                    float s0 = 0.f, s1 = 0.f, ms = 0.f;
#pragma unroll
                    for (int i = -RINT; i <= RINT; ++i)
#pragma unroll
                        for (int j = -RINT; j <= RINT; ++j) {
                            if (i * i + j * j > RINT * RINT) continue;
                            const float d = p[(ptrdiff_t)i * W + j];
                            s0 = __builtin_fmaf(d, (float)i, s0);
                            s1 = __builtin_fmaf(d, (float)j, s1);
                            ms = ms + d;
                        }
                    m = ms;
                    c0 = s0 / ms;
                    c1 = s1 / ms;
                    live = 1;
                }
                bool changed = false;
                if (c0 > sthr && u < H - 1) { u += 1; changed = true; }
                else if (c0 < -sthr && u > 0) { u -= 1; changed = true; }
                if (c1 > sthr && v < W - 1) { v += 1; changed = true; }
                else if (c1 < -sthr && v > 0) { v -= 1; changed = true; }
                if (!changed) break;
            }
        }
        if (m == 0.f) live = 0;
        if (!live) c0 = c1 = 0.f;

        for (int i0 = 0; i0 < n; i0 += G) {
            const int idx = min(i0 + grp, n - 1);   // the lane's row within the run
            const bool own = lane_in && i0 + grp < n;
            const int gu = __shfl(ue, idx, 64), gv = __shfl(ve, idx, 64);
            const int glive = __shfl(live, idx, 64);
            const float gm = __shfl(m, idx, 64), gc0 = __shfl(c0, idx, 64), gc1 = __shfl(c1, idx, 64);
            const uint64_t row = base + q0 + (uint32_t)idx;
            const int py0 = gu - RINT - R, px0 = gv - RINT - R;
            // a row without mass pulls nothing back: its (clamped) disk is
            // read but every weight is zero
            const float on1 = glive ? 1.f : 0.f;
            const float rm = glive ? 1.f / gm : 0.f;
            const int du = min(max(gu, RINT), max(H - 1 - RINT, RINT));
            const int dv = min(max(gv, RINT), max(W - 1 - RINT, RINT));
            double var[3] = {0.0, 0.0, 0.0};
            // EDGE: some patch of the group leaves the frame
            auto patches = [&](auto edge_c) {
                constexpr bool EDGE = decltype(edge_c)::value;
                // column pass
                float bw[D], wf[D], bf[D];
#pragma unroll
                for (int j = 0; j < D; ++j) {
                    const float fj = ((float)(j - RINT) - gc1) * rm;
                    if constexpr (EDGE) bw[j] = box_count(gv + j - RINT, px0 + c, R, W);
                    else bw[j] = abs(c - j - R) <= R ? 1.f : 0.f;
                    wf[j] = wl[j] * fj;
                    bf[j] = bw[j] * fj;
                }
                float sg[D], ug[D], sb[D], ub[D];
                const GLOBAL float* disk = P + (size_t)du * W + dv;
#pragma unroll
                for (int i = 0; i < D; ++i) {
                    sg[i] = ug[i] = sb[i] = ub[i] = 0.f;
#pragma unroll
                    for (int j = 0; j < D; ++j) {
                        if ((i - RINT) * (i - RINT) + (j - RINT) * (j - RINT) > RINT * RINT) continue;
                        const float on = disk[(ptrdiff_t)(i - RINT) * W + (j - RINT)] > 0.f ? on1 : 0.f;
                        sg[i] = __builtin_fmaf(on, wl[j], sg[i]);
                        ug[i] = __builtin_fmaf(on, wf[j], ug[i]);
                        sb[i] = __builtin_fmaf(on, bw[j], sb[i]);
                        ub[i] = __builtin_fmaf(on, bf[j], ub[i]);
                    }
                }
                // row pass: outputs y, x, mass; y's terms carry f_y(i)
                float yg[D], yb[D];
#pragma unroll
                for (int i = 0; i < D; ++i) {
                    const float fi = ((float)(i - RINT) - gc0) * rm;
                    yg[i] = fi * sg[i];
                    yb[i] = fi * sb[i];
                }
                const bool cin = px0 + c >= 0 && px0 + c < W;
                // first pixel of this lane's column (interior; rows that hold
                // no patch read the first one's)
                const GLOBAL T* col = I + (size_t)max(py0, 0) * W + max(px0, 0) + c;
                float* const jp = ao.jac ? ao.jac + (size_t)row * 3 * (S * S) + c : nullptr;
                // one patch row; run: the boxcar windows' running sums (interior)
                auto patch_row = [&](int r, const float (&run)[3]) {
                    float bo[3] = {run[0], run[1], run[2]};
                    if constexpr (EDGE) {
                        bo[0] = bo[1] = bo[2] = 0.f;
#pragma unroll
                        for (int i = 0; i < D; ++i) {
                            const float k = box_count(gu + i - RINT, py0 + r, R, H);
                            bo[0] = __builtin_fmaf(k, yb[i], bo[0]);
                            bo[1] = __builtin_fmaf(k, ub[i], bo[1]);
                            bo[2] = __builtin_fmaf(k, sb[i], bo[2]);
                        }
                    }
                    float ga = 0.f, gb = 0.f, gc = 0.f;
#pragma unroll
                    for (int i = 0; i < D; ++i) {
                        const int k = r - i - R;
                        if (k < -R || k > R) continue;
                        const float w = wd[k < 0 ? -k : k];
                        ga = __builtin_fmaf(w, yg[i], ga);
                        gb = __builtin_fmaf(w, ug[i], gb);
                        gc = __builtin_fmaf(w, sg[i], gc);
                    }
                    auto term = [&](float ga_, float bo_) {   // ga / gn^2 - bo / k^2
                        const float t = __builtin_fmaf(ga_, rgg_lo, ga_ * rgg);
                        return __builtin_fmaf(-bo_, rkk, __builtin_fmaf(-bo_, rkk_lo, t));
                    };
                    float jo[3] = {term(ga, bo[0]), term(gb, bo[1]), term(gc, bo[2])};
                    float pixel;
                    if constexpr (EDGE) {
                        const int ry = py0 + r, rx = px0 + c;
                        const bool in = cin && ry >= 0 && ry < H;
                        pixel = (float)I[(size_t)min(max(ry, 0), H - 1) * W + min(max(rx, 0), W - 1)];
#pragma unroll
                        for (int o = 0; o < 3; ++o) jo[o] = in ? jo[o] : 0.f;
                    } else {
                        pixel = (float)col[(size_t)r * W];
                    }
                    const double lam = (double)fmaxf(pixel, 0.f);
#pragma unroll
                    for (int o = 0; o < 3; ++o)
                        var[o] = __builtin_fma((double)jo[o] * (double)jo[o], lam, var[o]);
                    if (jp && own) {
#pragma unroll
                        for (int o = 0; o < 3; ++o) jp[o * (S * S) + r * S] = jo[o];
                    }
                };
                // boxcar windows: rows r < D the prefix 0..r, r > 2R the
                // suffix r - 2R .. D - 1 (from the last row upwards), in
                // between all
                float run[3] = {0.f, 0.f, 0.f};
#pragma unroll
                for (int r = 0; r <= 2 * R; ++r) {
                    if (r < D) { run[0] += yb[r]; run[1] += ub[r]; run[2] += sb[r]; }
                    patch_row(r, run);
                }
                run[0] = run[1] = run[2] = 0.f;
#pragma unroll
                for (int r = S - 1; r > 2 * R; --r) {
                    run[0] += yb[r - 2 * R]; run[1] += ub[r - 2 * R]; run[2] += sb[r - 2 * R];
                    patch_row(r, run);
                }
            };
            if (__ballot(py0 < 0 || px0 < 0 || py0 + S > H || px0 + S > W)) patches(std::true_type{});
            else patches(std::false_type{});
            // sum over the S lanes of the row
            constexpr int P2 = S > 32 ? 32 : S > 16 ? 16 : S > 8 ? 8 : S > 4 ? 4 : 2;
#pragma unroll
            for (int d = P2; d > 0; d >>= 1)
#pragma unroll
                for (int o = 0; o < 3; ++o) {
                    const double t = __shfl_down(var[o], d, 64);
                    if (c + d < S) var[o] += t;
                }
            if (own && c == 0) {
                // output order: y, x, mass
#pragma unroll
                for (int o = 0; o < 3; ++o) ao.sigma[row * 3 + o] = (float)sqrt(var[o]);
                ao.origin[row * 2 + 0] = py0;
                ao.origin[row * 2 + 1] = px0;
                ao.rowpos[row] = (int32_t)(frame_pos0 + f);
            }
        }
    }
}

// grad[f] = sum over the frame's rows, in row order, of
// gy * J_y + gx * J_x + gm * J_mass on each row's patch.  One wave per
// VT_W x VT_H tile of a frame: the frame's rows are tested 64 at a time, the
// patches that touch the tile are added in row order to the tile in LDS
// (every pixel receives its terms in that order, whatever the tiling), and
// the tile is written once.  Bound by the reads of the patches: 24 frames of
// 512^2 in 17 us (a workgroup per frame over its rows and a fill of the
// gradient before: about 250 us).
constexpr int VT_W = 64, VT_H = 32;
__global__ __launch_bounds__(64) void k_adjoint_vjp(const float* __restrict__ jac,
                                                   const int32_t* __restrict__ origin,
                                                   const uint64_t* __restrict__ frame_rows,
                                                   const float* __restrict__ grad_rows,
                                                   float* __restrict__ grad, int S, int H,
                                                   int W) {
    __shared__ float acc[VT_H * VT_W];
    const int lane = threadIdx.x;
    const int tx = (W + VT_W - 1) / VT_W, ty = (H + VT_H - 1) / VT_H;
    const uint32_t f = blockIdx.x / (uint32_t)(tx * ty);
    const int tile = (int)(blockIdx.x % (uint32_t)(tx * ty));
    const int x0 = tile % tx * VT_W, y0 = tile / tx * VT_H;
    const int SS = S * S;
#pragma unroll
    for (int r = 0; r < VT_H; ++r) acc[r * VT_W + lane] = 0.f;
    const uint64_t e = frame_rows[f + 1];
    for (uint64_t rb = frame_rows[f]; rb < e; rb += 64) {
        const uint64_t mine = min(rb + (uint64_t)lane, e - 1);
        const int oy = origin[mine * 2], ox = origin[mine * 2 + 1];
        const bool hit = rb + (uint64_t)lane < e && oy < y0 + VT_H && oy + S > y0 && ox < x0 + VT_W &&
                         ox + S > x0;
        for (uint64_t todo = __ballot(hit); todo; todo &= todo - 1) {
            const int q = __ffsll((long long)todo) - 1;
            const uint64_t row = rb + (uint64_t)q;
            const int py0 = __builtin_amdgcn_readlane(oy, q), px0 = __builtin_amdgcn_readlane(ox, q);
            const float gy = grad_rows[row * 3 + 0], gx = grad_rows[row * 3 + 1],
                        gm = grad_rows[row * 3 + 2];
            const float* jr = jac + row * 3 * (size_t)SS;
            // the part of the patch inside the tile
            const int ra = max(0, y0 - py0), rz = min(S, y0 + VT_H - py0);
            const int ca = max(0, x0 - px0), cw = min(S, x0 + VT_W - px0) - ca;
            const int cnt = (rz - ra) * cw;
            for (int p = lane; p < cnt; p += 64) {
                const int r = ra + p / cw, c = ca + p % cw;
                const int at = r * S + c;
                float v = gy * jr[at];
                v = __builtin_fmaf(gx, jr[SS + at], v);
                v = __builtin_fmaf(gm, jr[2 * SS + at], v);
                acc[(py0 + r - y0) * VT_W + (px0 + c - x0)] += v;
            }
            // the wave's LDS operations keep their order; so must the compiler
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
    __syncthreads();
    float* gf = grad + (size_t)f * H * W;
    if (x0 + lane < W) {
        for (int r = 0; r < min(VT_H, H - y0); ++r)
            gf[(size_t)(y0 + r) * W + x0 + lane] = acc[r * VT_W + lane];
    }
}

template <int RINT, int R>
hipError_t launch_adjoint_reg(const Batch& b, const Geom* d_geom, const AdjOut& ao,
                              uint32_t frame_pos0, hipStream_t s) {
    // about eight waves per SIMD in all, and enough of them where one frame
    // has all the rows
    const uint32_t per_frame = std::max(32u, std::min(512u, 8192u / std::max(b.nframes, 1u)));
    const dim3 grid(b.nframes, per_frame), block(64);
    if (b.in_type == IN_U16)
        hipLaunchKernelGGL((k_adjoint_reg<RINT, R, uint16_t>), grid, block, 0, s, b, d_geom, ao, frame_pos0);
    else if (b.in_type == IN_U8)
        hipLaunchKernelGGL((k_adjoint_reg<RINT, R, uint8_t>), grid, block, 0, s, b, d_geom, ao, frame_pos0);
    else
        hipLaunchKernelGGL((k_adjoint_reg<RINT, R, float>), grid, block, 0, s, b, d_geom, ao, frame_pos0);
    return hipGetLastError();
}

}  // namespace

int adjoint_patch(const Geom& g) { return 2 * (g.rint + g.R) + 1; }

bool adjoint_supported(const Geom& g) {
    return g.rint >= 0 && (2 * g.rint + 1) * (2 * g.rint + 1) <= ADJ_TAPS && g.R <= 16;
}

size_t adjoint_sep_lds(const Geom& g) {
    const size_t D = 2 * (size_t)g.rint + 1, S = (size_t)adjoint_patch(g), NW = 2 * (size_t)g.R + 1;
    return 4 * (D * D * 4 + 6 * D * S + 2 * S * D + NW);
}

hipError_t launch_adjoint(const Batch& b, const Geom& g, const Geom* d_geom, const AdjOut& ao,
                          uint32_t frame_pos0, hipStream_t s) {
    if (g.R == g.rint || g.R == g.rint + 1) {
        switch (2 * g.rint + (g.R - g.rint)) {
            case 2: return launch_adjoint_reg<1, 1>(b, d_geom, ao, frame_pos0, s);
            case 3: return launch_adjoint_reg<1, 2>(b, d_geom, ao, frame_pos0, s);
            case 4: return launch_adjoint_reg<2, 2>(b, d_geom, ao, frame_pos0, s);
            case 5: return launch_adjoint_reg<2, 3>(b, d_geom, ao, frame_pos0, s);
            case 6: return launch_adjoint_reg<3, 3>(b, d_geom, ao, frame_pos0, s);
            case 7: return launch_adjoint_reg<3, 4>(b, d_geom, ao, frame_pos0, s);
            case 8: return launch_adjoint_reg<4, 4>(b, d_geom, ao, frame_pos0, s);
            case 9: return launch_adjoint_reg<4, 5>(b, d_geom, ao, frame_pos0, s);
            case 10: return launch_adjoint_reg<5, 5>(b, d_geom, ao, frame_pos0, s);
            case 11: return launch_adjoint_reg<5, 6>(b, d_geom, ao, frame_pos0, s);
            case 12: return launch_adjoint_reg<6, 6>(b, d_geom, ao, frame_pos0, s);
            case 13: return launch_adjoint_reg<6, 7>(b, d_geom, ao, frame_pos0, s);
            case 14: return launch_adjoint_reg<7, 7>(b, d_geom, ao, frame_pos0, s);
            default: break;
        }
    }
    const size_t lds = adjoint_sep_lds(g);
    if (lds <= 48 * 1024)
        hipLaunchKernelGGL(k_adjoint_sep, dim3(b.nframes, 64), dim3(64), lds, s, b, d_geom, ao,
                           frame_pos0);
    else
        hipLaunchKernelGGL(k_adjoint, dim3(b.nframes, 64), dim3(64), 0, s, b, d_geom, ao,
                           frame_pos0);
    return hipGetLastError();
}

hipError_t launch_adjoint_vjp(const float* jac, const int32_t* origin, const uint64_t* frame_rows,
                              uint32_t nframes, const float* grad_rows, float* grad, int S, int H,
                              int W, hipStream_t s) {
    if (nframes == 0 || H <= 0 || W <= 0) return hipSuccess;
    const uint64_t tiles = (uint64_t)((W + VT_W - 1) / VT_W) * ((H + VT_H - 1) / VT_H);
    // a launch holds fewer than 2^31 workgroups: whole frames at a time
    const uint32_t most = (uint32_t)std::max<uint64_t>(1, (1ull << 30) / tiles);
    for (uint32_t f0 = 0; f0 < nframes; f0 += most) {
        const uint32_t nf = std::min(most, nframes - f0);
        hipLaunchKernelGGL(k_adjoint_vjp, dim3((uint32_t)(nf * tiles)), dim3(64), 0, s, jac, origin,
                           frame_rows + f0, grad_rows, grad + (size_t)f0 * H * W, S, H, W);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace gt
