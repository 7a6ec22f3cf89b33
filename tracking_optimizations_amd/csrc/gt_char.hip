// gt_char.hip -- characterisation columns of every output row:
//   cpu_processed  Rg, ecc, signal (execute_gpu.rs:165-172,286-299,346-352):
//                  products of the bandpassed disk at the candidate pixel with
//                  the host tables, each summed in ndarray's eight-accumulator
//                  order (full chunks of 8, pairwise fold, then the remainder
//                  in order), with the walked mass;
//   characterize   Rg_gpu, raw_mass_gpu, signal_gpu, ecc_gpu
//                  (centers.wgsl:64-80): sums over the candidate pixel's own
//                  disk in the shader's tap order.
//
// Runs after emit on the rows that are left, eight lanes to a row.  Lane q
// holds accumulator q of the host sums, and one of the shader's six running
// values (mass, Rg, raw mass, maximum, sine and cosine sums): those are serial
// chains over the taps, so they run side by side, as one multiply-add with
// the lane's own coefficient (x + d = fma(d, 1, x) exactly).  The eight lanes
// fetch their row's taps together, 64 at a time, and read them back from LDS:
// when every lane loaded every tap the address units were the bound (48
// frames of 1024^2 with 4.2 k rows each, d = 9: 131 us, 80 us so; one lane
// per candidate inside the refine kernel, with its own walk: 375 us).
#include <algorithm>

#include "gt_device.h"

#pragma clang fp contract(off)

namespace gt {

namespace {

constexpr int CH_WG = 256, CH_ROWS = CH_WG / 8;   // rows per workgroup and step
constexpr int CH_TAPS = 64;                       // taps staged at a time
constexpr int CH_LD = CH_TAPS + 1;                // rows on different banks

// Offsets (dy * W + dx) of a disk's taps in row-major order; lanes 0 .. 2r
// of one wave write one row each.
__device__ __forceinline__ void tap_offsets(int r, int W, int lane, int* off) {
    const int i = lane - r;
    int hw = -1;
    if (i <= r)
        while ((hw + 1) * (hw + 1) + i * i <= r * r) ++hw;
    const uint32_t n = (uint32_t)(2 * hw + 1);
    const uint32_t first = wave_incl_scan(hw >= 0 ? n : 0u, lane) - (hw >= 0 ? n : 0u);
    for (int j = -hw; j <= hw; ++j) off[first + (uint32_t)(j + hw)] = i * W + j;
}

template <typename T>
__global__ __launch_bounds__(CH_WG) void k_char(Batch b, const Geom* __restrict__ g) {
    extern __shared__ float s_tab[];
    const uint32_t f = blockIdx.x;
    const Frame fr = b.frames[f];
    const int H = (int)fr.H, W = (int)fr.W;
    const int tid = threadIdx.x, lane = tid & 63, q = lane & 7;
    const int first = lane & ~7;   // the row's first lane
    const int nc = g->ncols, band = g->band, rint = g->rint;
    const bool cpu = g->cpu_processed, gpu = g->characterize;
    const int ng = gpu ? g->ntap_gpu : 0, nh = cpu ? g->ntap_cpu : 0;
    const uint64_t base = b.frame_row_base[f];
    if (base >= b.rows_cap) return;
    const uint32_t nrows = (uint32_t)min((uint64_t)b.frame_rows[f], b.rows_cap - base);
    if (blockIdx.y * CH_ROWS >= nrows) return;   // workgroup-uniform
    // tables: the shader's disk, then the host's
    int* const goff = (int*)s_tab;
    float* const gr2 = s_tab + ng;
    float* const gsin = gr2 + ng;
    float* const gcos = gsin + ng;
    int* const hoff = (int*)(gcos + ng);
    float* const hr2 = (float*)hoff + nh;
    float* const hsin = hr2 + nh;
    float* const hcos = hsin + nh;
    float* const one = hcos + nh;
    // staged taps of this lane's row: bandpassed and raw pixels
    float* const sp = one + 1 + (tid / 8) * CH_LD;
    float* const sx = sp + CH_ROWS * CH_LD;
    auto wave_sync = [] {   // a wave's LDS operations keep their order; so must the compiler
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    if (tid < 64) {
        if (gpu) tap_offsets(rint, W, lane, goff);
        if (cpu) tap_offsets(band, W, lane, hoff);
    }
    for (int t = tid; t < ng; t += CH_WG) {
        gsin[t] = g->sin2_gpu[t];
        gcos[t] = g->cos2_gpu[t];
        gr2[t] = g->r2_gpu[t];
    }
    for (int t = tid; t < nh; t += CH_WG) {
        hr2[t] = g->r2_cpu[t];
        hsin[t] = g->sin_cpu[t];
        hcos[t] = g->cos_cpu[t];
    }
    if (tid == 0) *one = 1.0f;
    __syncthreads();

    const GLOBAL float* P = (const GLOBAL float*)fr.P;
    const GLOBAL T* I = (const GLOBAL T*)fr.in;
    // this lane's chain over the shader's disk: coefficients and their stride
    const float* const coef = q == 1 ? gr2 : q == 4 ? gsin : q == 5 ? gcos : one;
    const int step = q == 1 || q == 4 || q == 5 ? 1 : 0;
    for (uint32_t r = blockIdx.y * CH_ROWS + (uint32_t)tid / 8; ; r += gridDim.y * CH_ROWS) {
        const bool in = r < nrows;
        if (__ballot(in) == 0) break;   // wave-uniform
        const uint64_t row = base + (in ? r : nrows - 1);
        float* const o = b.rows + row * (uint64_t)nc;
        const uint32_t pix = (uint32_t)b.rows_cand[row];   // frames hold fewer than 2^30 pixels
        const int u0 = (int)(pix / (uint32_t)W), v0 = (int)(pix % (uint32_t)W);
        const GLOBAL float* p = P + pix;
        const float mid = *p;
        if (cpu) {
            const float mass = o[1];
            const int nfull = nh - nh % 8;
            float pr = 0.f, ps = 0.f, pc = 0.f, sig = mid;
#pragma unroll 8
            for (int t = q; t < nfull; t += 8) {
                const float d = p[hoff[t]];
                sig = d > sig ? d : sig;
                pr = pr + d * hr2[t];
                ps = ps + d * hsin[t];
                pc = pc + d * hcos[t];
            }
            // fold: (acc q + acc q + 4) for q = 0 .. 3, added in order to 0
            pr = pr + __shfl(pr, first + ((q + 4) & 7), 64);
            ps = ps + __shfl(ps, first + ((q + 4) & 7), 64);
            pc = pc + __shfl(pc, first + ((q + 4) & 7), 64);
            float rg = 0.f, ss = 0.f, cc = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                rg = rg + __shfl(pr, first + k, 64);
                ss = ss + __shfl(ps, first + k, 64);
                cc = cc + __shfl(pc, first + k, 64);
            }
            for (int t = nfull; t < nh; ++t) {
                const float d = p[hoff[t]];
                sig = d > sig ? d : sig;
                rg = rg + d * hr2[t];
                ss = ss + d * hsin[t];
                cc = cc + d * hcos[t];
            }
#pragma unroll
            for (int d = 1; d < 8; d <<= 1) {
                const float t = __shfl_xor(sig, d, 64);
                sig = t > sig ? t : sig;
            }
            // in order from the first tap: a NaN there stays, later ones are skipped
            const float lead = p[hoff[0]];
            sig = lead != lead ? lead : sig;
            ss = ss * ss;
            cc = cc * cc;
            const float ecc = sqrtf(ss + cc);
            if (in) {
                if (q == 0) o[4] = sqrtf(rg / mass);
                if (q == 1) o[5] = ecc / (mass - mid);
                if (q == 2) o[6] = sig;
            }
        }
        if (gpu) {
            float* const og = o + (nc - 4);   // the last four columns
            const bool inside = !(u0 - band < 0 || u0 + band >= H || v0 - band < 0 || v0 + band >= W);
            float acc = 0.f;
            const GLOBAL T* x = I + pix;
            const float* c = coef;
            for (int t0 = 0; t0 < ng; t0 += CH_TAPS) {
                const int n = min(CH_TAPS, ng - t0);
                if (inside) {   // every candidate pixel is
#pragma unroll
                    for (int k = 0; k < CH_TAPS / 8; ++k) {
                        const int t = q + 8 * k;
                        if (t < n) {
                            const int at = goff[t0 + t];
                            sp[t] = p[at];
                            sx[t] = (float)x[at];
                        }
                    }
                }
                wave_sync();
                if (inside) {
                    const float* v = q == 2 ? sx : sp;
#pragma unroll 8
                    for (int t = 0; t < n; ++t) {
                        const float d = v[t];
                        const float s = __builtin_fmaf(d, *c, acc);
                        acc = q == 3 ? (d > acc ? d : acc) : s;
                        c += step;
                    }
                }
                wave_sync();
            }
            const float ms = __shfl(acc, first + 0, 64), rg = __shfl(acc, first + 1, 64);
            float es = __shfl(acc, first + 4, 64), ec = __shfl(acc, first + 5, 64);
            es = es * es;
            ec = ec * ec;
            if (in) {
                if (q == 1) og[0] = inside ? sqrtf(rg / ms) : 0.f;
                if (q == 2) og[1] = acc;
                if (q == 3) og[2] = acc;
                if (q == 5) og[3] = inside ? sqrtf(es + ec) / (ms - mid) : 0.f;
            }
        }
    }
}

}  // namespace

hipError_t launch_char(const Batch& b, const Geom& g, const Geom* d_geom, hipStream_t s) {
    const size_t taps = (size_t)(g.characterize ? g.ntap_gpu : 0) + (g.cpu_processed ? g.ntap_cpu : 0);
    const size_t lds = (4 * taps + 1 + 2 * CH_ROWS * CH_LD) * sizeof(float);
    // every frame's rows over as many workgroups as give the chip four waves
    // per SIMD, and enough of them where one frame has all the rows
    const uint32_t per_frame = std::max(16u, std::min(256u, 1536u / std::max(b.nframes, 1u)));
    const dim3 grid(b.nframes, per_frame), block(CH_WG);
    if (b.in_type == IN_U16) hipLaunchKernelGGL(k_char<uint16_t>, grid, block, lds, s, b, d_geom);
    else if (b.in_type == IN_U8) hipLaunchKernelGGL(k_char<uint8_t>, grid, block, lds, s, b, d_geom);
    else hipLaunchKernelGGL(k_char<float>, grid, block, lds, s, b, d_geom);
    return hipGetLastError();
}

}  // namespace gt
