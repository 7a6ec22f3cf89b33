// gt_bandpass.hip -- launch of the locate path's bandpass (K1), and the
// two-pass form for what the streaming kernel (gt_bandpass.h) does not take.
#include "gt_bandpass.h"

#pragma clang fp contract(off)

namespace gt {

extern template hipError_t launch_bandpass_t<uint16_t>(int, const Batch&, const K1Params&, bool, hipStream_t);
extern template hipError_t launch_bandpass_t<uint8_t>(int, const Batch&, const K1Params&, bool, hipStream_t);
extern template hipError_t launch_bandpass_t<float>(int, const Batch&, const K1Params&, bool, hipStream_t);

// Bandpass without a Gaussian halo (R = 0) and of frames one pixel wide: two
// straightforward passes through a global temporary, each thread one pixel,
// taps in the shader's order.
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

bool bandpass_fast_path(int in_type, uint32_t min_w, const Geom& g) {
    return g.R >= 1 && g.R <= 16 && min_w >= 2 &&
           (in_type == IN_U16 || in_type == IN_U8 || in_type == IN_F32);
}

hipError_t launch_bandpass(const Batch& b, const Geom& g, const Geom* d_geom, int seg_rows,
                           hipStream_t s) {
    (void)d_geom;
    K1Params kp;
    for (int i = 0; i < 17; ++i) kp.w[i] = i <= g.R ? g.w[g.R + i] : 0.f;
    kp.gn = g.gn; kp.rgn = g.rgn; kp.rgn_lo = g.rgn_lo;
    kp.kk = g.kk; kp.rkk = g.rkk; kp.rkk_lo = g.rkk_lo;
    kp.seg = seg_rows;
    kp.hist = b.hist1 != nullptr && g.has_pct;
    const bool fast = g.fastdiv != 0;
    if (b.in_type == IN_U16) return launch_bandpass_t<uint16_t>(g.R, b, kp, fast, s);
    if (b.in_type == IN_F32) return launch_bandpass_t<float>(g.R, b, kp, fast, s);
    return launch_bandpass_t<uint8_t>(g.R, b, kp, fast, s);
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
