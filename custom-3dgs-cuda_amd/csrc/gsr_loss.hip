// gsr_loss.hip — the trainer's reconstruction loss
// (gaussian_splatting/utils/loss.py:12-33 of kmurungi/custom-3dgs-cuda):
//   loss = (1 - lambda) mean|gt - img| + lambda (1 - SSIM(clamp(img), clamp(gt)))
// with the SSIM of torchmetrics (>= 1.0, the reference's requirement; not
// vendored): an 11x11 Gaussian window of sigma 1.5 normalised to sum 1,
// C1 = (0.01)^2, C2 = (0.03)^2 for data range 1, per-window statistics
// sigma_x^2 = max(E[x^2] - mu_x^2, 0) (torchmetrics clamps both variances at 0
// since its releases after 1.0) and sigma_xy = E[xy] - mu_x mu_y, averaged over
// the windows whose 11x11 support lies inside the image (torchmetrics pads by
// reflection and crops the 5-pixel margin of the index map, which leaves
// exactly those windows) and over the 3 channels.  Images are [H, W, 3] fp32.
//
// Two kernels, each one pass over HBM, on tiles of 32x16 pixels with a halo of
// five, separable with the vertical pass first:
//   ssim_fwd_kernel   vertical: a thread per interleaved column (3 channels x 42
//                     columns, so its loads coalesce as the images lie in HBM)
//                     and half of the rows takes 18 rows of both images straight
//                     from memory, forms each product x^2, y^2, xy once and the
//                     five 11-tap sums of 8 rows, and leaves them in LDS;
//                     horizontal: a thread per four neighbouring windows of a
//                     channel takes their 14 columns of the sums from LDS, forms
//                     the moments, the SSIM index, and per window the three
//                     partial derivatives of the index with respect to mu_x,
//                     E[x^2] and E[xy] (stored for the backward);
//                     per-work-group sums of the index and of |gt - img|;
//   ssim_bwd_kernel   the same two passes over the derivative maps (the window is
//                     symmetric, so the adjoint of the moments' blur is the same
//                     blur), then
//                     dL/dimg = g ((1 - lambda)/(3HW) sgn(img - gt)
//                               - lambda/(3 n_win) [clamp mask] (B1 + 2 x B2 + y B3)).
// The images are not staged: what is staged per value is five words once, read
// 17.5 times, where a horizontal pass from staged images took 75 words of LDS
// per value.  1920x1080, same run, before and after: forward 78 and 60 us,
// backward 76 and 47 us.  VALU issue bounds both now (234 and 152 instructions
// per value, 0.68 and 0.55 of the slots), the loads' latency leaves the rest.
// Only the loss's own arithmetic is fp32-tolerance work: the convolutions use
// fused multiply-adds.
#include <hip/hip_runtime.h>

#include <cmath>

#include "gsr_common.h"
#include "gsr_internal.h"

namespace gsr {

namespace {

constexpr int kLossTW = 32, kLossTH = 16;  // output tile (columns x rows)
constexpr int kWinR = 5;                   // window radius: 11 taps
constexpr int kWinTaps = 2 * kWinR + 1;
constexpr int kInCols = 3 * (kLossTW + 2 * kWinR);  // 126 interleaved columns
constexpr int kRunV = 8;                            // rows a thread sums vertically
constexpr int kRunVIn = kRunV + kWinTaps - 1;       // from 18
constexpr int kRunH = 4;                            // windows a thread forms horizontally
constexpr int kRunHIn = kRunH + kWinTaps - 1;       // from 14 columns of their channel
constexpr int kRowRuns = 3 * (kLossTW / kRunH);     // 24 per row
constexpr int kHTasks = kRowRuns * kLossTH;         // 384
constexpr int kLossThreads = 384;
constexpr int kFinalThreads = 256;
constexpr int kPitch = kInCols + 1;                 // odd: the runs' lanes spread over the banks
static_assert(kHTasks == kLossThreads && kInCols <= 128 && kLossTH / kRunV * 128 <= kLossThreads,
              "one run of each kind per thread");
// A byte offset past every row (12 bytes per pixel, rows of at most 2^31 / 33
// pixels).
constexpr uint32_t kOutside = 0xffffff00u;
constexpr float kC1 = 0.01f * 0.01f, kC2 = 0.03f * 0.03f;

struct Window {
    float w[kWinTaps];
};

// torch.clamp(v, 0, 1): NaN stays NaN (IEEE 754-2019 maximum and minimum, one
// instruction each).
__device__ __forceinline__ float clamp01(float v) {
    return __builtin_elementwise_minimum(__builtin_elementwise_maximum(v, 0.0f), 1.0f);
}

// Windows whose support lies inside the image: centres in [5, H - 5) x [5, W - 5).
__device__ __forceinline__ bool interior(int y, int x, int H, int W) {
    return y >= kWinR && y < H - kWinR && x >= kWinR && x < W - kWinR;
}

// 1 / b for b in [C1, 4]: the hardware's (1 ulp) corrected once by its exact
// residual, a division's 0.5 ulp.
__device__ __forceinline__ float reciprocal(float b) {
    const float r = __builtin_amdgcn_rcpf(b);
    return __builtin_fmaf(__builtin_fmaf(-b, r, 1.0f), r, r);
}

// Adds input i's share, w[i - j] v, to the values j of a run it lies in: the
// vertical passes take the rows as their loads arrive.
template <int kRun>
__device__ __forceinline__ void run_add(float (&m)[kRun], const Window& win, int i, float v) {
#pragma clang fp contract(fast)
#pragma unroll
    for (int j = 0; j < kRun; ++j)
        if (i - j >= 0 && i - j < kWinTaps) m[j] += win.w[i - j] * v;
}

// The kRun neighbouring window sums of kRun + 10 values, each from the window's
// ends inwards: the large middle taps come last, so most additions round a small
// sum.  The horizontal passes, whose values lie in LDS, take them so.  In the
// order of the taps dL/dimg was 1.78e-6 from 64 bits at 1920x1080, where the
// horizontal pass first and a product w x times x per window had left 1.76e-6
// (x^2 formed once leaves its rounding in every window it lies in); so it is
// 1.42e-6, in the same time (62 and 47 us).  The vertical passes so as well gave
// 1.15e-6, but waited for the last row first: 63.5 and 48.3 us.
template <int kRun>
__device__ __forceinline__ void run_sums(float (&m)[kRun], const Window& win,
                                         const float (&v)[kRun + kWinTaps - 1]) {
#pragma clang fp contract(fast)
#pragma unroll
    for (int k = 0; k < kWinTaps; ++k) {
        const int tap = (k & 1) ? kWinTaps - 1 - k / 2 : k / 2;
#pragma unroll
        for (int j = 0; j < kRun; ++j)
            m[j] = k == 0 ? win.w[tap] * v[j + tap] : m[j] + win.w[tap] * v[j + tap];
    }
}

// The element at byte offset `at` of row y of a plane of interleaved pixels, 0
// for a row or a column (kOutside) outside the image: the row is a buffer of its
// own (a scalar descriptor, y is the wave's), so the halo needs no tests and no
// vector address arithmetic.
__device__ __forceinline__ float row_load(const float* plane, int y, int H, int W, uint32_t at) {
    const uint32_t bytes = (y >= 0 && y < H) ? (uint32_t)W * 12u : 0u;
    const float* row = plane + (ptrdiff_t)y * W * 3;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row), 0, (int)bytes,
                                                        0x00020000);
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)at, 0, 0));
}

// A thread's vertical run: two waves (126 of their lanes, one interleaved column
// each) take the tile's upper eight rows, two the lower.
struct VerticalRun {
    int q, r0;     // column of the halo, first row of the tile
    uint32_t at;   // the column's byte offset in a row
    bool active;
};
__device__ __forceinline__ VerticalRun vertical_run(int x0, int W) {
    VerticalRun v;
    const int pair = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 7);
    v.q = (int)threadIdx.x & 127;
    v.r0 = pair * kRunV;
    v.active = pair < kLossTH / kRunV && v.q < kInCols;
    const int gx = x0 - kWinR + v.q / 3;
    v.at = (gx >= 0 && gx < W) ? (uint32_t)((x0 - kWinR) * 3 + v.q) * 4u : kOutside;
    return v;
}

__global__ __launch_bounds__(kLossThreads)
__attribute__((amdgpu_waves_per_eu(5))) void ssim_fwd_kernel(
    int H, int W, const float* __restrict__ img, const float* __restrict__ gt, Window win,
    float* __restrict__ gmaps, float2* __restrict__ partial) {
#pragma clang fp contract(fast)
    __shared__ float s_v[5][kLossTH][kPitch];
    __shared__ float s_red[2][kLossThreads / kWave];
    const int tid = threadIdx.x;
    const int x0 = blockIdx.x * kLossTW, y0 = blockIdx.y * kLossTH;
    const size_t plane = (size_t)H * W * 3;

    float l1 = 0.0f;  // |gt - img| of the tile's own pixels
    const VerticalRun run = vertical_run(x0, W);
    if (run.active) {
        const int q = run.q, r0 = run.r0;
        const bool own = q >= 3 * kWinR && q < kInCols - 3 * kWinR;
        float xv[kRunVIn], yv[kRunVIn];
#pragma unroll
        for (int i = 0; i < kRunVIn; ++i) {
            xv[i] = row_load(img, y0 + r0 - kWinR + i, H, W, run.at);
            yv[i] = row_load(gt, y0 + r0 - kWinR + i, H, W, run.at);
        }
        float m[5][kRunV] = {};
#pragma unroll
        for (int i = 0; i < kRunVIn; ++i) {
            if (own && i >= kWinR && i < kWinR + kRunV) l1 += fabsf(yv[i] - xv[i]);
            const float x = clamp01(xv[i]), y = clamp01(yv[i]);
            run_add(m[0], win, i, x);
            run_add(m[1], win, i, y);
            run_add(m[2], win, i, x * x);
            run_add(m[3], win, i, y * y);
            run_add(m[4], win, i, x * y);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k)
#pragma unroll
            for (int j = 0; j < kRunV; ++j) s_v[k][r0 + j][q] = m[k][j];
    }
    __syncthreads();

    float ssum = 0.0f;
    {
        const int r = tid / kRowRuns, u = tid - r * kRowRuns, grp = u / 3, ch = u - 3 * grp;
        const int c = 3 * kRunH * grp + ch;  // the run's first window and input column
        float m[5][kRunH];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            float v[kRunHIn];
#pragma unroll
            for (int i = 0; i < kRunHIn; ++i) v[i] = s_v[k][r][c + 3 * i];
            run_sums(m[k], win, v);
        }
        const int gy = y0 + r;
#pragma unroll
        for (int j = 0; j < kRunH; ++j) {
            const int gx = x0 + kRunH * grp + j;
            if (gy >= H || gx >= W) continue;
            const bool window = interior(gy, gx, H, W);
            const float mux = m[0][j], muy = m[1][j];
            // the variances clamped at 0 (torch.clamp: NaN stays NaN)
            const float vxx = m[2][j] - mux * mux, vyy = m[3][j] - muy * muy;
            const float sxx = vxx < 0.0f ? 0.0f : vxx, syy = vyy < 0.0f ? 0.0f : vyy;
            const float sxy = m[4][j] - mux * muy;
            const float a1 = 2.0f * mux * muy + kC1, a2 = 2.0f * sxy + kC2;
            const float b1 = mux * mux + muy * muy + kC1, b2 = sxx + syy + kC2;
            const float rb1 = reciprocal(b1), rb2 = reciprocal(b2);
            const float inv = rb1 * rb2;
            const float s = a1 * a2 * inv;
            ssum += window ? s : 0.0f;
            if (gmaps) {
                // dS/dA1 = a2 inv, dS/dA2 = a1 inv, dS/dB1 = -S / b1, dS/dB2 = -S / b2;
                // A1 = 2 mux muy + C1, A2 = 2 (E[xy] - mux muy) + C2,
                // B1 = mux^2 + muy^2 + C1, B2 = E[x^2] - mux^2 + E[y^2] - muy^2 + C2
                const float dA1 = a2 * inv, dA2 = a1 * inv, dB1 = -s * rb1, dB2 = -s * rb2;
                // the clamp of sigma_x^2 passes its gradient where sigma_x^2 >= 0
                const float dBx = (vxx >= 0.0f) ? dB2 : 0.0f;
                const float g1 = 2.0f * muy * (dA1 - dA2) + 2.0f * mux * (dB1 - dBx);
                const size_t idx = ((size_t)gy * W + gx) * 3 + ch;
                gmaps[idx] = window ? g1 : 0.0f;              // dS/dmu_x
                gmaps[plane + idx] = window ? dBx : 0.0f;     // dS/dE[x^2]
                gmaps[2 * plane + idx] = window ? 2.0f * dA2 : 0.0f;  // dS/dE[xy]
            }
        }
    }
    const float ws = wave_sum(ssum), wl = wave_sum(l1);
    if ((tid & (kWave - 1)) == 0) {
        s_red[0][tid / kWave] = ws;
        s_red[1][tid / kWave] = wl;
    }
    __syncthreads();
    if (tid == 0) {
        float a = 0.0f, b = 0.0f;
        for (int w = 0; w < kLossThreads / kWave; ++w) {
            a += s_red[0][w];
            b += s_red[1][w];
        }
        partial[blockIdx.y * gridDim.x + blockIdx.x] = make_float2(a, b);
    }
}

// out[0] = loss, out[1] = SSIM, out[2] = mean |gt - img|, from the work-groups'
// partial sums (added in double, in work-group order: deterministic).
__global__ __launch_bounds__(kFinalThreads) void loss_finalize_kernel(
    int parts, const float2* __restrict__ partial, double n_win, double n_px, float lambda,
    float* __restrict__ out) {
    __shared__ double s_a[kFinalThreads], s_b[kFinalThreads];
    const int tid = threadIdx.x;
    double a = 0.0, b = 0.0;
    for (int i = tid; i < parts; i += kFinalThreads) {
        const float2 p = partial[i];
        a += (double)p.x;
        b += (double)p.y;
    }
    s_a[tid] = a;
    s_b[tid] = b;
    __syncthreads();
    for (int s = kFinalThreads / 2; s > 0; s >>= 1) {
        if (tid < s) {
            s_a[tid] += s_a[tid + s];
            s_b[tid] += s_b[tid + s];
        }
        __syncthreads();
    }
    if (tid == 0) {
        const double ssim = s_a[0] / n_win, l1 = s_b[0] / n_px;
        out[0] = (float)((1.0 - (double)lambda) * l1 + (double)lambda * (1.0 - ssim));
        out[1] = (float)ssim;
        out[2] = (float)l1;
    }
}

__global__ __launch_bounds__(kLossThreads) void ssim_bwd_kernel(
    int H, int W, const float* __restrict__ img, const float* __restrict__ gt, Window win,
    const float* __restrict__ gmaps, float c_l1, float c_ssim, const float* __restrict__ grad_loss,
    float* __restrict__ dimg) {
#pragma clang fp contract(fast)
    __shared__ float s_v[3][kLossTH][kPitch];
    const int tid = threadIdx.x;
    const int x0 = blockIdx.x * kLossTW, y0 = blockIdx.y * kLossTH;
    const size_t plane = (size_t)H * W * 3;
    const float g = grad_loss ? *grad_loss : 1.0f;
    // the run's own pixels, loaded ahead of the passes
    const int r = tid / kRowRuns, u = tid - r * kRowRuns, grp = u / 3, ch = u - 3 * grp;
    const int gy = y0 + r, gx = x0 + kRunH * grp;
    float xv[kRunH], yv[kRunH];
#pragma unroll
    for (int j = 0; j < kRunH; ++j) {
        const bool in = gy < H && gx + j < W;
        const size_t idx = ((size_t)gy * W + gx + j) * 3 + ch;
        xv[j] = in ? img[idx] : 0.0f;
        yv[j] = in ? gt[idx] : 0.0f;
    }
    // vertical: the derivative maps of the windows centred in the tile and its
    // halo (the forward stores 0 for windows that are not inside the image)
    const VerticalRun run = vertical_run(x0, W);
    if (run.active) {
        const int q = run.q, r0 = run.r0;
#pragma unroll
        for (int mp = 0; mp < 3; ++mp) {
            float v[kRunVIn], m[kRunV] = {};
#pragma unroll
            for (int i = 0; i < kRunVIn; ++i)
                v[i] = row_load(gmaps + mp * plane, y0 + r0 - kWinR + i, H, W, run.at);
#pragma unroll
            for (int i = 0; i < kRunVIn; ++i) run_add(m, win, i, v[i]);
#pragma unroll
            for (int j = 0; j < kRunV; ++j) s_v[mp][r0 + j][q] = m[j];
        }
    }
    __syncthreads();
    const int c = 3 * kRunH * grp + ch;
    float m[3][kRunH];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float v[kRunHIn];
#pragma unroll
        for (int i = 0; i < kRunHIn; ++i) v[i] = s_v[k][r][c + 3 * i];
        run_sums(m[k], win, v);
    }
#pragma unroll
    for (int j = 0; j < kRunH; ++j) {
        if (gy >= H || gx + j >= W) continue;
        const float x = xv[j], y = yv[j];
        const float xc = clamp01(x), yc = clamp01(y);
        // torch's clamp passes the gradient where 0 <= x <= 1
        const float ds = (x >= 0.0f && x <= 1.0f)
                             ? m[0][j] + 2.0f * xc * m[1][j] + yc * m[2][j]
                             : 0.0f;
        // d|gt - x|/dx = -sgn(gt - x) (0 at 0, as torch's abs backward)
        const float d = y - x;
        const float sg = (d > 0.0f) ? -1.0f : ((d < 0.0f) ? 1.0f : (d != d ? d : 0.0f));
        dimg[((size_t)gy * W + gx + j) * 3 + ch] = g * (c_l1 * sg - c_ssim * ds);
    }
}

Window gaussian_window() {
    Window w;
    double g[kWinTaps], sum = 0.0;
    for (int k = 0; k < kWinTaps; ++k) {
        const double d = (double)(k - kWinR) / 1.5;
        g[k] = std::exp(-0.5 * d * d);
        sum += g[k];
    }
    for (int k = 0; k < kWinTaps; ++k) w.w[k] = (float)(g[k] / sum);
    return w;
}

dim3 loss_grid(int H, int W) {
    return dim3((unsigned)((W + kLossTW - 1) / kLossTW), (unsigned)((H + kLossTH - 1) / kLossTH));
}

}  // namespace

size_t loss_partial_count(int H, int W) {
    const dim3 g = loss_grid(H, W);
    return (size_t)g.x * g.y;
}

hipError_t launch_l1_dssim_fwd(int H, int W, const float* img, const float* gt, float lambda,
                               float* gmaps, void* partial, float* out, hipStream_t st) {
    const dim3 grid = loss_grid(H, W);
    hipLaunchKernelGGL(ssim_fwd_kernel, grid, dim3(kLossThreads), 0, st, H, W, img, gt,
                       gaussian_window(), gmaps, static_cast<float2*>(partial));
    const double n_win = 3.0 * (double)(H - 2 * kWinR) * (double)(W - 2 * kWinR);
    const double n_px = 3.0 * (double)H * (double)W;
    hipLaunchKernelGGL(loss_finalize_kernel, dim3(1), dim3(kFinalThreads), 0, st,
                       (int)(grid.x * grid.y), static_cast<const float2*>(partial), n_win, n_px,
                       lambda, out);
    return hipGetLastError();
}

hipError_t launch_l1_dssim_bwd(int H, int W, const float* img, const float* gt, float lambda,
                               const float* gmaps, const float* grad_loss, float* dimg,
                               hipStream_t st) {
    const double n_win = 3.0 * (double)(H - 2 * kWinR) * (double)(W - 2 * kWinR);
    const double n_px = 3.0 * (double)H * (double)W;
    const float c_l1 = (float)((1.0 - (double)lambda) / n_px);
    const float c_ssim = (float)((double)lambda / n_win);
    hipLaunchKernelGGL(ssim_bwd_kernel, loss_grid(H, W), dim3(kLossThreads), 0, st, H, W, img,
                       gt, gaussian_window(), gmaps, c_l1, c_ssim, grad_loss, dimg);
    return hipGetLastError();
}

}  // namespace gsr
