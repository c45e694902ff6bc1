// gsr_blend.hip — front-to-back alpha blend and its backward.
//
// One work-group per 16x16 tile.  Layout template kPix (pixels per lane):
// 4 / kPix wave64s, each owning a 16 x (4 kPix) strip of the tile; lane l
// holds column l & 15 and rows (l >> 4) + 4p, p < kPix, of its strip.  More
// pixels per lane give each lane independent dependency chains and divide the
// per-pixel share of the batch loads and of the backward's wave reductions;
// more waves per tile shorten the longest tile's critical path.  A batch of
// one list entry per thread is staged in LDS as 48 B blend records (one
// record load per entry); lanes walk the batch with broadcast LDS reads.  The forward's per-pixel arithmetic is the reference's, operation
// for operation (rasterize.cu:241-270); the backward's decisions are too
// (rasterize_backward.cu:113-200).
//
// Exact strip culling: each record carries qthr, a bound on the quadratic
// form above which no pixel can reach alpha >= 1/255 (gsr_bin.hip).  When the
// batch is staged, each entry gets one bit per strip: clear when the least
// value of the quadratic form over the strip's rectangle exceeds qthr (with
// margins for the per-pixel fp32 rounding).  Every pixel of such a strip would
// skip the entry in the reference's own tests, so the wave skips it without
// changing any result.
//
// Forward early exit: a pixel is done once T < 1e-4; a wave leaves the batch
// when none of its pixels is live; the tile stops when all are done.
// Backward: the tile walks only entries [0, max n_contrib) of its list, back
// to front (the reference walks all K entries and skips the tail per pixel),
// and each wave skips entries beyond its own max n_contrib.  A batch holds only
// entries that a strip meets (fill_batch).  A wave takes its
// entries four at a time: their decisions in straight-line code, their colours'
// products with dL/dpixel by matrix instructions, and their nine gradient sums
// over the wave through one transposition in LDS (see group_sums).  The two
// waves' sums of an entry are added and stored with plain stores into the
// (Gaussian, tile) pair's own gradient slot
// (nine floats and a claim bit).  pair_grad_reduce_kernel adds each
// Gaussian's claimed slots.  Float atomics are used only for list entries
// that have no slot of their own: pairs outside the Gaussian's tile
// rectangle, and a repeated id within one tile's list (caller-supplied lists).
// Measured with a wave reduction per entry and so (same run): 229 and 213 us
// (100k Gaussians, 1080p), 288 and 275 us (1M), 96 and 76 us (10k, 256x256);
// VALU instructions per 1080p launch 1.38e8 and 1.09e8.  VALU issue takes 0.70
// of the slots; the waves' dependent chains (LDS, exp, compares and their
// masks) and the prologue's and batches' loads leave the rest.
//
// Work-groups take their tile from a launch order, longest estimated work
// first (tile_order_kernel), so long tiles do not start last.
#include <algorithm>
#include <cstdlib>

#include <mutex>

#include "gsr_internal.h"
#include "gsr_common.h"
#include "gsr_schedule.h"

namespace gsr {

namespace {

template <int kPix>
struct Layout {
    static constexpr int kWaves = 4 / kPix;
    static constexpr int kThreads = kWaves * kWave;
    static constexpr int kBatch = kThreads;
    static constexpr int kRows = 4 * kPix;  // rows per wave strip
};

template <int kPix>
struct Pixels {
    int px;
    int py[kPix];
    bool in[kPix];
};

template <int kPix>
__device__ __forceinline__ Pixels<kPix> pixels_of(int tile, int tiles_x, int W, int H) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    Pixels<kPix> p;
    p.px = tx * kTileSize + (lane & 15);
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
        p.py[k] = ty * kTileSize + wave * Layout<kPix>::kRows + (lane >> 4) + 4 * k;
        p.in[k] = p.px < W && p.py[k] < H;
    }
    return p;
}

// The backward's pixels: the same strips, a lane's two pixels in adjacent
// rows 2 (l >> 4) + k, so that a quad of lanes holds four columns of two
// adjacent rows (group_sums takes their moments).
__device__ __forceinline__ Pixels<2> bwd_pixels_of(int tile, int tiles_x, int W, int H) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    Pixels<2> p;
    p.px = tx * kTileSize + (lane & 15);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        p.py[k] = ty * kTileSize + wave * Layout<2>::kRows + 2 * (lane >> 4) + k;
        p.in[k] = p.px < W && p.py[k] < H;
    }
    return p;
}

// Minimum over the pixel rectangle [x0, x1] x [y0, y1] of the quadratic form
// q = A u^2 + 2 B u v + C v^2, (u, v) = (x - mx, y - my), for a positive
// definite conic (A > 0, AC > B^2): 0 when the mean is inside, else the least
// of the four edges' minima (each a clamped 1D quadratic).  The computed
// minimiser is off by a few ulp, which raises q only at second order; the
// evaluation's own rounding is covered by the caller's margin.
__device__ __forceinline__ float qmin_rect(float mx, float my, float A, float B, float C,
                                          float rA, float rC, float x0, float x1, float y0,
                                          float y1) {
    if (mx >= x0 && mx <= x1 && my >= y0 && my <= y1) return 0.0f;
    const float ux0 = x0 - mx, ux1 = x1 - mx, vy0 = y0 - my, vy1 = y1 - my;
    auto q = [&](float u, float v) { return A * u * u + 2.0f * B * u * v + C * v * v; };
    float best = q(fminf(fmaxf(-B * vy0 * rA, ux0), ux1), vy0);
    best = fminf(best, q(fminf(fmaxf(-B * vy1 * rA, ux0), ux1), vy1));
    best = fminf(best, q(ux0, fminf(fmaxf(-B * ux0 * rC, vy0), vy1)));
    best = fminf(best, q(ux1, fminf(fmaxf(-B * ux1 * rC, vy0), vy1)));
    return best;
}

// Staged strip bits: bit w for wave w of the tile, and the record's flags
// (plain_record) where its quadratic form's |terms| sum to at most kPlainTerms over
// the tile, so that exp's argument reduction holds and gives 0 or a denormal far
// below the range, an alpha below 1/255 either way.
constexpr float kPlainTerms = 4e6f;

// Bit w set: some pixel of strip w may reach alpha >= 1/255.  A strip is
// culled when the least q over its rectangle, lowered by 1e-5 of the largest
// sum of |terms| there (the fp32 rounding of the per-pixel q and of this
// bound are each within ~1e-6 of that sum), still exceeds qthr.  Conics that
// are not positive definite, and NaN anywhere, cull nothing.  With the
// flags of a plain entry.
template <int kPix>
__device__ __forceinline__ uint32_t strip_bits(const BlendRec& r, int tile, int tiles_x) {
    constexpr uint32_t kAll = (1u << Layout<kPix>::kWaves) - 1u;
    // the conic from the record's scaled coefficients (exact)
    const float A = -2.0f * r.a.z, B = -2.0f * r.c.y, C = -2.0f * r.b.x, thr = r.c.z;
    if (!(A > 0.0f) || !(C > 0.0f) || !((double)A * C - (double)B * B > 0.0)) return kAll;
    const float mx = r.a.x, my = r.a.y;
    const float rA = 1.0f / A, rC = 1.0f / C;
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const float x0 = (float)(tx * kTileSize), x1 = x0 + (float)(kTileSize - 1);
    const float dxm = fmaxf(fabsf(x0 - mx), fabsf(x1 - mx));
    uint32_t bits = 0;
    float most = 0.0f;  // the largest sum of |terms| over the tile
#pragma unroll 1
    for (int w = 0; w < Layout<kPix>::kWaves; ++w) {
        const float y0 = (float)(ty * kTileSize + w * Layout<kPix>::kRows);
        const float y1 = y0 + (float)(Layout<kPix>::kRows - 1);
        const float dym = fmaxf(fabsf(y0 - my), fabsf(y1 - my));
        const float absq = A * dxm * dxm + 2.0f * fabsf(B) * dxm * dym + C * dym * dym;
        const float q = qmin_rect(mx, my, A, B, C, rA, rC, x0, x1, y0, y1) - 1e-5f * absq;
        const bool skip = q > thr;  // false for NaN
        bits |= skip ? 0u : (1u << w);
        most = (absq <= most) ? most : absq;  // NaN stays
    }
    return bits | (most <= kPlainTerms ? __float_as_uint(r.c.w) : 0u);
}

// The record of list entry g, zeros for an id outside [0, n) (such entries are
// skipped: rasterize_backward.cu:79-86).
__device__ __forceinline__ BlendRec load_record(const BlendRec* __restrict__ recs, int g, int n) {
    BlendRec r;
    if (g >= 0 && g < n) {
        r = recs[g];
    } else {
        r.a = r.b = r.c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    return r;
}

// A staged entry of the forward: the record's a and b words, and of c the blue
// channel and the strip bits (c.y is a.w / 2, exactly; qthr has served).
template <int kPix>
__device__ __forceinline__ void stage_entry(const BlendRec* __restrict__ recs, int g, int n,
                                            int tile, int tiles_x, float4* s_a, float4* s_b,
                                            float2* s_c, int slot) {
    const BlendRec r = load_record(recs, g, n);
    const bool ok = g >= 0 && g < n;
    s_a[slot] = r.a;
    s_b[slot] = r.b;
    const uint32_t bits = ok ? strip_bits<kPix>(r, tile, tiles_x) : 0u;
    s_c[slot] = make_float2(r.c.x, __uint_as_float(bits));
}

// Forward pixel state.  A pixel is done once a blend takes T below 1e-4
// (rasterize.cu:264-267); T only changes on a blend, so "done" is T < 1e-4
// and needs no flag (pixels off the screen start with T = 0).
struct FwdPixel {
    float T, C0, C1, C2;
    int last;
};

__device__ __forceinline__ bool live(const FwdPixel& p) { return p.T >= kTransmittanceMin; }

// power = -0.5 (cx dx^2 + 2 cy dx dy + cz dy^2) (rasterize.cu:249-251) with
// its two additions fused, from the record's coefficients a = -cx/2 (A.z),
// b = -cy (A.w), c = -cz/2 (B.x): fma(c dy, dy, fma(b dx, dy, (a dx) dx)).
__device__ __forceinline__ float blend_power(float dx, float dy, const float4& A,
                                             const float4& B) {
    return __builtin_fmaf(B.x * dy, dy, __builtin_fmaf(A.w * dx, dy, (A.z * dx) * dx));
}

// One pixel's forward step for one list entry (rasterize.cu:243-268), with the
// reference's skips as selects: the same fp32 operations in the same order,
// the colour sums fused (pix_color += colour * weight).  `on` is live(p), the
// lane mask the caller's early-exit ballot already holds.
__device__ __forceinline__ void fwd_step(FwdPixel& p, bool on, float fx, float fy,
                                         const float4& A, const float4& B, float cb,
                                         int contributor) {
    const float dx = fx - A.x;
    const float dy = fy - A.y;
    const float power = blend_power(dx, dy, A, B);
    const float alpha = fminf(kAlphaMax, B.y * exp_blend_noclamp(power));
    const bool blend = on & !(power > 0.0f) & !(alpha < kAlphaMin);
    const float w = alpha * p.T;
    const float Tn = p.T * (1.0f - alpha);
    p.C0 = blend ? __builtin_fmaf(B.z, w, p.C0) : p.C0;
    p.C1 = blend ? __builtin_fmaf(B.w, w, p.C1) : p.C1;
    p.C2 = blend ? __builtin_fmaf(cb, w, p.C2) : p.C2;
    p.T = blend ? Tn : p.T;
    p.last = blend ? contributor : p.last;
}

// fwd_step of the next kCount plain entries (kPlainBit, or kClampBit with kClamp;
// no kColourBit) of `todo` in list order, bit for bit: a plain entry's power is
// never positive, its alpha never clamped (kClamp: one minimum), exp needs no range
// select, and one select of alpha serves the colours and T (a weight of 0 adds
// nothing, T times 1 is T): 28 VALU per pixel and entry instead of 35.  The alphas
// do not depend on T: all of the group's are formed first, in straight-line code
// with independent chains, then blended in order.
// Measured with a step per entry and so (same run): 140 and 123 us (100k
// Gaussians, 1080p), 180 and 157 us (1M), 48 and 41 us (10k, 256x256).  With half of the
// opacities from 0.99 on, by fwd_step and so: 97 and 88 us (100k, 1080p), 53 and 43
// us (10k, 256x256).
constexpr int kFwdGroup = 4;
template <int kPix, int kCount, bool kClamp>
__device__ __forceinline__ void fwd_steps_plain(FwdPixel (&p)[kPix], float fx,
                                                const float (&fy)[kPix], const float4* s_a,
                                                const float4* s_b, const float2* s_c, int c0,
                                                uint64_t& todo, int cbase) {
    float alpha[kCount][kPix];
    int at[kCount];
#pragma unroll
    for (int s = 0; s < kCount; ++s) {
        at[s] = c0 + (int)__builtin_ctzll(todo);
        todo &= todo - 1;
        const float4 A = s_a[at[s]];
        const float2 B = *reinterpret_cast<const float2*>(s_b + at[s]);
        const float dx = fx - A.x;
        const float adxdx = (A.z * dx) * dx, bdx = A.w * dx;  // blend_power's column terms
#pragma unroll
        for (int k = 0; k < kPix; ++k) {
            const float dy = fy[k] - A.y;
            const float power = __builtin_fmaf(B.x * dy, dy, __builtin_fmaf(bdx, dy, adxdx));
            float a = B.y * exp_core(power);
            if constexpr (kClamp) a = fminf(kAlphaMax, a);
            alpha[s][k] = (a < kAlphaMin) ? 0.0f : a;
        }
    }
#pragma unroll
    for (int s = 0; s < kCount; ++s) {
        const float2 rg = *(reinterpret_cast<const float2*>(s_b + at[s]) + 1);
        const float cb = s_c[at[s]].x;
#pragma unroll
        for (int k = 0; k < kPix; ++k) {
            const float a = live(p[k]) ? alpha[s][k] : 0.0f;
            const float w = a * p[k].T;
            p[k].C0 = __builtin_fmaf(rg.x, w, p[k].C0);
            p[k].C1 = __builtin_fmaf(rg.y, w, p[k].C1);
            p[k].C2 = __builtin_fmaf(cb, w, p[k].C2);
            p[k].T = p[k].T * (1.0f - a);
            p[k].last = (a > 0.0f) ? cbase + at[s] : p[k].last;
        }
    }
}

template <int kPix>
__device__ __forceinline__ bool any_live(const FwdPixel (&p)[kPix]) {
    bool l = false;
#pragma unroll
    for (int k = 0; k < kPix; ++k) l |= live(p[k]);
    return l;
}

// Steps `todo`'s entries, all of them plain, while a pixel is live.
template <int kPix, bool kClamp>
__device__ __forceinline__ void fwd_walk_plain(FwdPixel (&p)[kPix], float fx,
                                               const float (&fy)[kPix], const float4* s_a,
                                               const float4* s_b, const float2* s_c, int c0,
                                               uint64_t& todo, int cbase) {
    // two at a time where four would take more registers than eight waves per SIMD
    // leave (71 of 64)
    constexpr int kCount = kClamp && kPix == 2 ? 2 : kFwdGroup;
    int left = popc64(todo);
    for (; left >= kCount && ballot(any_live(p)) != 0; left -= kCount)
        fwd_steps_plain<kPix, kCount, kClamp>(p, fx, fy, s_a, s_b, s_c, c0, todo, cbase);
    for (; left > 0 && ballot(any_live(p)) != 0; --left)
        fwd_steps_plain<kPix, 1, kClamp>(p, fx, fy, s_a, s_b, s_c, c0, todo, cbase);
}

template <int kPix>
__global__ __launch_bounds__(Layout<kPix>::kThreads) void blend_fwd_kernel(
    int n, int H, int W, int tiles_x, uint64_t m, const int2* __restrict__ ranges,
    const int32_t* __restrict__ ids, const BlendRec* __restrict__ recs, float* __restrict__ img,
    float* __restrict__ finalT, int32_t* __restrict__ ncontrib,
    const uint32_t* __restrict__ order) {
    constexpr int kBatch = Layout<kPix>::kBatch;
    __shared__ float4 s_a[kBatch];
    __shared__ float4 s_b[kBatch];
    __shared__ float2 s_c[kBatch];
    const int tile = order ? (int)order[blockIdx.x] : (int)blockIdx.x;
    // a launch order is a permutation of the tiles; nothing else is touched
    if ((unsigned)tile >= (unsigned)(tiles_x * ((H + kTileSize - 1) / kTileSize))) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: uniform branches
    const uint32_t my_bit = 1u << wave;
    const Pixels<kPix> pp = pixels_of<kPix>(tile, tiles_x, W, H);
    float fx = (float)pp.px;
    asm volatile("" : "+v"(fx));
    float fy[kPix];
    FwdPixel p[kPix];
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
        fy[k] = (float)pp.py[k];
        p[k] = FwdPixel{pp.in[k] ? 1.0f : 0.0f, 0.0f, 0.0f, 0.0f, 0};
        asm volatile("" : "+v"(fy[k]));  // kept as floats, not converted again per entry
    }
    int start, end;
    clamp_range(ranges[tile], m, start, end);
    // the range is the work-group's: scalar, so the loop counters are scalar
    start = __builtin_amdgcn_readfirstlane(start);
    end = __builtin_amdgcn_readfirstlane(end);

    // each batch's ids are loaded while the batch before it is blended
    int next_id = (start + tid < end) ? ids[start + tid] : -1;
    for (int b0 = start; b0 < end; b0 += kBatch) {
        // scalar, so the entry loop's counter is scalar
        const int cnt = __builtin_amdgcn_readfirstlane(min(kBatch, end - b0));
        const int g = next_id;
        __syncthreads();
        if (tid < cnt)
            stage_entry<kPix>(recs, g, n, tile, tiles_x, s_a, s_b, s_c, tid);
        if (b0 + kBatch + tid < end) next_id = ids[b0 + kBatch + tid];
        __syncthreads();
        if (ballot(any_live(p)) != 0) {
            const int cbase = b0 - start + 1;
            // 64 entries at a time: one ballot gives the entries this wave's
            // strip meets (lane e holds entry c0 + e), walked in order with a
            // scalar find-first; strip-culled entries cost nothing
            bool done = false;
            for (int c0 = 0; c0 < cnt && !done; c0 += kWave) {
                const int e = c0 + lane;
                const uint32_t bits = e < cnt ? __float_as_uint(s_c[min(e, kBatch - 1)].y) : 0u;
                uint64_t todo = ballot((bits & my_bit) != 0u);
                constexpr uint32_t kAny = kPlainBit | kClampBit | kColourBit;
                const uint64_t odd = todo & ballot((bits & kAny) != kPlainBit);
                // the wave stops once no pixel is live, tested before each group
                // or entry with the same compares the steps' skips use
                if (odd == 0) {
                    fwd_walk_plain<kPix, false>(p, fx, fy, s_a, s_b, s_c, c0, todo, cbase);
                } else if ((odd & ballot((bits & kAny) != kClampBit)) == 0) {
                    fwd_walk_plain<kPix, true>(p, fx, fy, s_a, s_b, s_c, c0, todo, cbase);
                } else {
                    while (todo && ballot(any_live(p)) != 0) {
                        const int j = c0 + (int)__builtin_ctzll(todo);
                        todo &= todo - 1;
                        const float4 A = s_a[j];
                        const float4 B = s_b[j];
                        const float cb = s_c[j].x;
#pragma unroll
                        for (int k = 0; k < kPix; ++k)
                            fwd_step(p[k], live(p[k]), fx, fy[k], A, B, cb, cbase + j);
                    }
                }
                done = todo != 0;
            }
        }
        if (__syncthreads_and(!any_live(p))) break;
    }
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
        if (!pp.in[k]) continue;
        const size_t q = (size_t)pp.py[k] * W + pp.px;
        img[3 * q] = p[k].C0;
        img[3 * q + 1] = p[k].C1;
        img[3 * q + 2] = p[k].C2;
        finalT[q] = p[k].T;
        ncontrib[q] = p[k].last;
    }
}

// Backward pixel state: dL/dpixel, T (unwound back to front from final_T),
// accg = sum over channels of dL/dpixel * the reconstructed colour of what lies
// behind (the reference keeps the colour, accum_rec, and only ever uses its
// dot product with dL/dpixel), and n_contrib.
struct BwdPixel {
    float g0, g1, g2, T, accg;
    int last;
};

// Per pixel and list entry the walk forms dL/dpower = alpha dL/dalpha
// (rasterize_backward.cu:155-161: 0 for a clamped or skipped entry) and the
// colour weight alpha T; dL/dopacity = G dL/dalpha is dL/dpower / opacity,
// formed once per (tile, entry) at the flush.
struct BwdTerms {
    float aT;   // alpha * T_before: dL/dcolour = aT * dL/dpixel
    float dpw;  // dL/dpower
};

// One pixel's decision for one list entry (rasterize_backward.cu:117-140):
// G = exp(power), alpha = min(0.99, opacity G), and whether the entry blends
// (within n_contrib, power <= 0, alpha >= 1/255).  ae = alpha if it blends,
// else 0.  `within`: the lanes whose n_contrib the entry is within.  Each returns
// the lanes that blend it.
//
// The forward's own evaluation: exp_blend and the same fp32 operations, so
// every skip agrees with the forward bit for bit.
__device__ __forceinline__ uint64_t decide_exact(float power, float o, uint64_t within,
                                                 float& ae) {
    const float araw = o * exp_blend(power);
    const float alpha = fminf(kAlphaMax, araw);
    const uint64_t act =
        within & ballot(!(power > 0.0f)) & ballot(!(alpha < kAlphaMin));
    ae = __builtin_amdgcn_inverse_ballot_w64(act) ? alpha : 0.0f;
    return act;
}

// For a plain entry (kPlainBit: its power is never positive): G from the
// hardware exp2, which is within 1e-6 relative of exp_blend wherever alpha can
// reach 1/255 (power in [-5.6, 0]), so the alpha >= 1/255 test agrees with the
// exact one unless alpha lies within kNearAlpha of 1/255; alpha <= opacity <
// 0.99 is never clamped.  Alpha at or above kAlphaMin + kNearAlpha passes the
// test, below kAlphaMin - kNearAlpha fails it; `near` holds the lanes in
// neither case (near the threshold, or a NaN alpha), which need the exact
// evaluation.  Two compares per pixel, each ballot a compare's own mask.
constexpr float kNearAlpha = kAlphaMin * 2e-5f;
constexpr float kAlphaLo = kAlphaMin - kNearAlpha, kAlphaHi = kAlphaMin + kNearAlpha;
__device__ __forceinline__ uint64_t decide_fast(float power, float o, uint64_t within,
                                                float& ae, uint64_t& near) {
    const float alpha = o * __builtin_amdgcn_exp2f(power * 1.44269504088896341f);
    const uint64_t pass = ballot(alpha >= kAlphaHi);
    const uint64_t act = within & pass;
    ae = __builtin_amdgcn_inverse_ballot_w64(act) ? alpha : 0.0f;
    near |= ballot(!(alpha < kAlphaLo)) & ~pass;
    return act;
}

// One pixel's gradient step for a decided entry (rasterize_backward.cu:
// 141-198); cg is the entry's colour . dL/dpixel.  A skipped entry enters with
// ae = 0, which leaves T (x / 1) and accg unchanged and gives zero terms.
// dL/dpower is alpha T (colour . dL/dpixel less what lies behind); the caller
// zeroes it where alpha is clamped.  This arithmetic only has to meet the fp32
// gradient tolerance and may use fused multiply-adds.
__device__ __forceinline__ BwdTerms bwd_update(BwdPixel& p, float ae, float cg) {
#pragma clang fp contract(fast)
    BwdTerms t;
    // T / (1 - alpha) with 1 - alpha in [0.01, 1]: the reference's 1e-4 floor
    // never applies.  The hardware reciprocal (1 ulp) times T: about 1.5 ulp
    // per entry where a division is 0.5, so over the two thousand entries of
    // the benchmark scene's longest lists T drifts by a few 1e-5, against the
    // 1e-5 that the reference's own fp32 division reaches there; both lie
    // within the 1e-4 gradient bar.  A correction step from the exact residual
    // T - q (1 - alpha) (two fused multiply-adds on the entry's dependency
    // chain) brought the quotient to a division's 0.5 ulp and cost 15 us of
    // the bench frame's 229 us backward blend; on c5's distributions (walks
    // of 1.5e4 entries) it left the gradients unchanged to 1e-3 of their
    // error against float64, as did the forward's own alpha in place of the
    // fast one.  A skipped entry (alpha 0) leaves T unchanged: the reciprocal
    // of 1 is exact.
    const float den = 1.0f - ae;
    const float Tb = p.T * __builtin_amdgcn_rcpf(den);
    const float diff = cg - p.accg;
    t.aT = ae * Tb;
    t.dpw = ae * (diff * Tb);
    p.accg = __builtin_fmaf(ae, diff, p.accg);
    p.T = Tb;
    return t;
}

__device__ __forceinline__ BwdPixel load_bwd_pixel(bool in, int px, int py, int W,
                                                   const float* __restrict__ grad,
                                                   const GradStrides& gst,
                                                   const float* __restrict__ finalT,
                                                   const int32_t* __restrict__ ncontrib) {
    BwdPixel p{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0};
    if (in) {
        const float* g = grad + (int64_t)py * gst.h + (int64_t)px * gst.w;
        p.g0 = g[0];
        p.g1 = g[gst.c];
        p.g2 = g[2 * gst.c];
        const size_t q = (size_t)py * W + px;
        p.T = finalT[q];
        p.last = max(ncontrib[q], 0);
    }
    return p;
}

// Per (tile, entry) the wave sums nine values over its 128 pixels, from
// dpw = dL/dpower and aT = alpha T of each: S0 = sum dpw, P1 = sum dpw e,
// P2 = sum dpw dy, Q1 = sum dpw e^2, Q2 = sum dpw e dy, P5 = sum dpw dy^2 and
// the colours C = sum aT dL/dpixel, where e = dx + rho dy with the entry's
// rho = cy / cx (ridge_slope).  The pixel's offset times the conic is then
//   wx = cx dx + cy dy = cx e + r dy,   r = cy - cx rho,
//   wy = cy dx + cz dy = cy e + k dy,   k = cz - cy rho,
// exactly for any rho (r and k are one fused multiply-add each), and the
// reference's sums (rasterize_backward.cu:163-176, 211-221) are dL/dmean =
// sum dpw (wx, wy), dL/dcov2d = sum dpw (wx^2 / 2, wx wy, wy^2 / 2) (the
// conversion from dL/dconic, a congruence), dL/dcolour = C and dL/dopacity =
// S0 / opacity.  With rho = 0 they are sums about dx and dy, whose second
// moments a needle-shaped splat's conic cancels to a small remainder (wx^2
// from cx^2 dx^2, cx cy dx dy and cy^2 dy^2); along the ridge they do not
// cancel.
// kGroup entries are walked and summed together, so that the sums' share per
// entry is a quarter of one reduction:
// - walking, a lane forms its two pixels' terms of the four entries and leaves
//   them in LDS, the dpw pairs and then the alpha T pairs;
// - each is read back transposed, lane 4b + j taking entry j's terms of the
//   four lanes of quad b (four columns, two rows);
// - it sums the quad's dpw moments about entry j's mean: about a centre shared by
//   the entries a matrix product could form them, but where little beyond one
//   pixel beside the mean blends, e^2 would be the difference of numbers
//   thousands of times its size;
// - the colours' weights dL/dpixel are no entry's own, so their products are
//   matrix instructions (v_mfma_f32_4x4x1, fp32: sixteen 4x4 outer products,
//   one per quad, accumulated over the quad's eight pixels);
// - the sixteen quads are summed (permlane swaps and row rotations).
constexpr int kTerms = 9;
constexpr int kGroup = 4;               // entries per matrix-instruction group
constexpr int kGroupPitch = kWave + 1;  // float2s per entry; +1: transposed reads hit all banks
constexpr int kS0 = 0, kP1 = 1, kQ1 = 2, kP2 = 3, kQ2 = 4, kP5 = 5, kC0 = 6, kC1 = 7, kC2 = 8;

// Which of the nine sums lane l holds after group_sums, of entry l & 3 (-1:
// none): by row l >> 4 and quad of the row (l >> 2) & 3.
__device__ __forceinline__ int group_value_of_lane(int l) {
    const int row = l >> 4;
    switch ((l >> 2) & 3) {
        case 0: return row == 0 ? kS0 : row == 1 ? kP1 : row == 2 ? kC0 : kC1;
        case 1: return row == 0 ? kQ1 : row == 1 ? kP2 : row == 2 ? kC2 : kP5;
        case 2: return row == 0 ? kQ2 : -1;
        default: return -1;
    }
}

// The weights of the quad's colour products, element i = l & 3 of lane l:
// dL/dpixel (r, g, b, 0) of quad lane s's pixel k.
struct GroupWeights {
    float g[2][4];
};

template <int kLane>
__device__ __forceinline__ float quad_lane(float v) {
    return dpp_move<kLane * 0x55>(v);  // quad_perm [kLane x 4]
}

__device__ __forceinline__ GroupWeights group_weights(const BwdPixel (&p)[2]) {
    const int i = lane_id() & 3;
    GroupWeights w;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        auto pick = [&](float r, float g, float b) {
            return i == 0 ? r : i == 1 ? g : i == 2 ? b : 0.0f;
        };
        w.g[k][0] = pick(quad_lane<0>(p[k].g0), quad_lane<0>(p[k].g1), quad_lane<0>(p[k].g2));
        w.g[k][1] = pick(quad_lane<1>(p[k].g0), quad_lane<1>(p[k].g1), quad_lane<1>(p[k].g2));
        w.g[k][2] = pick(quad_lane<2>(p[k].g0), quad_lane<2>(p[k].g1), quad_lane<2>(p[k].g2));
        w.g[k][3] = pick(quad_lane<3>(p[k].g0), quad_lane<3>(p[k].g1), quad_lane<3>(p[k].g2));
    }
    return w;
}

// The nine sums of a group's entries over the wave's pixels; lane l returns
// sum group_value_of_lane(l) of entry l & 3.  terms: the wave's LDS; x0: the
// quad's first column, y: its rows; mean, rho: of entry l & 3.  All 64 lanes must
// be active.
__device__ __forceinline__ float group_sums(float2* terms, const GroupWeights& wt,
                                            const BwdTerms (&q)[kGroup][2], float x0,
                                            const float (&y)[2], const float2& mean, float rho) {
#pragma clang fp contract(fast)
    const int l = lane_id();
    const float2* mine = terms + (l & 3) * kGroupPitch + (l & ~3);
    // the wave's own stores, read by its other lanes: LDS serves a wave's
    // accesses in order, and the compiler keeps them so
    auto order = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int s = 0; s < kGroup; ++s)
        terms[s * kGroupPitch + l] = make_float2(q[s][0].dpw, q[s][1].dpw);
    order();
    const float dx0 = x0 - mean.x, dy0 = y[0] - mean.y, dy1 = y[1] - mean.y;
    const float b0 = dx0 + rho * dy0, b1 = dx0 + rho * dy1;
    float S[2], P[2], Q[2];  // per row: sums of dpw, dpw e, dpw e^2
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const float2 t = mine[s];
        const float e0 = b0 + (float)s, e1 = b1 + (float)s;
        const float f0 = e0 * t.x, f1 = e1 * t.y;
        S[0] = s == 0 ? t.x : S[0] + t.x;
        S[1] = s == 0 ? t.y : S[1] + t.y;
        P[0] = s == 0 ? f0 : P[0] + f0;
        P[1] = s == 0 ? f1 : P[1] + f1;
        Q[0] = s == 0 ? e0 * f0 : Q[0] + e0 * f0;
        Q[1] = s == 0 ? e1 * f1 : Q[1] + e1 * f1;
    }
    order();
#pragma unroll
    for (int s = 0; s < kGroup; ++s)
        terms[s * kGroupPitch + l] = make_float2(q[s][0].aT, q[s][1].aT);
    order();
    f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const float2 t = mine[s];
        c = __builtin_amdgcn_mfma_f32_4x4x1f32(wt.g[0][s], t.x, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_4x4x1f32(wt.g[1][s], t.y, c, 0, 0, 0);
    }
    order();
    const float S0 = S[0] + S[1], P1 = P[0] + P[1], Q1 = Q[0] + Q[1];
    const float g0 = dy0 * S[0], g1 = dy1 * S[1];
    const float P2 = g0 + g1;
    const float P5 = dy0 * g0 + dy1 * g1;
    const float Q2 = dy0 * P[0] + dy1 * P[1];
    // over the quads: lanes 0-31 keep the first of each pair, 32-63 the second
    const float f0 = fold32(S0, c[0]);
    const float f1 = fold32(P1, c[1]);
    const float f2 = fold32(Q1, c[2]);
    const float f3 = fold32(P2, P5);
    // Q2 alone: its swaps take a register that is no longer needed (what it
    // leaves in lanes 32-63 and in rows 1 and 3 is kept by nobody)
    const float f4 = fold32(Q2, g0);
    float h0 = fold16(f0, f1);  // rows: S0, P1, C0, C1
    float h1 = fold16(f2, f3);  // rows: Q1, P2, C2, P5
    float h2 = fold16(f4, g1);  // row 0: Q2
    h0 += dpp_move<kDppRowRor8>(h0);
    h1 += dpp_move<kDppRowRor8>(h1);
    h2 += dpp_move<kDppRowRor8>(h2);
    h0 += dpp_move<kDppRowRor4>(h0);
    h1 += dpp_move<kDppRowRor4>(h1);
    h2 += dpp_move<kDppRowRor4>(h2);
    // formed with every lane active: the selects below must not draw the last
    // adds into branches, away from their lane moves
    asm volatile("" : "+v"(h0), "+v"(h1), "+v"(h2));
    const int r = (l >> 2) & 3;
    return r == 0 ? h0 : r == 1 ? h1 : h2;
}

// The slope rho of a staged entry's ridge, from the record's a = -cx/2 (A.z) and
// b = -cy (A.w); 0 where the conic is not positive in x or the slope no number.
__device__ __forceinline__ float ridge_slope(const float4& A) {
    const float rho = (0.5f * A.w) / A.z;
    return (A.z < 0.0f && fabsf(rho) < 1e6f) ? rho : 0.0f;
}

// Long tiles' backward runs as two work items (tile_order_kernel picks them).
// The back part walks entries [mid, maxc) from the final transmittance, as a
// whole tile does.  The front part walks the same entries first with the
// pixel state only (state_walk) (the T and accumulated-colour steps of
// rasterize_backward.cu:141-198, no gradient sums), which hands it the exact
// state the sequential walk has at mid, then walks [0, mid) in full.  Both
// parts' gradients are bit for bit the whole tile's.  mid = 0.30 maxc: the two
// parts then take about as long (at 0.23, 0.27, 0.30, 0.37 and 0.44: 73.8, 73.1,
// 72.6, 75.7 and 79.3 us, 10k Gaussians at 256x256; six bands of lists of 350k
// entries 3.72, 3.77, 3.79, 3.84 and 3.88 ms; 720p between 121 and 124 us at all).
constexpr int kPartWhole = 0, kPartBack = 1, kPartFront = 2;
constexpr int kSplitNum = 30, kSplitDen = 100;
// Most tiles split per backward launch (the launch has this many extra groups).
constexpr int kSplitMax = 256;

// A batch of the backward in LDS: list entries that some strip of the tile meets
// within its n_contrib, back to front, and per wave the list of those it walks:
// the byte offsets of their places in `a` (the flag kListExact in the low bits),
// filled up with the none entry to a whole number of groups.
template <int kPix, int kBatch>
struct BwdBatch {
    static constexpr int kWaves = Layout<kPix>::kWaves;
    // one place more than the batch: the none entry, whose opacity is 0, so
    // that no pixel blends it
    float4 a[kBatch + 1];   // the record's a and b words
    float4 b[kBatch + 1];
    float blue[kBatch + 1];
    float rho[kBatch + 1];  // ridge_slope
    int id[kBatch];
    __attribute__((aligned(16))) int list[kWaves][kBatch + kGroup];
    // two windows' ballots: per wave of the entries its threads hold, those that
    // each strip meets
    uint64_t met[2][kWaves][kWaves];
};
constexpr int kListExact = 1;  // not a plain entry
constexpr int kListFlags = 15;

template <int kPix, int kBatch>
__device__ __forceinline__ void stage_none(BwdBatch<kPix, kBatch>& s) {
    s.a[kBatch] = s.b[kBatch] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    s.blue[kBatch] = s.rho[kBatch] = 0.0f;
}

// The tile's list as the backward fills its batches from it, back to front:
// positions [lo, hi) are left, next_id is thread t's id of position hi - 1 - t
// (-1: none).
struct BwdSource {
    const int32_t* ids;  // of the tile's first entry
    const BlendRec* recs;
    int n, tile, tiles_x;
    int lo, hi, next_id;
    int width;        // entries of the next window
    uint32_t window;  // windows taken so far
    __device__ __forceinline__ int id_below(int p, int t) const {
        return p - 1 - t >= lo ? ids[p - 1 - t] : -1;
    }
};

// Fills the batch from the list, a window of 128 entries (or 64, below) at a
// time, one per thread: each forms its entry's strip bits, and only entries with
// one are staged, in order, until the batch is at least half full or the list
// ends; what does not fit stays for the next batch.  So the barriers, the partial
// sums and their flush are paid for entries that are walked, and groups fill up
// across the windows: of a needle-shaped cloud's entries 4% meet a strip, of
// uniform clouds' 45%.  Staging 64 or 128 list entries as they came, with groups
// within 64 of them (1.57 places per entry of the needles), and so (same run):
// blend_bwd 3.67 and 2.42 ms (5M needles, 4K), 254 and 248 us (1M Gaussians,
// 1080p), 179 and 174 us (100k), 118 and 115 us (720p).
// The 64-entry batch takes windows of 64 while more than 3/4 of them meet a
// strip: of 128 half would be looked at twice (the benchmark frame, of whose
// entries 85% do, 200 us so and 196).
// strip_last: each strip's largest n_contrib; least_last: the least of this
// wave's pixels.  Returns how many entries are staged; `first`: per pixel the
// byte offset of the first of them within its n_contrib; `listed`: those that this
// wave walks, and whether all of them are plain.  All threads of the work-group,
// whose reads of the batch before end at its first barrier.
template <int kPix, int kBatch>
__device__ __forceinline__ int fill_batch(BwdBatch<kPix, kBatch>& s, BwdSource& src,
                                          const int (&strip_last)[Layout<kPix>::kWaves],
                                          int least_last, const BwdPixel (&px)[kPix],
                                          int (&first)[kPix], int& listed, bool& plain) {
    constexpr int kWaves = Layout<kPix>::kWaves, kThreads = Layout<kPix>::kThreads;
    static_assert(kBatch <= kThreads, "an empty batch takes at least one entry of a window");
    const int tid = (int)threadIdx.x, lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int count = 0, in_list[kWaves] = {};
#pragma unroll
    for (int k = 0; k < kPix; ++k) first[k] = 0;
    do {
        const int width = src.width, hi = src.hi;
        const int g = tid < width ? src.next_id : -1;
        const int p = hi - 1 - tid;
        // the window below, if this one fits
        src.next_id = src.id_below(hi - width, tid);
        const BlendRec r = load_record(src.recs, g, src.n);
        uint32_t bits = (g >= 0 && g < src.n) ? strip_bits<kPix>(r, src.tile, src.tiles_x) : 0u;
        uint64_t met[kWaves][kWaves];  // [threads' wave][strip]
        uint64_t* out = s.met[src.window & 1u][wave];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            if (p >= strip_last[w]) bits &= ~(1u << w);
            const uint64_t m = ballot(((bits >> w) & 1u) != 0u);
            if (lane == 0) out[w] = m;
        }
        __syncthreads();
        uint64_t any[kWaves];
        int total = 0;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            any[v] = 0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                met[v][w] = uniform64(s.met[src.window & 1u][v][w]);
                any[v] |= met[v][w];
            }
            total += popc64(any[v]);
        }
        ++src.window;
        if (count + total > kBatch) {
            // the first entry that does not fit, and all after it, stay
            int room = kBatch - count, taken = 0;
#pragma unroll
            for (int v = 0; v < kWaves; ++v) {
                const int here = popc64(any[v]);
                if (room >= 0 && here > room) {
                    const uint64_t first = ballot(((any[v] >> lane) & 1u) != 0u &&
                                                  popc_below(any[v]) == room);
                    taken = v * kWave + (int)__builtin_ctzll(first);
                    any[v] &= (first - 1);
                    room = -1;
                } else if (room < 0) {
                    any[v] = 0;
                } else {
                    room -= here;
                }
            }
            src.hi -= taken;
            src.next_id = src.id_below(src.hi, tid);
        } else {
            src.hi -= min(width, hi - src.lo);
        }
        if constexpr (kBatch < kThreads) src.width = 4 * total > 3 * width ? kBatch : kThreads;
        if (hi > least_last) {  // some pixel's n_contrib ends in or below the window
#pragma unroll
            for (int k = 0; k < kPix; ++k) {
#pragma unroll
                for (int v = 0; v < kWaves; ++v) {
                    const int c = min(hi - px[k].last - v * kWave, kWave);
                    first[k] += c > 0 ? popc64(any[v] << (kWave - c)) : 0;
                }
            }
        }
        int before = count;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            if (v == wave && ((any[v] >> lane) & 1u) != 0u) {
                const int slot = before + popc_below(any[v]);
                s.a[slot] = r.a;
                s.b[slot] = r.b;
                s.blue[slot] = r.c.x;
                s.rho[slot] = ridge_slope(r.a);
                s.id[slot] = g;
                const int entry =
                    slot * (int)sizeof(float4) | ((bits & kPlainBit) ? 0 : kListExact);
#pragma unroll
                for (int w = 0; w < kWaves; ++w)
                    if ((bits >> w) & 1u)
                        s.list[w][in_list[w] + popc_below(met[v][w] & any[v])] = entry;
            }
            before += popc64(any[v]);
#pragma unroll
            for (int w = 0; w < kWaves; ++w) in_list[w] += popc64(met[v][w] & any[v]);
        }
        count = before;
    } while (count < kBatch / 2 && src.hi > src.lo);
#pragma unroll
    for (int k = 0; k < kPix; ++k) first[k] *= (int)sizeof(float4);
    listed = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) listed = w == wave ? in_list[w] : listed;
    if (lane < kGroup - 1) s.list[wave][listed + lane] = kBatch * (int)sizeof(float4);
    __syncthreads();
    int flags = 0;
    for (int e = lane; e < listed; e += kWave) flags |= s.list[wave][e];
    plain = ballot((flags & kListFlags) != 0) == 0;
    return count;
}

template <int kPix>
__device__ __forceinline__ bool all_within(const int (&first)[kPix]) {
    int some = 0;
#pragma unroll
    for (int k = 0; k < kPix; ++k) some |= first[k];
    return ballot(some != 0) == 0;
}

template <typename T>
__device__ __forceinline__ T staged(const void* base, int offset) {
    return *reinterpret_cast<const T*>(static_cast<const char*>(base) + offset);
}

// colour . dL/dpixel of the group's entries for the lane's pixels, [pixel][entry]:
// the entries' colours (lane l reads entry l & 3's, at `own`) by the lanes' own
// dL/dpixel, as three outer products per pixel (v_mfma_f32_4x4x1; lane l keeps
// its pixel's column).
template <int kPix, int kBatch>
__device__ __forceinline__ void group_colours(int own, const BwdBatch<kPix, kBatch>& st,
                                              const BwdPixel (&p)[kPix], f32x4 (&cg)[kPix]) {
    const float2 rg = staged<float2>(st.b, own + (int)sizeof(float2));
    const float b = staged<float>(st.blue, own / 4);
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
        f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
        c = __builtin_amdgcn_mfma_f32_4x4x1f32(rg.x, p[k].g0, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_4x4x1f32(rg.y, p[k].g1, c, 0, 0, 0);
        cg[k] = __builtin_amdgcn_mfma_f32_4x4x1f32(b, p[k].g2, c, 0, 0, 0);
    }
}

// The wave's decisions for a group's entries, all of them in straight-line code
// (independent chains, one test for the whole group): the fast evaluation, then
// the exact one for the whole wave for every entry that is not plain or has a
// lane near the threshold.  at: the group's part of the wave's list; within: the
// whole batch lies within every pixel's n_contrib.
template <int kPix>
struct GroupDecision {
    float ae[kGroup][kPix];
    bool any;      // some pixel blends an entry
    bool clamped;  // an alpha may be clamped: it is then kAlphaMax itself, and only then
};
__device__ __forceinline__ float staged_power(const float4& A, float c, float fx, float fy) {
    // the forward's power, bit for bit (blend_power)
    const float dx = fx - A.x, dy = fy - A.y;
    return __builtin_fmaf(c * dy, dy, __builtin_fmaf(A.w * dx, dy, (A.z * dx) * dx));
}
template <int kPix, int kBatch>
__device__ __forceinline__ void decide_group(GroupDecision<kPix>& d, const int4& at, bool plain,
                                             bool within, const int (&first)[kPix], float fx,
                                             const float (&fy)[kPix],
                                             const BwdBatch<kPix, kBatch>& st) {
    int off[kGroup] = {at.x, at.y, at.z, at.w};
    bool exact[kGroup] = {};
    if (!plain) {
#pragma unroll
        for (int s = 0; s < kGroup; ++s) {
            exact[s] = (__builtin_amdgcn_readfirstlane(off[s]) & kListExact) != 0;
            off[s] &= ~kListFlags;
        }
    }
    float4 A[kGroup];
    float2 B[kGroup];
#pragma unroll
    for (int s = 0; s < kGroup; ++s) {
        A[s] = staged<float4>(st.a, off[s]);
        B[s] = staged<float2>(st.b, off[s]);
    }
    uint64_t in[kGroup][kPix];
#pragma unroll
    for (int s = 0; s < kGroup; ++s)
#pragma unroll
        for (int k = 0; k < kPix; ++k) in[s][k] = ~0ull;
    if (!within) {
#pragma unroll
        for (int s = 0; s < kGroup; ++s) {
#pragma unroll
            for (int k = 0; k < kPix; ++k) in[s][k] = ballot(off[s] >= first[k]);
        }
    }
    uint64_t act = 0, odd[kGroup], odd_any = 0;
#pragma unroll
    for (int s = 0; s < kGroup; ++s) {
        odd[s] = 0;
#pragma unroll
        for (int k = 0; k < kPix; ++k)
            act |= decide_fast(staged_power(A[s], B[s].x, fx, fy[k]), B[s].y, in[s][k],
                               d.ae[s][k], odd[s]);
        odd_any |= odd[s];
    }
    d.clamped = false;
    if (odd_any != 0 || !plain) {
#pragma unroll
        for (int s = 0; s < kGroup; ++s) {
            if (odd[s] == 0 && !exact[s]) continue;
            d.clamped |= exact[s];
            const float4 a = staged<float4>(st.a, off[s]);
            const float2 b = staged<float2>(st.b, off[s]);
#pragma unroll
            for (int k = 0; k < kPix; ++k)
                act |= decide_exact(staged_power(a, b.x, fx, fy[k]), b.y, in[s][k], d.ae[s][k]);
        }
    }
    // act may hold an entry's fast decision that the exact one took back: the
    // group is then summed for nothing
    d.any = act != 0;
}

// The pixel state's walk over the source's entries: the same decisions and T /
// accumulated-colour steps as the full walk, no sums.
template <int kPix, int kBatch>
__device__ __forceinline__ void state_walk(BwdSource src,
                                           const int (&strip_last)[Layout<kPix>::kWaves],
                                           int least_last, float fx, const float (&fy)[kPix],
                                           BwdPixel (&p)[kPix], BwdBatch<kPix, kBatch>& st) {
    const int* list = st.list[__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)];
    while (src.hi > src.lo) {
        int listed, first[kPix];
        bool plain;
        if (fill_batch(st, src, strip_last, least_last, p, first, listed, plain) == 0) break;
        const bool within = all_within(first);
        for (int i = 0; i < listed; i += kGroup) {
            const int4 at = *reinterpret_cast<const int4*>(list + i);
            GroupDecision<kPix> d;
            decide_group(d, at, plain, within, first, fx, fy, st);
            if (!d.any) continue;  // as the full walk
            f32x4 cg[kPix];
            group_colours(list[i + (lane_id() & 3)] & ~kListFlags, st, p, cg);
#pragma unroll
            for (int s = 0; s < kGroup; ++s) {
#pragma unroll
                for (int k = 0; k < kPix; ++k) (void)bwd_update(p[k], d.ae[s][k], cg[k][s]);
            }
        }
    }
}

template <int kPix, int kBatch, bool kSplit>
__global__ __launch_bounds__(Layout<kPix>::kThreads)
__attribute__((amdgpu_waves_per_eu(kBatch == 64 ? 6 : 4))) void blend_bwd_kernel(
    int n, int H, int W, int tiles_x, uint64_t m, const float* __restrict__ grad, GradStrides gst,
    const int2* __restrict__ ranges, const int32_t* __restrict__ ids,
    const BlendRec* __restrict__ recs, const float* __restrict__ finalT,
    const int32_t* __restrict__ ncontrib, float* __restrict__ dmean, float* __restrict__ dcov,
    float* __restrict__ dcol, float* __restrict__ dalpha, GradSlots gs,
    const uint32_t* __restrict__ order) {
    constexpr int kWaves = Layout<kPix>::kWaves;
    __shared__ BwdBatch<kPix, kBatch> st;
    // +1: the none entry, and a group's writers hit different banks
    __shared__ float s_part[kWaves][kTerms][kBatch + 1];
    __shared__ float2 s_terms[kWaves][kGroup * kGroupPitch];
    __shared__ int s_max[kWaves];

    // Work item.  kSplit (a schedule is given): items 2i and 2i + 1 (i < K) are
    // the back and front parts of the schedule's i-th tile, and the later
    // items its tiles from K on, whole; order[T] holds K (at most kSplitMax).
    const int T = tiles_x * ((H + kTileSize - 1) / kTileSize);
    int part = kPartWhole, tile;
    if constexpr (kSplit) {
        const int K = (int)min((uint32_t)kSplitMax,
                               (uint32_t)__builtin_amdgcn_readfirstlane((int)order[T]));
        const int item = (int)blockIdx.x;
        if (item < 2 * K) {
            part = (item & 1) ? kPartFront : kPartBack;
            tile = (int)order[item >> 1];
        } else {
            const int idx = item - K;
            if (idx >= T) return;
            tile = (int)order[idx];
        }
    } else {
        tile = order ? (int)order[blockIdx.x] : (int)blockIdx.x;
    }
    tile = __builtin_amdgcn_readfirstlane(tile);
    // a launch order is a permutation of the tiles; nothing else is touched
    if ((unsigned)tile >= (unsigned)T) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: uniform branches
    static_assert(kPix == 2, "group_sums takes two pixels per lane");
    const Pixels<kPix> pp = bwd_pixels_of(tile, tiles_x, W, H);
    const int tx = tile % tiles_x, ty = tile / tiles_x;
    const float fx = (float)pp.px;
    float fy[kPix];
    BwdPixel p[kPix];
    int my_last = 0, my_least = 0x7fffffff;
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
        fy[k] = (float)pp.py[k];
        p[k] = load_bwd_pixel(pp.in[k], pp.px, pp.py[k], W, grad, gst, finalT, ncontrib);
        my_last = max(my_last, p[k].last);
        my_least = min(my_least, p[k].last);
    }
    int start, end;
    clamp_range(ranges[tile], m, start, end);
    const int wave_last = __builtin_amdgcn_readfirstlane((int)wave_max_u32((uint32_t)my_last));
    const int least_last = 0x7fffffff - __builtin_amdgcn_readfirstlane(
        (int)wave_max_u32(0x7fffffffu - (uint32_t)my_least));
    if (lane == 0) s_max[wave] = wave_last;
    __syncthreads();
    int strip_last[kWaves], tile_last = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        strip_last[w] = __builtin_amdgcn_readfirstlane(s_max[w]);
        tile_last = max(tile_last, strip_last[w]);
    }
    start = __builtin_amdgcn_readfirstlane(start);
    const int maxc = min(tile_last, __builtin_amdgcn_readfirstlane(end) - start);
    const int my_value = group_value_of_lane(lane);
    const GroupWeights wt = group_weights(p);
    const float x0 = (float)(tx * kTileSize + (lane & 12));  // the quad's first column
    if (tid == 0) stage_none(st);  // before the first batch's barriers
    float2* terms = s_terms[wave];
    const int* list = st.list[wave];
    // the entries [lo, hi) this item walks with gradients; the front part first
    // walks [mid, maxc) for the pixel state only
    BwdSource src{ids + start, recs, n, tile, tiles_x, 0, maxc, -1, kBatch, 0u};
    if constexpr (kSplit) {
        const int mid = (int)(((int64_t)maxc * kSplitNum) / kSplitDen);
        if (part == kPartBack) src.lo = mid;
        if (part == kPartFront) {
            BwdSource behind = src;
            behind.lo = mid;
            behind.next_id = behind.id_below(maxc, tid);
            state_walk(behind, strip_last, least_last, fx, fy, p, st);
            src.hi = mid;
        }
    }

    src.next_id = src.id_below(src.hi, tid);
    while (src.hi > src.lo) {
        // the flush's addresses are formed again per batch: kept through the
        // walk they cost it registers, then scratch
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        int listed, first[kPix];
        bool plain;
        const int cnt = fill_batch(st, src, strip_last, least_last, p, first, listed, plain);
        if (cnt == 0) break;
        // this wave's partial sums of the batch start at zero: entries it does
        // not walk add nothing
        for (int e = lane; e < cnt; e += kWave)
#pragma unroll
            for (int k = 0; k < kTerms; ++k) s_part[wave][k][e] = 0.0f;
        const bool within = all_within(first);
        for (int i = 0; i < listed; i += kGroup) {
            const int4 at = *reinterpret_cast<const int4*>(list + i);
            const int own = list[i + (lane & 3)] & ~kListFlags;
            GroupDecision<kPix> d;
            decide_group(d, at, plain, within, first, fx, fy, st);
            // no pixel blends an entry: the state stays and the sums are zero
            if (!d.any) continue;
            f32x4 cg[kPix];
            group_colours(own, st, p, cg);
            BwdTerms q[kGroup][kPix];
#pragma unroll
            for (int s = 0; s < kGroup; ++s)
#pragma unroll
                for (int k = 0; k < kPix; ++k)
                    q[s][k] = bwd_update(p[k], d.ae[s][k], cg[k][s]);
            if (d.clamped) {
#pragma unroll
                for (int s = 0; s < kGroup; ++s)
#pragma unroll
                    for (int k = 0; k < kPix; ++k)
                        q[s][k].dpw = d.ae[s][k] == kAlphaMax ? 0.0f : q[s][k].dpw;
            }
            const float sum = group_sums(terms, wt, q, x0, fy, staged<float2>(st.a, own),
                                         staged<float>(st.rho, own / 4));
            if (my_value >= 0) s_part[wave][my_value][own / (int)sizeof(float4)] = sum;
        }
        __syncthreads();
        if (tid < cnt) {
            const int g = st.id[tid];
            float tot[kTerms];
            bool any = false;
#pragma unroll
            for (int k = 0; k < kTerms; ++k) {
                float acc = 0.0f;
#pragma unroll
                for (int w = 0; w < kWaves; ++w) acc += s_part[w][k][tid];
                tot[k] = acc;
                any |= acc != 0.0f;
            }
            if (any) {
                float t[kTerms];
                // the record's -cx/2 (A.z), -cy (A.w), -cz/2 (B.x), opacity (B.y)
                const float cx = -2.0f * st.a[tid].z, cy = -st.a[tid].w, cz = -2.0f * st.b[tid].x;
                const float o = st.b[tid].y, rho = st.rho[tid];
                const float r = __builtin_fmaf(-cx, rho, cy), k = __builtin_fmaf(-cy, rho, cz);
                const float S0 = tot[kS0], P1 = tot[kP1], P2 = tot[kP2];
                const float Q1 = tot[kQ1], Q2 = tot[kQ2], P5 = tot[kP5];
                t[0] = cx * P1 + r * P2;  // dL/dmean: sums of dpw wx, dpw wy
                t[1] = cy * P1 + k * P2;
                // dL/dcov2d, formed per (tile, entry) as the reference converts
                // each flushed batch (rasterize_backward.cu:211-221): what
                // cancels for a near-singular covariance then cancels at one
                // tile's magnitude instead of at the Gaussian's total
                t[2] = 0.5f * (cx * (cx * Q1 + 2.0f * r * Q2) + r * r * P5);
                t[3] = cx * (cy * Q1 + k * Q2) + r * (cy * Q2 + k * P5);
                t[4] = 0.5f * (cy * (cy * Q1 + 2.0f * k * Q2) + k * k * P5);
                t[5] = tot[kC0];                  // dL/dcolour
                t[6] = tot[kC1];
                t[7] = tot[kC2];
                // dL/dopacity: every dpw carries a factor opacity (no pixel
                // blends the entry when the opacity is 0)
                t[8] = (S0 == 0.0f) ? 0.0f : S0 / o;
                // the pair's slot: goff[g] + this tile's index in g's rectangle
                const uint2 rc = gs.rects[g];
                const int rx0 = (int)(rc.x & 0xffffu), rx1 = (int)(rc.x >> 16);
                const int ry0 = (int)(rc.y & 0xffffu), ry1 = (int)(rc.y >> 16);
                const uint64_t slot = (uint64_t)gs.goff[g] +
                                      (uint64_t)((ty - ry0) * (rx1 - rx0) + (tx - rx0));
                bool own = tx >= rx0 && tx < rx1 && ty >= ry0 && ty < ry1 && slot < gs.slots;
                if (own) {
                    // claim the slot: its flag bit.  Only an id repeated
                    // within this tile's list finds it claimed already.
                    const uint32_t bit = 1u << (uint32_t)(slot & 31u);
                    own = (atomicOr(gs.flags + (slot >> 5), bit) & bit) == 0u;
                }
                if (own) {
                    float* d = gs.sums + 9 * slot;
#pragma unroll
                    for (int k = 0; k < kTerms; ++k) d[k] = t[k];
                } else {
                    // no slot of its own (outside the rectangles, or a repeated
                    // id): straight to the outputs
                    unsafeAtomicAdd(&dmean[2 * (size_t)g], t[0]);
                    unsafeAtomicAdd(&dmean[2 * (size_t)g + 1], t[1]);
                    unsafeAtomicAdd(&dcov[3 * (size_t)g], t[2]);
                    unsafeAtomicAdd(&dcov[3 * (size_t)g + 1], t[3]);
                    unsafeAtomicAdd(&dcov[3 * (size_t)g + 2], t[4]);
                    unsafeAtomicAdd(&dcol[3 * (size_t)g], t[5]);
                    unsafeAtomicAdd(&dcol[3 * (size_t)g + 1], t[6]);
                    unsafeAtomicAdd(&dcol[3 * (size_t)g + 2], t[7]);
                    unsafeAtomicAdd(&dalpha[g], t[8]);
                }
            }
        }
    }
}

// Sum over the kLanes (16 or 8) lanes of each row, result in every lane of
// the row.
template <int kLanes>
__device__ __forceinline__ float row_sum(float x) {
    if constexpr (kLanes == 16) x += dpp_move<kDppRowRor8>(x);
    x += lane_xor4(x);
    x += dpp_move<kDppQuadXor2>(x);
    x += dpp_move<kDppQuadXor1>(x);
    return x;
}

// One row of lanes per Gaussian: the nine sums of its flagged
// slots (d mean2d, d cov2d, d colour, d opacity), added to the outputs (which
// hold zeros and any fallback atomics from the blend).
// kReduceRowLanes per Gaussian: 16, or 8 when Gaussians have few slots (half the
// waves then wait on the dependent loads).  Each lane reads the flag bits of
// kGroup consecutive slots per step: 8 (one byte) when Gaussians average a
// few hundred slots or fewer, 64 (one word) beyond, where claimed slots are
// sparse and a row then covers 1024 slots per step.
template <int kReduceRowLanes, int kGroup>
__device__ __forceinline__ void reduce_row(int n, int g, const GradSlots& gs,
                                           float* __restrict__ dmean, float* __restrict__ dcov,
                                           float* __restrict__ dcol, float* __restrict__ dalpha) {
    static_assert(kReduceRowLanes == 16 || kReduceRowLanes == 8, "rows of 16 or 8 lanes");
    static_assert(kGroup == 8 || kGroup == 64, "flag groups of 8 or 64 slots");
    const int sub = threadIdx.x & (kReduceRowLanes - 1);
    // the flag bits of slots [grp, grp + kGroup), grp a multiple of kGroup
    // (the flag array is 256-byte aligned and padded to 64-bit words)
    auto group_bits = [&](uint64_t grp) -> uint64_t {
        if constexpr (kGroup == 8)
            return reinterpret_cast<const uint8_t*>(gs.flags)[grp >> 3];
        else
            return reinterpret_cast<const uint64_t*>(gs.flags)[grp >> 6];
    };
    float v[kTerms] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    bool claimed = false;
    if (g < n) {
        const uint64_t base = gs.goff[g];
        const uint64_t end = min(base + (uint64_t)gs.counts[g], gs.slots);
        // each group's flags are loaded while the group before is summed, and
        // the sums of two flagged slots are loaded together
        uint64_t grp = (base & ~(uint64_t)(kGroup - 1)) + (uint64_t)kGroup * sub;
        uint64_t bits = (grp < end) ? group_bits(grp) : 0ull;
        while (grp < end) {
            const uint64_t nxt = grp + (uint64_t)kGroup * kReduceRowLanes;
            const uint64_t nbits = (nxt < end) ? group_bits(nxt) : 0ull;
            // only the flags of [base, end)
            if (grp < base) bits &= ~0ull << (base - grp);
            if (end - grp < (uint64_t)kGroup) bits &= ~(~0ull << (end - grp));
            claimed |= bits != 0;
            while (bits) {
                const uint64_t s0 = grp + (uint64_t)__builtin_ctzll(bits);
                bits &= bits - 1;
                const bool two = bits != 0;
                const uint64_t s1 = two ? grp + (uint64_t)__builtin_ctzll(bits) : s0;
                if (two) bits &= bits - 1;
                const float* d0 = gs.sums + 9 * s0;
                const float* d1 = gs.sums + 9 * s1;
                float a[kTerms], b[kTerms];
#pragma unroll
                for (int k = 0; k < kTerms; ++k) {
                    a[k] = d0[k];
                    b[k] = d1[k];
                }
#pragma unroll
                for (int k = 0; k < kTerms; ++k) v[k] += two ? a[k] + b[k] : a[k];
            }
            grp = nxt;
            bits = nbits;
        }
    }
    // a Gaussian without claimed slots adds nothing: its outputs are not read or
    // written, and a wave without any skips the row sums
    const uint64_t wave_claims = ballot(claimed);
    if (wave_claims == 0ull) return;
    // every lane takes part in the row sums (rows past n add zeros)
    float t[kTerms];
#pragma unroll
    for (int k = 0; k < kTerms; ++k) t[k] = row_sum<kReduceRowLanes>(v[k]);
    const uint64_t row_claims =
        (wave_claims >> (lane_id() & (64 - kReduceRowLanes))) & ((1ull << kReduceRowLanes) - 1);
    if (g < n && sub == 0 && row_claims != 0) {
        const float m0 = dmean[2 * (size_t)g], m1 = dmean[2 * (size_t)g + 1];
        const float c0 = dcov[3 * (size_t)g], c1 = dcov[3 * (size_t)g + 1],
                    c2 = dcov[3 * (size_t)g + 2];
        const float k0 = dcol[3 * (size_t)g], k1 = dcol[3 * (size_t)g + 1],
                    k2 = dcol[3 * (size_t)g + 2];
        const float a0 = dalpha[g];
        dmean[2 * (size_t)g] = m0 + t[0];
        dmean[2 * (size_t)g + 1] = m1 + t[1];
        dcov[3 * (size_t)g] = c0 + t[2];
        dcov[3 * (size_t)g + 1] = c1 + t[3];
        dcov[3 * (size_t)g + 2] = c2 + t[4];
        dcol[3 * (size_t)g] = k0 + t[5];
        dcol[3 * (size_t)g + 1] = k1 + t[6];
        dcol[3 * (size_t)g + 2] = k2 + t[7];
        dalpha[g] = a0 + t[8];
    }
}

template <int kReduceRowLanes, int kGroup>
__global__ __launch_bounds__(256) void pair_grad_reduce_kernel(
    int n, GradSlots gs, float* __restrict__ dmean, float* __restrict__ dcov,
    float* __restrict__ dcol, float* __restrict__ dalpha) {
    const int g = blockIdx.x * (256 / kReduceRowLanes) + (int)(threadIdx.x / kReduceRowLanes);
    reduce_row<kReduceRowLanes, kGroup>(n, g, gs, dmean, dcov, dcol, dalpha);
}

// The same sums where claimed slots are few: each wave looks through the claim
// bits of 16 Gaussians, four lanes and four words at a time, and only those with
// a claimed slot get a row.  In a 4K frame of 5M Gaussians (112 slots each, most
// behind opaque ones) a row per Gaussian spent 425 us almost wholly on loading
// bits that are zero; here 174 us.  8 Gaussians per wave: 204.
constexpr int kSparseGaussians = 16;  // per wave

template <int kGroup>
__global__ __launch_bounds__(256) void pair_grad_reduce_sparse_kernel(
    int n, GradSlots gs, float* __restrict__ dmean, float* __restrict__ dcov,
    float* __restrict__ dcol, float* __restrict__ dalpha) {
    const int lane = lane_id();
    const int g0 = (int)(blockIdx.x * 4u + (threadIdx.x >> 6)) * kSparseGaussians;
    const int i = g0 + (lane >> 2);
    bool any = false;
    if (i < n) {
        const uint64_t base = gs.goff[i];
        const uint64_t end = min(base + (uint64_t)gs.counts[i], gs.slots);
        const uint64_t* words = reinterpret_cast<const uint64_t*>(gs.flags);
        for (uint64_t w = (base >> 6) + (uint64_t)(lane & 3); w << 6 < end; w += 4) {
            uint64_t bits = words[w];
            if (w << 6 < base) bits &= ~0ull << (base - (w << 6));
            if (end - (w << 6) < 64u) bits &= ~(~0ull << (end - (w << 6)));
            any |= bits != 0;
        }
    }
    // bit 4 j: Gaussian g0 + j has a claimed slot
    uint64_t claimed = ballot(any);
    claimed |= claimed >> 1;
    claimed |= claimed >> 2;
    claimed &= 0x1111111111111111ull;
    while (claimed) {
        // the next four, one per 16-lane row
        int g = n;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (claimed && (lane >> 4) == r) g = g0 + (int)(__builtin_ctzll(claimed) >> 2);
            claimed &= claimed - 1;
        }
        reduce_row<16, kGroup>(n, g, gs, dmean, dcov, dcol, dalpha);
    }
}

// ---- tile scheduling: work-groups start in descending order of estimated
// work, so the longest tiles do not start last and set the kernel's tail.
// The order changes no result: every tile's pixels are computed by one
// work-group on their own. ----

// Backward work of a tile: its list entries up to the largest n_contrib
// (tile_work_bwd_wave, one wave per tile).  Run here, or by the backward
// records kernel in work-groups of its own launch.
__global__ __launch_bounds__(kWorkTilesPerBlock * kWave) void tile_work_bwd_kernel(BwdWork b) {
    const int tile = blockIdx.x * kWorkTilesPerBlock + (int)(threadIdx.x >> 6);
    if (tile >= b.T) return;  // whole waves
    tile_work_bwd_wave(b, tile);
}

// Forward work of a tile: the list entries it takes until two sample pixels
// (on the diagonal, a quarter of the way in from opposite corners) are done
// (T < 1e-4), or the whole list when one never is (the forward walks a tile's
// list until every pixel is done).  An ordering heuristic only: it uses the
// hardware exp and log and no culling.  Measured against five points and a
// 1024-entry cap, it costs less than it loses in ordering (render -5 us at
// 1080p, -11 us at 720p on the bench scene, +3 us on c3).  Ordering by list
// length alone (no walk) made the bench scene's forward blend 32 us slower;
// one centre point cost c4's blend 5 us.
constexpr int kEstPoints = 2;

// One wave per tile, 64 entries per step, the next step's ids prefetched.  A
// sample pixel still live after kEstCap entries counts as never done.  256
// orders as well as 512 and 1024 on the bench scene, c3 and c4 and walks
// less (the estimate 22 to 19 us on the bench scene); 128 orders worse.
constexpr int kEstTilesPerBlock = 4;
constexpr int kEstCap = 256;

__global__ __launch_bounds__(kEstTilesPerBlock * kWave) void tile_work_fwd_kernel(
    int T, int tiles_x, int n, uint64_t m, const int2* __restrict__ ranges,
    const int32_t* __restrict__ ids, const BlendRec* __restrict__ recs,
    uint32_t* __restrict__ work) {
    constexpr float kLnTmin = -9.21034037f;  // ln(1e-4)
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * kEstTilesPerBlock + (int)(threadIdx.x >> 6);
    if (tile >= T) return;  // whole waves
    int start, end;
    clamp_range(ranges[tile], m, start, end);
    const int len = end - start;
    const float x0 = (float)((tile % tiles_x) * kTileSize);
    const float y0 = (float)((tile / tiles_x) * kTileSize);
    const float sx[kEstPoints] = {x0 + 3.0f, x0 + 12.0f};
    const float sy[kEstPoints] = {y0 + 3.0f, y0 + 12.0f};
    float carry[kEstPoints] = {0.0f, 0.0f};
    int sat[kEstPoints] = {-1, -1};
    int next = (lane < len) ? ids[start + lane] : -1;
    for (int c = 0; c < min(len, kEstCap); c += kWave) {
        const int g = next;
        const bool ok = g >= 0 && g < n;  // false past the list end as well
        BlendRec r;
        if (ok) r = recs[g];
        next = (c + kWave + lane < len) ? ids[start + c + kWave + lane] : -1;
        bool all = true;
#pragma unroll
        for (int q = 0; q < kEstPoints; ++q) {
            float l = 0.0f;
            if (ok) {
                const float dx = sx[q] - r.a.x, dy = sy[q] - r.a.y;
                const float power = blend_power(dx, dy, r.a, r.b);
                const float alpha = fminf(kAlphaMax, r.b.y * __expf(power));
                l = (power <= 0.0f && alpha >= kAlphaMin) ? __logf(1.0f - alpha) : 0.0f;
            }
            const float incl = wave_inclusive_scan_f(l);
            const uint64_t below = ballot(c + lane < len && carry[q] + incl < kLnTmin);
            if (sat[q] < 0 && below != 0) sat[q] = c + (int)__builtin_ctzll(below);
            carry[q] += __shfl(incl, 63, kWave);
            all &= sat[q] >= 0;
        }
        if (all) break;
    }
    if (lane == 0) {
        int w = 0;
        bool open = false;
#pragma unroll
        for (int q = 0; q < kEstPoints; ++q) {
            if (sat[q] < 0) open = true;
            else w = max(w, sat[q] + 1);
        }
        work[tile] = (uint32_t)(open ? len : w);
    }
}

// 256 buckets, ordered like the value: 5-bit exponent, 3-bit mantissa.
__device__ __forceinline__ uint32_t work_bucket(uint32_t w) {
    if (w == 0) return 0;
    const uint32_t e = 31u - (uint32_t)__builtin_clz(w);
    const uint32_t mant = (e >= 3) ? (w >> (e - 3)) & 7u : (w << (3 - e)) & 7u;
    return min(255u, e * 8u + mant + 1u);
}

constexpr int kOrderThreads = 1024;
constexpr int kOrderHeld = 8;  // 8192 tiles held in registers (1080p: 8160)
constexpr uint32_t kSplitBuckets = 5;
constexpr uint32_t kSplitMinWork = 256;
// A tile alone on a CU runs at roughly a quarter of the CU's rate.
constexpr uint64_t kSplitLoad = 4;

// order[i] = tiles by descending work bucket (one work-group); with split_max
// >= 0 also order[T], the backward's split count (below).  work == null:
// the forward's estimate, the tile's list length.
__global__ __launch_bounds__(kOrderThreads) void tile_order_kernel(
    int T, uint64_t m, const int2* __restrict__ ranges, const uint32_t* __restrict__ work,
    uint32_t* __restrict__ order, int split_max, int cus) {
    __shared__ uint32_t s_cnt[256];
    __shared__ uint32_t s_scan[4];
    __shared__ uint32_t s_top;
    __shared__ unsigned long long s_sum;
    __shared__ uint32_t s_wmax;
    const int tid = threadIdx.x;
    auto work_of = [&](int t) -> uint32_t {
        if (work) return work[t];
        int start, end;
        clamp_range(ranges[t], m, start, end);
        return (uint32_t)(end - start);
    };
    auto bucket = [](uint32_t w) -> uint32_t { return 255u - work_bucket(w); };  // descending
    auto bucket_of = [&](int t) -> uint32_t { return bucket(work_of(t)); };
    if (tid < 256) s_cnt[tid] = 0;
    if (tid == 0) {
        s_sum = 0ull;
        s_wmax = 0u;
    }
    // the first kOrderHeld tiles per thread are read once, all loads in
    // flight together, and their work kept for the scatter
    auto held_tile = [&](int i) { return tid + i * kOrderThreads; };
    uint32_t held[kOrderHeld];
#pragma unroll
    for (int i = 0; i < kOrderHeld; ++i) {
        const int t = held_tile(i);
        held[i] = (t < T) ? work_of(t) : 0u;
    }
    __syncthreads();
    uint64_t wsum = 0;
    uint32_t wmax = 0;
#pragma unroll
    for (int i = 0; i < kOrderHeld; ++i) {
        if (held_tile(i) < T) atomicAdd(&s_cnt[bucket(held[i])], 1u);
        wsum += held[i];
        wmax = max(wmax, held[i]);
    }
    for (int t = tid + kOrderHeld * kOrderThreads; t < T; t += kOrderThreads) {
        const uint32_t w = work_of(t);
        atomicAdd(&s_cnt[bucket(w)], 1u);
        wsum += w;
        wmax = max(wmax, w);
    }
    if (split_max > 0) {
        // one atomic per wave
        const uint64_t ws = wave_sum_u64(wsum);
        const uint32_t wm = wave_max_u32(wmax);
        if ((tid & 63) == 0) {
            atomicAdd(&s_sum, (unsigned long long)ws);
            atomicMax(&s_wmax, wm);
        }
    }
    __syncthreads();
    uint32_t c = 0, inc = 0;
    if (tid < 256) {
        c = s_cnt[tid];
        inc = wave_inclusive_scan(c);
        if ((tid & 63) == 63) s_scan[tid >> 6] = inc;
    }
    __syncthreads();
    if (tid < 256) {
        uint32_t pre = 0;
        for (int w = 0; w < (tid >> 6); ++w) pre += s_scan[w];
        s_cnt[tid] = pre + inc - c;  // first slot of the bucket
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOrderHeld; ++i) {
        const int t = held_tile(i);
        if (t < T) {
            const uint32_t pos = atomicAdd(&s_cnt[bucket(held[i])], 1u);
            if (pos < (uint32_t)T) order[pos] = (uint32_t)t;
        }
    }
    for (int t = tid + kOrderHeld * kOrderThreads; t < T; t += kOrderThreads) {
        const uint32_t pos = atomicAdd(&s_cnt[bucket_of(t)], 1u);
        if (pos < (uint32_t)T) order[pos] = (uint32_t)t;
    }
    if (split_max == 0 && tid == 0) order[T] = 0u;
    if (split_max > 0) {
        // order[T] = how many of the first tiles the backward splits: those
        // within kSplitBuckets sub-buckets (a factor 2^(5/8) ~ 1.5) of the
        // longest, if it has kSplitMinWork entries or more and a long tail
        // (below).  s_cnt[b] now holds the end of bucket b, so the first
        // non-zero one is the top.
        if (tid == 0) s_top = 256u;
        __syncthreads();
        if (tid < 256 && s_cnt[tid] > 0u) atomicMin(&s_top, (uint32_t)tid);
        __syncthreads();
        if (tid == 0) {
            const uint32_t top = s_top;
            uint32_t k = 0;
            // only when the longest tile outlasts the balanced share of the
            // work: kSplitLoad x its work x the CUs against the total
            const bool tail = (uint64_t)s_wmax * (uint64_t)max(cus, 1) * kSplitLoad >= s_sum;
            if (tail && top < 256u && 255u - top >= work_bucket(kSplitMinWork))
                k = min(s_cnt[min(top + kSplitBuckets, 255u)], (uint32_t)split_max);
            order[T] = k;
        }
    }
}

// Splitting the backward's longest tiles in two (on unless GSR_BWD_SPLIT=0;
// read on every call, so a test can compare both).
bool bwd_split() {
    const char* v = std::getenv("GSR_BWD_SPLIT");
    return !(v && v[0] == '0');
}

// Per-device launch facts, looked up once per device and kept in a fixed
// table (no allocation after the first call): the compute units, and how many
// work-groups of the 64-entry-batch backward kernel fit on the device at once.
constexpr int kMaxDevices = 64;
struct DeviceFacts {
    int cus = 0;
    unsigned fwd_resident = 0;
    unsigned bwd_resident = 0;
};
DeviceFacts device_facts() {
    static std::mutex mu;
    static DeviceFacts table[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return DeviceFacts{1, 1, 1};
    std::lock_guard<std::mutex> lock(mu);
    DeviceFacts& f = table[dev];
    if (f.cus == 0) {
        int per_cu = 0, fwd_per_cu = 0, cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, reinterpret_cast<const void*>(&blend_bwd_kernel<2, 64, false>),
                Layout<2>::kThreads, 0) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &fwd_per_cu, reinterpret_cast<const void*>(&blend_fwd_kernel<2>),
                Layout<2>::kThreads, 0) != hipSuccess)
            return DeviceFacts{1, 1, 1};
        f.cus = std::max(1, cus);
        f.fwd_resident = (unsigned)std::max(1, fwd_per_cu * f.cus);
        f.bwd_resident = (unsigned)std::max(1, per_cu * f.cus);
    }
    return f;
}

int cu_count() { return device_facts().cus; }

// Whether the forward's whole grid of tiles, two pixels per lane, is resident
// on the device at once.
bool fwd_grid_fits(unsigned tiles) { return tiles <= device_facts().fwd_resident; }

// Whether the backward's grid of tiles is resident on the device at once, or
// so nearly (4/3 of what fits: 4096 tiles) that its longest tiles set its
// length and the 128-entry batch with the split pays: 256x256 76 us so and 110
// with 64-entry batches, 720p (3600 tiles) 122 and 127, 1080p (8160 tiles) 215 and
// 214, with a million Gaussians 276 and 266.
bool bwd_grid_fits(unsigned tiles) {
    return (uint64_t)tiles * 3 <= (uint64_t)device_facts().bwd_resident * 4;
}

// Lists that average this many entries per tile or more (the screen bands of
// config c5 average ~350k) are walked like a resident grid's: 128-entry
// batches with the longest tiles split.  Their longest tiles set the kernel's
// length there (blend_bwd 4.14 ms per frame with 64-entry batches, 3.84 so), while
// the 64-entry batch without the split stays ahead at 1080p (1.6k entries per
// tile) and for the 4K needles of the depth-prefix frame (11k): 266 us against
// 276, 2.45 ms against 2.62.
constexpr uint64_t kLongListAvg = 32768;
bool bwd_long_lists(unsigned tiles, uint64_t pairs) {
    return pairs >= kLongListAvg * (uint64_t)tiles;
}

// Whether the backward walks 128-entry batches and may split long tiles.
bool bwd_wide(unsigned tiles, uint64_t pairs) {
    return bwd_grid_fits(tiles) || bwd_long_lists(tiles, pairs);
}

}  // namespace

hipError_t launch_fwd_schedule(int n, int H, int W, const int32_t* ranges, const int32_t* ids,
                               uint64_t m, const void* recs, uint32_t* work, uint32_t* order,
                               hipStream_t st) {
    const int tiles_x = (W + kTileSize - 1) / kTileSize;
    const unsigned tiles = (unsigned)(tiles_x * ((H + kTileSize - 1) / kTileSize));
    if (tiles == 0) return hipSuccess;
    const auto* r = reinterpret_cast<const int2*>(ranges);
    hipLaunchKernelGGL(tile_work_fwd_kernel,
                       dim3((tiles + kEstTilesPerBlock - 1) / kEstTilesPerBlock),
                       dim3(kEstTilesPerBlock * kWave), 0, st, (int)tiles, tiles_x, n, m, r, ids,
                       static_cast<const BlendRec*>(recs), work);
    hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(kOrderThreads), 0, st, (int)tiles, m, r,
                       work, order, -1, 1);
    return hipGetLastError();
}

hipError_t launch_blend_fwd(int n, int H, int W, const int32_t* ranges, const int32_t* ids,
                            uint64_t m, const void* recs, float* img, float* finalT,
                            int32_t* ncontrib, const uint32_t* order, hipStream_t st) {
    const int tiles_x = (W + kTileSize - 1) / kTileSize;
    const int tiles_y = (H + kTileSize - 1) / kTileSize;
    const unsigned tiles = (unsigned)(tiles_x * tiles_y);
    if (tiles == 0) return hipSuccess;
    const auto* r = reinterpret_cast<const int2*>(ranges);
    const auto* rc = static_cast<const BlendRec*>(recs);
    // Two pixels per lane share each entry's record reads, column terms and
    // loop, which pays when the total work sets the kernel's length (1080p:
    // 135.4 -> 129.6 us with a step per entry).  Where the longest tiles set it (a grid resident at
    // once, or lists averaging 32k entries per tile), one pixel per lane in
    // four 16x4 strips culls finer and exits sooner per wave (720p bench frame
    // 0.4615 ms with two pixels per lane against 0.430; c5's blend_fwd 4.86
    // against 4.3 ms per frame).
    if (fwd_grid_fits(tiles) || bwd_long_lists(tiles, m))
        hipLaunchKernelGGL(blend_fwd_kernel<1>, dim3(tiles), dim3(Layout<1>::kThreads), 0, st,
                           n, H, W, tiles_x, m, r, ids, rc, img, finalT, ncontrib, order);
    else
        hipLaunchKernelGGL(blend_fwd_kernel<2>, dim3(tiles), dim3(Layout<2>::kThreads), 0, st,
                           n, H, W, tiles_x, m, r, ids, rc, img, finalT, ncontrib, order);
    return hipGetLastError();
}

hipError_t launch_bwd_schedule(int H, int W, const int32_t* ranges, uint64_t num_pairs,
                               const int32_t* ncontrib, uint32_t* work, uint32_t* order,
                               hipStream_t st, bool work_ready) {
    const int tiles_x = (W + kTileSize - 1) / kTileSize;
    const unsigned tiles = (unsigned)(tiles_x * ((H + kTileSize - 1) / kTileSize));
    if (tiles == 0) return hipSuccess;
    const auto* r = reinterpret_cast<const int2*>(ranges);
    if (!work_ready)
        hipLaunchKernelGGL(tile_work_bwd_kernel,
                           dim3((tiles + kWorkTilesPerBlock - 1) / kWorkTilesPerBlock),
                           dim3(kWorkTilesPerBlock * kWave), 0, st,
                           make_bwd_work(H, W, ranges, num_pairs, ncontrib, work));
    hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(kOrderThreads), 0, st, (int)tiles,
                       num_pairs, r, work, order,
                       (bwd_split() && bwd_wide(tiles, num_pairs)) ? kSplitMax : 0,
                       cu_count());
    return hipGetLastError();
}

hipError_t launch_blend_bwd(int n, int H, int W, const float* grad, const GradStrides& gst,
                            const int32_t* ranges,
                            const int32_t* ids, uint64_t num_pairs, const void* recs,
                            const float* finalT, const int32_t* ncontrib, float* dmean,
                            float* dcov, float* dcol, float* dalpha, const GradSlots& gs,
                            const uint32_t* order, hipStream_t st) {
    const int tiles_x = (W + kTileSize - 1) / kTileSize;
    const int tiles_y = (H + kTileSize - 1) / kTileSize;
    const unsigned tiles = (unsigned)(tiles_x * tiles_y);
    if (tiles == 0) return hipSuccess;
    const auto* r = reinterpret_cast<const int2*>(ranges);
    const auto* rc = static_cast<const BlendRec*>(recs);
    // With a schedule and the grid (nearly) resident at once, or lists long
    // enough that the longest tiles set the kernel's length, up to kSplitMax
    // of the longest run as two items each.  Otherwise the total work does,
    // and the split's extra state-only walk costs more than it saves.
    const bool wide = bwd_wide(tiles, num_pairs);
    const bool split = order && bwd_split() && wide;
    // The 64-entry batch takes 12.3 KB of LDS and 80 registers (6 waves per SIMD,
    // 12 work-groups per CU); it pays when the grid does not fit on the device
    // at once.  When it would, the 128-entry batch (20 KB) leaves part of the
    // grid to be placed as CUs free up, which balances the long tiles better.
    if (!wide)
        hipLaunchKernelGGL((blend_bwd_kernel<2, 64, false>), dim3(tiles),
                           dim3(Layout<2>::kThreads), 0, st, n, H, W, tiles_x, num_pairs, grad, gst,
                           r, ids, rc, finalT, ncontrib, dmean, dcov, dcol, dalpha, gs, order);
    else if (split)
        hipLaunchKernelGGL((blend_bwd_kernel<2, 128, true>), dim3(tiles + kSplitMax),
                           dim3(Layout<2>::kThreads), 0, st, n, H, W, tiles_x, num_pairs, grad, gst,
                           r, ids, rc, finalT, ncontrib, dmean, dcov, dcol, dalpha, gs, order);
    else
        hipLaunchKernelGGL((blend_bwd_kernel<2, 128, false>), dim3(tiles),
                           dim3(Layout<2>::kThreads), 0, st, n, H, W, tiles_x, num_pairs, grad, gst,
                           r, ids, rc, finalT, ncontrib, dmean, dcov, dcol, dalpha, gs, order);
    return hipGetLastError();
}

hipError_t launch_pair_grad_reduce(int n, const GradSlots& gs, float* dmean, float* dcov,
                                   float* dcol, float* dalpha, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    // 8-lane rows when a Gaussian averages at most 64 slots (one flag load per
    // lane); word-sized flag groups beyond 256 slots per Gaussian.  Beyond 64
    // slots, from 2^19 Gaussians on (2^15 waves of the sparse kernel, four times
    // what the chip holds), a tile's list averages over 1000 entries at 4K: mostly
    // they end behind what hides them, and the sparse kernel is the faster, 51
    // against 72 us (600k Gaussians of 78 slots, opacity 0.5) and 174 against
    // 425.  A cloud faint enough to be seen through is summed 5% slower, 284
    // against 264 us (600k of opacity 0.02), 337 against 313 (0.05), 450 against
    // 428 (540k wider ones), as its waves, four times as long, end less evenly:
    // 0.2% of those frames (13 ms and more); which of them a frame is, only the
    // blend knows.
    if (gs.slots <= 64ull * (uint64_t)n)
        hipLaunchKernelGGL((pair_grad_reduce_kernel<8, 8>), dim3((unsigned)((n + 31) / 32)),
                           dim3(256), 0, st, n, gs, dmean, dcov, dcol, dalpha);
    else if (n >= (1 << 19) && gs.slots <= 256ull * (uint64_t)n)
        hipLaunchKernelGGL((pair_grad_reduce_sparse_kernel<8>), dim3((unsigned)((n + 63) / 64)),
                           dim3(256), 0, st, n, gs, dmean, dcov, dcol, dalpha);
    else if (n >= (1 << 19))
        hipLaunchKernelGGL((pair_grad_reduce_sparse_kernel<64>), dim3((unsigned)((n + 63) / 64)),
                           dim3(256), 0, st, n, gs, dmean, dcov, dcol, dalpha);
    else if (gs.slots <= 256ull * (uint64_t)n)
        hipLaunchKernelGGL((pair_grad_reduce_kernel<16, 8>), dim3((unsigned)((n + 15) / 16)),
                           dim3(256), 0, st, n, gs, dmean, dcov, dcol, dalpha);
    else
        hipLaunchKernelGGL((pair_grad_reduce_kernel<16, 64>), dim3((unsigned)((n + 15) / 16)),
                           dim3(256), 0, st, n, gs, dmean, dcov, dcol, dalpha);
    return hipGetLastError();
}

}  // namespace gsr
