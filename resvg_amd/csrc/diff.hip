// The differentiable f32 form of the pixel pipeline: a forward renderer and
// hand-written adjoint kernels for the scene model below, for one scene or a stack
// of equally shaped scenes.  Everything is f32, premultiplied RGBA; a thread takes one
// pixel, in the blurs four or eight.
//
// Model (the reference's operations restated in f32, resvg 0.48.1):
//   * path i covers pixel p with c_i(p): either coverage_u8 / 255, the anti-aliased
//     coverage of its outline (tiny-skia fill_path, path.rs:26-75) computed by the
//     u8 rasterizer and fixed (no gradient to the geometry), or, in the analytic
//     mode, min(1, |∫ winding|) over the pixel of the path's flattened cubics mapped
//     by its affine transform, whose gradient flows to the control points and the
//     transform through the boundary term;
//   * its paint is a pad-spread linear gradient (path.rs:118-177) along
//     (x0, y0) -> (x1, y1) with 4 stops (offset, unpremultiplied RGBA), times a
//     per-path RGB tint, times a per-path opacity (the group opacity of
//     render.rs:133); the premultiplied source is (rgb·tint·A, A), A = c·opacity·a;
//   * paths composite with SourceOver in order onto a transparent canvas S;
//   * the filter chain is feGaussianBlur (a separable Gaussian of radius
//     ceil(3σ), at most kMaxRadius, zero outside the image) -> feColorMatrix (4x5
//     on the demultiplied colour, clamped, premultiplied; color_matrix.rs:11-110)
//     -> composite over SourceGraphic (filter/mod.rs:731-793): out = F + (1 - F_a)·S.
//
// Parameters (f32, device): per path kDiffPathParams values (tint r, g, b;
// opacity; 4 stop colours r, g, b, a; 4 stop offsets), then σ, then the 20 matrix
// entries.  Gradients come in the same layout.
//
// Checkpointing: the forward stores the canvas before every kSeg-th path and the
// blur intermediates; the backward recomputes each segment of kSeg paths per pixel
// in registers and walks it in reverse.  Parameter gradients are summed per block
// into partial rows and reduced by a second kernel, so they are deterministic.
#include "rvk_internal.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int kSeg = 8;          // paths per checkpoint segment
constexpr int kThreads = 1024;   // pixels per block (one thread each)
constexpr int kWaves = kThreads / 64;
constexpr int kMaxRadius = 48;   // 3 * the largest σ the model accepts (16)
constexpr int kPP = RVK_DIFF_PATH_PARAMS;
constexpr int kGlobalParams = 1 + 20;  // σ, matrix

struct Dims {
    uint32_t w, h, n;        // width, height, paths
    uint32_t nblk;           // blocks of the per-pixel kernels
    uint32_t tx, ntile;      // pixel squares of the path kernels: per row of squares, in all
    uint32_t k;              // cubics per path (analytic mode), else 0
    size_t ws;               // workspace bytes per scene
    float qscale;            // analytic mode: fixed-point scale of the area accumulation
};

// A batch holds scenes of one shape, stacked: scene blockIdx.y finds its parameters,
// geometry, gradient ends, coverage planes, workspace and images at blockIdx.y times
// the per-scene size of each (a null pointer stays null).
// (char arithmetic, not an integer round trip, so that the compiler keeps the
// pointer in the global address space: scalar loads for uniform values)
template <class T> __device__ __forceinline__ T *scene_at(T *p, size_t bytes) {
    using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return reinterpret_cast<T *>(reinterpret_cast<B *>(p) + (size_t)blockIdx.y * bytes);
}
// the same for a pointer that may be null (an optional buffer)
template <class T> __device__ __forceinline__ T *scene_of(T *p, size_t bytes) {
    return p ? scene_at(p, bytes) : p;
}
__device__ __forceinline__ size_t params_bytes(const Dims &d) {
    return ((size_t)d.n * kPP + kGlobalParams) * sizeof(float);
}
__device__ __forceinline__ size_t geom_bytes(const Dims &d) {
    return (size_t)d.n * (6 + 2 * (3 * d.k + 1)) * sizeof(float);
}
__device__ __forceinline__ size_t image_bytes(const Dims &d) { return (size_t)d.w * d.h * sizeof(float4); }

// Where the coverage of path i at pixel p comes from: u8 planes (coverage / 255), or
// the winding-area planes of the analytic mode (coverage min(1, |area|); row stride
// w + 2, see k_diff_accum).  In the analytic mode the backward also writes
// dL/d(area) per path and pixel into gW.
struct Cov {
    const uint8_t *u8;
    const float *area;
    float *gW;
};
__device__ __forceinline__ Cov scene_cov(const Cov &cv, const Dims &d) {
    return Cov{scene_of(cv.u8, (size_t)d.n * d.w * d.h), scene_of(cv.area, d.ws), scene_of(cv.gW, d.ws)};
}
// ---- the path kernels' pixels -------------------------------------------------
// A block of 4 waves covers a 64 x 4 pixel rectangle, each wave 16 x 4 of it (not 64 x 1: a
// path's outline then crosses a third of the waves, and a wave's pixels mostly share a
// stop interval).  Four such blocks share a CU, so the barriers and the loads at a
// segment's start hold up one of them, not the CU's only block.
constexpr int kSquareW = 64, kSquareH = 4, kWaveW = 16, kWaveH = 4;
constexpr int kPathThreads = kSquareW * kSquareH, kPathWaves = kPathThreads / 64;
static_assert(kWaveW * kWaveH == 64 && kPathThreads % 64 == 0, "a thread per pixel");
struct Pixel {
    uint32_t x, y;
    size_t p;
    bool live;
};
__device__ __forceinline__ Pixel square_pixel(const Dims &d) {
    const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    Pixel q;
    q.x = blockIdx.x % d.tx * kSquareW + wave % (kSquareW / kWaveW) * kWaveW + lane % kWaveW;
    q.y = blockIdx.x / d.tx * kSquareH + wave / (kSquareW / kWaveW) * kWaveH + lane / kWaveW;
    q.live = q.x < d.w && q.y < d.h;
    q.p = (size_t)q.y * d.w + q.x;
    return q;
}

__device__ __forceinline__ size_t area_index(const Dims &d, uint32_t i, const Pixel &q) {
    return ((size_t)i * d.h + q.y) * (d.w + 2) + q.x;
}
// The segment's coverage at a pixel (0 past the last path and outside the image) and, in
// the analytic mode, its signed winding areas; the loads are issued together.
template <bool kArea>
__device__ __forceinline__ void segment_coverage(const Cov &cv, const Dims &d, uint32_t i0, const Pixel &q,
                                                 float (&cov)[kSeg], float (&area)[kSeg]) {
    float raw[kSeg];
    const size_t at = q.live ? (kArea ? area_index(d, i0, q) : (size_t)i0 * d.w * d.h + q.p) : 0;
    const size_t step = kArea ? (size_t)d.h * (d.w + 2) : (size_t)d.w * d.h;
#pragma unroll
    for (int j = 0; j < kSeg; j++) {
        const size_t o = i0 + j < d.n ? at + j * step : 0;  // the last segment may be short
        raw[j] = kArea ? cv.area[o] : (float)cv.u8[o];
    }
#pragma unroll
    for (int j = 0; j < kSeg; j++) {
        const bool on = q.live & (i0 + j < d.n);
        area[j] = kArea && on ? raw[j] : 0.0f;
        cov[j] = !on ? 0.0f : (kArea ? fminf(1.0f, fabsf(raw[j])) : raw[j] * (1.0f / 255.0f));
    }
}

// ---- paint ------------------------------------------------------------------
// What the path kernels read of a path, in scalar registers (written by k_diff_prepare): the
// gradient's start and direction, its squared length and that one's reciprocal, tint,
// opacity and offsets; `one`, whether the wave may draw it by one interval's record; then per
// stop interval its lower offset, width, the width's reciprocal and the two stops.
struct Interval {
    float lo, span, rs, pad;
    float c0[4], c1[4];
};
struct PathHead {
    float x0, y0, dx, dy, dd, rdd, opacity, tint[3], o0, o1, o2, o3, one, pad;
};
struct PathRec {
    PathHead head;
    Interval iv[3];
};
__device__ __forceinline__ float scalar(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}
// A uniform record by scalar loads: in the constant address space (nothing writes it during
// the kernel) whatever the kernel stores between them, and each value by readfirstlane, as
// the compiler turns a choice between two loaded values into one vector load at a chosen
// address.
template <class T> __device__ __forceinline__ T scalar_rec(const T *p) {
    typedef const float __attribute__((address_space(4))) *Constant;
    const uintptr_t at = (uintptr_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32));
    const Constant f = (Constant)((uintptr_t)hi << 32 | lo);
    T r;
    float *o = reinterpret_cast<float *>(&r);
#pragma unroll
    for (size_t k = 0; k < sizeof(T) / sizeof(float); k++) o[k] = scalar(f[k]);
    return r;
}
// 1 / d for div_by, 0 where d is too small or large for it (or not a width at all)
__device__ __forceinline__ float div_ready(float d) { return d > 0x1p-60f && d < 0x1p60f ? 1.0f / d : 0.0f; }
// n / d by the rounded reciprocal r and one exact residual (Markstein): the quotient that
// the division rounds to, in 3 operations instead of 10; q must not overflow
__device__ __forceinline__ float div_by(float n, float d, float r) {
    const float q = n * r;
    return fmaf(fmaf(-q, d, n), r, q);
}

// Where a wave's pixels lie along a path's gradient: t, and as lane masks whether t is past
// offsets 1 and 2 (the stop interval is 0, 1 or 2) and strictly inside the stops.  Before the
// first stop the interval is 0 at u = 0, after the last 2 at u = 1.
struct Along {
    float t;
    uint64_t past1, past2, inside;
};
__device__ __forceinline__ Along along_path(const PathHead &h, float px, float py) {
    Along e;
    const float num = fmaf(px - h.x0, h.dx, (py - h.y0) * h.dy);
    float t = 0.0f;
    if (h.rdd != 0.0f) t = div_by(num, h.dd, h.rdd);  // uniform
    else if (h.dd > 0.0f) t = num / h.dd;
    t = fminf(fmaxf(t, 0.0f), 1.0f);
    e.t = t;
    const uint64_t before = __ballot(t <= h.o0), after = ~before & __ballot(t >= h.o3);
    e.past1 = ~before & (after | __ballot(!(t < h.o1)));  // not below: also where an offset is a NaN
    e.past2 = e.past1 & (after | __ballot(!(t < h.o2)));
    e.inside = __ballot(t > h.o0) & __ballot(t < h.o3);
    return e;
}
// Whether the covered pixels of the wave (touched, not none) share a stop interval, k0, and
// the path's record is one for it: widths that div_by takes, and paint whose products with
// a zero coverage are zeros (a non-finite value would reach the uncovered pixels, which
// only the form for several intervals keeps apart).
__device__ __forceinline__ bool one_interval(const PathHead &h, const Along &e, uint64_t touched, int &k0) {
    const uint64_t a = e.past1 & touched, b = e.past2 & touched;
    k0 = __builtin_amdgcn_readfirstlane(b != 0 ? 2 : (a != 0 ? 1 : 0));
    return (a == 0 || a == touched) && (b == 0 || b == touched) && h.one != 0.0f;
}

// A pixel's stop colour (unpremultiplied) and where it lies between the stops.
struct Stop {
    float rgba[4];
    float u;
};
// the wave's pixels in one interval: outside the stops the quotient leaves [0, 1]
__device__ __forceinline__ Stop stop_in(const Interval &iv, float t) {
    Stop s;
    s.u = fminf(fmaxf(div_by(t - iv.lo, iv.span, iv.rs), 0.0f), 1.0f);
    const float v = 1.0f - s.u;
#pragma unroll
    for (int ch = 0; ch < 4; ch++) s.rgba[ch] = fmaf(s.u, iv.c1[ch], v * iv.c0[ch]);
    return s;
}
// pixels of several intervals, or an interval without width
__device__ __forceinline__ int lane_interval(const Along &e, int lane) {
    return (e.past2 >> lane) & 1 ? 2 : ((e.past1 >> lane) & 1 ? 1 : 0);
}
__device__ __noinline__ Stop stop_any(const PathRec *rec, int k, float t, float o0, float o3) {
    const Interval &iv = rec->iv[k];
    Stop s;
    s.u = t <= o0 ? 0.0f : (t >= o3 ? 1.0f : (iv.span > 0.0f ? (t - iv.lo) / iv.span : 0.0f));
    const float v = 1.0f - s.u;
    for (int ch = 0; ch < 4; ch++) s.rgba[ch] = fmaf(s.u, iv.c1[ch], v * iv.c0[ch]);
    return s;
}

// SourceOver of the path at coverage c (0: s unchanged); `touched`: the wave's covered
// pixels, not none
__device__ __forceinline__ float4 draw_path(const PathRec *rec, const PathHead &h, float c, uint64_t touched, float px,
                                            float py, float4 s, int lane) {
    const Along e = along_path(h, px, py);
    int k0;
    Stop st;
    if (one_interval(h, e, touched, k0)) st = stop_in(scalar_rec(&rec->iv[k0]), e.t);
    else st = stop_any(rec, lane_interval(e, lane), e.t, h.o0, h.o3);
    const float A = c * h.opacity * st.rgba[3], ia = 1.0f - A;
    const float4 o = make_float4(fmaf(ia, s.x, st.rgba[0] * h.tint[0] * A), fmaf(ia, s.y, st.rgba[1] * h.tint[1] * A),
                                 fmaf(ia, s.z, st.rgba[2] * h.tint[2] * A), fmaf(ia, s.w, A));
    return c != 0.0f ? o : s;
}

__device__ __forceinline__ float wave_sum(float v) {
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// Sums 32 values over the 64 lanes of a wave with a halving butterfly: at each step
// a lane keeps half of its values and adds a partner lane's copy of that half, so
// 16 + 8 + 4 + 2 + 1 exchanges and one final one replace 32 full reductions.  The
// exchanges stay in registers (no LDS): v_permlane16_swap pairs the 16-lane rows
// (values i and 16 + i), then DPP row rotations by 1, 2, 4 and 8 pair, within each
// row, the lanes with that lane bit clear with those with it set (a bijection that
// keeps the lower lane bits, which already select the values a lane holds), and
// v_permlane32_swap adds the two halves of the wave.  Returns, in every lane, the
// wave sum of value (lane & 31).
template <int N>
__device__ __forceinline__ float row_ror(float x) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x120 + N, 0xf, 0xf, false));
}
template <int B, int M>  // lane bit B in {1, 2, 4, 8}: M values in, M / 2 out
__device__ __forceinline__ void halve_row(const float (&v)[M], float (&o)[M / 2], bool up) {
#pragma unroll
    for (int k = 0; k < M / 2; k++) {
        const float lo = v[2 * k] + row_ror<B>(v[2 * k]);
        const float hi = v[2 * k + 1] + row_ror<B>(v[2 * k + 1]);
        o[k] = up ? hi : lo;
    }
}
__device__ __forceinline__ float wave_sum32(const float (&v)[32], int lane) {
    float a[16], b[8], c[4], d[2], e[1];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        // rows 0 and 2 end with value i, rows 1 and 3 with value 16 + i
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[16 + i]), false, false);
        a[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    halve_row<1, 16>(a, b, (lane & 1) != 0);
    halve_row<2, 8>(b, c, (lane & 2) != 0);
    halve_row<4, 4>(c, d, (lane & 4) != 0);
    halve_row<8, 2>(d, e, (lane & 8) != 0);
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(e[0]), __float_as_uint(e[0]), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The same for 16 values: lane l returns the sum of value (l & 7) + 8 * (bit 4 of l).
__device__ __forceinline__ float wave_sum16(const float (&v)[16], int lane) {
    float a[8], b[4], c[2], d[1];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[8 + i]), false, false);
        a[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    halve_row<1, 8>(a, b, (lane & 1) != 0);
    halve_row<2, 4>(b, c, (lane & 2) != 0);
    halve_row<4, 2>(c, d, (lane & 4) != 0);
    const float e = d[0] + row_ror<8>(d[0]);
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(e), __float_as_uint(e), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Inclusive sum over the wave's lanes (wrapping), in six DPP additions.
template <int CTRL, int ROWS>
__device__ __forceinline__ int add_dpp(int v) {
    return (int)((uint32_t)v + (uint32_t)__builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ int wave_prefix(int v) {
    v = add_dpp<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
    v = add_dpp<0x112, 0xf>(v);
    v = add_dpp<0x114, 0xf>(v);
    v = add_dpp<0x118, 0xf>(v);
    v = add_dpp<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    return add_dpp<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}

// ---- forward: paths -----------------------------------------------------------
// Bound by the latency of its loads more than by the VALU, so the next path's record is
// loaded while a path is drawn, a segment's coverage at once, and a CU holds several blocks.
// 1024^2, 256 paths: 0.50 -> 0.31 ms (VALU 36% busy before); 16 scenes of 512^2 with 128
// paths of analytic coverage 1.45 -> 0.86 ms.
template <bool kArea>
__global__ __launch_bounds__(kPathThreads) void k_diff_paths_fwd(Dims d, Cov cv, const PathRec *__restrict__ rec,
                                                                 float4 *canvas, float4 *ck) {
    cv = scene_cov(cv, d);
    rec = scene_at(rec, d.ws);
    canvas = scene_at(canvas, d.ws);
    ck = scene_at(ck, d.ws);
    const size_t np = (size_t)d.w * d.h;
    const Pixel q = square_pixel(d);
    const int lane = (int)(threadIdx.x % 64);
    const float px = (float)q.x + 0.5f, py = (float)q.y + 0.5f;
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    PathHead next = scalar_rec(&rec->head);
    for (uint32_t i0 = 0; i0 < d.n; i0 += kSeg) {
        if (q.live) ck[(size_t)(i0 / kSeg) * np + q.p] = s;
        float c[kSeg], area[kSeg];
        segment_coverage<kArea>(cv, d, i0, q, c, area);
#pragma unroll
        for (int j = 0; j < kSeg; j++) {
            const PathHead h = next;
            next = scalar_rec(&rec[min(i0 + j + 1, d.n - 1)].head);
            const uint64_t touched = __ballot(c[j] != 0.0f);
            if (touched != 0) s = draw_path(rec + i0 + j, h, c[j], touched, px, py, s, lane);
        }
    }
    if (q.live) canvas[q.p] = s;
}

// ---- blur weights from σ (block 0) and the paths' records (the other blocks) ----
// wts[0] = R (as a float), then w_k and, kWeightSpan further, dw_k/dσ for k = -R .. R, each
// between kWeightPad zeros, with w_k = g_k / Σg, g_k = exp(-k² / (2σ²)), σ clamped to
// [0.05, 16]; dw_k/dσ = w_k (k² - Σ_j w_j j²) / σ³.
constexpr int kWeightPad = 8, kWeightSpan = 2 * kMaxRadius + 1 + 2 * kWeightPad;
__global__ void k_diff_prepare(Dims d, const float *params, const float4 *ends, float *wts, PathRec *rec) {
    __shared__ float g[2 * kMaxRadius + 1];
    __shared__ float sums[2];
    params = scene_at(params, params_bytes(d));
    if (blockIdx.x > 0) {
        ends = scene_at(ends, (size_t)d.n * sizeof(float4));
        rec = scene_at(rec, d.ws);
        const uint32_t i = (blockIdx.x - 1) * blockDim.x + threadIdx.x;
        if (i >= d.n) return;
        const float4 e = ends[i];
        const float *pp = params + (size_t)i * kPP, *off = pp + 20;
        PathRec r;
        PathHead &h = r.head;
        h.x0 = e.x;
        h.y0 = e.y;
        h.dx = e.z - e.x;
        h.dy = e.w - e.y;
        h.dd = h.dx * h.dx + h.dy * h.dy;
        h.rdd = div_ready(h.dd);
        for (int k = 0; k < 3; k++) h.tint[k] = pp[k];
        h.opacity = pp[3];
        h.o0 = off[0];
        h.o1 = off[1];
        h.o2 = off[2];
        h.o3 = off[3];
        h.one = 1.0f;
        for (int k = 0; k < 20; k++)
            if (!(fabsf(pp[k]) < 0x1p60f)) h.one = 0.0f;
        h.pad = 0.0f;
        for (int k = 0; k < 3; k++) {
            Interval &iv = r.iv[k];
            iv.lo = off[k];
            iv.span = off[k + 1] - off[k];
            iv.rs = div_ready(iv.span);
            iv.pad = 0.0f;
            if (iv.rs == 0.0f) h.one = 0.0f;
            for (int ch = 0; ch < 4; ch++) {
                iv.c0[ch] = pp[4 + 4 * k + ch];
                iv.c1[ch] = pp[8 + 4 * k + ch];
            }
        }
        rec[i] = r;
        return;
    }
    wts = scene_at(wts, d.ws);
    const float raw = params[(size_t)d.n * kPP];
    const float sigma = fminf(fmaxf(raw, 0.05f), 16.0f);
    const float live = raw > 0.05f && raw < 16.0f ? 1.0f : 0.0f;  // no σ gradient where it is clamped
    const int R = min((int)ceilf(3.0f * sigma), kMaxRadius);
    const int t = threadIdx.x;
    if (t <= 2 * R) {
        const float k = (float)(t - R);
        g[t] = expf(-k * k / (2.0f * sigma * sigma));
    }
    __syncthreads();
    if (t == 0) {
        float z = 0.0f, m2 = 0.0f;
        for (int j = 0; j <= 2 * R; j++) {
            const float k = (float)(j - R);
            z += g[j];
            m2 += g[j] * k * k;
        }
        sums[0] = z;
        sums[1] = m2 / z;  // E[k²]
        wts[0] = (float)R;
    }
    __syncthreads();
    for (int j = t; j < 2 * R + 1 + 2 * kWeightPad; j += (int)blockDim.x) {
        const int i = j - kWeightPad;  // weight i - R
        const bool in = i >= 0 && i <= 2 * R;
        const float k = (float)(i - R);
        const float w = in ? g[i] / sums[0] : 0.0f;
        wts[1 + j] = w;
        wts[1 + kWeightSpan + j] = in ? live * w * (k * k - sums[1]) / (sigma * sigma * sigma) : 0.0f;
    }
}

// ---- blur passes: conv(in, w) along x or y, zero padding --------------------------
// A launch does one or two jobs (blockIdx.z): `out` = conv(in, w), or the block's share of
// the pass's σ derivative, Σ_p dot(gdot[p], conv(in, w')[p]), into part[blockIdx.x].
//
// A thread makes 8 outputs along y, or 4 along x, and reads each input once for all of them
// (one thread per output read 2 R + 1 float4 values from L1: 41 us a pass at 1024^2, σ 4,
// and 81 us for 16 images of 512^2, σ 2.5).  Every output adds its taps in order of k.  The
// weights are symmetric and padded with zeros, so an input's 8 (4) weights are consecutive
// and come by one scalar load.
struct BlurJob {
    const float4 *in;
    float4 *out;
    const float4 *gdot;
    float *part;
};
constexpr int kBlurY = 8, kBlurX = 4;
constexpr int kBlurWaves = 4;
// pixels of a block: 64 x 32 for the pass along y, 256 x 4 along x
inline uint32_t blur_blocks_y(uint32_t w, uint32_t h) { return ((w + 63) / 64) * ((h + 31) / 32); }
inline uint32_t blur_blocks_x(uint32_t w, uint32_t h) { return ((w + 255) / 256) * ((h + 3) / 4); }

template <int N> struct Weights { float w[N]; };

// adds input i's value v to outputs lo .. hi - 1 of N: weight k = o - i (or its mirror i - o)
template <int N>
__device__ __forceinline__ void blur_add(float4 (&acc)[N], const float *w, int R, int i, float4 v, int lo, int hi) {
    const Weights<N> k = scalar_rec(reinterpret_cast<const Weights<N> *>(w + kWeightPad + R - i));
#pragma unroll
    for (int o = 0; o < N; o++) {
        if (o < lo || o >= hi) continue;
        acc[o].x = fmaf(k.w[o], v.x, acc[o].x);
        acc[o].y = fmaf(k.w[o], v.y, acc[o].y);
        acc[o].z = fmaf(k.w[o], v.z, acc[o].z);
        acc[o].w = fmaf(k.w[o], v.w, acc[o].w);
    }
}
// All inputs -R .. R + N - 1 of N outputs.  The first and last N - 1 of them are further
// than R from some outputs, which then take nothing (a zero weight times an infinity would
// be a NaN).
template <int N, typename F> __device__ __forceinline__ void blur_taps(float4 (&acc)[N], const float *w, int R, F at) {
    if (2 * R + 1 >= N) {
#pragma unroll
        for (int j = 0; j < N - 1; j++) blur_add<N>(acc, w, R, j - R, at(j - R), 0, j + 1);
        for (int i = N - 1 - R; i <= R; i++) blur_add<N>(acc, w, R, i, at(i), 0, N);
#pragma unroll
        for (int j = 1; j < N; j++) blur_add<N>(acc, w, R, R + j, at(R + j), j, N);
    } else {
        for (int i = -R; i < R + N; i++) blur_add<N>(acc, w, R, i, at(i), i - R, i + R + 1);
    }
}
__device__ __forceinline__ void blur_part(float dot, float *part, float *red) {
    dot = wave_sum(dot);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = dot;
    __syncthreads();
    if (threadIdx.x == 0) {
        float s = 0.0f;
        for (int i = 0; i < kBlurWaves; i++) s += red[i];
        part[blockIdx.x] = s;
    }
}
__device__ __forceinline__ float dot4(float4 a, float4 b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }

__global__ __launch_bounds__(64 * kBlurWaves) void k_diff_blur_y(Dims d, BlurJob job0, BlurJob job1,
                                                                 const float *__restrict__ wts) {
    __shared__ float red[kBlurWaves];
    const BlurJob job = blockIdx.z ? job1 : job0;
    const float4 *in = scene_at(job.in, d.ws);
    wts = scene_at(wts, d.ws);
    const int R = __builtin_amdgcn_readfirstlane((int)wts[0]);
    const float *w = wts + 1 + (job.gdot ? kWeightSpan : 0);
    const uint32_t bx = (d.w + 63) / 64;
    const int x = (int)(blockIdx.x % bx * 64 + threadIdx.x % 64);
    const int y0 = (int)(blockIdx.x / bx * 32 + threadIdx.x / 64 * kBlurY);
    const bool live = x < (int)d.w;
    float4 acc[kBlurY];
#pragma unroll
    for (int o = 0; o < kBlurY; o++) acc[o] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    blur_taps<kBlurY>(acc, w, R, [&](int i) {
        const int y = y0 + i;
        return live && y >= 0 && y < (int)d.h ? in[(size_t)y * d.w + x] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    });
    float dot = 0.0f;
#pragma unroll
    for (int o = 0; o < kBlurY; o++) {
        const int y = y0 + o;
        if (!live || y >= (int)d.h) continue;
        const size_t p = (size_t)y * d.w + x;
        if (job.gdot) dot += dot4(scene_at(job.gdot, d.ws)[p], acc[o]);
        else scene_at(job.out, d.ws)[p] = acc[o];
    }
    if (job.gdot) blur_part(dot, scene_at(job.part, d.ws), red);
}

__global__ __launch_bounds__(64 * kBlurWaves) void k_diff_blur_x(Dims d, BlurJob job0, BlurJob job1,
                                                                 const float *__restrict__ wts) {
    // a wave's row segment and its halo; a pad after every 4 pixels keeps the lanes' reads,
    // 4 pixels apart, on different banks
    constexpr int kSpan = 64 * kBlurX + 2 * kMaxRadius;
    __shared__ float4 rows[kBlurWaves][kSpan + kSpan / kBlurX];
    __shared__ float red[kBlurWaves];
    const BlurJob job = blockIdx.z ? job1 : job0;
    const float4 *in = scene_at(job.in, d.ws);
    wts = scene_at(wts, d.ws);
    const int R = __builtin_amdgcn_readfirstlane((int)wts[0]);
    const float *w = wts + 1 + (job.gdot ? kWeightSpan : 0);
    const uint32_t bx = (d.w + 255) / 256;
    const int lane = (int)(threadIdx.x % 64);
    const int x0 = (int)(blockIdx.x % bx * 256), y = (int)(blockIdx.x / bx * 4 + threadIdx.x / 64);
    float4 *row = rows[threadIdx.x / 64];
    if (y < (int)d.h) {
        for (int c = lane; c < 64 * kBlurX + 2 * R; c += 64) {
            const int x = x0 - R + c;
            row[c + c / kBlurX] =
                x >= 0 && x < (int)d.w ? in[(size_t)y * d.w + x] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    __syncthreads();
    float4 acc[kBlurX];
#pragma unroll
    for (int o = 0; o < kBlurX; o++) acc[o] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float dot = 0.0f;
    if (y < (int)d.h) {
        blur_taps<kBlurX>(acc, w, R, [&](int i) {
            const int c = kBlurX * lane + i + R;
            return row[c + c / kBlurX];
        });
#pragma unroll
        for (int o = 0; o < kBlurX; o++) {
            const int x = x0 + kBlurX * lane + o;
            if (x >= (int)d.w) continue;
            const size_t p = (size_t)y * d.w + x;
            if (job.gdot) dot += dot4(scene_at(job.gdot, d.ws)[p], acc[o]);
            else scene_at(job.out, d.ws)[p] = acc[o];
        }
    }
    if (job.gdot) blur_part(dot, scene_at(job.part, d.ws), red);
}

// ---- colour matrix on the demultiplied colour ----------------------------------
struct CmEval {
    float v[4];  // demultiplied input (r, g, b, a)
    float o[4];  // matrix output before clamping
    float q[4];  // clamped
};
// The colour is demultiplied by max(a, 1/255): exact for every alpha a u8 pixmap can
// hold (its non-zero alphas are >= 1/255), and below that a continuous ramp to zero,
// so that alphas which are rounding residue (the blur's far tails, cancelled winding
// sums) cannot turn into full-strength colours.
constexpr float kAlphaFloor = 1.0f / 255.0f;
__device__ __forceinline__ CmEval cm_eval(const float *m, float4 b) {
    CmEval e;
    const float a = b.w, r = 1.0f / fmaxf(a, kAlphaFloor);
    e.v[0] = b.x * r;
    e.v[1] = b.y * r;
    e.v[2] = b.z * r;
    e.v[3] = a;
    for (int c = 0; c < 4; c++) {
        const float *r = m + 5 * c;
        e.o[c] = r[0] * e.v[0] + r[1] * e.v[1] + r[2] * e.v[2] + r[3] * e.v[3] + r[4];
        e.q[c] = fminf(fmaxf(e.o[c], 0.0f), 1.0f);
    }
    return e;
}

// final = F + (1 - F_a) S with F = premultiply(clamp(M v(B)))
__global__ __launch_bounds__(kThreads) void k_diff_cm_fwd(Dims d, const float4 *__restrict__ B,
                                                          const float4 *__restrict__ S,
                                                          const float *__restrict__ params, float4 *out) {
    B = scene_at(B, d.ws);
    S = scene_at(S, d.ws);
    params = scene_at(params, params_bytes(d));
    out = scene_at(out, image_bytes(d));
    const size_t np = (size_t)d.w * d.h;
    const size_t p = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (p >= np) return;
    const float *m = params + (size_t)d.n * kPP + 1;
    const CmEval e = cm_eval(m, B[p]);
    const float fa = e.q[3];
    const float4 s = S[p];
    out[p] = make_float4(e.q[0] * fa + (1.0f - fa) * s.x, e.q[1] * fa + (1.0f - fa) * s.y,
                         e.q[2] * fa + (1.0f - fa) * s.z, fa + (1.0f - fa) * s.w);
}

// Backward of the colour matrix and the final composite: from dL/dout, writes
// dL/dB and dL/dS (the composite's direct term) and the block's matrix partials
// into part[blockIdx.x * 20 ..].
__global__ __launch_bounds__(kThreads) void k_diff_cm_bwd(Dims d, const float4 *__restrict__ B,
                                                          const float4 *__restrict__ S,
                                                          const float *__restrict__ params,
                                                          const float4 *__restrict__ gout, float4 *gB, float4 *gS,
                                                          float *part) {
    __shared__ float red[kWaves][20];
    B = scene_at(B, d.ws);
    S = scene_at(S, d.ws);
    params = scene_at(params, params_bytes(d));
    gout = scene_at(gout, image_bytes(d));
    gB = scene_at(gB, d.ws);
    gS = scene_at(gS, d.ws);
    part = scene_at(part, d.ws);
    const size_t np = (size_t)d.w * d.h;
    const size_t p = (size_t)blockIdx.x * kThreads + threadIdx.x;
    const float *m = params + (size_t)d.n * kPP + 1;
    float gm[32];  // 20 matrix entries, padded for the butterfly
#pragma unroll
    for (int j = 0; j < 32; j++) gm[j] = 0.0f;
    if (p < np) {
        const float4 b = B[p], s = S[p], g = gout[p];
        const CmEval e = cm_eval(m, b);
        const float fa = e.q[3];
        // out_c = F_c + (1 - F_a) s_c ; F_c = q_c q_a (c < 3), F_a = q_a
        gS[p] = make_float4(g.x * (1.0f - fa), g.y * (1.0f - fa), g.z * (1.0f - fa), g.w * (1.0f - fa));
        const float gfa = g.w - (g.x * s.x + g.y * s.y + g.z * s.z + g.w * s.w);  // includes dF_a/dF_a = 1
        float gq[4] = {g.x * fa, g.y * fa, g.z * fa, gfa + g.x * e.q[0] + g.y * e.q[1] + g.z * e.q[2]};
        float go[4];
        for (int c = 0; c < 4; c++) go[c] = (e.o[c] > 0.0f && e.o[c] < 1.0f) ? gq[c] : 0.0f;
        float gv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int c = 0; c < 4; c++) {
            for (int j = 0; j < 4; j++) {
                gm[5 * c + j] = go[c] * e.v[j];
                gv[j] += go[c] * m[5 * c + j];
            }
            gm[5 * c + 4] = go[c];
        }
        const float a = b.w, r = 1.0f / fmaxf(a, kAlphaFloor);
        float4 gb;
        gb.x = gv[0] * r;
        gb.y = gv[1] * r;
        gb.z = gv[2] * r;
        // v_c = b_c / a depends on a only above the floor
        gb.w = a > kAlphaFloor ? gv[3] - (gv[0] * e.v[0] + gv[1] * e.v[1] + gv[2] * e.v[2]) * r : gv[3];
        gB[p] = gb;
    }
    const int lane = (int)(threadIdx.x % 64);
    const float v = wave_sum32(gm, lane);
    if (lane < 20) red[threadIdx.x / 64][lane] = v;
    __syncthreads();
    if (threadIdx.x < 20) {
        float s = 0.0f;
        for (int i = 0; i < kWaves; i++) s += red[i][threadIdx.x];
        part[(size_t)blockIdx.x * 20 + threadIdx.x] = s;
    }
}

// ---- backward: paths ----------------------------------------------------------
// dL/dS arrives as gS (direct term) + gS2 (through the blur).  Segments are walked
// from the last; each is recomputed from its checkpoint, then reversed.  The block's
// sums of the per-path gradients go to part[(blockIdx.x * n + i) * kPP ..].
// VALU instructions and load latency bound it: a wave within one stop interval (nearly all
// are) reads that interval's record and reduces 14 sums instead of 24, quotients use the
// record's reciprocals, and 4-wave blocks leave a CU other blocks to run at a segment's
// barriers.  5 waves per SIMD over u8 planes; over areas that would spill (4.3 against 3.2
// ms), so 4.  1024^2, 256 paths 1.60 -> 0.86 ms (6.6e8 -> 3.1e8 wave instructions); 16
// scenes of 512^2 with 128 paths of analytic coverage 4.92 -> 3.20 ms.
template <bool kArea>
__global__ __launch_bounds__(kPathThreads, kArea ? 4 : 5) void k_diff_paths_bwd(Dims d, Cov cv, const PathRec *__restrict__ rec,
                                                                 const float4 *__restrict__ ck,
                                                                 const float4 *__restrict__ gS,
                                                                 const float4 *__restrict__ gS2, float *part) {
    __shared__ float red[kPathWaves][kSeg][kPP];  // per wave, the segment's path sums
    cv = scene_cov(cv, d);
    rec = scene_at(rec, d.ws);
    ck = scene_at(ck, d.ws);
    gS = scene_at(gS, d.ws);
    gS2 = scene_at(gS2, d.ws);
    part = scene_at(part, d.ws);
    const size_t np = (size_t)d.w * d.h;
    const Pixel q = square_pixel(d);
    const size_t p = q.p;
    const bool live = q.live;
    const int lane = (int)(threadIdx.x % 64), wave = (int)(threadIdx.x / 64);
    const float px = (float)q.x + 0.5f, py = (float)q.y + 0.5f;
    // where this lane's parameter sits among wave_sum16's values when the wave's pixels are
    // in stop interval k: 0-2 tint, 3 opacity, 4-7 stop k, 8-11 stop k + 1, 12, 13 their
    // offsets (14: none)
    auto value_lane = [&](int k) {
        const int st = (lane - 4) >> 2, o = lane - 20;
        int v = 14;
        if (lane < 4) v = lane;
        else if (lane < 20) v = st == k ? 4 + (lane & 3) : (st == k + 1 ? 8 + (lane & 3) : 14);
        else v = o == k ? 12 : (o == k + 1 ? 13 : 14);
        return (v & 7) + ((v & 8) << 1);
    };
    float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (live) {
        const float4 a = gS[p], b = gS2[p];
        g = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
    }
    const uint32_t nseg = (d.n + kSeg - 1) / kSeg;
    for (int32_t sg = (int32_t)nseg - 1; sg >= 0; sg--) {
        const uint32_t i0 = (uint32_t)__builtin_amdgcn_readfirstlane(sg) * kSeg;
        float4 canv[kSeg + 1];
        float cov[kSeg], area[kSeg];  // the segment's coverage (and signed area) at this pixel, read once
        canv[0] = live ? ck[(size_t)sg * np + p] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        segment_coverage<kArea>(cv, d, i0, q, cov, area);
        PathHead next = scalar_rec(&rec[i0].head);
#pragma unroll
        for (int j = 0; j < kSeg; j++) {
            canv[j + 1] = canv[j];
            const PathHead h = next;
            // the segment's last path is the first of the walk back
            next = scalar_rec(&rec[min(i0 + j + (j + 1 < kSeg ? 1 : 0), d.n - 1)].head);
            const uint64_t touched = __ballot(cov[j] != 0.0f);
            if (touched != 0) canv[j + 1] = draw_path(rec + i0 + j, h, cov[j], touched, px, py, canv[j], lane);
        }
#pragma unroll
        for (int j = kSeg - 1; j >= 0; j--) {
            const uint32_t i = i0 + j;
            const PathHead h = next;
            next = scalar_rec(&rec[min(i0 + (j > 0 ? j - 1 : 0), d.n - 1)].head);
            if (i >= d.n) continue;  // uniform
            const float c = cov[j];
            float gcov = 0.0f;  // dL/d(coverage)
            float v = 0.0f;     // this wave's sum of the path's gradient `lane`
            const uint64_t touched = __ballot(c != 0.0f);
            if (touched != 0) {
                // every lane evaluates; those without coverage contribute zeros, whatever
                // their dL/dS and canvas hold: A is 0 there and gc and gA are set to it
                const Along e = along_path(h, px, py);
                const float4 sb = canv[j];
                int k0;
                const bool one = one_interval(h, e, touched, k0);
                const PathRec *r = rec + i;
                const int k = lane_interval(e, lane);
                Interval iv;
                Stop st;
                if (one) {
                    iv = scalar_rec(&r->iv[k0]);
                    st = stop_in(iv, e.t);
                } else {
                    st = stop_any(r, k, e.t, h.o0, h.o3);
                }
                float A = c * h.opacity * st.rgba[3];
                if (!one && c == 0.0f) A = 0.0f;  // with `one` it is
                // after = (rgb·tint·A, A) + (1 - A)·before
                const bool on = c != 0.0f;
                const float gc[3] = {on ? g.x : 0.0f, on ? g.y : 0.0f, on ? g.z : 0.0f};
                float gA = g.w - fmaf(g.w, sb.w, fmaf(g.z, sb.z, fmaf(g.y, sb.y, g.x * sb.x)));
                gA = on ? gA : 0.0f;
                float gt[4];    // tint, opacity
                float gcol[4];  // interpolated stop colour and alpha
#pragma unroll
                for (int ch = 0; ch < 3; ch++) {
                    const float ga = gc[ch] * A;
                    gA = fmaf(gc[ch] * st.rgba[ch], h.tint[ch], gA);
                    gt[ch] = ga * st.rgba[ch];
                    gcol[ch] = ga * h.tint[ch];
                }
                const float gAc = gA * c, gAo = gA * h.opacity;
                gt[3] = gAc * st.rgba[3];
                gcol[3] = gAc * h.opacity;
                gcov = on ? gAo * st.rgba[3] : 0.0f;
                const float ia = 1.0f - A;
                g = make_float4(g.x * ia, g.y * ia, g.z * ia, g.w * ia);
                const bool in = (e.inside >> lane) & 1;
                // u = (t - lo) / span inside the stops (constant outside); du: the colour's
                // slope along u, stop k+1 - stop k, dotted with gcol
                if (one) {
                    float gu = gcol[0] * (iv.c1[0] - iv.c0[0]);
#pragma unroll
                    for (int ch = 1; ch < 4; ch++) gu = fmaf(gcol[ch], iv.c1[ch] - iv.c0[ch], gu);
                    const float q = gu * iv.rs;  // div_by, but an overflow stays an infinity
                    const float gs = !in ? 0.0f : (fabsf(q) < INFINITY ? fmaf(fmaf(-q, iv.span, gu), iv.rs, q) : q);
                    // one stop interval: 14 sums instead of 24
                    float gp[16];
                    const float w1 = st.u, w0 = 1.0f - w1;
#pragma unroll
                    for (int ch = 0; ch < 4; ch++) {
                        gp[ch] = gt[ch];
                        gp[4 + ch] = gcol[ch] * w0;
                        gp[8 + ch] = gcol[ch] * w1;
                    }
                    gp[12] = gs * -w0;  // (t - hi) / span = u - 1
                    gp[13] = gs * -w1;
                    gp[14] = gp[15] = 0.0f;
                    v = __shfl(wave_sum16(gp, lane), value_lane(k0), 64);
                } else {
                    const Interval &lv = r->iv[k];
                    float gu = 0.0f;
                    for (int ch = 0; ch < 4; ch++) gu = fmaf(gcol[ch], lv.c1[ch] - lv.c0[ch], gu);
                    float ga_lo = 0.0f, ga_hi = 0.0f;
                    if (in && lv.span > 0.0f && on) {
                        ga_lo = gu * -(1.0f - st.u) / lv.span;
                        ga_hi = gu * -st.u / lv.span;
                    }
                    float gp[32];  // kPP gradients, padded to 32 for the butterfly
                    const float w1 = st.u, w0 = 1.0f - w1;
                    const float ws[4] = {k == 0 ? w0 : 0.0f, k == 1 ? w0 : (k == 0 ? w1 : 0.0f),
                                         k == 2 ? w0 : (k == 1 ? w1 : 0.0f), k == 2 ? w1 : 0.0f};
#pragma unroll
                    for (int ch = 0; ch < 4; ch++) {
                        gp[ch] = on ? gt[ch] : 0.0f;
#pragma unroll
                        for (int q = 0; q < 4; q++) gp[4 + 4 * q + ch] = on ? gcol[ch] * ws[q] : 0.0f;
                    }
                    gp[20] = k == 0 ? ga_lo : 0.0f;
                    gp[21] = k == 1 ? ga_lo : (k == 0 ? ga_hi : 0.0f);
                    gp[22] = k == 2 ? ga_lo : (k == 1 ? ga_hi : 0.0f);
                    gp[23] = k == 2 ? ga_hi : 0.0f;
#pragma unroll
                    for (int z = kPP; z < 32; z++) gp[z] = 0.0f;
                    v = wave_sum32(gp, lane);
                }
            }
            if (kArea && live) {
                // coverage = min(1, |area|): d/d(area) = sign(area) inside (0, 1), else 0
                const float ar = area[j];
                const float da = fabsf(ar) < 1.0f ? (ar > 0.0f ? 1.0f : (ar < 0.0f ? -1.0f : 0.0f)) : 0.0f;
                cv.gW[(size_t)i * np + p] = gcov * da;
            }
            if (lane < kPP) red[wave][j][lane] = v;
        }
        // block sums of the segment's paths
        __syncthreads();
        for (int q = threadIdx.x; q < kSeg * kPP; q += kPathThreads) {
            const int j = q / kPP, k = q % kPP;
            if (i0 + j < d.n) {
                float s = 0.0f;
                for (int w = 0; w < kPathWaves; w++) s += red[w][j][k];
                part[((size_t)blockIdx.x * d.n + i0 + j) * kPP + k] = s;
            }
        }
        __syncthreads();
    }
}

// ---- analytic coverage (geometry mode) ---------------------------------------
// A path is a closed chain of k cubics: user-space points P0 .. P3k (geom floats
// after the path's 6 affine values sx, ky, kx, sy, tx, ty; device = (sx x + kx y +
// tx, ky x + sy y + ty)), each cubic flattened into kFlat segments at uniform t,
// and the polygon closed by a line from P3k back to P0.  Vertex j of path i:
// vert[i * nv + j], nv = k * kFlat + 1.
constexpr int kFlat = 16;

__device__ __forceinline__ void bern(float t, float b[4]) {
    const float u = 1.0f - t;
    b[0] = u * u * u;
    b[1] = 3.0f * u * u * t;
    b[2] = 3.0f * u * t * t;
    b[3] = t * t * t;
}

// vertex j of a path of k cubics
__device__ __forceinline__ float2 flat_vertex(const float *g, uint32_t k, uint32_t j) {
    const uint32_t c = j / kFlat < k ? j / kFlat : k - 1;  // the last vertex is t = 1 of the last cubic
    const float t = (float)(j - c * kFlat) / (float)kFlat;
    float b[4];
    bern(t, b);
    float x = 0.0f, y = 0.0f;
    for (int m = 0; m < 4; m++) {
        x += b[m] * g[6 + 2 * (3 * c + m)];
        y += b[m] * g[6 + 2 * (3 * c + m) + 1];
    }
    return make_float2(g[0] * x + g[2] * y + g[4], g[1] * x + g[3] * y + g[5]);
}

// A thread per vertex and, of the kFlat edges of each cubic and the closing one, the least and
// the largest y of their ends (everything where one of them is a NaN):
// bounds[i * (k + 1) + j / kFlat].
__global__ __launch_bounds__(256) void k_diff_flatten(Dims d, const float *__restrict__ geom, float2 *vert,
                                                      float2 *bounds) {
    static_assert(kFlat == 16, "a group's lanes are a row of 16");
    geom = scene_at(geom, geom_bytes(d));
    vert = scene_at(vert, d.ws);
    bounds = scene_at(bounds, d.ws);
    const uint32_t k = d.k, nv = k * kFlat + 1, lanes = (k + 1) * kFlat;
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t i = gid / lanes, j = gid % lanes;
    float lo = INFINITY, hi = -INFINITY;
    if (i < d.n && j < nv) {
        const float *g = geom + (size_t)i * (6 + 2 * (3 * k + 1));
        const float2 v = flat_vertex(g, k, j);
        vert[(size_t)i * nv + j] = v;
        // the group's last edge ends at the next group's first vertex, or closes the path
        const float e = j % kFlat == kFlat - 1 || j + 1 == nv ? flat_vertex(g, k, j + 1 == nv ? 0 : j + 1).y : v.y;
        const bool nan = v.y != v.y || e != e;
        lo = nan ? -INFINITY : fminf(v.y, e);
        hi = nan ? INFINITY : fmaxf(v.y, e);
    }
    for (int m = 1; m < kFlat; m <<= 1) {
        lo = fminf(lo, __shfl_xor(lo, m, kFlat));
        hi = fmaxf(hi, __shfl_xor(hi, m, kFlat));
    }
    if (i < d.n && j % kFlat == 0) bounds[(size_t)i * (k + 1) + j / kFlat] = make_float2(lo, hi);
}

__global__ void k_diff_zero(float *p, size_t n, size_t stride) {
    p = scene_at(p, stride);
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.0f;
}

// One straight piece of an edge within a pixel row (x in [0, w], dd its signed share
// of the row's height): adds the differences whose prefix sum along the row is the
// piece's contribution to each pixel's winding area (the trapezoid right of the
// piece, split by the pixel columns).  The differences are added in fixed point
// (round(v * q), integer atomics), so the sums do not depend on the order in which
// edges arrive.
__device__ __forceinline__ void add_q(int *cell, float v, float q) { atomicAdd(cell, __float2int_rn(v * q)); }
__device__ __forceinline__ void accum_piece(int *row, float xa, float xb, float dd, float q) {
    const float x0 = fminf(xa, xb), x1 = fmaxf(xa, xb);
    const float x0f = floorf(x0);
    const int x0i = (int)x0f;
    const float x1c = ceilf(x1);
    if (x1c <= x0f + 1.0f) {  // within one column
        const float xm = 0.5f * (xa + xb) - x0f;
        add_q(row + x0i, dd * (1.0f - xm), q);
        add_q(row + x0i + 1, dd * xm, q);
        return;
    }
    const float sl = 1.0f / (x1 - x0);
    const float fx0 = x0 - x0f;
    const float a0 = 0.5f * sl * (1.0f - fx0) * (1.0f - fx0);
    const float fx1 = x1 - x1c + 1.0f;
    const float am = 0.5f * sl * fx1 * fx1;
    const int x1i = (int)x1c;
    add_q(row + x0i, dd * a0, q);
    if (x1i == x0i + 2) {
        add_q(row + x0i + 1, dd * (1.0f - a0 - am), q);
    } else {
        const float a1 = sl * (1.5f - fx0);
        add_q(row + x0i + 1, dd * (a1 - a0), q);
        for (int xi = x0i + 2; xi < x1i - 1; xi++) add_q(row + xi, dd * sl, q);
        const float a2 = a1 + (float)(x1i - x0i - 3) * sl;
        add_q(row + x1i - 1, dd * (1.0f - a2 - am), q);
    }
    add_q(row + x1i, dd * am, q);
}

// The part of one polygon edge (a above b, winding dir) in pixel row y, added to `row`
// (w + 2 cells): the row's share of the edge's winding is split between the cells its x
// range touches so that the prefix sum along the row is the winding-weighted area of each
// pixel (the exact area coverage of the polygon's winding number).  The stretch is cut
// where it crosses x = 0 and x = w: a piece left of the canvas is moved onto x = 0 (cell 0,
// so it changes the winding of every pixel of the row alike), a piece right of it lands in
// cell w, beyond the prefix, so the planes are exact whatever lies outside.
__device__ __forceinline__ void accum_row(int *row, const Dims &d, float2 a, float2 b, float dxdy, float dir, int y) {
    const float W = (float)d.w;
    const float ya = fmaxf(a.y, (float)y), yb = fminf(b.y, (float)(y + 1));
    const float dy = yb - ya;
    if (!(dy > 0.0f)) return;
    const float xa = a.x + dxdy * (ya - a.y), xb = a.x + dxdy * (yb - a.y);
    const float dd = dy * dir;
    // cut points (fractions of the stretch) at x = 0 and x = w, in order
    float c0 = 2.0f, c1 = 2.0f;
    if (xb != xa) {
        const float u = (0.0f - xa) / (xb - xa), v = (W - xa) / (xb - xa);
        const float lo = fminf(u, v), hi = fmaxf(u, v);
        if (lo > 0.0f && lo < 1.0f) c0 = lo;
        if (hi > 0.0f && hi < 1.0f) {
            if (c0 > 1.0f) c0 = hi;
            else c1 = hi;
        }
    }
    const float cuts[4] = {0.0f, c0 < 1.0f ? c0 : 1.0f, c1 < 1.0f ? c1 : 1.0f, 1.0f};
    for (int q = 0; q < 3; q++) {
        const float t0 = cuts[q], t1 = cuts[q + 1];
        if (!(t1 > t0)) continue;
        const float pa = fminf(fmaxf(xa + t0 * (xb - xa), 0.0f), W);
        const float pb = fminf(fmaxf(xa + t1 * (xb - xa), 0.0f), W);
        accum_piece(row, pa, pb, dd * (t1 - t0), d.qscale);
    }
}

// edge j of path i with its upper end first; false when it is horizontal
__device__ __forceinline__ bool edge_down(const float2 *vert, uint32_t nv, uint32_t i, uint32_t j, float2 &a, float2 &b,
                                          float &dir) {
    a = vert[(size_t)i * nv + j];
    b = vert[(size_t)i * nv + (j + 1 == nv ? 0 : j + 1)];
    dir = 1.0f;
    if (a.y == b.y) return false;
    if (a.y > b.y) {
        const float2 t = a;
        a = b;
        b = t;
        dir = -1.0f;
    }
    return true;
}

// The winding areas of a band of `rows` pixel rows of one path, in LDS from the edges to the
// prefix sums: of the cubics whose bounds meet the band the edges that do are gathered,
// kAreaEdges at a time, a thread per gathered (edge, row) adds the row's differences, then a
// wave per row sums along it in exact integer arithmetic and writes the floats.  The planes
// are written once (they were cleared, added to with global atomics, read and written
// again); the integers, and so the areas, are the same.  For rows of at most kAreaCells cells.
// Bound by the planes' stores with few cubics (16 scenes of 512^2 with 128 paths of 8 cubics:
// 2.15 GB, 1.92 -> 0.61 ms), by the gathers with many: looking at every edge for every row
// instead, a forward of 16 wobbly circles of 4096 cubics at 64 x 4096 took 5.9 ms, where the
// form below, which visits an edge's own rows, took 0.20; now 0.15 (32 of 512 cubics at
// 512^2: 0.38, 0.12 and 0.09).  Cubics through all of the canvas, 32 of 512 at 512^2: 0.43,
// 0.75 and 0.17.
constexpr int kAreaCells = 8192;  // 32 KB of LDS
constexpr int kAreaEdges = 512;
constexpr int kAreaGroups = 512;  // cubics looked at together

// Appends `value` of the lanes with `keep` to a list in LDS of which `count` entries are used.
__device__ __forceinline__ void gather(bool keep, uint32_t value, uint16_t *list, uint32_t &count, int lane) {
    const uint64_t m = __ballot(keep);
    uint32_t at = 0;
    if (lane == 0 && m != 0) at = atomicAdd(&count, (uint32_t)__popcll(m));
    at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    if (keep) list[at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)value;
}
// whether rows y0 .. y1 - 1 meet a stretch from lo down to hi, as k_diff_area's rows take it
// (a NaN lo is above them all, a NaN hi ends before them)
__device__ __forceinline__ bool meets_rows(float lo, float hi, uint32_t y0, uint32_t y1) {
    return !(floorf(lo) >= (float)y1) && ceilf(hi) > (float)y0;
}
__global__ __launch_bounds__(256) void k_diff_area(Dims d, const float2 *__restrict__ vert,
                                                   const float2 *__restrict__ bounds, float *area, uint32_t rows,
                                                   uint32_t bands) {
    __shared__ int cells[kAreaCells];
    __shared__ uint16_t groups[kAreaGroups], list[kAreaEdges];  // cubics; 16 * a cubic's place in its batch + edge
    __shared__ uint32_t ngroups, nedges;
    vert = scene_at(vert, d.ws);
    bounds = scene_at(bounds, d.ws);
    area = scene_at(area, d.ws);
    const uint32_t i = blockIdx.x / bands, y0 = blockIdx.x % bands * rows, y1 = min(y0 + rows, d.h);
    const uint32_t stride = d.w + 2, nv = d.k * kFlat + 1, batch = kAreaEdges / kFlat;
    const int lane = (int)(threadIdx.x % 64);
    for (uint32_t c = threadIdx.x; c < rows * stride; c += 256) cells[c] = 0;
    for (uint32_t c0 = 0; c0 <= d.k; c0 += kAreaGroups) {
        if (d.k < batch) {  // all of them fit a batch: their edges are looked at anyway
            if (threadIdx.x <= d.k) groups[threadIdx.x] = (uint16_t)threadIdx.x;
            if (threadIdx.x == 0) ngroups = d.k + 1, nedges = 0;
        } else {
            __syncthreads();
            if (threadIdx.x == 0) ngroups = nedges = 0;
            __syncthreads();
            for (uint32_t k = threadIdx.x; k < kAreaGroups; k += 256) {
                bool meets = false;
                if (c0 + k <= d.k) {
                    const float2 b = bounds[(size_t)i * (d.k + 1) + c0 + k];
                    meets = meets_rows(b.x, b.y, y0, y1);
                }
                gather(meets, c0 + k, groups, ngroups, lane);
            }
        }
        __syncthreads();
        for (uint32_t g0 = 0; g0 < ngroups; g0 += batch) {
            for (uint32_t k = threadIdx.x; k < kAreaEdges; k += 256) {
                bool meets = false;
                if (g0 + k / kFlat < ngroups) {
                    const uint32_t j = groups[g0 + k / kFlat] * kFlat + k % kFlat;
                    float2 a, b;
                    float dir;
                    meets = j < nv && edge_down(vert, nv, i, j, a, b, dir) && meets_rows(a.y, b.y, y0, y1);
                }
                gather(meets, k, list, nedges, lane);
            }
            __syncthreads();
            // a thread per edge where there are enough of them, else per edge and row
            const uint32_t split = nedges < 256 ? rows : 1;
            for (uint32_t q = threadIdx.x; q < nedges * split; q += 256) {
                const uint32_t k = list[q / split], j = groups[g0 + k / kFlat] * kFlat + k % kFlat;
                float2 a, b;
                float dir;
                if (!edge_down(vert, nv, i, j, a, b, dir)) continue;
                // the rows that the edge spans
                int ya = max((int)y0, (int)floorf(a.y)), yb = min((int)y1, (int)ceilf(b.y));
                if (split > 1) {
                    const int y = (int)(y0 + q % split);
                    ya = max(ya, y);
                    yb = min(yb, y + 1);
                }
                for (int y = ya; y < yb; y++)
                    accum_row(cells + ((uint32_t)y - y0) * stride, d, a, b, (b.x - a.x) / (b.y - a.y), dir, y);
            }
            __syncthreads();
            if (g0 + batch < ngroups) {  // uniform
                if (threadIdx.x == 0) nedges = 0;
                __syncthreads();
            }
        }
    }
    __syncthreads();
    const float inv = 1.0f / d.qscale;
    for (uint32_t r = threadIdx.x / 64; r < y1 - y0; r += 4) {
        const int *c = cells + r * stride;
        float *o = area + ((size_t)i * d.h + y0 + r) * stride;
        int carry = 0;
        // four 64-column chunks at a time: their scans are independent chains
        for (uint32_t x0 = 0; x0 < d.w; x0 += 256) {
            int v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t x = x0 + 64 * k + lane;
                v[k] = x < d.w ? c[x] : 0;
            }
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = wave_prefix(v[k]);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t x = x0 + 64 * k + lane;
                if (x < d.w) o[x] = (float)(int)((uint32_t)carry + (uint32_t)v[k]) * inv;
                carry = (int)((uint32_t)carry + (uint32_t)__builtin_amdgcn_readlane(v[k], 63));
            }
        }
    }
}

// Rows too long for LDS: signed area accumulation of one polygon edge into its path's plane
// (row stride w + 2).  The planes hold fixed-point integers (scale d.qscale) until
// k_diff_prefix.
__global__ void k_diff_accum(Dims d, const float2 *__restrict__ vert, int *area) {
    vert = scene_at(vert, d.ws);
    area = scene_at(area, d.ws);
    const uint32_t nv = d.k * kFlat + 1;
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= d.n * nv) return;
    const uint32_t i = gid / nv;
    float2 a, b;
    float dir;
    if (!edge_down(vert, nv, i, gid % nv, a, b, dir)) return;
    const float dxdy = (b.x - a.x) / (b.y - a.y);
    int *plane = area + (size_t)i * d.h * (d.w + 2);
    const int y0 = max(0, (int)floorf(a.y)), y1 = min((int)d.h, (int)ceilf(b.y));
    for (int y = y0; y < y1; y++) accum_row(plane + (size_t)y * (d.w + 2), d, a, b, dxdy, dir, y);
}

// Prefix sums along each row of the area planes (one wave per row), in place: the
// fixed-point differences are summed in wrapping integer arithmetic (exact, and
// every prefix, a pixel's winding area, is within range) and written back as floats.
__global__ void k_diff_prefix(Dims d, float *area) {
    area = scene_at(area, d.ws);
    const uint32_t row = blockIdx.x;  // over n * h
    const int lane = threadIdx.x;
    float *r = area + (size_t)row * (d.w + 2);
    const int *ri = (const int *)r;
    const float inv = 1.0f / d.qscale;
    uint32_t carry = 0;
    // four 64-column chunks at a time: their loads are issued together and their
    // scans are independent chains
    for (uint32_t x0 = 0; x0 < d.w; x0 += 256) {
        uint32_t v[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint32_t x = x0 + 64 * c + lane;
            v[c] = x < d.w ? (uint32_t)ri[x] : 0u;
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint32_t t = __shfl_up(v[c], o, 64);
                if (lane >= o) v[c] += t;
            }
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint32_t x = x0 + 64 * c + lane;
            if (x < d.w) r[x] = (float)(int)(carry + v[c]) * inv;
            carry += __shfl(v[c], 63, 64);
        }
    }
}

// dL/d(area) through one edge: the boundary term.  Moving the edge point x(s) =
// a + s (b - a) by δx changes the winding area of the pixel it crosses by
// δx · (-(b-a).y, (b-a).x) ds, so per pixel crossed on s in [s0, s1]:
// dA/da = n ∫(1 - s) ds, dA/db = n ∫ s ds.  The pixels are walked in order along
// the edge; pixels outside the canvas are skipped.  Writes (dL/da, dL/db) per edge.
__global__ void k_diff_boundary(Dims d, const float2 *__restrict__ vert, const float *__restrict__ gW,
                                float4 *egrad) {
    vert = scene_at(vert, d.ws);
    gW = scene_at(gW, d.ws);
    egrad = scene_at(egrad, d.ws);
    const uint32_t nv = d.k * kFlat + 1;
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= d.n * nv) return;
    const uint32_t i = gid / nv, j = gid % nv;
    const float2 a = vert[gid], b = vert[(size_t)i * nv + (j + 1 == nv ? 0 : j + 1)];
    const float tx = b.x - a.x, ty = b.y - a.y;
    float wa = 0.0f, wb = 0.0f;
    // the part of the edge inside the canvas, s in [s0, s1] (Liang-Barsky): the walk
    // below then crosses at most w + h + 2 pixels whatever the edge's length, and its
    // step count is capped at w + h + 3 even for non-finite end points (reads stay
    // behind the bounds check)
    float s0 = 0.0f, s1 = 1.0f;
    bool inside = tx != 0.0f || ty != 0.0f;
    if (tx != 0.0f) {
        const float u = -a.x / tx, v = ((float)d.w - a.x) / tx;
        s0 = fmaxf(s0, fminf(u, v));
        s1 = fminf(s1, fmaxf(u, v));
    } else {
        inside = inside && a.x >= 0.0f && a.x < (float)d.w;
    }
    if (ty != 0.0f) {
        const float u = -a.y / ty, v = ((float)d.h - a.y) / ty;
        s0 = fmaxf(s0, fminf(u, v));
        s1 = fminf(s1, fmaxf(u, v));
    } else {
        inside = inside && a.y >= 0.0f && a.y < (float)d.h;
    }
    if (inside && s0 < s1) {
        const float *g = gW + (size_t)i * d.w * d.h;
        const float px = fminf(fmaxf(a.x + s0 * tx, 0.0f), (float)d.w - 1.0f);
        const float py = fminf(fmaxf(a.y + s0 * ty, 0.0f), (float)d.h - 1.0f);
        int ix = (int)floorf(px), iy = (int)floorf(py);
        const int sx = tx > 0.0f ? 1 : -1, sy = ty > 0.0f ? 1 : -1;
        const float inf = 3.0e38f;
        float tmx = tx != 0.0f ? ((float)(ix + (sx > 0 ? 1 : 0)) - a.x) / tx : inf;
        float tmy = ty != 0.0f ? ((float)(iy + (sy > 0 ? 1 : 0)) - a.y) / ty : inf;
        const float tdx = tx != 0.0f ? fabsf(1.0f / tx) : inf, tdy = ty != 0.0f ? fabsf(1.0f / ty) : inf;
        float s = s0;
        const int steps = (int)fminf((s1 - s0) * (fabsf(tx) + fabsf(ty)), (float)(d.w + d.h)) + 3;
        for (int q = 0; q < steps && s < s1; q++) {
            const float sn = fminf(fminf(tmx, tmy), s1);
            if (ix >= 0 && ix < (int)d.w && iy >= 0 && iy < (int)d.h) {
                const float G = g[(size_t)iy * d.w + ix];
                const float i1 = sn - s, i2 = 0.5f * (sn * sn - s * s);
                wa += G * (i1 - i2);
                wb += G * i2;
            }
            s = sn;
            if (tmx < tmy) {
                ix += sx;
                tmx += tdx;
            } else {
                iy += sy;
                tmy += tdy;
            }
        }
    }
    // n = (-t.y, t.x)
    egrad[gid] = make_float4(-ty * wa, tx * wa, -ty * wb, tx * wb);
}

// Per path (one wave): vertex gradients from the edge gradients, through the flattening
// (Bernstein weights) to the device control points, a lane each, then through the affine to
// the user-space points and, summed over the wave, the affine's six values (one thread per
// path took 229 us for 2048 paths of 8 cubics).
__global__ __launch_bounds__(64) void k_diff_geom_chain(Dims d, const float *__restrict__ geom,
                                                        const float4 *__restrict__ egrad, float *ggeom) {
    geom = scene_at(geom, geom_bytes(d));
    egrad = scene_at(egrad, d.ws);
    ggeom = scene_at(ggeom, geom_bytes(d));
    const uint32_t k = d.k, i = blockIdx.x, lane = threadIdx.x;
    const uint32_t nv = k * kFlat + 1, np = 3 * k + 1;
    const float *g = geom + (size_t)i * (6 + 2 * np);
    float *o = ggeom + (size_t)i * (6 + 2 * np);
    const float4 *e = egrad + (size_t)i * nv;
    float aff[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t pi = lane; pi < np; pi += 64) {
        float dx = 0.0f, dy = 0.0f;  // dL/d(device point)
        // point 3 of a cubic is point 0 of the next
        for (uint32_t part = 0; part < 2; part++) {
            const uint32_t m = part == 0 ? (pi % 3 == 0 ? 3 : pi % 3) : 0;
            if (part == 0 ? pi == 0 : pi % 3 != 0 || pi == 3 * k) continue;
            const uint32_t c = (pi - m) / 3;
            const uint32_t last = c + 1 == k ? kFlat : kFlat - 1;  // t = 1 belongs to the last cubic
            for (uint32_t q = 0; q <= last; q++) {
                // vertex j starts edge j and ends edge j - 1 (edge nv - 1 closes to vertex 0)
                const uint32_t j = c * kFlat + q;
                const float4 ea = e[j], eb = e[j == 0 ? nv - 1 : j - 1];
                float b[4];
                bern((float)q / (float)kFlat, b);
                const float bm = m == 0 ? b[0] : (m == 1 ? b[1] : (m == 2 ? b[2] : b[3]));
                dx += bm * (ea.x + eb.z);
                dy += bm * (ea.y + eb.w);
            }
        }
        const float ux = g[6 + 2 * pi], uy = g[6 + 2 * pi + 1];
        // device = (sx x + kx y + tx, ky x + sy y + ty)
        o[6 + 2 * pi] = g[0] * dx + g[1] * dy;
        o[6 + 2 * pi + 1] = g[2] * dx + g[3] * dy;
        aff[0] += dx * ux;
        aff[1] += dy * ux;
        aff[2] += dx * uy;
        aff[3] += dy * uy;
        aff[4] += dx;
        aff[5] += dy;
    }
#pragma unroll
    for (int q = 0; q < 6; q++) {
        const float s = wave_sum(aff[q]);
        if (lane == 0) o[q] = s;
    }
}

// Sums partial rows into the gradients, in a fixed order: a block of 16 columns x 64 row
// lanes, each lane summing every 64th row of a column in eight sums, then those and the
// lanes in pairs, which keeps the rounding of many rows down.  Blocks
// below `blocks` take the paths' partial rows; the last two σ (both passes' block sums, one
// column) and the matrix (20 columns).
struct ReducePart {
    const float *part;
    float *out;
    uint32_t rows, cols;
};
__global__ __launch_bounds__(1024) void k_diff_reduce(ReducePart paths, ReducePart sigma, ReducePart matrix,
                                                      uint32_t blocks, size_t part_stride, size_t out_stride) {
    __shared__ float acc[64][17];
    ReducePart r = paths;
    uint32_t c = blockIdx.x * 16;
    if (blockIdx.x >= blocks) {
        r = blockIdx.x == blocks ? sigma : matrix;
        c = blockIdx.x <= blocks + 1 ? 0 : 16;
    }
    const float *part = scene_at(r.part, part_stride);
    const uint32_t tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    c += tx;
    float s[8] = {};
    if (c < r.cols) {
        uint32_t row = ty;
        for (; row + 7 * 64 < r.rows; row += 512) {
#pragma unroll
            for (uint32_t k = 0; k < 8; k++) s[k] += part[(size_t)(row + 64 * k) * r.cols + c];
        }
        // the last ones: loads without a branch, which go out together
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) {
            const float v = part[(size_t)min(row + 64 * k, r.rows - 1) * r.cols + c];
            s[k] += row + 64 * k < r.rows ? v : 0.0f;
        }
    }
    acc[ty][tx] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    for (uint32_t half = 32; half > 0; half >>= 1) {
        __syncthreads();
        if (ty < half) acc[ty][tx] += acc[ty + half][tx];
    }
    if (ty == 0 && c < r.cols) scene_at(r.out, out_stride)[c] = acc[0][tx];
}

// Workspace layout (bytes, 256-aligned): canvas S | T | B | gB | gS | gS2 | weights |
// path records | checkpoints | partial rows (paths) | partial rows (matrix) | σ partials (2 rows).
struct Layout {
    size_t S, T, B, gB, gS, gS2, wts, rec, ck, part_p, part_m, part_s, area, gW, vert, egrad, bounds, total;
};
uint32_t squares(uint32_t side, int square) { return (side + square - 1) / square; }
Layout layout(uint32_t w, uint32_t h, uint32_t n, uint32_t k) {
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t img = al((size_t)w * h * sizeof(float4));
    const size_t nblk = ((size_t)w * h + kThreads - 1) / kThreads;
    Layout L;
    L.S = 0;
    L.T = L.S + img;
    L.B = L.T + img;
    L.gB = L.B + img;
    L.gS = L.gB + img;
    L.gS2 = L.gS + img;
    L.wts = L.gS2 + img;
    L.rec = L.wts + al((1 + 2 * kWeightSpan) * sizeof(float));
    L.ck = L.rec + al((size_t)n * sizeof(PathRec));
    L.part_p = L.ck + al((size_t)((n + kSeg - 1) / kSeg) * w * h * sizeof(float4));
    L.part_m = L.part_p + al((size_t)squares(w, kSquareW) * squares(h, kSquareH) * n * kPP * sizeof(float));
    L.part_s = L.part_m + al(nblk * 20 * sizeof(float));
    L.area = L.part_s + al((size_t)(blur_blocks_y(w, h) + blur_blocks_x(w, h)) * sizeof(float));
    const size_t nv = (size_t)k * kFlat + 1;
    L.gW = L.area + (k ? al((size_t)n * h * (w + 2) * sizeof(float)) : 0);
    L.vert = L.gW + (k ? al((size_t)n * w * h * sizeof(float)) : 0);
    L.egrad = L.vert + (k ? al((size_t)n * nv * sizeof(float2)) : 0);
    L.bounds = L.egrad + (k ? al((size_t)n * nv * sizeof(float4)) : 0);
    L.total = L.bounds + (k ? al((size_t)n * (k + 1) * sizeof(float2)) : 0);
    return L;
}

// Fixed-point scale of the area accumulation: a pixel's winding area is at most half
// the polygon's edge count (k * kFlat + 1) in magnitude, so with q = 2^(30 - ceil(log2
// of that + 1)) every prefix fits a 32-bit integer; at most 2^24 (a resolution of
// 6e-8, f32's near 1).  8-cubic paths: 2^23.
float area_qscale(uint32_t k) {
    const uint64_t edges = (uint64_t)k * kFlat + 1;
    int bits = 0;
    while ((1ull << bits) < edges / 2 + 1) bits++;
    const int sh = 30 - bits < 24 ? 30 - bits : 24;
    return std::ldexp(1.0f, sh);
}

Dims dims_of(uint32_t w, uint32_t h, uint32_t n, uint32_t k, size_t ws) {
    const uint32_t tx = squares(w, kSquareW);
    return Dims{w, h, n, (uint32_t)(((size_t)w * h + kThreads - 1) / kThreads), tx, tx * squares(h, kSquareH), k, ws,
                area_qscale(k)};
}

// The kernels index vertices (path_count x (16 cubics + 1)) and prefix rows
// (path_count x height) with 32-bit grid and thread indices.
bool scene_ok(const rvk_diff_scene *s, const float *geom) {
    return s && s->width > 0 && s->height > 0 && s->path_count > 0 && s->dev_gradient_ends &&
           (s->cubics ? geom != nullptr && s->cubics <= 4096 : s->dev_coverage != nullptr) &&
           (uint64_t)s->width * s->height <= (1ull << 30) &&
           (uint64_t)s->path_count * ((uint64_t)s->cubics * kFlat + 1) < (1ull << 31) &&
           (uint64_t)s->path_count * s->height < (1ull << 31);
}

}  // namespace

extern "C" {

rvk_status rvk_diff_workspace_size(uint32_t width, uint32_t height, uint32_t path_count, uint32_t cubics,
                                   size_t *bytes) {
    if (!bytes || width == 0 || height == 0 || path_count == 0 || cubics > 4096) return RVK_ERR_INVALID_ARGUMENT;
    *bytes = layout(width, height, path_count, cubics).total;
    return RVK_OK;
}

rvk_status rvk_diff_forward_batch(rvk_context *ctx, const rvk_diff_scene *scene, uint32_t batch,
                                  const float *dev_params, const float *dev_geom, void *dev_workspace,
                                  float *dev_out) {
    if (!ctx || !scene_ok(scene, dev_geom) || !dev_params || !dev_workspace || !dev_out || batch == 0 ||
        batch > 65535)
        return RVK_ERR_INVALID_ARGUMENT;
    const uint32_t w = scene->width, h = scene->height, n = scene->path_count, k = scene->cubics;
    const Layout L = layout(w, h, n, k);
    uint8_t *ws = (uint8_t *)dev_workspace;
    const Dims d = dims_of(w, h, n, k, L.total);
    float4 *S = (float4 *)(ws + L.S), *T = (float4 *)(ws + L.T), *B = (float4 *)(ws + L.B);
    float *wts = (float *)(ws + L.wts);
    const double px_bytes = (double)w * h * batch;
    Cov cv{scene->dev_coverage, nullptr, nullptr};
    if (k) {
        // analytic coverage: flatten, accumulate winding area, prefix along rows
        float *area = (float *)(ws + L.area);
        float2 *vert = (float2 *)(ws + L.vert), *bounds = (float2 *)(ws + L.bounds);
        const size_t nv = (size_t)k * kFlat + 1, cells = (size_t)n * h * (w + 2);
        const unsigned ge = (unsigned)((n * nv + 255) / 256);
        const unsigned gz = (unsigned)((cells + 255) / 256 < 65535 ? (cells + 255) / 256 : 65535);
        rvk::timed_launch(ctx, "diff_coverage", (double)cells * 8.0 * batch, [&] {
            const size_t lanes = (size_t)n * (k + 1) * kFlat;
            hipLaunchKernelGGL(k_diff_flatten, dim3((unsigned)((lanes + 255) / 256), batch), dim3(256), 0, ctx->stream,
                               d, dev_geom, vert, bounds);
            const uint32_t rows = std::min<uint32_t>({(uint32_t)kAreaCells / (w + 2), 16u, h});
            if (rows > 0) {
                const uint32_t bands = (h + rows - 1) / rows;
                hipLaunchKernelGGL(k_diff_area, dim3(n * bands, batch), dim3(256), 0, ctx->stream, d,
                                   (const float2 *)vert, (const float2 *)bounds, area, rows, bands);
            } else {
                hipLaunchKernelGGL(k_diff_zero, dim3(gz, batch), dim3(256), 0, ctx->stream, area, cells, L.total);
                hipLaunchKernelGGL(k_diff_accum, dim3(ge, batch), dim3(256), 0, ctx->stream, d, (const float2 *)vert,
                                   (int *)area);
                hipLaunchKernelGGL(k_diff_prefix, dim3(n * h, batch), dim3(64), 0, ctx->stream, d, area);
            }
        });
        cv = Cov{nullptr, area, nullptr};
    }
    PathRec *rec = (PathRec *)(ws + L.rec);
    rvk::timed_launch(ctx, "diff_prepare", 0.0, [&] {
        const unsigned threads = 2 * kMaxRadius + 1;
        hipLaunchKernelGGL(k_diff_prepare, dim3(1 + (n + threads - 1) / threads, batch), dim3(threads), 0, ctx->stream,
                           d, dev_params, (const float4 *)scene->dev_gradient_ends, wts, rec);
    });
    rvk::timed_launch(ctx, "diff_paths_fwd", px_bytes * (16.0 + n), [&] {
        hipLaunchKernelGGL(k ? k_diff_paths_fwd<true> : k_diff_paths_fwd<false>, dim3(d.ntile, batch), dim3(kPathThreads),
                           0, ctx->stream, d, cv, (const PathRec *)rec, S, (float4 *)(ws + L.ck));
    });
    const uint32_t by = blur_blocks_y(w, h), bx = blur_blocks_x(w, h);
    rvk::timed_launch(ctx, "diff_blur", px_bytes * 32.0, [&] {
        const BlurJob job{S, T, nullptr, nullptr};
        hipLaunchKernelGGL(k_diff_blur_x, dim3(bx, batch), dim3(64 * kBlurWaves), 0, ctx->stream, d, job, job,
                           (const float *)wts);
    });
    rvk::timed_launch(ctx, "diff_blur", px_bytes * 32.0, [&] {
        const BlurJob job{T, B, nullptr, nullptr};
        hipLaunchKernelGGL(k_diff_blur_y, dim3(by, batch), dim3(64 * kBlurWaves), 0, ctx->stream, d, job, job,
                           (const float *)wts);
    });
    rvk::timed_launch(ctx, "diff_cm_fwd", px_bytes * 48.0, [&] {
        hipLaunchKernelGGL(k_diff_cm_fwd, dim3(d.nblk, batch), dim3(kThreads), 0, ctx->stream, d, (const float4 *)B,
                           (const float4 *)S, dev_params, (float4 *)dev_out);
    });
    RVK_HIP_CHECK(hipGetLastError());
    return RVK_OK;
}

rvk_status rvk_diff_forward(rvk_context *ctx, const rvk_diff_scene *scene, const float *dev_params,
                            const float *dev_geom, void *dev_workspace, float *dev_out) {
    return rvk_diff_forward_batch(ctx, scene, 1, dev_params, dev_geom, dev_workspace, dev_out);
}

rvk_status rvk_diff_backward_batch(rvk_context *ctx, const rvk_diff_scene *scene, uint32_t batch,
                                   const float *dev_params, const float *dev_geom, void *dev_workspace,
                                   const float *dev_grad_out, float *dev_grad_params, float *dev_grad_geom) {
    if (!ctx || !scene_ok(scene, dev_geom) || !dev_params || !dev_workspace || !dev_grad_out || !dev_grad_params ||
        (scene->cubics && !dev_grad_geom) || batch == 0 || batch > 65535)
        return RVK_ERR_INVALID_ARGUMENT;
    const uint32_t w = scene->width, h = scene->height, n = scene->path_count, k = scene->cubics;
    const Layout L = layout(w, h, n, k);
    uint8_t *ws = (uint8_t *)dev_workspace;
    Cov cv{scene->dev_coverage, nullptr, nullptr};
    if (k) cv = Cov{nullptr, (const float *)(ws + L.area), (float *)(ws + L.gW)};
    const Dims d = dims_of(w, h, n, k, L.total);
    const float4 *S = (const float4 *)(ws + L.S), *T = (const float4 *)(ws + L.T), *B = (const float4 *)(ws + L.B);
    float4 *gB = (float4 *)(ws + L.gB), *gS = (float4 *)(ws + L.gS), *gS2 = (float4 *)(ws + L.gS2);
    const float *wts = (const float *)(ws + L.wts);
    float *part_p = (float *)(ws + L.part_p), *part_m = (float *)(ws + L.part_m), *part_s = (float *)(ws + L.part_s);
    const double px_bytes = (double)w * h * batch;
    const dim3 grid(d.nblk, batch);
    rvk::timed_launch(ctx, "diff_cm_bwd", px_bytes * 80.0, [&] {
        hipLaunchKernelGGL(k_diff_cm_bwd, grid, dim3(kThreads), 0, ctx->stream, d, B, S, dev_params,
                           (const float4 *)dev_grad_out, gB, gS, part_m);
    });
    // B = V(T): dL/dT = V(gB) (into gS2 for now); σ term Σ gB · V'(T)
    const uint32_t by = blur_blocks_y(w, h), bx = blur_blocks_x(w, h);
    rvk::timed_launch(ctx, "diff_blur_bwd", px_bytes * 80.0, [&] {
        hipLaunchKernelGGL(k_diff_blur_y, dim3(by, batch, 2), dim3(64 * kBlurWaves), 0, ctx->stream, d,
                           BlurJob{gB, gS2, nullptr, nullptr}, BlurJob{T, nullptr, gB, part_s}, wts);
    });
    // T = H(S): dL/dS += H(dL/dT) (into gB, free now); σ term Σ dL/dT · H'(S)
    rvk::timed_launch(ctx, "diff_blur_bwd", px_bytes * 80.0, [&] {
        hipLaunchKernelGGL(k_diff_blur_x, dim3(bx, batch, 2), dim3(64 * kBlurWaves), 0, ctx->stream, d,
                           BlurJob{gS2, gB, nullptr, nullptr}, BlurJob{S, nullptr, gS2, part_s + by}, wts);
    });
    rvk::timed_launch(ctx, "diff_paths_bwd", px_bytes * (48.0 + 2.0 * n), [&] {
        hipLaunchKernelGGL(k ? k_diff_paths_bwd<true> : k_diff_paths_bwd<false>, dim3(d.ntile, batch), dim3(kPathThreads),
                           0, ctx->stream, d, cv, (const PathRec *)(ws + L.rec),
                           (const float4 *)(ws + L.ck), (const float4 *)gS, (const float4 *)gB, part_p);
    });
    const uint32_t np_params = n * kPP;
    const size_t pstride = ((size_t)np_params + kGlobalParams) * sizeof(float);
    rvk::timed_launch(ctx, "diff_reduce", 0.0, [&] {
        const uint32_t blocks = (np_params + 15) / 16;
        const ReducePart paths{part_p, dev_grad_params, d.ntile, np_params};
        const ReducePart sigma{part_s, dev_grad_params + np_params, by + bx, 1u};
        const ReducePart matrix{part_m, dev_grad_params + np_params + 1, d.nblk, 20u};
        hipLaunchKernelGGL(k_diff_reduce, dim3(blocks + 3, batch), dim3(1024), 0, ctx->stream, paths, sigma, matrix,
                           blocks, L.total, pstride);
    });
    if (k) {
        const size_t nv = (size_t)k * kFlat + 1;
        const unsigned ge = (unsigned)((n * nv + 255) / 256);
        float4 *egrad = (float4 *)(ws + L.egrad);
        rvk::timed_launch(ctx, "diff_boundary", (double)n * w * h * 4.0 * batch, [&] {
            hipLaunchKernelGGL(k_diff_boundary, dim3(ge, batch), dim3(256), 0, ctx->stream, d,
                               (const float2 *)(ws + L.vert), (const float *)(ws + L.gW), egrad);
            hipLaunchKernelGGL(k_diff_geom_chain, dim3(n, batch), dim3(64), 0, ctx->stream, d, dev_geom,
                               (const float4 *)egrad, dev_grad_geom);
        });
    }
    RVK_HIP_CHECK(hipGetLastError());
    return RVK_OK;
}

rvk_status rvk_diff_backward(rvk_context *ctx, const rvk_diff_scene *scene, const float *dev_params,
                             const float *dev_geom, void *dev_workspace, const float *dev_grad_out,
                             float *dev_grad_params, float *dev_grad_geom) {
    return rvk_diff_backward_batch(ctx, scene, 1, dev_params, dev_geom, dev_workspace, dev_grad_out,
                                   dev_grad_params, dev_grad_geom);
}

}  // extern "C"
