// Box blur (crates/resvg/src/filter/box_blur.rs).  Five rounds of
// [vertical pass, horizontal pass]; every pass rounds to u8, so the ten passes are
// run in the reference's order.  One kernel per round: a 2-D tile plus its halo is
// staged in LDS, the vertical running sums fill an LDS intermediate, and the
// horizontal running sums read it back, so each round reads and writes HBM once.
// The per-pass arithmetic is the reference's: exact integer window sums (zero
// outside the image), times f32 1/(2r+1), round-to-nearest-even, cast to u8.
#include "rvk_internal.h"
#include "device_math.h"
#include <mutex>

using namespace rvkd;

namespace {

constexpr int TW = 64;        // output tile width
constexpr int TH = 32;        // output tile height
constexpr int kThreads = 256;
constexpr int kMaxFusedR = 24;  // halo limit of the fused kernel (LDS budget)

// Back buffer of rvk_box_blur_noalloc: 64 MiB, a 4096 x 4096 RGBA8 image.
constexpr size_t kNoAllocScratchBytes = rvk::kNoAllocBoxBlurBytes;
__device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

__device__ __forceinline__ uint32_t round_pass(uint32_t s, float iarr) {
    // round() of box_blur.rs:327-331 is round-to-nearest-even on [0, 2^22].
    return (uint32_t)rintf((float)s * iarr);
}

// The same integer, as the low byte of a float's bits: the product plus 1.5 * 2^23, whose
// unit in the last place is 1.  The product isn't rounded by itself first, which makes no
// difference: s / (2 r + 1) has an odd divisor and so stays 1 / (4 r + 2), at least 0.01,
// away from every tie, and both products lie within 2^-15 of it.
__device__ __forceinline__ uint32_t round_pass_bits(uint32_t s, float iarr) {
    return __float_as_uint(__builtin_fmaf((float)s, iarr, 12582912.0f));
}

// Sums four u8 channels of packed pixels into four 16-bit lanes of two u32s.
struct Acc {
    uint32_t rb, ga;  // (r | b << 16), (g | a << 16)
    // byte selects (v_perm_b32; selector 0x0c gives a zero byte)
    __device__ __forceinline__ static uint32_t lo(uint32_t p) { return __builtin_amdgcn_perm(0u, p, 0x0c020c00u); }
    __device__ __forceinline__ static uint32_t hi(uint32_t p) { return __builtin_amdgcn_perm(0u, p, 0x0c030c01u); }
    __device__ __forceinline__ void zero() { rb = 0; ga = 0; }
    __device__ __forceinline__ void add(uint32_t p) { rb += lo(p); ga += hi(p); }
    __device__ __forceinline__ void sub(uint32_t p) { rb -= lo(p); ga -= hi(p); }
    __device__ __forceinline__ uint32_t out(float iarr) const {
        const uint32_t r = round_pass_bits(rb & 0xffffu, iarr), g = round_pass_bits(ga & 0xffffu, iarr);
        const uint32_t b = round_pass_bits(rb >> 16, iarr), a = round_pass_bits(ga >> 16, iarr);
        return __builtin_amdgcn_perm(g, r, 0x0c0c0400u) | __builtin_amdgcn_perm(a, b, 0x04000c0cu);
    }
};

// One round: dst = H_rh(V_rv(src)).  Tile covers output [x0, x0+TW) x [y0, y0+TH).
// LDS: in[TH + 2 rv rows][TW + 2 rh cols, to whole chunks], mid[TH rows][(TW + 2 rh) | 1
// cols].  Bound by the vector instructions of the passes and of the staging (a copy of a 4096^2
// image takes 27 us): with LDS addresses by division and a checked store a pixel a round
// of radii 3 took 46.4 us there, now 42.1; 1601 x 1131 9.3 us, now 8.3.
__global__ __launch_bounds__(kThreads) void k_box_round(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst,
                                                        uint32_t w, uint32_t h, int rh, int rv) {
    extern __shared__ __align__(16) uint32_t lds[];
    const int cw = TW + 2 * rh;   // staged columns
    const int ch_ = TH + 2 * rv;  // staged rows
    const int ms = cw | 1;  // odd row stride of mid: the horizontal pass's lanes (rows) hit distinct banks
    const uint2 tile = xcd_tile();
    const int x0 = (int)tile.x * TW, y0 = (int)tile.y * TH;
    // the input tile with zero padding outside the image (fv = lv = 0), in chunks of 4
    // pixels: chunk c of a tile row holds global x in [a0 + 4c, a0 + 4c + 3] and goes to
    // LDS whole, so a row there starts up to 3 columns before the tile
    const int gx0 = x0 - rh, gy0 = y0 - rv;
    const int a0 = gx0 & ~3;
    const int nc = (gx0 + cw - a0 + 3) >> 2, is = 4 * nc;
    uint32_t *in = lds;
    uint32_t *mid = lds + is * ch_;
    // 16-byte loads (which need 4-byte alignment only) where the chunk lies inside the
    // image, single pixels elsewhere
    {
        const float inv_nc = 1.0f / (float)nc;  // (i + 0.5) / nc truncates exactly for these sizes
        const bool inner = a0 >= 0 && a0 + is <= (int)w && gy0 >= 0 && gy0 + ch_ <= (int)h;
        const uint32_t *corner = src + ((int64_t)gy0 * w + a0);  // dereferenced inside the image only
        for (uint32_t i = threadIdx.x; i < (uint32_t)(ch_ * nc); i += kThreads) {
            const uint32_t ly = (uint32_t)(((float)i + 0.5f) * inv_nc), c = i - __umul24(ly, nc);
            uint4 v;
            const uint32_t at = __umul24(ly, w) + 4 * c;  // ly < 2^7, w <= 2^16
            const int gy = gy0 + (int)ly, gx = a0 + 4 * (int)c;
            if (inner || (gy >= 0 && gy < (int)h && gx >= 0 && gx + 3 < (int)w)) {
                const px4 q = *reinterpret_cast<const px4 *>(corner + at);
                v = make_uint4(q[0], q[1], q[2], q[3]);
            } else {
                auto px = [&](int x) {
                    return gy >= 0 && gy < (int)h && x >= 0 && x < (int)w ? src[(size_t)gy * w + x] : 0u;
                };
                v = make_uint4(px(gx), px(gx + 1), px(gx + 2), px(gx + 3));
            }
            reinterpret_cast<uint4 *>(in)[i] = v;
        }
    }
    in += gx0 - a0;
    __syncthreads();
    // vertical pass: each thread walks one staged column over TH/segs rows
    if (rv == 0) {
        for (int i = threadIdx.x; i < cw * TH; i += kThreads) {
            const int ly = i / cw;
            mid[ly * ms + (i - ly * cw)] = in[ly * is + (i - ly * cw)];
        }
    } else {
        const float iarr = 1.0f / (float)(2 * rv + 1);
        // two segments of TH / 2 rows per column: every column's 2 jobs fit one pass of
        // the block (cw <= 112), and the window sum is started (2 rv + 1 adds) only twice
        constexpr int segs = 2, seg_len = TH / segs;
        static_assert(segs * (TW + 2 * kMaxFusedR) <= kThreads, "a job a thread");
        const int seg = (int)threadIdx.x >= cw, col = (int)threadIdx.x - (seg ? cw : 0);
        if (col < cw) {
            const uint32_t *head = in + seg * seg_len * is + col, *tail = head;
            uint32_t *m = mid + seg * seg_len * ms + col;
            Acc acc; acc.zero();
            for (int k = 0; k <= 2 * rv; k++, head += is) acc.add(*head);
            *m = acc.out(iarr);
#pragma unroll 5
            for (int t = 1; t < seg_len; t++) {
                acc.add(*head);
                acc.sub(*tail);
                head += is, tail += is, m += ms;
                *m = acc.out(iarr);
            }
        }
    }
    __syncthreads();
    // horizontal pass: each thread walks a row segment of 8 outputs
    constexpr int segw = 8, nseg = TW / segw;
    const float iarr = 1.0f / (float)(2 * rh + 1);
    for (int job = threadIdx.x; job < TH * nseg; job += kThreads) {
        int row = job % TH, seg = job / TH;
        int gy = y0 + row;
        if (gy >= (int)h) continue;
        const uint32_t *m = mid + row * ms;
        int c0 = seg * segw;
        uint32_t outv[segw];
        if (rh == 0) {
            for (int k = 0; k < segw; k++) outv[k] = m[c0 + k];
        } else {
            Acc acc; acc.zero();
            for (int k = 0; k <= 2 * rh; k++) acc.add(m[c0 + k]);
            outv[0] = acc.out(iarr);
            for (int k = 1; k < segw; k++) {
                acc.add(m[c0 + k + 2 * rh]);
                acc.sub(m[c0 + k - 1]);
                outv[k] = acc.out(iarr);
            }
        }
        int gx = x0 + c0;
        uint32_t *d = dst + (size_t)gy * w + gx;
        if (gx + segw <= (int)w) {
            reinterpret_cast<px4 *>(d)[0] = px4{outv[0], outv[1], outv[2], outv[3]};
            reinterpret_cast<px4 *>(d)[1] = px4{outv[4], outv[5], outv[6], outv[7]};
        } else {
            for (int k = 0; k < segw; k++)
                if (gx + k < (int)w) d[k] = outv[k];
        }
    }
}

// 32-bit per-channel sums for the large-radius fallback (255 * (2r + 1) may exceed 16 bits).
struct Acc32 {
    uint32_t c[4];
    __device__ __forceinline__ void zero() { c[0] = c[1] = c[2] = c[3] = 0; }
    __device__ __forceinline__ void add(uint32_t p) { for (int i = 0; i < 4; i++) c[i] += (p >> (8 * i)) & 0xffu; }
    __device__ __forceinline__ void sub(uint32_t p) { for (int i = 0; i < 4; i++) c[i] -= (p >> (8 * i)) & 0xffu; }
    __device__ __forceinline__ uint32_t out(float iarr) const {
        return pack(round_pass(c[0], iarr), round_pass(c[1], iarr), round_pass(c[2], iarr), round_pass(c[3], iarr));
    }
};

// Fallback for radii beyond the fused kernel's LDS budget: one thread per column
// (vertical) or per row (horizontal) with a running sum read straight from memory.
__global__ void k_box_vert(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, uint32_t w, uint32_t h,
                           int r, int chunk) {
    uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t y0 = blockIdx.y * chunk;
    if (x >= w || y0 >= h) return;
    uint32_t y1 = min(h, y0 + (uint32_t)chunk);
    const float iarr = 1.0f / (float)(2 * r + 1);
    auto at = [&](int64_t y) -> uint32_t { return (y >= 0 && y < (int64_t)h) ? src[(size_t)y * w + x] : 0u; };
    Acc32 acc; acc.zero();
    for (int64_t k = (int64_t)y0 - r; k <= (int64_t)y0 + r; k++) acc.add(at(k));
    dst[(size_t)y0 * w + x] = acc.out(iarr);
    for (uint32_t y = y0 + 1; y < y1; y++) {
        acc.add(at((int64_t)y + r));
        acc.sub(at((int64_t)y - r - 1));
        dst[(size_t)y * w + x] = acc.out(iarr);
    }
}

__global__ void k_box_horz(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, uint32_t w, uint32_t h,
                           int r, int chunk) {
    uint32_t y = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t x0 = blockIdx.y * chunk;
    if (y >= h || x0 >= w) return;
    uint32_t x1 = min(w, x0 + (uint32_t)chunk);
    const float iarr = 1.0f / (float)(2 * r + 1);
    const uint32_t *row = src + (size_t)y * w;
    auto at = [&](int64_t x) -> uint32_t { return (x >= 0 && x < (int64_t)w) ? row[x] : 0u; };
    Acc32 acc; acc.zero();
    for (int64_t k = (int64_t)x0 - r; k <= (int64_t)x0 + r; k++) acc.add(at(k));
    dst[(size_t)y * w + x0] = acc.out(iarr);
    for (uint32_t x = x0 + 1; x < x1; x++) {
        acc.add(at((int64_t)x + r));
        acc.sub(at((int64_t)x - r - 1));
        dst[(size_t)y * w + x] = acc.out(iarr);
    }
}

}  // namespace

namespace rvk {

// create_box_gauss (box_blur.rs:37-71), evaluated in f32 exactly as the reference.
static void box_gauss_sizes(float sigma, int32_t out[5]) {
    if (sigma > 0.0f) {
        const float n = 5.0f;
        float w_ideal = std::sqrt(12.0f * sigma * sigma / n) + 1.0f;
        float fl = std::floor(w_ideal);
        int32_t wl = fl >= 2147483647.0f ? INT32_MAX : (int32_t)fl;
        if (wl % 2 == 0) wl -= 1;
        int32_t wu = wl + 2;
        float wlf = (float)wl;
        float m_ideal = (12.0f * sigma * sigma - n * wlf * wlf - 4.0f * n * wlf - 3.0f * n) / (-4.0f * wlf - 4.0f);
        float mr = std::round(m_ideal);
        size_t m = mr > 0.0f ? (size_t)mr : 0;
        for (size_t i = 0; i < 5; i++) out[i] = i < m ? wl : wu;
    } else {
        for (int i = 0; i < 5; i++) out[i] = 1;
    }
}

// one fused round, a to b (both radii at most kMaxFusedR)
static rvk_status box_round(rvk_context *ctx, const uint32_t *a, uint32_t *b, uint32_t w, uint32_t h, int rh, int rv) {
    // a staged row: at most 3 columns before and 3 behind the tile's
    size_t lds = (size_t)(((TW + 2 * rh + 6) & ~3) * (TH + 2 * rv) + ((TW + 2 * rh) | 1) * TH) * 4;
    dim3 grid(div_up(w, TW), div_up(h, TH));
    // algorithmic bytes: the image read once and written once per blur (8 B/px,
    // whatever the pass count), split evenly over the five rounds
    timed_launch(ctx, "box_blur_round", 8.0 * (double)w * h / 5.0, [&] {
        hipLaunchKernelGGL(k_box_round, grid, dim3(kThreads), lds, ctx->stream, a, b, w, h, rh, rv);
    });
    RVK_HIP_CHECK(hipGetLastError());
    return RVK_OK;
}

// The five rounds with `tmp` (w * h * 4 bytes of device memory) as the back buffer;
// allocates nothing.
static rvk_status box_blur_with(rvk_context *ctx, uint8_t *px, uint32_t w, uint32_t h, double sx, double sy,
                                void *tmp) {
    int32_t bh[5], bv[5];
    box_gauss_sizes((float)sx, bh);
    box_gauss_sizes((float)sy, bv);
    const size_t bytes = (size_t)w * h * 4;
    uint32_t *a = (uint32_t *)px, *b = (uint32_t *)tmp;
    rvk_status st = RVK_OK;
    const double round_bytes = 8.0 * (double)w * h / 5.0;  // as in box_round
    for (int i = 0; i < 5 && st == RVK_OK; i++) {
        int rh = (bh[i] - 1) / 2, rv = (bv[i] - 1) / 2;
        if (rh <= kMaxFusedR && rv <= kMaxFusedR) {
            st = box_round(ctx, a, b, w, h, rh, rv);
            std::swap(a, b);
        } else {
            const int chunk = 256;
            // vertical: a -> b, horizontal: b -> a
            if (rv == 0) {
                if (hipMemcpyAsync(b, a, bytes, hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess) { st = RVK_ERR_HIP; break; }
            } else {
                timed_launch(ctx, "box_blur_vert", round_bytes / 2.0, [&] {
                    hipLaunchKernelGGL(k_box_vert, dim3(div_up(w, 64), div_up(h, chunk)), dim3(64), 0, ctx->stream,
                                       a, b, w, h, rv, chunk);
                });
            }
            if (rh == 0) {
                if (hipMemcpyAsync(a, b, bytes, hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess) { st = RVK_ERR_HIP; break; }
            } else {
                timed_launch(ctx, "box_blur_horz", round_bytes / 2.0, [&] {
                    hipLaunchKernelGGL(k_box_horz, dim3(div_up(h, 64), div_up(w, chunk)), dim3(64), 0, ctx->stream,
                                       b, a, w, h, rh, chunk);
                });
            }
            if (hipGetLastError() != hipSuccess) { st = RVK_ERR_HIP; break; }
        }
    }
    if (st == RVK_OK && a != (uint32_t *)px) {
        if (hipMemcpyAsync(px, a, bytes, hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess) st = RVK_ERR_HIP;
    }
    return st;
}

rvk_status launch_box_blur_to(rvk_context *ctx, uint8_t *src, uint8_t *dst, uint8_t *tmp, uint32_t w, uint32_t h,
                              double sx, double sy) {
    int32_t bh[5], bv[5];
    box_gauss_sizes((float)sx, bh);
    box_gauss_sizes((float)sy, bv);
    uint8_t *work = tmp ? tmp : src;
    for (int i = 0; i < 5; i++) {
        if ((bh[i] - 1) / 2 <= kMaxFusedR && (bv[i] - 1) / 2 <= kMaxFusedR) continue;
        RVK_TRY(launch_copy(ctx, dst, src, (size_t)w * h * 4));
        return box_blur_with(ctx, dst, w, h, sx, sy, work);
    }
    // the odd number of rounds ends in dst: no copy in front, none behind
    const uint32_t *from = (const uint32_t *)src;
    for (int i = 0; i < 5; i++) {
        uint32_t *to = (uint32_t *)(i % 2 == 0 ? dst : work);
        RVK_TRY(box_round(ctx, from, to, w, h, (bh[i] - 1) / 2, (bv[i] - 1) / 2));
        from = to;
    }
    return RVK_OK;
}

rvk_status launch_box_blur(rvk_context *ctx, uint8_t *px, uint32_t w, uint32_t h, double sx, double sy) {
    void *tmp = nullptr;
    RVK_TRY(scratch_alloc(ctx, (size_t)w * h * 4, &tmp));
    const rvk_status st = box_blur_with(ctx, px, w, h, sx, sy, tmp);
    scratch_release(ctx, tmp);
    return st;
}

// ---------------------------------------------------------------------------
// The no-allocation form: the back buffer is a file-scope device array, one per GPU
// for the life of the process.  Its address is looked up once per device, with that
// device current, when a context is created on it; host code uses only that address
// (the array's own name is a host-side stand-in, not a device pointer).
// ---------------------------------------------------------------------------
constexpr int kMaxDevices = 64;
static std::mutex g_noalloc_mu;
static void *g_noalloc_ptr[kMaxDevices] = {};

rvk_status noalloc_init(int device) {
    if (device < 0 || device >= kMaxDevices) return RVK_ERR_INVALID_ARGUMENT;
    std::lock_guard<std::mutex> g(g_noalloc_mu);
    if (g_noalloc_ptr[device]) return RVK_OK;
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
        (void)hipGetLastError();
        set_last_error("hipGetSymbolAddress(scratch)", __FILE__);
        return RVK_ERR_HIP;
    }
    g_noalloc_ptr[device] = p;
    return RVK_OK;
}

rvk_status launch_box_blur_noalloc(rvk_context *ctx, uint8_t *px, uint32_t w, uint32_t h, double sx, double sy) {
    if ((size_t)w * h * 4 > kNoAllocScratchBytes) return RVK_ERR_TOO_LARGE;
    void *tmp = nullptr;
    if (ctx->device >= 0 && ctx->device < kMaxDevices) {
        std::lock_guard<std::mutex> g(g_noalloc_mu);
        tmp = g_noalloc_ptr[ctx->device];
    }
    if (!tmp) return RVK_ERR_HIP;  // the context's set-up could not look the array up
    return box_blur_with(ctx, px, w, h, sx, sy, tmp);
}

}  // namespace rvk
