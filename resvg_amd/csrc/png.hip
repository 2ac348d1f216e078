// PNG scanlines of a pixmap: the device part of tiny-skia's Pixmap::encode_png, which
// resvg's CLI calls to write its output (crates/resvg/src/main.rs:108 and :113).
//
// Every pixel is demultiplied the way PremultipliedColorU8::demultiply does it:
// alpha 255 unchanged, otherwise each colour channel c / (a / 255) + 0.5 in f64 and
// cast to u8 (saturating, NaN to 0) -- the reference's test harness restates the same
// rule at crates/resvg/tests/integration/main.rs:204-211.  On the device a channel is
// floor(c * r(a) + 0.5) in f32, fused, with an r(a) near 255 / a that gives the f64 rule's value
// for all 256 channel values (checked on the host by the same function, png_demul.h); the six
// alphas whose ties no single r gets right have their 256 values in a table.  Each row is
// then filtered with one of the five PNG filter types (ISO/IEC 15948 section 9: None, Sub,
// Up, Average, Paeth; 4 bytes per pixel, bytes left of the row and the row above the
// first count as 0), chosen per row as the type whose filtered bytes, read as signed,
// have the smallest sum of magnitudes (the minimum-sum heuristic of adaptive PNG
// encoders; ties go to the lower type).  The output is the zlib input of the IDAT
// stream: per row its filter type byte, then its 4 * w filtered bytes.
//
// One 256-thread block per row: the straight pixels of the row and the one above (an L2
// hit: it is the previous block's row) go to LDS, a first pass sums the five candidates
// over the row, a second writes the chosen one, all on packed pixels (four bytes a word,
// Paeth on 16-bit pairs).  Rows too long for LDS are read and demultiplied again instead.
// Bound by the VALU (Paeth is half of it).  With byte-wise filters, a 64 KB table read
// three times a pixel, twice a pass, and a launch to build it: 92 us at 3001 x 2003.
#include "png_demul.h"
#include "rvk_internal.h"

using namespace rvk_png;

namespace {

constexpr int kPngBlock = 256;
constexpr uint32_t kPngLdsWidth = 4096;  // widest row whose pixels stay in LDS (two rows: 32 KB)

// the straight pixel of p
__device__ __forceinline__ uint32_t straight(const float *r, const uint8_t (*special)[256], uint32_t p) {
    const float f = r[p >> 24];
    auto ch = [&](uint32_t c) { return straight_channel(c, f); };
    uint32_t v = ch(p & 0xffu) | (ch((p >> 8) & 0xffu) << 8) | (ch((p >> 16) & 0xffu) << 16);
    if (by_table(f)) {
        const uint8_t *row = special[table_row(f)];
        v = (uint32_t)row[p & 0xffu] | ((uint32_t)row[(p >> 8) & 0xffu] << 8) | ((uint32_t)row[(p >> 16) & 0xffu] << 16);
    }
    return v | (p & 0xff000000u);
}

// byte-wise x - y (modulo 256)
__device__ __forceinline__ uint32_t sub4(uint32_t x, uint32_t y) {
    return ((x | 0x80808080u) - (y & 0x7f7f7f7fu)) ^ ((x ^ ~y) & 0x80808080u);
}
typedef short i16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bits(i16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ i16x2 pair(uint32_t v) { return __builtin_bit_cast(i16x2, v); }
// Paeth's choice among left a, above b and upper-left c, two bytes in 16-bit fields: with
// pa = |b - c|, pb = |a - c|, pc = |a + b - 2 c|, a where pa is the least, else b where pb
// is at most pc, else c
__device__ __forceinline__ uint32_t paeth2(uint32_t a, uint32_t b, uint32_t c) {
    const i16x2 va = pair(b) - pair(c), vb = pair(a) - pair(c), vc = va + vb;
    const i16x2 pa = __builtin_elementwise_max(va, -va), pb = __builtin_elementwise_max(vb, -vb),
                pc = __builtin_elementwise_max(vc, -vc);
    const i16x2 bc = __builtin_elementwise_min(pb, pc);
    // 0 where the comparison holds, else -1 in every bit of the field
    const uint32_t not_b = bits((pc - pb) >> 15), not_a = bits((bc - pa) >> 15);
    const uint32_t q = (b & ~not_b) | (c & not_b);
    return (a & ~not_a) | (q & not_a);
}
// the bytes that filter type t subtracts from the pixel (left a, above b, upper-left c)
__device__ __forceinline__ uint32_t paeth4(uint32_t a, uint32_t b, uint32_t c) {
    const uint32_t m = 0x00ff00ffu;
    return paeth2(a & m, b & m, c & m) | (paeth2((a >> 8) & m, (b >> 8) & m, (c >> 8) & m) << 8);
}
__device__ __forceinline__ uint32_t mean4(uint32_t a, uint32_t b) { return __builtin_amdgcn_lerp(a, b, 0u); }
// s + the sum of the bytes' magnitudes, read as signed
__device__ __forceinline__ uint32_t add_mag(uint32_t v, uint32_t s) {
    return __builtin_amdgcn_sad_u8(v ^ 0x80808080u, 0x80808080u, s);
}

template <bool kLds>
__global__ __launch_bounds__(kPngBlock) void k_png_rows(const uint32_t *px, uint32_t w, uint32_t h, Demul t,
                                                       uint8_t *out) {
    typedef uint32_t __attribute__((aligned(1))) unaligned_u32;
    extern __shared__ uint32_t rows[];  // the row and the row above, straight, each after one 0
    __shared__ float rec[256];
    __shared__ uint8_t special[kSpecial][256];
    __shared__ uint32_t part[kPngBlock / 64][5];
    const uint32_t y = blockIdx.x;
    const int tid = (int)threadIdx.x, lane = tid % 64;
    const uint32_t *row = px + (size_t)y * w;
    const uint32_t *up = y > 0 ? row - w : nullptr;
    uint8_t *dst = out + (size_t)y * (4u * (size_t)w + 1u);
    rec[tid] = t.r[tid];
    for (int k = 0; k < kSpecial; k++) special[k][tid] = t.special[k][tid];
    __syncthreads();
    uint32_t *xs = rows, *bs = rows + w + 1;
    if (kLds) {
        for (uint32_t i = tid; i < w; i += kPngBlock) {
            xs[i + 1] = straight(rec, special, row[i]);
            bs[i + 1] = up ? straight(rec, special, up[i]) : 0u;
        }
        if (tid == 0) xs[0] = bs[0] = 0u;
        __syncthreads();
    }
    // pixel i, its left neighbour a, the one above b and the one above its left c
    auto load = [&](uint32_t i, uint32_t &x, uint32_t &a, uint32_t &b, uint32_t &c) {
        if (kLds) {
            x = xs[i + 1];
            a = xs[i];
            b = bs[i + 1];
            c = bs[i];
        } else {
            x = straight(rec, special, row[i]);
            a = i ? straight(rec, special, row[i - 1]) : 0u;
            b = up ? straight(rec, special, up[i]) : 0u;
            c = up && i ? straight(rec, special, up[i - 1]) : 0u;
        }
    };
    uint32_t sum[5] = {0, 0, 0, 0, 0};
    for (uint32_t i = tid; i < w; i += kPngBlock) {
        uint32_t x, a, b, c;
        load(i, x, a, b, c);
        sum[0] = add_mag(x, sum[0]);
        sum[1] = add_mag(sub4(x, a), sum[1]);
        sum[2] = add_mag(sub4(x, b), sum[2]);
        sum[3] = add_mag(sub4(x, mean4(a, b)), sum[3]);
        sum[4] = add_mag(sub4(x, paeth4(a, b, c)), sum[4]);
    }
    // the row's sums: waves reduce by shuffles, then across the block's four waves
    for (int k = 0; k < 5; k++) {
        uint32_t s = sum[k];
        for (int o = 32; o > 0; o >>= 1) s += (uint32_t)__shfl_xor((int)s, o, 64);
        if (lane == 0) part[tid / 64][k] = s;
    }
    __syncthreads();
    uint32_t best = 0;
    uint64_t best_sum = ~0ull;
    for (uint32_t k = 0; k < 5; k++) {
        uint64_t s = 0;
        for (int wv = 0; wv < kPngBlock / 64; wv++) s += part[wv][k];
        if (s < best_sum) { best_sum = s; best = k; }
    }
    best = (uint32_t)__builtin_amdgcn_readfirstlane((int)best);
    if (tid == 0) dst[0] = (uint8_t)best;
    for (uint32_t i = tid; i < w; i += kPngBlock) {
        uint32_t x, a, b, c;
        load(i, x, a, b, c);
        uint32_t v = x;
        if (best == 1) v = sub4(x, a);
        else if (best == 2) v = sub4(x, b);
        else if (best == 3) v = sub4(x, mean4(a, b));
        else if (best == 4) v = sub4(x, paeth4(a, b, c));
        *(unaligned_u32 *)(dst + 1 + 4u * (size_t)i) = v;
    }
}

}  // namespace

extern "C" {

rvk_status rvk_png_filter_rows(rvk_context *ctx, const uint8_t *px, uint32_t w, uint32_t h, uint8_t *out) {
    if (!ctx || !px || !out || !rvk::valid_dims(w, h)) return RVK_ERR_INVALID_ARGUMENT;
    RVK_HIP_CHECK(hipSetDevice(ctx->device));
    static const Demul table = [] {
        Demul t{};
        if (!make_demul(t)) t.r[0] = -100.0f;
        return t;
    }();
    if (table.r[0] < 0.0f) return RVK_ERR_UNSUPPORTED;
    // algorithmic bytes: each pixel read once, 4 bytes per pixel and 1 per row written
    const double bytes = 4.0 * (double)w * h + (4.0 * (double)w + 1.0) * h;
    rvk::timed_launch(ctx, "png_rows", bytes, [&] {
        if (w <= kPngLdsWidth)
            hipLaunchKernelGGL(k_png_rows<true>, dim3(h), dim3(kPngBlock), 8 * ((size_t)w + 1), ctx->stream,
                               (const uint32_t *)px, w, h, table, out);
        else
            hipLaunchKernelGGL(k_png_rows<false>, dim3(h), dim3(kPngBlock), 0, ctx->stream, (const uint32_t *)px, w, h,
                               table, out);
    });
    RVK_HIP_CHECK(hipGetLastError());
    return RVK_OK;
}

}  // extern "C"
