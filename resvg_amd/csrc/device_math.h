// Device-side numeric helpers with the reference's Rust semantics.  All HIP code
// is compiled with -ffp-contract=off so a*b+c is never fused, matching Rust.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace rvkd {

// four pixels, moved by 16-byte accesses of any 4-byte alignment
typedef uint32_t px4 __attribute__((ext_vector_type(4), aligned(4)));

// Which of `count` pieces of an image a block takes, given its place in dispatch order.
// Blocks go to the 8 XCDs in turn, and an XCD reads what it wrote itself from its own L2,
// what another wrote from beyond it.  So each XCD takes one contiguous eighth of the
// image, in every filter pass and whatever the shape of its pieces: a pass then finds
// its input, and a tile its neighbours' halo, in the L2 at hand (a copy of 12.6 MB that
// the kernel before it wrote: 3.9 us in 16-byte accesses, against 8.4-10.9 with the eighths
// mixed).
__device__ __forceinline__ uint32_t xcd_piece(uint32_t block, uint32_t count) {
    const uint32_t xcd = block & 7u, each = count >> 3, more = count & 7u;
    return xcd * each + min(xcd, more) + (block >> 3);
}
// the piece of a grid whose blocks tile the image row by row: (column, row) of the tile
__device__ __forceinline__ uint2 xcd_tile() {
    const uint32_t i = xcd_piece(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y), r = i / gridDim.x;
    return make_uint2(i - r * gridDim.x, r);
}

// Rust `f32 as u8`: saturating, NaN -> 0, truncation toward zero.
__device__ __forceinline__ uint32_t as_u8(float v) {
    return (uint32_t)fminf(fmaxf(v, 0.0f), 255.0f);  // fmaxf gives 0 for a NaN
}
__device__ __forceinline__ uint32_t as_u8d(double v) {
    if (!(v > 0.0)) return 0u;
    if (v >= 255.0) return 255u;
    return (uint32_t)v;
}
__device__ __forceinline__ int32_t as_i32(float v) {
    if (v != v) return 0;
    if (v >= 2147483647.0f) return 2147483647;
    if (v <= -2147483648.0f) return (-2147483647 - 1);
    return (int32_t)v;
}
__device__ __forceinline__ int32_t as_i32d(double v) {
    if (v != v) return 0;
    if (v >= 2147483647.0) return 2147483647;
    if (v <= -2147483648.0) return (-2147483647 - 1);
    return (int32_t)v;
}

// f32_bound (crates/resvg/src/filter/mod.rs:242-254)
__device__ __forceinline__ float f32_bound(float mn, float v, float mx) {
    if (v > mx) return mx;
    if (v >= mn) return v;
    return mn;
}

// strict-num ApproxEqUlps (crates/usvg/src/tree/geom.rs:9-24)
__device__ __forceinline__ bool approx_eq_ulps(float a, float b, int32_t ulps) {
    if (a == b) return true;
    if (signbit(a) != signbit(b)) return false;
    int32_t d = (int32_t)(__float_as_uint(a) - __float_as_uint(b));
    return d >= -ulps && d <= ulps;
}
__device__ __forceinline__ bool approx_zero_ulps(float a, int32_t ulps) { return approx_eq_ulps(a, 0.0f, ulps); }

__device__ __forceinline__ uint32_t pack(uint32_t r, uint32_t g, uint32_t b, uint32_t a) {
    return r | (g << 8) | (b << 16) | (a << 24);
}
__device__ __forceinline__ uint32_t ch(uint32_t p, int c) { return (p >> (8 * c)) & 0xffu; }

// x / d, correctly rounded, from r = 1 / d: the product, corrected once by its remainder
// (exact in a fused multiply-add).  Holds for the bytes divided here, which a test runs
// through all of; an IEEE division is ten instructions, this is three.
__device__ __forceinline__ float div_r(float x, float d, float r) {
    const float q = x * r;
    return __builtin_fmaf(__builtin_fmaf(-q, d, x), r, q);
}
// c / 255 of a byte
__device__ __forceinline__ float unit(uint32_t c) { return div_r((float)c, 255.0f, 1.0f / 255.0f); }

// multiply_alpha / demultiply_alpha on one packed pixel (filter/mod.rs:129-146)
__device__ __forceinline__ uint32_t premul_px(uint32_t p) {
    float a = unit(ch(p, 3));
    uint32_t r = as_u8((float)ch(p, 0) * a + 0.5f);
    uint32_t g = as_u8((float)ch(p, 1) * a + 0.5f);
    uint32_t b = as_u8((float)ch(p, 2) * a + 0.5f);
    return pack(r, g, b, ch(p, 3));
}
__device__ __forceinline__ uint32_t demul_px(uint32_t p) {
    const float a = unit(ch(p, 3));
    float y = __builtin_amdgcn_rcpf(a);
    y = __builtin_fmaf(__builtin_fmaf(-a, y, 1.0f), y, y);
    if (ch(p, 3) == 0u) y = 1e30f;  // c / 0: 255 for every c but 0
    uint32_t r = as_u8(div_r((float)ch(p, 0), a, y) + 0.5f);
    uint32_t g = as_u8(div_r((float)ch(p, 1), a, y) + 0.5f);
    uint32_t b = as_u8(div_r((float)ch(p, 2), a, y) + 0.5f);
    return pack(r, g, b, ch(p, 3));
}

}  // namespace rvkd
