// Device rasterizer: curve expansion, anti-aliased coverage and the fused
// shade/composite of draw lists.
//
// Expansion (k_expand): tiny-skia's quadratic / cubic update loop (Skia's forward
// differencing in 16.16 fixed point) from the state the host left after the first piece,
// a lane per edge, then a lane per segment for its line piece; every non-empty piece is
// written in order.
//
// Coverage (k_coverage): a block of eight 64-lane waves per (coverage job, band of 8
// pixel rows), one wave per row.  The block's threads leave the crossings of the band's
// edges with its sub-scanlines in LDS and sort the edges once (keys: x in the middle of the
// band, edge id, winding); each wave brings its row's four sub-scanlines into order from
// that one by exchanges of neighbours and turns them into span events (tiny-skia's
// walk_edges spans); the SuperBlitter contributions (16 per covered sub-column of a partial
// pixel, 64 or 63 for a fully covered pixel) are accumulated per 1024- or 512-pixel window
// in LDS, prefix-summed and clamped to 255.  Coverage leaves the kernel as 8 x 8 tiles
// aligned to the target: a u16 table entry per tile (empty, full, or the slot of a partial
// tile's 64 bytes), so only tiles that an edge crosses cost memory.  Bands that more edges
// meet than a block holds take one wave each (k_coverage_many).
//
// Compositing (k_draw): one thread per target pixel, one wave per 8 x 8 tile,
// looping over the draw items in order with the pixel in a register: tile-table
// entry -> coverage -> gradient or solid shade (tiny-skia lowp stages) -> SourceOver
// into the target (direct items) or into an elided layer pixel that is then
// composited in f32 with the group's opacity and blend mode (draw_pixmap semantics).
#include <type_traits>
#include "rvk_internal.h"
#include "blend_ops.h"
#include "raster.h"

using namespace rvkd;
using rvkr::CovJob;
using rvkr::DrawCull;
using rvkr::DrawItem;
using rvkr::EdgeCov;
using rvkr::EdgeRec;
using rvkr::HairLine;
using rvkr::PieceDev;
using rvkr::ShaderParams;
using rvkr::ShaderHead;
using rvkr::JobRef;
using rvkr::kMaxStops;

namespace {

constexpr int kWave = 64;
constexpr int kMaxKeys = (int)rvkr::kCoverageKeys[2];  // crossings per sub-scanline of the widest variant
constexpr int kWin = 512;         // pixels k_coverage_many accumulates per window
constexpr int kMaxSub = 4;        // sub-scanlines per pixel row

// ---------------------------------------------------------------------------
// expansion
// ---------------------------------------------------------------------------
__device__ __forceinline__ int32_t fdot6_round(int32_t x) { return (x + 32) >> 6; }
__device__ __forceinline__ int32_t fdot6_to_fixed(int32_t x) { return (int32_t)((uint32_t)x << 10); }
__device__ __forceinline__ int32_t fixed_mul(int32_t a, int32_t b) {
    return (int32_t)(((int64_t)a * (int64_t)b) >> 16);
}
// (a << 16) / b truncated towards zero and saturated, b > 0.  The dividend has at most 47
// bits, so the f64 quotient is off by less than 1 / 64 of the distance 1 / b that a
// non-integral one keeps from the next integer, and its truncation is the integer
// quotient (a 64-bit integer division takes ten times the instructions).
__device__ __forceinline__ int32_t fdot6_div(int32_t a, int32_t b) {
    return as_i32d((double)a * 65536.0 / (double)b);
}

// SkEdge::updateLine on 16.16 inputs
__device__ __forceinline__ bool line_piece(int32_t x0, int32_t y0, int32_t x1, int32_t y1, PieceDev &p) {
    y0 >>= 10;
    y1 >>= 10;
    const int32_t top = fdot6_round(y0), bot = fdot6_round(y1);
    if (top == bot) return false;
    x0 >>= 10;
    x1 >>= 10;
    const int32_t slope = fdot6_div(x1 - x0, y1 - y0);
    const int32_t dy = ((top << 6) + 32) - y0;
    p.x = fdot6_to_fixed(x0 + fixed_mul(slope, dy));
    p.dx = slope;
    p.first_y = top;
    p.last_y = bot - 1;
    return true;
}

struct ExpandArgs {
    const EdgeRec *edges;
    uint32_t nedges;
    const EdgeCov *cov;
    PieceDev *pieces;
    uint32_t *npieces;
    int32_t *overflow;
};

constexpr int kExpandSteps = 64;   // curve segments after the first piece (MAX_COEFF_SHIFT 6: at most 63)

// One wave per E edges (4 or 16, see launch_expand).  A lane per edge runs the curve's update steps, which only add
// and shift, into LDS; then each half of the wave takes an edge at a time, a lane per
// segment: the slope's division (most of the work), and the non-empty pieces compacted in
// order and stored together.  One thread per edge doing both took 15-30 us however few
// edges there were (29.8 -> 11.6 us per launch of a 2048^2 document's clip paths).
template <int E>
__global__ __launch_bounds__(kWave) void k_expand(ExpandArgs a) {
    __shared__ int2 pts[E][kExpandSteps + 1];  // 16.16 points, the first piece's end first
    __shared__ int4 head[E];                   // segments, first piece slot, row bound, the first piece's last row
    const int lane = threadIdx.x;
    const uint32_t first = blockIdx.x * E;
    if (lane < E && first + lane < a.nedges) {
        const EdgeRec e = a.edges[first + lane];
        const int32_t bound = a.cov[first + lane].ymax;
        a.pieces[e.piece_offset] = PieceDev{e.x, e.dx, e.first_y, e.last_y};
        int n = 0;
        int2 at = make_int2(e.cx, e.cy);
        pts[lane][0] = at;
        if (e.type == 1) {  // SkQuadraticEdge::updateQuadratic, repeated until exhausted
            int32_t dx = e.d1x, dy = e.d1y;
            for (int32_t count = e.count; count > 0 && n < kExpandSteps;) {
                if (--count > 0) {
                    at.x += dx >> e.shift;
                    dx += e.d2x;
                    at.y += dy >> e.shift;
                    dy += e.d2y;
                } else {
                    at = make_int2(e.lx, e.ly);
                }
                pts[lane][++n] = at;
            }
        } else if (e.type == 2) {  // SkCubicEdge::updateCubic
            int32_t d1x = e.d1x, d1y = e.d1y, d2x = e.d2x, d2y = e.d2y;
            for (int32_t count = e.count; count < 0 && n < kExpandSteps;) {
                const int32_t oldy = at.y;
                if (++count < 0) {
                    at.x += d1x >> e.dshift;
                    d1x += d2x >> e.shift;
                    d2x += e.d3x;
                    at.y += d1y >> e.dshift;
                    d1y += d2y >> e.shift;
                    d2y += e.d3y;
                } else {
                    at = make_int2(e.lx, e.ly);
                }
                at.y = max(at.y, oldy);
                pts[lane][++n] = at;
            }
        }
        head[lane] = make_int4(n, (int)e.piece_offset, bound, e.last_y);
    }
    __syncthreads();
    const int half = lane >> 5, hl = lane & 31;
    for (int k = half; k < E; k += 2) {
        const uint32_t i = first + (uint32_t)k;
        if (i >= a.nedges) break;
        const int4 h = head[k];
        const int n = h.x;
        PieceDev *out = a.pieces + (uint32_t)h.y;
        uint32_t count = 1;
        bool over = h.w > h.z;
        for (int j0 = 0; j0 < n; j0 += 32) {
            const int j = j0 + hl;
            PieceDev p;
            bool ok = false;
            if (j < n) {
                const int2 u = pts[k][j], v = pts[k][j + 1];
                ok = line_piece(u.x, u.y, v.x, v.y, p);
            }
            const uint32_t m = (uint32_t)(__ballot(ok) >> (32 * half));
            if (ok) {
                out[count + __popc(m & ((1u << hl) - 1u))] = p;
                over = over || p.last_y > h.z;
            }
            count += __popc(m);
        }
        if (hl == 0) a.npieces[i] = count;
        // the host's row bound must cover every piece (else rows would miss the edge)
        if (over) atomicAdd(a.overflow, 1);
    }
}

// ---------------------------------------------------------------------------
// coverage
// ---------------------------------------------------------------------------
struct CovArgs {
    const uint2 *bands;  // (job, band) of each block of this launch
    const CovJob *jobs;
    const EdgeCov *edges;
    const uint2 *windows;
    const PieceDev *pieces;
    const uint32_t *npieces;
    uint16_t *table;
    uint8_t *arena;
    int32_t *overflow;
};

// Inclusive sum over the wave's lanes in six DPP additions (shifts within the 16-lane
// rows, then the row totals broadcast to the rows after them); no LDS traffic.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_from(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ int wave_incl_scan(int v) {
    v += dpp_from<0x111, 0xf>(v);  // row_shr:1
    v += dpp_from<0x112, 0xf>(v);
    v += dpp_from<0x114, 0xf>(v);
    v += dpp_from<0x118, 0xf>(v);
    v += dpp_from<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v += dpp_from<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    return v;
}

// set bits of `m` below this lane
__device__ __forceinline__ int lanes_below(uint64_t m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Lane exchange across xor distance LD (1..32) for the bitonic network, all in the VALU
// (the coverage kernel's LDS pipe is busy with keys and accumulators): DPP patterns
// within the 16-lane rows, row and half swaps across them.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_perm(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, true);
}
template <int LD>
__device__ __forceinline__ uint32_t xor_lane(uint32_t v, int lane) {
    if constexpr (LD == 1) return dpp_perm<0xB1>(v);                    // quad_perm [1, 0, 3, 2]
    else if constexpr (LD == 2) return dpp_perm<0x4E>(v);               // quad_perm [2, 3, 0, 1]
    else if constexpr (LD == 4) return dpp_perm<0x1B>(dpp_perm<0x141>(v));  // mirror of 8, then of 4
    else if constexpr (LD == 8) return dpp_perm<0x128>(v);              // row_ror:8
    else if constexpr (LD == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (lane & 16) ? r[0] : r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (lane & 32) ? r[0] : r[1];
    }
}

// One stage (k, jj) of an ascending bitonic network over S independent arrays of
// 64*K keys, element e = lane*K + j of array s in v[s][j].
template <int K, int S, int k, int jj>
__device__ __forceinline__ void bitonic_stage(uint64_t (&v)[S][K], int lane) {
    if constexpr (jj >= K) {
        constexpr int ld = jj / K;
        // e & k and e & jj depend on the lane only; keep the smaller key when the pair
        // is ascending and this is its lower element, or descending and upper
        const bool up = k >= kWave * K ? true : (lane & (k / K)) == 0;
        const bool keep_min = up == ((lane & ld) == 0);
#pragma unroll
        for (int s = 0; s < S; s++)
#pragma unroll
            for (int j = 0; j < K; j++) {
                const uint64_t x = v[s][j];
                const uint64_t o = ((uint64_t)xor_lane<ld>((uint32_t)(x >> 32), lane) << 32) |
                                   xor_lane<ld>((uint32_t)x, lane);
                v[s][j] = ((o < x) == keep_min) ? o : x;
            }
    } else {
#pragma unroll
        for (int j = 0; j < K; j++) {
            if ((j & jj) == 0) {
                const int p = j | jj;
                const bool up = k >= K ? (k >= kWave * K ? true : (lane & (k / K)) == 0) : (j & k) == 0;
#pragma unroll
                for (int s = 0; s < S; s++) {
                    const uint64_t x = v[s][j], y = v[s][p];
                    const bool sw = (x > y) == up;
                    v[s][j] = sw ? y : x;
                    v[s][p] = sw ? x : y;
                }
            }
        }
    }
}

template <int K, int S, int k, int jj>
__device__ __forceinline__ void bitonic_from(uint64_t (&v)[S][K], int lane) {
    bitonic_stage<K, S, k, jj>(v, lane);
    if constexpr (jj > 1) bitonic_from<K, S, k, jj / 2>(v, lane);
    else if constexpr (k < kWave * K) bitonic_from<K, S, k * 2, k>(v, lane);
}

// Sorts the S sub-scanlines' keys (n[s] each, in keys[s]) together and writes each
// one's span events (pixel-rounded supersampled columns; starts and ends alternate)
// over its own key area.  Returns the event counts in nev.
// A column chunk of the row (crossings rounded to [c0, c1) only) starts from the
// backdrop winding base[s] of the crossings left of it: inside a span there, the
// events get a leading start at c0, and a span still open after the last crossing
// gets an end at c1.  The whole row is the chunk with base 0 (closed paths end
// outside).
template <int K, int S, int MK>
__device__ __forceinline__ void spans_of(uint64_t (*keys)[MK], const int *n, bool evenodd, int *nev, int lane,
                                         const int *base, int32_t c0, int32_t c1) {
    static_assert(K * 64 <= MK, "each lane's K keys stay inside its sub-scanline's key row");
    uint64_t v[S][K];
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int e = lane * K + j;
            v[s][j] = e < n[s] ? keys[s][e] : ~0ull;
        }
    __syncthreads();  // every key is in registers before the key areas are reused for events
    bitonic_from<K, S, 2, 1>(v, lane);
#pragma unroll
    for (int s = 0; s < S; s++) {
        int w[K], local = 0;
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int e = lane * K + j;
            w[j] = e < n[s] ? ((v[s][j] & 1) ? 1 : -1) : 0;
            local += w[j];
        }
        const int incl = wave_incl_scan(local);
        int before = base[s] + incl - local;
        const bool in0 = evenodd ? (base[s] & 1) != 0 : base[s] != 0;
        const int total = base[s] + __shfl(incl, kWave - 1, kWave);
        const bool in1 = evenodd ? (total & 1) != 0 : total != 0;
        bool evt[K];
        int nevt = 0;
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int after = before + w[j];
            const bool in_b = evenodd ? (before & 1) != 0 : before != 0;
            const bool in_a = evenodd ? (after & 1) != 0 : after != 0;
            evt[j] = w[j] != 0 && in_b != in_a;
            nevt += evt[j] ? 1 : 0;
            before = after;
        }
        const int eincl = wave_incl_scan(nevt);
        int pos = eincl - nevt + (in0 ? 1 : 0);
        int32_t *ev = reinterpret_cast<int32_t *>(keys[s]);
#pragma unroll
        for (int j = 0; j < K; j++)
            if (evt[j]) {
                const int32_t x = (int32_t)((uint32_t)(v[s][j] >> 32) ^ 0x80000000u);
                ev[pos++] = (x + 0x8000) >> 16;
            }
        const int ne = (in0 ? 1 : 0) + __shfl(eincl, kWave - 1, kWave);
        if (lane == 0 && in0) ev[0] = c0;
        if (lane == 0 && in1) ev[ne] = c1;
        nev[s] = ne + (in1 ? 1 : 0);
    }
}

// tile state of k_coverage_many (u16): 0..255 a tile whose rows so far are all
// that value, kStatePartial + k a partial tile holding slot k
constexpr uint32_t kStatePartial = 256u;
static_assert(rvkr::kMaxTilesX + kStatePartial <= 65536u, "a partial tile's state fits 16 bits");
static_assert(kWin == 8 * kWave, "a lane holds one 8-pixel tile row of a window");

// ---- coverage of a band, one wave per pixel row ----
constexpr int32_t kOpenEnd = 0x3fffffff;  // the end of a span that its sub-scanline leaves open
// exchanges of neighbours tried before a full sort: a 4096^2 render of 2000 paths takes
// 105.2, 102.9, 101.9, 101.6, 101.6 and 102.0 ms with 1, 2, 4, 6, 10 and 20
constexpr int kSettlePasses = 6;

// The low word of an edge's key: its id (orders equal x), its slot in the band's list and
// its direction (1: downwards).  The host keeps jobs of more than 2^22 edges out of
// k_coverage, whose slots fit 9 bits.
__device__ __forceinline__ uint32_t edge_low(int32_t id, int slot, int32_t winding) {
    return ((uint32_t)id << 10) | ((uint32_t)slot << 1) | (winding > 0 ? 1u : 0u);
}
__device__ __forceinline__ int low_slot(uint32_t lo) { return (int)((lo >> 1) & 511u); }
__device__ __forceinline__ uint64_t edge_key(int32_t x, uint32_t lo) {
    return ((uint64_t)((uint32_t)x ^ 0x80000000u) << 32) | lo;
}

// A key of the next lane (~0 past the last) and of the one before (0 before the first).
__device__ __forceinline__ uint64_t next_lane(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)(uint32_t)v, 0x130, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)(uint32_t)(v >> 32), 0x130, 0xf, 0xf, false);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t prev_lane(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, 0x138, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), 0x138, 0xf, 0xf, false);
    return ((uint64_t)hi << 32) | lo;
}

// Sorts 64 J keys (element lane * J + j in v[0][j]) that are nearly in order: neighbours
// are exchanged until none is out of order, or the full network sorts them after
// kSettlePasses rounds.
template <int J>
__device__ __forceinline__ void settle(uint64_t (&v)[1][J], int lane) {
    uint64_t(&u)[J] = v[0];
    auto order = [&](int a, int b) {
        const bool sw = u[a] > u[b];
        const uint64_t x = sw ? u[b] : u[a];
        u[b] = sw ? u[a] : u[b];
        u[a] = x;
    };
    for (int pass = 0;; pass++) {
        bool bad = u[J - 1] > next_lane(u[0]);
#pragma unroll
        for (int j = 0; j + 1 < J; j++) bad = bad || u[j] > u[j + 1];
        if (__ballot(bad) == 0) return;
        if (pass == kSettlePasses) break;
        if constexpr (J == 1) {
            // lanes 2 i, 2 i + 1, then 2 i + 1, 2 i + 2
#pragma unroll
            for (int odd = 0; odd < 2; odd++) {
                const uint64_t up = next_lane(u[0]), down = prev_lane(u[0]);
                if ((lane & 1) == odd) u[0] = up < u[0] ? up : u[0];
                else u[0] = down > u[0] ? down : u[0];
            }
        } else {
#pragma unroll
            for (int j = 0; j + 1 < J; j += 2) order(j, j + 1);
#pragma unroll
            for (int j = 1; j + 1 < J; j += 2) order(j, j + 1);
            const uint64_t up = next_lane(u[0]), down = prev_lane(u[J - 1]);
            u[J - 1] = up < u[J - 1] ? up : u[J - 1];
            u[0] = down > u[0] ? down : u[0];
        }
    }
    bitonic_from<J, 1, 2, 1>(v, lane);
}

// The span events of one row's sub-scanlines (pixel-rounded supersampled columns; starts
// and ends alternate) and their counts in nev.  ev[s][slot] holds the x of the band's edge
// `slot` on sub-scanline s, and is replaced by the events; bit shift + s of act[slot] says
// that the edge crosses it (where it does not, x is that of its nearer end, so the order
// stays the same from one sub-scanline to the next); ord holds the edges' low words in the
// order of their x in the middle of the band.
// Each sub-scanline starts from the order of the one before it, which is nearly always
// its own: of the full sorts that took 1300 of 2100 VALU instructions a row (128 edges;
// 8000 of 9000 with 512), a check or a few exchanges of neighbours remain.
// Every crossing changes the winding by one, so with U downward crossings among the A
// before an element the winding there is 2 U - A, and ballots give every prefix; under
// the even-odd rule every crossing is an event.
template <int J, int STRIDE>
__device__ __forceinline__ void row_spans(int32_t (*ev)[STRIDE], const uint32_t *act, int shift, const uint32_t *ord,
                                          int nact, int nsub, bool evenodd, int *nev, int lane) {
    uint32_t lo[J];
    bool off = false, on_any = false;
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int e = lane * J + j;
        lo[j] = ord[e < nact ? e : 0];
        const uint32_t bits = (act[low_slot(lo[j])] >> shift) & 15u;
        off = off || (e < nact && bits != (nsub == 1 ? 1u : 15u));
        on_any = on_any || (e < nact && bits != 0);
    }
    const bool all = __ballot(off) == 0;  // every edge crosses every sub-scanline of the row
    if (__ballot(on_any) == 0) return;
#pragma unroll
    for (int s = 0; s < kMaxSub; s++) {
        if (s >= nsub) break;
        uint64_t v[1][J];
#pragma unroll
        for (int j = 0; j < J; j++)
            v[0][j] = lane * J + j < nact ? edge_key(ev[s][low_slot(lo[j])], lo[j]) : ~0ull;
        settle<J>(v, lane);
        bool on[J], up[J];
        int32_t x[J];
        int below = 0, before = 0;
#pragma unroll
        for (int j = 0; j < J; j++) {
            const bool real = lane * J + j < nact;
            x[j] = ((int32_t)((uint32_t)(v[0][j] >> 32) ^ 0x80000000u) + 0x8000) >> 16;
            if (real) lo[j] = (uint32_t)v[0][j];
            on[j] = real && (all || ((act[low_slot(lo[j])] >> (shift + s)) & 1u) != 0);
            up[j] = on[j] && (lo[j] & 1u) != 0;
            below += lanes_below(__ballot(on[j]));
            before += 2 * lanes_below(__ballot(up[j]));
        }
        before -= below;
        int pos = 0, total = 0;
        bool evt[J];
        if (evenodd) {
            pos = below;
#pragma unroll
            for (int j = 0; j < J; j++) {
                evt[j] = on[j];
                total += __popcll(__ballot(on[j]));
            }
        } else {
#pragma unroll
            for (int j = 0; j < J; j++) {
                const int after = before + (up[j] ? 1 : -1);
                evt[j] = on[j] && (before == 0 || after == 0);
                before = on[j] ? after : before;
                const uint64_t m = __ballot(evt[j]);
                pos += lanes_below(m);
                total += __popcll(m);
            }
        }
#pragma unroll
        for (int j = 0; j < J; j++)
            if (evt[j]) ev[s][pos++] = x[j];
        if (total & 1) {
            if (lane == 0) ev[s][total] = kOpenEnd;
            total++;
        }
        nev[s] = total;
    }
}

constexpr int kRowWaves = rvkr::kBandRows;        // waves of a block: one per pixel row of the band
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// MK: edges that the band holds (128, 256 or 512).  The host sends a band to the
// smallest variant that holds the edges whose rows meet it.
//
// Block b handles band bands[b].y (8 pixel rows) of job bands[b].x, wave r its row r.
// * The 512 threads pick the band's active edges out of its window.  Then MK / 64
//   threads share an edge: each walks the pieces over its J rows and leaves the crossing
//   of every sub-scanline in LDS (x by sub-scanline and edge, and an edge's sub-scanlines
//   as a bit mask).
// * One wave sorts the edges by their x in the middle of the band (a bitonic network over
//   64 J keys held in registers, exchanged in the VALU).  From that order each wave settles
//   its row's sub-scanlines one after the other (row_spans) and turns them into span events,
//   which take the crossings' place in LDS.
// * Per 512- or 1024-pixel window a wave adds its spans' coverage as differences (16 bit,
//   two pixels a word, exact modulo 2^32), each lane prefix-sums one or two 8-pixel tile
//   rows, and the waves agree on which of the window's tiles are all 0, all 255 or partial
//   through 64-bit masks; each writes its row of the partial tiles.
// Windows alternate between three mask slots, so one barrier a window is enough.
//
// Why a wave per row: a row's work is a chain of dependent steps (piece loads, sort
// stages, window scans), and one wave walking its band's 8 rows took 90-200 us however
// small the launch, with the wider variants' few bands leaving the chip idle (the 512
// variant's VALU 13% busy).  Per row the old form issued 2400 VALU, 1600 SALU and 450 LDS
// wave instructions, the LDS pipe as busy as the VALU; scans and sort exchanges moved to
// DPP, winding prefixes to ballots, and differences instead of two packed sums.  With
// 37 KB of LDS and 38 VGPRs the 128 variant runs 8 waves per SIMD (4 before).  Renders:
// 4096^2, 2000 paths 150.4 -> 120.7 ms; 1201x843, 64 paths 3.36 -> 1.95 ms; 2048^2 with
// 150 clipped or masked groups 90.1 -> 64.6 ms; 64 documents in a batch 109 -> 87 ms.
template <int MK>
__global__ __launch_bounds__(kRowWaves * kWave) void k_coverage(CovArgs a) {
    constexpr int J = MK / kWave;          // keys per lane, and rows per thread of the gather
    constexpr int PARTS = rvkr::kBandRows / J;
    constexpr int kThreads = kRowWaves * kWave;
    static_assert(PARTS * MK == kThreads, "a thread per edge and J rows");
    // tiles per lane of a window: 1024 pixels (a fifth fewer instructions a row), or 512
    // where the larger accumulators would cost a block per CU (256: 23% slower with 1024)
    constexpr int T = MK <= 128 ? 2 : 1;
    constexpr int32_t kRowWin = rvkr::kTile * kWave * T;
    constexpr int kAccWords = kRowWin / 2 + 4;  // a window's pixel differences, two per word, and their spill
    constexpr int kStride = MK + 4;        // a row of crossings, and its events with an open end
    __shared__ __align__(16) int32_t xs[rvkr::kBandRows * kMaxSub][kStride];
    __shared__ uint32_t act[PARTS][MK];    // bits (row in the part) * 4 + sub-scanline
    __shared__ uint32_t meta[MK];          // low words by slot
    __shared__ uint32_t list[MK];          // edges by slot, then the low words in x order
    __shared__ __align__(16) uint32_t acc[kRowWaves][kAccWords];
    __shared__ int wcount[kRowWaves];
    __shared__ __align__(16) uint64_t masks[3][2 * T];  // tiles of the window that are 0 / 255 in every row so far
    const int tid = threadIdx.x, lane = tid % kWave;
    const int r = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint2 bj = a.bands[blockIdx.x];
    const CovJob job = a.jobs[bj.x];
    const uint32_t band = bj.y;
    const int shift = job.aa ? 2 : 0, nsub = 1 << shift;
    const bool evenodd = job.rule == RVK_FILL_EVENODD;
    const int32_t row0 = job.gy0 + (int32_t)band * rvkr::kBandRows;
    const int32_t ry0 = max(row0, job.y0), ry1 = min(row0 + rvkr::kBandRows, job.y0 + job.h);  // covered rows
    const EdgeCov *edges = a.edges + job.edge_offset;

    // ---- the band's active edges ----
    const int32_t sb0 = ry0 << shift, sb1 = (ry1 << shift) - 1;  // covered sub-scanlines
    const uint2 win = a.windows[job.window_offset + band];
    for (int i = tid; i < kRowWaves * kAccWords; i += kThreads) (&acc[0][0])[i] = 0;
    if (tid < 6 * T) masks[tid / (2 * T)][tid % (2 * T)] = ~0ull;
    int nact = 0;
    for (uint32_t base = win.x; base < win.y; base += kThreads) {
        const uint32_t i = base + (uint32_t)tid;
        bool meets = false;
        if (i < win.y) {
            const int2 rows = *reinterpret_cast<const int2 *>(&edges[i].first_y);  // first_y, ymax
            meets = rows.x <= sb1 && rows.y >= sb0;
        }
        const uint64_t m = __ballot(meets);
        if (lane == 0) wcount[r] = __popcll(m);
        __syncthreads();
        int pos = nact + lanes_below(m);
#pragma unroll
        for (int w = 0; w < kRowWaves; w++) {
            const int c = wcount[w];
            if (w < r) pos += c;
            nact += c;
        }
        if (meets && pos < MK) list[pos] = i;
        __syncthreads();
    }
    if (nact > MK) {  // the host's count was too small: reported, the rest dropped
        if (tid == 0) atomicAdd(a.overflow, 1);
        nact = MK;
    }
    // ---- their crossings ----
    {
        const int slot = tid % MK, part = tid / MK;
        if (slot < nact) {
            const uint32_t i = list[slot];
            const EdgeCov e = edges[i];
            const PieceDev *pc = a.pieces + e.piece_offset;
            const uint32_t n = a.npieces[job.edge_offset + i];
            const int32_t y0 = row0 + part * J;
            const int32_t s0 = max(y0, ry0) << shift, s1 = min(y0 + J, ry1) << shift;
            uint32_t bits = 0;
            if (part == 0) meta[slot] = edge_low(e.id, slot, e.winding);
            if (s0 < s1) {
                uint32_t k = 0;
                if (e.first_y < s0) {  // the first piece that reaches s0, or the last one
                    uint32_t hi = n - 1;
                    while (k < hi) {
                        const uint32_t mid = (k + hi) >> 1;
                        if (pc[mid].last_y < s0) k = mid + 1;
                        else hi = mid;
                    }
                }
                PieceDev p = pc[k];
                for (int32_t sy = s0; sy < s1; sy++) {
                    while (p.last_y < sy && k + 1 < n) p = pc[++k];
                    const int32_t y = sy >> shift, s = sy - (y << shift);
                    const int32_t at = min(max(sy, p.first_y), p.last_y);
                    xs[(y - row0) * kMaxSub + s][slot] =
                        (int32_t)((uint32_t)p.x + (uint32_t)(at - p.first_y) * (uint32_t)p.dx);
                    if (at == sy) bits |= 1u << ((y - y0) * kMaxSub + s);
                }
            }
            act[part][slot] = bits;
        }
    }
    __syncthreads();
    // ---- their order in the middle of the band ----
    if (r == 0 && nact > 0) {
        const int32_t sm = (sb0 + sb1) >> 1, ym = sm >> shift;
        const int32_t *xm = xs[(ym - row0) * kMaxSub + (sm - (ym << shift))];
        auto sort_slots = [&](auto &v, auto jc) {
            constexpr int JJ = decltype(jc)::value;
#pragma unroll
            for (int j = 0; j < JJ; j++) {
                const int e = lane * JJ + j;
                v[0][j] = e < nact ? edge_key(xm[e], meta[e]) : ~0ull;
            }
            bitonic_from<JJ, 1, 2, 1>(v, lane);
#pragma unroll
            for (int j = 0; j < JJ; j++)
                if (lane * JJ + j < nact) list[lane * JJ + j] = (uint32_t)v[0][j];
        };
        if (J > 1 && nact <= kWave) {
            uint64_t v[1][1];
            sort_slots(v, std::integral_constant<int, 1>());
        } else {
            uint64_t v[1][J];
            sort_slots(v, std::integral_constant<int, J>());
        }
    }
    __syncthreads();
    // ---- this row's span events ----
    int32_t(*ev)[kStride] = &xs[r * kMaxSub];
    int nev[kMaxSub] = {0, 0, 0, 0};
    if (nact > 0 && row0 + r >= ry0 && row0 + r < ry1) {
        if (J > 1 && nact <= kWave)
            row_spans<1>(ev, act[r / J], r % J * kMaxSub, list, nact, nsub, evenodd, nev, lane);
        else
            row_spans<J>(ev, act[r / J], r % J * kMaxSub, list, nact, nsub, evenodd, nev, lane);
    }
    // ---- windows ----
    const int sl = lane >> 4;  // lanes 16 s .. 16 s + 15 look at sub-scanline s's spans
    const int nspl = (sl < 2 ? (sl == 0 ? nev[0] : nev[1]) : (sl == 2 ? nev[2] : nev[3])) >> 1;
    const int32_t *evl = ev[sl];
    const bool any = (nev[0] | nev[1] | nev[2] | nev[3]) != 0;
    const int32_t maxv = job.aa ? (sl == 3 ? 63 : 64) : 255;
    const int32_t rx0 = job.x0, rx1 = job.x0 + job.w;  // covered columns
    const int32_t cw = (int32_t)job.tiles_x * rvkr::kTile;
    uint32_t *wacc = acc[r];
    uint16_t *tab = a.table + job.table_offset + (size_t)band * job.tiles_x;
    uint8_t *slots = a.arena + job.cov_offset + (size_t)band * job.tiles_x * 64u;
    uint32_t nslots = 0;  // partial tiles of the band so far
    int kst = 0;          // the first span of this lane's sub-scanline not behind the windows
    int mslot = 0, wi = 0;
    for (int32_t wx0 = 0; wx0 < cw; wx0 += kRowWin, wi++) {
        const int32_t ww = min(kRowWin, cw - wx0);  // a multiple of kTile
        const int32_t wabs = job.gx0 + wx0;
        uint32_t w[2 * T] = {};  // this lane's tile rows, 8 bytes each
        if (any) {
            // spans cut to the window and to the job's columns (coverage is 0 outside)
            const int32_t colbase = wabs << shift, wend = colbase + (ww << shift);
            const int32_t lo = max(0, rx0 - wabs) << shift, hi = max(0, min(ww, rx1 - wabs)) << shift;
            // the next 16 spans of each sub-scanline: those that start before the window's
            // end are a prefix of them, as are those that end at or before it
            // (a sub-scanline whose 16 spans all end there is looked at again)
            bool live = true;
            do {
                const int k = kst + (lane & 15);
                int32_t L = INT32_MAX, R = INT32_MAX;
                if (live && k < nspl) {
                    L = evl[2 * k];
                    R = evl[2 * k + 1];
                }
                const bool in = L < wend;
                if (in) {
                    const int32_t l = max(L - colbase, lo), h = min(R - colbase, hi);
                    if (h > l) {
                        auto add = [&](int32_t p, int32_t d) { atomicAdd(&wacc[p >> 1], (uint32_t)d << ((p & 1) * 16)); };
                        if (!job.aa) {
                            add(l, 255);
                            add(h, -255);
                        } else {
                            const int32_t pl = l >> 2, pr = h >> 2, fb = l & 3, fe = (h & 3) * 16;
                            if (pl == pr) {
                                const int32_t d = fe - fb * 16;
                                add(pl, d);
                                add(pl + 1, -d);
                            } else {
                                const int32_t first = fb ? 64 - fb * 16 : maxv;  // pixel pl; then full ones, then fe
                                add(pl, first);
                                if (pr > pl + 1) {
                                    if (first != maxv) add(pl + 1, maxv - first);
                                    add(pr, fe - maxv);
                                } else {
                                    add(pr, fe - first);
                                }
                                if (fe) add(pr + 1, -fe);
                            }
                        }
                    }
                }
                const uint64_t mdone = __ballot(R <= wend);
                const uint32_t half = sl < 2 ? (uint32_t)mdone : (uint32_t)(mdone >> 32);
                const uint32_t done = (half >> (16 * (sl & 1))) & 0xffffu;
                kst += __popc(done);
                live = done == 0xffffu;
            } while (__ballot(live) != 0);
            // ---- prefix sum: lane l holds pixels [8 T l, 8 T (l + 1)), T tile rows; the
            // accumulator is cleared behind the read ----
            uint32_t q[4 * T];
#pragma unroll
            for (int t = 0; t < T; t++) {
                uint4 *at = reinterpret_cast<uint4 *>(&wacc[4 * (T * lane + t)]);
                const uint4 u = *at;
                *at = make_uint4(0, 0, 0, 0);
                q[4 * t] = u.x;
                q[4 * t + 1] = u.y;
                q[4 * t + 2] = u.z;
                q[4 * t + 3] = u.w;
            }
            if (lane == 0) wacc[kRowWin / 2] = 0;
            // a word is lo + 65536 hi of two signed differences, so the words' sum is the
            // sums of both, and word * 65537 the running pair
            uint32_t sum = 0;
#pragma unroll
            for (int i = 0; i < 4 * T; i++) sum += q[i];
            const int32_t slo = (int32_t)(int16_t)sum;
            const int32_t loc = slo + ((int32_t)(sum - (uint32_t)slo) >> 16);
            uint32_t before = (uint32_t)(wave_incl_scan(loc) - loc) << 16;  // the pixel before, in the high half
#pragma unroll
            for (int i = 0; i < 4 * T; i++) {
                before = (q[i] << 16) + __builtin_amdgcn_perm(before, before, 0x03020302u) + q[i];
                q[i] = before;
            }
            // each field is a pixel's coverage, at most 256: 256 becomes 255
            auto clamp2 = [](uint32_t p) {
                const u16x2 c = {255, 255};
                return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, p), c));
            };
#pragma unroll
            for (int i = 0; i < 2 * T; i++)
                w[i] = __builtin_amdgcn_perm(clamp2(q[2 * i + 1]), clamp2(q[2 * i]), 0x06040200u);
        }
        // ---- the window's tiles: T masks (tile T l + t in bit l of mask t) ----
        uint64_t mz[T], mf[T];
#pragma unroll
        for (int t = 0; t < T; t++) {
            const bool valid = 8 * (T * lane + t) < ww;
            mz[t] = __ballot(!valid || (w[2 * t] | w[2 * t + 1]) == 0u);
            mf[t] = __ballot(valid && (w[2 * t] & w[2 * t + 1]) == ~0u);
        }
        if (lane < 2 * T) {
            uint64_t m = lane & 1 ? mf[0] : mz[0];
            if (T > 1 && lane >= 2) m = lane & 1 ? mf[T - 1] : mz[T - 1];
            atomicAnd((unsigned long long *)&masks[mslot][lane], (unsigned long long)m);
        }
        const int next = mslot == 2 ? 0 : mslot + 1;
        if (tid < 2 * T) masks[next][tid] = ~0ull;  // last read before the previous barrier
        __syncthreads();
        uint64_t part[T];
        uint32_t k = nslots;
#pragma unroll
        for (int t = 0; t < T; t++) {
            mz[t] = masks[mslot][2 * t];
            part[t] = ~(mz[t] | masks[mslot][2 * t + 1]);
            k += (uint32_t)lanes_below(part[t]);
            nslots += (uint32_t)__popcll(part[t]);
        }
#pragma unroll
        for (int t = 0; t < T; t++) {
            const bool mine = (part[t] >> lane) & 1ull;
            if (mine) *reinterpret_cast<uint2 *>(slots + (size_t)k * 64u + r * 8) = make_uint2(w[2 * t], w[2 * t + 1]);
            if (r == ((T * wi + t) & (kRowWaves - 1)) && 8 * (T * lane + t) < ww)
                tab[wx0 / rvkr::kTile + T * lane + t] =
                    (uint16_t)(mine ? rvkr::kTileSlot0 + k
                                    : ((mz[t] >> lane) & 1ull ? rvkr::kTileEmpty : rvkr::kTileFull));
            k += mine ? 1u : 0u;
        }
        mslot = next;
    }
}

// A band that more edges meet than k_coverage<kMaxKeys> holds (many short edges, such as
// the arcs of round joins): one 64-lane wave per band, row by row over every edge of the
// band's window, with up to kMaxKeys crossings per sub-scanline sorted at a time.  A
// sub-scanline with more is redone in narrower column chunks.  The spans are accumulated
// per 512-pixel window in LDS, prefix-summed and clamped to 255.  Each lane then holds
// one 8-pixel row of a tile, which is tracked as uniform (every pixel so far one value)
// or partial: a tile turns partial at the first row that differs, takes the band's next
// slot, and from then on its rows are written there (the earlier, uniform rows are filled
// in at that point); at the end of the band the tile table gets empty, full or the slot.
__global__ __launch_bounds__(kWave) void k_coverage_many(CovArgs a) {
    constexpr int MK = kMaxKeys;
    __shared__ uint64_t keys[kMaxSub][MK];  // crossings; reused for span events
    __shared__ __align__(16) int32_t acc[kWin + 8];  // acc (low 16 bits) + run difference (high 16 bits)
    __shared__ uint16_t tstate[rvkr::kChunkTiles];
    const int lane = threadIdx.x;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint2 bj = a.bands[blockIdx.x];
    const CovJob job = a.jobs[bj.x];
    const uint32_t band = bj.y;
    const int shift = job.aa ? 2 : 0;
    const int nsub_aa = 1 << shift;
    const bool evenodd = job.rule == RVK_FILL_EVENODD;
    const int32_t row0 = job.gy0 + (int32_t)band * rvkr::kBandRows;
    const int32_t ry0 = max(row0, job.y0), ry1 = min(row0 + rvkr::kBandRows, job.y0 + job.h);  // covered rows
    uint16_t *tab = a.table + job.table_offset + (size_t)band * job.tiles_x;
    uint8_t *slots = a.arena + job.cov_offset + (size_t)band * job.tiles_x * 64u;
    const int32_t rx0 = job.x0, rx1 = job.x0 + job.w;  // covered columns
    const EdgeCov *edges = a.edges + job.edge_offset;
    const uint32_t *npieces = a.npieces + job.edge_offset;

    for (int i = lane; i < kWin + 8; i += kWave) acc[i] = 0;  // each window clears it behind its read
    const uint2 win = a.windows[job.window_offset + band];

    uint32_t nslots = 0;  // partial tiles of the band so far
    // The band is processed in column chunks of up to kChunkTiles tiles.  Normally a
    // row's every crossing is sorted; when a sub-scanline holds more crossings than its
    // key area (MK), the chunk is redone at half the width, and from then on each
    // chunk keeps only the crossings that round into its columns and starts from the
    // winding of those left of it (down to single tiles).
    uint32_t chunk_tiles = rvkr::kChunkTiles;
    bool cut = false;  // chunks keep only their own crossings
    for (uint32_t ct0 = 0; ct0 < job.tiles_x;) {
        const uint32_t ctn = min(chunk_tiles, job.tiles_x - ct0);
        const int32_t cx0 = job.gx0 + (int32_t)ct0 * rvkr::kTile;  // first column of the chunk
        const int32_t cw = (int32_t)ctn * rvkr::kTile;
        const int32_t c0s = cut ? cx0 * nsub_aa : INT32_MIN, c1s = cut ? (cx0 + cw) * nsub_aa : INT32_MAX;
        const uint32_t nslots0 = nslots;
        bool redo = false;
        for (int r = 0; r < rvkr::kBandRows && !redo; r++) {
            const int32_t y = row0 + r;
            const bool row_in = y >= ry0 && y < ry1;
            int nev[kMaxSub] = {0, 0, 0, 0};
            if (row_in) {
                // ---- the crossings of the row's sub-scanlines ----
                const int32_t sy0 = y * nsub_aa;
                int cnt[kMaxSub] = {0, 0, 0, 0};
                int bd[kMaxSub] = {0, 0, 0, 0};  // winding of the crossings left of the chunk
                // the crossings of edge i on the row's sub-scanlines, stepping its piece
                // index k forward; those in the chunk are compacted into the key areas in
                // lane order, those left of it are summed into bd
                auto gather = [&](bool valid, uint32_t i, uint32_t &k) {
                    uint64_t key[kMaxSub];
                    bool act[kMaxSub] = {false, false, false, false};
                    int left[kMaxSub] = {0, 0, 0, 0};
                    if (valid) {
                        const EdgeCov e = edges[i];
                        const PieceDev *pc = a.pieces + e.piece_offset;
                        const uint32_t n = npieces[i];
                        if (e.first_y <= sy0 + nsub_aa - 1 && e.ymax >= sy0 && k < n) {
                            PieceDev p = pc[k];
                            for (int s = 0; s < nsub_aa; s++) {
                                const int32_t sy = sy0 + s;
                                while (p.last_y < sy && k + 1 < n) p = pc[++k];
                                if (p.first_y <= sy && p.last_y >= sy) {
                                    const int32_t x = (int32_t)((uint32_t)p.x + (uint32_t)(sy - p.first_y) * (uint32_t)p.dx);
                                    const int32_t xr = (x + 0x8000) >> 16;  // the sub-column of its event
                                    if (xr < c0s) {
                                        left[s] = e.winding > 0 ? 1 : -1;
                                    } else if (xr < c1s) {
                                        key[s] = ((uint64_t)((uint32_t)x ^ 0x80000000u) << 32) |
                                                 ((uint64_t)(uint32_t)e.id << 1) | (e.winding > 0 ? 1u : 0u);
                                        act[s] = true;
                                    }
                                }
                            }
                        }
                    }
                    for (int s = 0; s < nsub_aa; s++) {
                        const uint64_t m = __ballot(act[s]);
                        const int pos = cnt[s] + __popcll(m & below);
                        if (act[s] && pos < MK) keys[s][pos] = key[s];
                        cnt[s] += __popcll(m);
                        if (cut) bd[s] += __popcll(__ballot(left[s] > 0)) - __popcll(__ballot(left[s] < 0));
                    }
                };
                // every edge of the window, its piece found by binary search
                for (uint32_t base = win.x; base < win.y; base += kWave) {
                    const uint32_t i = base + (uint32_t)lane;
                    uint32_t k = 0;
                    if (i < win.y) {
                        const EdgeCov e = edges[i];
                        if (e.first_y < sy0) {
                            const PieceDev *pc = a.pieces + e.piece_offset;
                            uint32_t hi = npieces[i];
                            while (k < hi) {
                                const uint32_t mid = (k + hi) >> 1;
                                if (pc[mid].last_y < sy0) k = mid + 1;
                                else hi = mid;
                            }
                        }
                    }
                    gather(i < win.y, i, k);
                }
                __syncthreads();
                // ---- sort the sub-scanlines together and turn them into span events ----
                int nmax = 0;
                for (int s = 0; s < nsub_aa; s++) nmax = max(nmax, cnt[s]);
                if (nmax > MK) {
                    if (ctn > 1) {  // too many crossings: this chunk again, narrower
                        redo = true;
                        break;
                    }
                    // more than MK crossings round into one tile's columns: kept
                    // truncated, and the render reports it
                    if (lane == 0) atomicAdd(a.overflow, 1);
                    for (int s = 0; s < nsub_aa; s++) cnt[s] = min(cnt[s], MK);
                    nmax = MK;
                }
                // keys per lane: the smallest network that holds the fullest sub-scanline
                // (cnt is at most MK, so none needs more than MK / 64 = 8 keys per lane)
                // (a cut chunk with no crossings inside can still lie inside a span)
                if (nmax == 0 && !cut) {
                } else if (nsub_aa == 1) {
                    if (nmax <= 64) spans_of<1, 1, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                    else if (nmax <= 128) spans_of<2, 1, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                    else if (nmax <= 256) spans_of<4, 1, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                    else spans_of<8, 1, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                } else {
                    if (nmax <= 64) spans_of<1, kMaxSub, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                    else if (nmax <= 128) spans_of<2, kMaxSub, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                    else if (nmax <= 256) spans_of<4, kMaxSub, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                    else spans_of<8, kMaxSub, MK>(keys, cnt, evenodd, nev, lane, bd, c0s, c1s);
                }
                __syncthreads();
            }
            const int nsub = row_in ? nsub_aa : 0;
            int kst[kMaxSub] = {0, 0, 0, 0};  // per sub-scanline: the first span not yet behind the windows
            for (int32_t wx0 = 0; wx0 < cw; wx0 += kWin) {
                const int32_t ww = min(kWin, cw - wx0);  // a multiple of kTile
                // ---- the spans that reach this window, cut to it and to the job's
                // columns (coverage is 0 outside them) ----
                const int32_t wabs = cx0 + wx0;
                const int32_t colbase = wabs * nsub_aa;
                const int32_t wend = colbase + ww * nsub_aa;  // first sub-column past the window
                const int32_t lo = max(0, rx0 - wabs) * nsub_aa, hi = max(0, min(ww, rx1 - wabs)) * nsub_aa;
                // lanes 16 s .. 16 s + 15 look at the next 16 spans of sub-scanline s: the
                // spans that start before the window's end are a prefix of them (spans
                // are ordered), as are those that end at or before it (behind every
                // later window); all the window's spans are then accumulated in one
                // pass, one per lane
                int nin[kMaxSub] = {0, 0, 0, 0}, off[kMaxSub + 1] = {0, 0, 0, 0, 0};
                bool more = false;
                if (nsub > 0 && hi > lo) {
                    const int sl = lane >> 4;
                    const int kk = kst[sl] + (lane & 15);
                    const int nspl = sl < nsub ? nev[sl] >> 1 : 0;
                    int32_t La = 0, Ra = 0;
                    if (kk < nspl) {
                        const int32_t *ev = reinterpret_cast<const int32_t *>(keys[sl]);
                        La = ev[2 * kk];
                        Ra = ev[2 * kk + 1];
                    }
                    const uint64_t min_ = __ballot(kk < nspl && La < wend);
                    const uint64_t mdone = __ballot(kk < nspl && Ra <= wend);
                    for (int q = 0; q < kMaxSub; q++) {
                        nin[q] = __popcll((min_ >> (16 * q)) & 0xffffull);
                        more = more || nin[q] == 16;
                        off[q + 1] = off[q] + nin[q];
                    }
                    for (int q = 0; q < kMaxSub; q++) kst[q] += __popcll((mdone >> (16 * q)) & 0xffffull);
                    // the accumulation of one span (window-relative sub-columns)
                    auto add_span = [&](int q, int32_t La2, int32_t Ra2) {
                        const int32_t maxv = job.aa ? (64 - (((q & 3) + 1) >> 2)) : 255;
                        int32_t L = max(La2 - colbase, lo), R = min(Ra2 - colbase, hi);
                        if (R <= L) return;
                        if (!job.aa) {
                            atomicAdd(&acc[L], 255 << 16);
                            atomicAdd(&acc[R], -(255 << 16));
                            return;
                        }
                        const int32_t fb = L & 3, fe = R & 3;
                        int32_t c = (R >> 2) - (L >> 2) - 1;
                        if (c < 0) {
                            atomicAdd(&acc[L >> 2], (fe - fb) * 16);
                        } else {
                            int32_t st = L >> 2;
                            if (fb == 0) c += 1;
                            else { atomicAdd(&acc[st], (4 - fb) * 16); st += 1; }
                            if (c > 0) {
                                atomicAdd(&acc[st], maxv << 16);
                                atomicAdd(&acc[st + c], -(maxv << 16));
                            }
                            if (fe) atomicAdd(&acc[R >> 2], fe * 16);
                        }
                    };
                    if (lane < off[kMaxSub]) {
                        const int q = (lane >= off[1]) + (lane >= off[2]) + (lane >= off[3]);
                        const int k = kst[q] - __popcll((mdone >> (16 * q)) & 0xffffull) + (lane - off[q]);
                        const int32_t *ev = reinterpret_cast<const int32_t *>(keys[q]);
                        add_span(q, ev[2 * k], ev[2 * k + 1]);
                    }
                    if (more) {
                        // a sub-scanline with 16 or more spans in this window: the rest of
                        // them, 64 at a time
                        for (int q = 0; q < nsub; q++) {
                            if (nin[q] < 16) continue;
                            const int32_t *ev = reinterpret_cast<const int32_t *>(keys[q]);
                            const int nsp = nev[q] >> 1;
                            const int k0q = kst[q] - __popcll((mdone >> (16 * q)) & 0xffffull) + 16;
                            int extra_done = 0;
                            for (int kb = k0q; kb < nsp; kb += kWave) {
                                const int k = kb + lane;
                                int32_t La2 = 0, Ra2 = 0;
                                if (k < nsp) {
                                    La2 = ev[2 * k];
                                    Ra2 = ev[2 * k + 1];
                                }
                                const bool in = k < nsp && La2 < wend;
                                extra_done += __popcll(__ballot(k < nsp && Ra2 <= wend));
                                if (in) add_span(q, La2, Ra2);
                                if (__ballot(in) != ~0ull) break;
                            }
                            kst[q] += extra_done;
                        }
                    }
                }
                __syncthreads();
                // ---- prefix sum: lane l holds pixels [8 l, 8 l + 8) of the window, one
                // tile row; the window's accumulator is cleared behind the read ----
                const int32_t p0 = 8 * lane;
                const bool valid = p0 < ww;
                const int4 qa = *reinterpret_cast<const int4 *>(&acc[p0]);
                const int4 qb = *reinterpret_cast<const int4 *>(&acc[p0 + 4]);
                *reinterpret_cast<int4 *>(&acc[p0]) = make_int4(0, 0, 0, 0);
                *reinterpret_cast<int4 *>(&acc[p0 + 4]) = make_int4(0, 0, 0, 0);
                if (lane == 0) acc[kWin] = 0;
                const int32_t packed8[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
                int v[8], d[8], loc = 0;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int32_t packed = valid ? packed8[q] : 0;
                    v[q] = packed & 0xffff;
                    d[q] = packed >> 16;
                    loc += d[q];
                }
                const int incl = wave_incl_scan(loc);
                int run = incl - loc;
                uint32_t w0 = 0, w1 = 0;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    run += d[q];
                    const uint32_t c = (uint32_t)min(255, v[q] + run);
                    if (q < 4) w0 |= c << (8 * q);
                    else w1 |= c << (8 * (q - 4));
                }
                // ---- the tile of this row of 8 pixels ----
                const uint32_t t = (uint32_t)wx0 / rvkr::kTile + (uint32_t)lane;  // tile in the chunk
                const uint32_t v0 = w0 & 0xffu;
                const bool tuni = w0 == v0 * 0x01010101u && w1 == w0;
                const uint32_t st = valid && r > 0 ? (uint32_t)tstate[t] : 0u;
                const bool was_partial = r > 0 && st >= kStatePartial;
                const bool fresh = valid && !was_partial && (r == 0 ? !tuni : !(tuni && v0 == st));
                const uint64_t m = __ballot(fresh);
                const uint32_t k = was_partial ? st - kStatePartial : nslots + (uint32_t)__popcll(m & below);
                nslots += (uint32_t)__popcll(m);
                if (valid && (was_partial || fresh)) {
                    uint2 *tp = reinterpret_cast<uint2 *>(slots + (size_t)k * 64u);
                    tp[r] = make_uint2(w0, w1);
                    if (fresh) {  // the tile's earlier rows were all st
                        const uint32_t u = st * 0x01010101u;
                        for (int rr = 0; rr < r; rr++) tp[rr] = make_uint2(u, u);
                        tstate[t] = (uint16_t)(kStatePartial + k);
                    }
                } else if (valid && r == 0) {
                    tstate[t] = (uint16_t)v0;
                }
                __syncthreads();
            }
        }
        if (redo) {
            chunk_tiles = max(ctn / 2, 1u);
            cut = true;
            nslots = nslots0;
            __syncthreads();
            continue;
        }
        // ---- the chunk's tile table entries ----
        for (uint32_t t0 = 0; t0 < ctn; t0 += kWave) {
            const uint32_t t = t0 + (uint32_t)lane;
            const bool valid = t < ctn;
            const uint32_t st = valid ? (uint32_t)tstate[t] : 0u;
            // a uniform tile of another value than 0 or 255 (rows of different sub-row
            // spans, or a partial pixel value everywhere) gets a slot of its own
            const bool fill = valid && st < kStatePartial && st != 0u && st != 255u;
            const uint64_t m = __ballot(fill);
            const uint32_t k = nslots + (uint32_t)__popcll(m & below);
            nslots += (uint32_t)__popcll(m);
            uint32_t e = rvkr::kTileEmpty;
            if (st >= kStatePartial) {
                e = rvkr::kTileSlot0 + (st - kStatePartial);
            } else if (fill) {
                uint4 *tp = reinterpret_cast<uint4 *>(slots + (size_t)k * 64u);
                const uint32_t v4 = st * 0x01010101u;
                for (int q = 0; q < 4; q++) tp[q] = make_uint4(v4, v4, v4, v4);
                e = rvkr::kTileSlot0 + k;
            } else if (st == 255u) {
                e = rvkr::kTileFull;
            }
            if (valid) tab[ct0 + t] = (uint16_t)e;
        }
        __syncthreads();
        ct0 += ctn;
    }
}

// ---------------------------------------------------------------------------
// shading (tiny-skia lowp) and compositing
// ---------------------------------------------------------------------------
// lowp arithmetic on packed pixels, two channels per 24-bit multiply (one full-rate
// VALU operation): channels 0 and 2 sit in bits 0-7 and 16-23 of one word, 1 and 3 in
// bits 8-15 and 24-31 of the other, and each 16-bit field's value (at most
// 255 * 255 + 255) never carries into the next.  div255(v) = (v + 255) >> 8.
constexpr uint32_t kEven = 0x00ff00ffu;

// div255(c_k * m) for every channel k of c (m <= 255)
__device__ __forceinline__ uint32_t scale_px(uint32_t c, uint32_t m) {
    const uint32_t lo = ((__umul24(c & kEven, m) + kEven) >> 8) & kEven;
    const uint32_t hi = (__umul24((c >> 8) & kEven, m) + kEven) & ~kEven;
    return lo | hi;
}

// div255(d_k * (255 - m) + s_k * m) for every channel k (lowp lerp, m <= 255)
__device__ __forceinline__ uint32_t lerp_px(uint32_t d, uint32_t s, uint32_t m) {
    const uint32_t im = 255u - m;
    const uint32_t lo = ((__umul24(d & kEven, im) + __umul24(s & kEven, m) + kEven) >> 8) & kEven;
    const uint32_t hi = (__umul24((d >> 8) & kEven, im) + __umul24((s >> 8) & kEven, m) + kEven) & ~kEven;
    return lo | hi;
}
__device__ __forceinline__ float clamp01(float v) { return fminf(fmaxf(v, 0.0f), 1.0f); }

// the spread mode applied to a gradient coordinate (m: the shader's mode word)
__device__ __forceinline__ float spread_t(uint32_t m, float t) {
    const uint32_t spread = (m >> rvkr::kModeSpreadShift) & 3u;
    if (spread == RVK_SPREAD_REFLECT) {
        const float u = t - 1.0f;
        t = clamp01(fabsf(u - 2.0f * floorf(u * 0.5f) - 1.0f));
    } else if (spread == RVK_SPREAD_REPEAT) {
        t = clamp01(t - floorf(t));
    } else if (m & rvkr::kModePadClamp) {
        t = clamp01(t);
    }
    return t;
}

// sqrtf, correctly rounded, for a wave of values: away from 0 < x < 2^-96 (where the
// residuals below would underflow; the whole wave then takes sqrtf) the hardware root is
// within one unit in the last place, and the signs of the exact residuals at its two
// neighbours say which of the three is nearest (Tuckerman's test).  0, infinity and NaN
// fail both comparisons and stay as they are.
__device__ __forceinline__ float wave_sqrt(float x) {
    if (__ballot(x < 0x1p-96f && x > 0.0f) != 0) return sqrtf(x);
    const float s = __builtin_amdgcn_sqrtf(x);
    const float lo = __uint_as_float(__float_as_uint(s) - 1u), hi = __uint_as_float(__float_as_uint(s) + 1u);
    // sqrt(x) <= s - half a unit: s * lo >= x; sqrt(x) > s + half a unit: s * hi < x
    float r = fmaf(-lo, s, x) <= 0.0f ? lo : s;
    return fmaf(-hi, s, x) > 0.0f ? hi : r;
}

// gradient coordinate t of a linear or concentric radial shader at the pixel centre
// (x, y)
__device__ __forceinline__ float grad_t(const ShaderHead &s, uint32_t m, float x, float y) {
    const float tx = x * s.sx + (y * s.kx + s.tx);
    float t = tx;
    if (m & rvkr::kModeRadial) {
        const float ty = x * s.ky + (y * s.sy + s.ty);
        t = wave_sqrt(tx * tx + ty * ty);
        if (m & rvkr::kModeRTwist) t = (t - s.r_scale) / s.r_bias;
    }
    return spread_t(m, t);
}

// gradient coordinate t of a two-point conical shader; `degenerate` is set where the
// gradient is undefined (tiny-skia mask_2pt_conical_degenerates: t <= 0 or NaN, with t
// forced to 0)
__device__ __forceinline__ float grad_t_focal(const ShaderHead &s, int32_t px, int32_t py, bool &degenerate) {
    const float x = (float)px + 0.5f, y = (float)py + 0.5f;
    const float tx = x * s.sx + (y * s.kx + s.tx);
    const float ty = x * s.ky + (y * s.sy + s.ty);
    float t;
    if (s.focal == rvkr::kFocalOnCircle) t = tx + ty * ty / tx;
    else if (s.focal == rvkr::kFocalWellBehaved) t = sqrtf(tx * tx + ty * ty) - tx * s.p0;
    else t = sqrtf(tx * tx - ty * ty) - tx * s.p0;
    degenerate = false;
    if (s.focal != rvkr::kFocalWellBehaved) {
        degenerate = t <= 0.0f || t != t;
        if (degenerate) t = 0.0f;
    }
    return spread_t(s.mode, t);
}

// the gradient's colour at t (tiny-skia's gradient / evenly_spaced_2_stop_gradient
// stages, f32, before any clamp)
__device__ __forceinline__ void grad_color(const ShaderParams &sp, uint32_t m, float t, float c[4]) {
    if (m & rvkr::kModeTwoStop) {
        for (int k = 0; k < 4; k++) c[k] = t * sp.f[0][k] + sp.b[0][k];
    } else {
        // the thresholds are read four at a time; those past the last stop are NaN, which
        // no t reaches
        const uint32_t nstops = m >> rvkr::kModeStopsShift;
        uint32_t idx = 0;
        for (uint32_t i = 1; i < nstops; i += 4) {
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) idx += t >= sp.t[i + k] ? 1u : 0u;
        }
        for (int k = 0; k < 4; k++) c[k] = t * sp.f[idx][k] + sp.b[idx][k];
    }
}

// premultiplied u8 source colour of a shader at the pixel centre (x, y), packed
// (tiny-skia lowp)
__device__ __forceinline__ uint32_t shade(const ShaderParams &sp, uint32_t m, float x, float y) {
    if ((m & rvkr::kModeKind) == 1u) return sp.rgba;
    float c[4];
    grad_color(sp, m, grad_t(sp, m, x, y), c);
    uint32_t o = 0;
    for (int k = 0; k < 4; k++) {
        const float v = clamp01(c[k]);  // fmaxf(NaN, 0) = 0
        o |= (uint32_t)(v * 255.0f + 0.5f) << (8 * k);
    }
    // premultiply: every colour channel times alpha / 255 (alpha's own field is empty)
    if (!(m & rvkr::kModeOpaque)) o = scale_px(o & 0x00ffffffu, o >> 24) | (o & 0xff000000u);
    return o;
}

// One texel of a pattern pixmap at pixmap coordinates (u, v): Repeat tiling (none for
// Pad), then gather_ix (clamped to the last texel) and load_8888 (v * (1/255)).
__device__ __forceinline__ F4 tile_texel(const ShaderHead &s, const uint32_t *tile, float u, float v) {
    const float fw = (float)s.tile_w, fh = (float)s.tile_h;
    if (s.spread == RVK_SPREAD_REPEAT) {
        u = u - floorf(u * s.tile_iw) * fw;
        v = v - floorf(v * s.tile_ih) * fh;
    }
    // the largest float below the size (ulp_sub)
    u = fminf(fmaxf(u, 0.0f), __uint_as_float(__float_as_uint(fw) - 1u));
    v = fminf(fmaxf(v, 0.0f), __uint_as_float(__float_as_uint(fh) - 1u));
    const uint32_t p = tile[(uint32_t)(int32_t)v * s.tile_w + (uint32_t)(int32_t)u];
    const float k = 1.0f / 255.0f;
    return F4{(float)(p & 0xffu) * k, (float)((p >> 8) & 0xffu) * k, (float)((p >> 16) & 0xffu) * k,
              (float)(p >> 24) * k};
}

// The premultiplied colour of a pattern shader at pixel (px, py) (tiny-skia's f32
// seed_shader and transform, then repeat (Repeat spread) + gather for nearest
// sampling, bilinear, or bicubic + clamp_0 + clamp_a, then scale_1_float by the
// opacity).
__device__ F4 pattern_color(const ShaderHead &s, int32_t px, int32_t py) {
    const float x = (float)px + 0.5f, y = (float)py + 0.5f;
    const float tx = x * s.sx + (y * s.kx + s.tx);
    const float ty = x * s.ky + (y * s.sy + s.ty);
    const uint32_t *tile = (const uint32_t *)s.tile;
    F4 o;
    if (s.quality == 0) {
        o = tile_texel(s, tile, tx, ty);
    } else if (s.quality == 1) {
        // bilinear: weights 1 - f, f of the fractions of x + 0.5 and y + 0.5 over the
        // 2 x 2 texels from (x - 0.5, y - 0.5); no clamp stages follow
        const float fx = (tx + 0.5f) - floorf(tx + 0.5f), fy = (ty + 0.5f) - floorf(ty + 0.5f);
        o = F4{0.0f, 0.0f, 0.0f, 0.0f};
        float v = ty - 0.5f;
#pragma unroll 1
        for (int j = 0; j < 2; j++) {
            float u = tx - 0.5f;
            const float wyj = j == 0 ? 1.0f - fy : fy;
#pragma unroll 1
            for (int i = 0; i < 2; i++) {
                const F4 c = tile_texel(s, tile, u, v);
                const float wgt = (i == 0 ? 1.0f - fx : fx) * wyj;
                o.r = wgt * c.r + o.r; o.g = wgt * c.g + o.g; o.b = wgt * c.b + o.b; o.a = wgt * c.a + o.a;
                u = u + 1.0f;
            }
            v = v + 1.0f;
        }
    } else {
        // weights far(1 - f), near(1 - f), near(f), far(f) of the fractions of x + 0.5
        // and y + 0.5: near(t) = ((-21/18 t + 27/18) t + 9/18) t + 1/18, far(t) =
        // t^2 (7/18 t - 6/18); texels from (x - 1.5, y - 1.5) in steps of 1
        auto near_w = [](float t) {
            return t * (t * ((-21.0f / 18.0f) * t + 27.0f / 18.0f) + 9.0f / 18.0f) + 1.0f / 18.0f;
        };
        auto far_w = [](float t) { return (t * t) * ((7.0f / 18.0f) * t + -6.0f / 18.0f); };
        const float fx = (tx + 0.5f) - floorf(tx + 0.5f), fy = (ty + 0.5f) - floorf(ty + 0.5f);
        auto weight = [&](int k, float f) {
            return k == 0 ? far_w(1.0f - f) : k == 1 ? near_w(1.0f - f) : k == 2 ? near_w(f) : far_w(f);
        };
        o = F4{0.0f, 0.0f, 0.0f, 0.0f};
        float v = ty - 1.5f;
        // rolled loops with the weights formed in place keep the compositor's register
        // budget (the kernel is sized for the deepest call it makes)
#pragma unroll 1
        for (int j = 0; j < 4; j++) {
            float u = tx - 1.5f;
            const float wyj = weight(j, fy);
#pragma unroll 1
            for (int i = 0; i < 4; i++) {
                const F4 c = tile_texel(s, tile, u, v);
                const float wgt = weight(i, fx) * wyj;
                o.r = wgt * c.r + o.r; o.g = wgt * c.g + o.g; o.b = wgt * c.b + o.b; o.a = wgt * c.a + o.a;
                u = u + 1.0f;
            }
            v = v + 1.0f;
        }
        o.r = fmaxf(o.r, 0.0f); o.g = fmaxf(o.g, 0.0f); o.b = fmaxf(o.b, 0.0f); o.a = fmaxf(o.a, 0.0f);
        o.a = fminf(o.a, 1.0f);
        o.r = fminf(o.r, o.a); o.g = fminf(o.g, o.a); o.b = fminf(o.b, o.a);
    }
    if (s.pattern_opacity != 1.0f) {
        o.r *= s.pattern_opacity; o.g *= s.pattern_opacity; o.b *= s.pattern_opacity; o.a *= s.pattern_opacity;
    }
    return o;
}

// A covered pixel under a shader of tiny-skia's f32 pipeline (a two-point conical
// gradient: gradient, premultiply, apply_vector_mask; or a pattern), then
// scale_1_float by c / 255, SourceOver onto d, store (kept out of line: the
// compositor's common paths do not carry it)
template <bool kPatterns>
__device__ __noinline__ uint32_t paint_px_hp(const ShaderParams &sp, const ShaderHead &s, int32_t px, int32_t py,
                                             uint32_t c, uint32_t d) {
    F4 src;
    if (kPatterns && s.kind == 3) {
        src = pattern_color(s, px, py);
    } else {
        bool degenerate;
        const float t = grad_t_focal(s, px, py, degenerate);
        float col[4];
        grad_color(sp, s.mode, t, col);
        if (!s.opaque) { col[0] *= col[3]; col[1] *= col[3]; col[2] *= col[3]; }
        src = degenerate ? F4{0.0f, 0.0f, 0.0f, 0.0f} : F4{col[0], col[1], col[2], col[3]};
    }
    if (c != 255u) {
        const float cf = (float)c * (1.0f / 255.0f);
        src.r *= cf; src.g *= cf; src.b *= cf; src.a *= cf;
    }
    return store_px(blend(RVK_BLEND_SOURCE_OVER, src, load_px(d)));
}

// lowp: scale by coverage (unless full), then SourceOver onto `d`; an opaque shader
// composites with Source instead (full coverage stores, partial coverage lerps).  A
// premultiplied colour never exceeds its alpha, so SourceOver's per-channel sums stay
// within 255.
__device__ __forceinline__ uint32_t over_lowp(uint32_t src, uint32_t cov, uint32_t d, bool as_source) {
    if (as_source) return cov == 255 ? src : lerp_px(d, src, cov);
    if (cov != 255) src = scale_px(src, cov);
    return src + scale_px(d, 255u - (src >> 24));
}

// ---- the same arithmetic on pixels held as four floats with whole values 0 .. 255 ----
// Products of two such values plus 255 stay below 2^24, so fma and the division by 256
// are exact and floor((v + 255) / 256) is div255(v); nothing is converted or packed
// between one draw item and the next.
__device__ __forceinline__ F4 px_floats(uint32_t p) {
    return F4{(float)ch(p, 0), (float)ch(p, 1), (float)ch(p, 2), (float)ch(p, 3)};
}
__device__ __forceinline__ uint32_t px_pack(F4 v) {
    return pack((uint32_t)v.r, (uint32_t)v.g, (uint32_t)v.b, (uint32_t)v.a);
}
__device__ __forceinline__ float div256f(float v) { return floorf(v * (1.0f / 256.0f)); }
__device__ __forceinline__ float scale_f(float v, float m) { return div256f(fmaf(v, m, 255.0f)); }
__device__ __forceinline__ F4 scale_f4(F4 v, float m) {
    return F4{scale_f(v.r, m), scale_f(v.g, m), scale_f(v.b, m), scale_f(v.a, m)};
}

// `shade` without the packing
__device__ __forceinline__ F4 shade_f(const ShaderParams &sp, uint32_t m, float x, float y) {
    if ((m & rvkr::kModeKind) == 1u) return px_floats(sp.rgba);
    float c[4];
    const float t = grad_t(sp, m, x, y);
    // (the clamp repeated in both forms folds into the addition before it)
    if (m & rvkr::kModeTwoStop) {
        for (int k = 0; k < 4; k++) c[k] = clamp01(t * sp.f[0][k] + sp.b[0][k]);
    } else {
        grad_color(sp, m & ~rvkr::kModeTwoStop, t, c);
        for (int k = 0; k < 4; k++) c[k] = clamp01(c[k]);
    }
    for (int k = 0; k < 4; k++) c[k] = floorf(c[k] * 255.0f + 0.5f);
    if (!(m & rvkr::kModeOpaque))
        for (int k = 0; k < 3; k++) c[k] = scale_f(c[k], c[3]);
    return F4{c[0], c[1], c[2], c[3]};
}

// `over_lowp`: the colour at coverage c (`full`: c is 255 everywhere) onto d
__device__ __forceinline__ void over_f(F4 s, float c, bool full, F4 &d, bool as_source) {
    if (as_source) {
        if (full) {
            d = s;
        } else {
            const float ic = 255.0f - c;
            d.r = div256f(fmaf(s.r, c, fmaf(d.r, ic, 255.0f)));
            d.g = div256f(fmaf(s.g, c, fmaf(d.g, ic, 255.0f)));
            d.b = div256f(fmaf(s.b, c, fmaf(d.b, ic, 255.0f)));
            d.a = div256f(fmaf(s.a, c, fmaf(d.a, ic, 255.0f)));
        }
    } else {
        if (!full) s = scale_f4(s, c);
        const float ia = 255.0f - s.a;
        d.r = s.r + scale_f(d.r, ia);
        d.g = s.g + scale_f(d.g, ia);
        d.b = s.b + scale_f(d.b, ia);
        d.a = s.a + scale_f(d.a, ia);
    }
}

// SourceOver of a layer pixel with the layer's opacity (in [0, 1]) onto d: load_px,
// blend and store_px.  The sum of a channel exceeds 1 by rounding only, so times 255 it
// rounds to 255 without the clamp.
__device__ __forceinline__ void layer_over_f(float s, float ia, float &d) {
    d = rintf((s + d * (1.0f / 255.0f) * ia) * 255.0f);
}
__device__ __forceinline__ void layer_f(F4 s, float opacity, bool scaled, F4 &d) {
    const float k = 1.0f / 255.0f;
    s.r *= k; s.g *= k; s.b *= k; s.a *= k;
    if (scaled) { s.r *= opacity; s.g *= opacity; s.b *= opacity; s.a *= opacity; }
    const float ia = 1.0f - s.a;
    layer_over_f(s.r, ia, d.r);
    layer_over_f(s.g, ia, d.g);
    layer_over_f(s.b, ia, d.b);
    layer_over_f(s.a, ia, d.a);
}

// one covered pixel (lx, ly), centre (cx, cy), of a draw item: Clear, or the shaded
// colour composited with over_lowp, or for a shader of the f32 pipeline (two-point
// conical gradients, patterns) in f32 (scale_1_float by c / 255, SourceOver, store);
// the colour is shaded only when needed
template <bool kPatterns>
__device__ __forceinline__ uint32_t paint_px(const ShaderParams &sp, const ShaderHead &sh, int32_t lx, int32_t ly,
                                             float cx, float cy, uint32_t c, uint32_t d, uint32_t &src,
                                             bool &shaded) {
    const uint32_t m = sh.mode;
    if (m & rvkr::kModeClear) return scale_px(d, 255u - c);
    if (m & rvkr::kModeF32) return paint_px_hp<kPatterns>(sp, sh, lx, ly, c, d);
    if (!shaded) {
        src = shade(sp, m, cx, cy);
        shaded = true;
    }
    return over_lowp(src, c, d, (m & rvkr::kModeAsSource) != 0);
}

// tile-table entry of target tile (tx, ty) in a job's grid (origin gx0, gy0, gw x gh
// tiles); empty outside the grid (and for no job, whose grid is 0 x 0)
__device__ __forceinline__ uint32_t tile_entry(const uint16_t *table, int32_t gx0, int32_t gy0, uint32_t gw,
                                               uint32_t gh, uint32_t first, int32_t tx, int32_t ty) {
    const uint32_t cx = (uint32_t)(tx - gx0), cy = (uint32_t)(ty - gy0);
    return cx < gw && cy < gh ? (uint32_t)table[first + cy * gw + cx] : rvkr::kTileEmpty;
}

// coverage of a pixel of target tile row ty from its tile-table entry e (`pix` is the
// pixel's index within its 8 x 8 tile)
__device__ __forceinline__ uint32_t tile_cov(const JobRef &r, const uint8_t *arena, uint32_t e, int32_t ty,
                                             uint32_t pix) {
    if (e == rvkr::kTileEmpty) return 0u;
    if (e == rvkr::kTileFull) return 255u;
    const size_t slot = (size_t)(uint32_t)(ty - r.y0) * r.w + (e - rvkr::kTileSlot0);
    return arena[r.cov_offset + slot * 64u + pix];
}

// Coverage of one hairline blit at pixel (x, y) (see HairLine); 0 when the line does
// not blit the pixel.
__device__ __forceinline__ uint32_t hair_alpha(const HairLine &L, int32_t x, int32_t y) {
    const bool ymaj = (L.flags & rvkr::kHairYMajor) != 0;
    const int32_t major = ymaj ? y : x, minor = ymaj ? x : y;
    if (major < L.istart || major >= L.istop) return 0;
    if ((L.flags & rvkr::kHairClipped) && (x < L.cl || x >= L.cr || y < L.ct || y >= L.cb)) return 0;
    const int32_t k = major - L.istart;
    int32_t mod = 64;
    if (k == 0) mod = L.scale_start;
    else if (L.scale_stop > 0 && major == L.istop - 1) mod = L.scale_stop;
    const int32_t f = (int32_t)((uint32_t)L.fstart + (uint32_t)k * (uint32_t)L.slope + 0x8000u);
    const int32_t lo = f >> 16;
    const int32_t a = (f >> 8) & 0xff;
    if (minor == lo) return (uint32_t)((a * mod) >> 6);
    if (minor == lo - 1) return (uint32_t)(((255 - a) * mod) >> 6);
    return 0;
}

struct DrawArgs {
    const DrawItem *items;
    const DrawCull *cull;
    uint32_t nitems;
    const uint16_t *table;
    const uint8_t *arena;
    const ShaderParams *shaders;
    const uint32_t *hair_tiles, *hair_bins;
    const HairLine *hair_lines;
};

// One thread per target pixel; each 64-lane wave covers one 8 x 8 coverage tile and a
// block of 4 waves a 16 x 16 square.  A wave first culls a run of 64 items, one lane
// per item (its tile rect and its jobs' tile-table entries for the wave's tile, loaded
// side by side), then composites the items that touch its tile in order: an empty
// tile costs nothing, a full one no coverage load, a partial one one 64-byte load.
constexpr int kWaveW = rvkr::kTile, kWaveH = rvkr::kTile;  // pixels of one 64-lane wave
constexpr int TX = 16, TY = 16;                            // pixels of one block (four waves)
constexpr int kWavesX = TX / kWaveW;
static_assert(kWaveW * kWaveH == 64 && (TX / kWaveW) * (TY / kWaveH) == 4, "four 64-pixel waves per tile");

// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Block b is
// mapped to a square so that each XCD gets runs of kChunk horizontally adjacent
// row-major squares (which read neighbouring coverage and pixel cache lines), the
// runs interleaved over the draw rect so the XCDs share the work evenly; squares past
// the last whole round of runs keep their own index.
constexpr uint32_t kXcds = 8, kChunk = 4;

// kPatterns: the draw list holds pattern shaders.  The pattern sampler makes the
// out-of-line f32 path (and with it the whole kernel, which is sized for its deepest
// call) need more registers, so lists without patterns use the variant without it.
template <bool kPatterns>
__global__ __launch_bounds__(256) void k_draw(uint32_t *px, uint32_t w, uint32_t h, int32_t otx, int32_t oty,
                                              uint32_t blocks_x, DrawArgs a) {
    const uint32_t b = blockIdx.x;
    const uint32_t round = kXcds * kChunk, full = gridDim.x / round * round;
    const uint32_t xcd = b % kXcds, k = b / kXcds;
    const uint32_t sq = b < full ? (k / kChunk) * round + xcd * kChunk + k % kChunk : b;
    const uint32_t bx = sq % blocks_x, by = sq / blocks_x;
    const int lane = (int)(threadIdx.x % 64);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));  // uniform: tile math stays scalar
    // this wave's target tile and pixel
    const int32_t ttx = otx + (int32_t)bx * kWavesX + wv % kWavesX, tty = oty + (int32_t)by * (TY / kWaveH) + wv / kWavesX;
    const int32_t x = ttx * kWaveW + lane % kWaveW, y = tty * kWaveH + lane / kWaveW;
    const uint32_t pix = (uint32_t)lane;  // = (y % 8) * 8 + x % 8
    const float fx = (float)x + 0.5f, fy = (float)y + 0.5f;
    const bool inside = x < (int32_t)w && y < (int32_t)h;
    const uint32_t d0 = inside ? px[(size_t)y * w + x] : 0u;
    F4 df = px_floats(d0);
    for (uint32_t base = 0; base < a.nitems; base += kWave) {
        // ---- cull 64 items, one per lane ----
        const uint32_t i = base + (uint32_t)lane;
        uint32_t ef = 0, es = 0;
        bool keep = false;
        if (i < a.nitems) {
            const DrawCull c = a.cull[i];
            if (ttx >= c.tx0 && ttx < c.tx1 && tty >= c.ty0 && tty < c.ty1) {
                ef = tile_entry(a.table, c.fx0, c.fy0, c.fw, c.fh, c.ftable, ttx, tty);
                es = tile_entry(a.table, c.sx0, c.sy0, c.sw, c.sh, c.stable, ttx, tty);
                keep = ef != rvkr::kTileEmpty || es != rvkr::kTileEmpty || c.hair != 0;
            }
        }
        // ---- composite the kept items in order ----
        for (uint64_t m = __ballot(keep); m != 0; m &= m - 1) {
            const int kl = __builtin_ctzll(m);
            const uint32_t efk = (uint32_t)__builtin_amdgcn_readlane((int)ef, kl);
            const uint32_t esk = (uint32_t)__builtin_amdgcn_readlane((int)es, kl);
            const DrawItem &item = a.items[base + (uint32_t)kl];  // with its jobs' grids and tables
            const uint32_t im = item.mode;
            // the pixel centre in layer coordinates, exact in f32 (|x|, |lx| < 2^23)
            const float cx = fx - item.flx, cy = fy - item.fly;
            if (im & rvkr::kItemPlain) {
                // gradients and solids of the u8 pipeline, SourceOver.  Coverage 0 leaves
                // every value as it is, so the whole wave goes through together
                const bool swap = (im & rvkr::kItemStrokeFirst) != 0;
                auto shaded = [&](bool stroke, uint32_t e, float &c, uint32_t &sm) {
                    const ShaderParams &sp = a.shaders[stroke ? item.stroke_shader : item.fill_shader];
                    if (e != rvkr::kTileFull) c = (float)tile_cov(stroke ? item.sj : item.fj, a.arena, e, tty, pix);
                    sm = sp.mode;
                    return shade_f(sp, sm, cx, cy);
                };
                // the first of fill and stroke in drawing order that touches the tile,
                // then the other
                const uint32_t e0 = swap ? esk : efk, e1 = swap ? efk : esk;
                const bool one = e0 == rvkr::kTileEmpty || e1 == rvkr::kTileEmpty;
                const bool first = (e0 == rvkr::kTileEmpty) != swap;  // the first is the stroke
                const uint32_t ea = e0 == rvkr::kTileEmpty ? e1 : e0;
                float c = 255.0f;
                uint32_t sm;
                F4 t = shaded(first, ea, c, sm);
                if (im & rvkr::kItemLayer) {
                    // onto a transparent layer pixel: the colour scaled by its coverage
                    if (ea != rvkr::kTileFull) t = scale_f4(t, c);
                    if (!one) {
                        const F4 u = shaded(!first, e1, c = 255.0f, sm);
                        over_f(u, c, e1 == rvkr::kTileFull, t, (sm & rvkr::kModeAsSource) != 0);
                    }
                    layer_f(t, item.opacity, (im & rvkr::kItemScaled) != 0, df);
                } else {
                    over_f(t, c, ea == rvkr::kTileFull, df, (sm & rvkr::kModeAsSource) != 0);
                    if (!one) {
                        const F4 u = shaded(!first, e1, c = 255.0f, sm);
                        over_f(u, c, e1 == rvkr::kTileFull, df, (sm & rvkr::kModeAsSource) != 0);
                    }
                }
                continue;
            }
            if (!inside) continue;
            uint32_t d = px_pack(df);
            const int32_t lx = x - item.lx, ly = y - item.ly;
            const uint32_t cf = tile_cov(item.fj, a.arena, efk, tty, pix);
            uint32_t cs = 0, hb = 0, he = 0;
            if (item.stroke_hair) {
                // the hairline lines binned to this pixel's tile, in drawing order
                const uint32_t cx = (uint32_t)(lx - item.sj.x0), cy = (uint32_t)(ly - item.sj.y0);
                if (cx < item.sj.w && cy < item.sj.h) {
                    const uint32_t t = item.sj.table + cy / rvkr::kHairTile * item.sj.stride + cx / rvkr::kHairTile;
                    hb = a.hair_tiles[t];
                    he = a.hair_tiles[t + 1];
                }
            } else {
                cs = tile_cov(item.sj, a.arena, esk, tty, pix);
            }
            if ((cf | cs) != 0 || hb != he) {
                uint32_t target = item.layer ? 0u : d;
                for (int pass = 0; pass < 2; pass++) {
                    const bool stroke = (pass == 0) == (item.stroke_first != 0);
                    const ShaderParams &sp = a.shaders[stroke ? item.stroke_shader : item.fill_shader];
                    const ShaderHead &sh = sp;
                    uint32_t src = 0;
                    bool shaded = false;
                    if (stroke && item.stroke_hair) {
                        // every blit of the hairline at this pixel, composited in order
                        for (uint32_t kk = hb; kk < he; kk++) {
                            const uint32_t c = hair_alpha(a.hair_lines[a.hair_bins[kk]], lx, ly);
                            if (c) target = paint_px<kPatterns>(sp, sh, lx, ly, cx, cy, c, target, src, shaded);
                        }
                        continue;
                    }
                    const uint32_t c = stroke ? cs : cf;
                    if (c) target = paint_px<kPatterns>(sp, sh, lx, ly, cx, cy, c, target, src, shaded);
                }
                if (!item.layer) {
                    d = target;
                } else {
                    F4 s = load_px(target);
                    if (item.opacity != 1.0f) {
                        s.r *= item.opacity; s.g *= item.opacity; s.b *= item.opacity; s.a *= item.opacity;
                    }
                    d = store_px(blend(item.blend_mode, s, load_px(d)));
                }
                df = px_floats(d);
            }
        }
    }
    const uint32_t d = px_pack(df);
    if (inside && d != d0) px[(size_t)y * w + x] = d;
}

}  // namespace

namespace rvk {

rvk_status launch_expand(rvk_context *ctx, const EdgeRec *edges, uint32_t nedges, const EdgeCov *cov,
                         PieceDev *pieces, uint32_t *npieces, int32_t *overflow, double algo_bytes) {
    if (nedges == 0) return RVK_OK;
    ExpandArgs a{edges, nedges, cov, pieces, npieces, overflow};
    // few edges: four a wave, so that there are enough waves (the clip paths above took
    // 16.4 us with 16 a wave, 11.6 with 4); past 1024 waves of 16 the chip is full either
    // way and the second half of the kernel fills more lanes
    timed_launch(ctx, "expand", algo_bytes, [&] {
        if (nedges > 16384u) hipLaunchKernelGGL(k_expand<16>, dim3(div_up(nedges, 16)), dim3(kWave), 0, ctx->stream, a);
        else hipLaunchKernelGGL(k_expand<4>, dim3(div_up(nedges, 4)), dim3(kWave), 0, ctx->stream, a);
    });
    RVK_HIP_CHECK(hipGetLastError());
    return RVK_OK;
}

rvk_status launch_coverage(rvk_context *ctx, const CovJob *jobs, const uint2 *const bands[rvkr::kBandLists],
                           const uint64_t n_bands[rvkr::kBandLists], const EdgeCov *edges, const uint2 *windows,
                           const PieceDev *pieces, const uint32_t *npieces, uint16_t *table, uint8_t *arena,
                           int32_t *overflow, double algo_bytes) {
    // the algorithmic bytes are split between the launches by their band counts
    double total = 0.0;
    for (int t = 0; t < rvkr::kBandLists; t++) total += (double)n_bands[t];
    auto launch = [&](auto kernel, int t, int threads) -> rvk_status {
        if (n_bands[t] == 0) return RVK_OK;
        CovArgs a{bands[t], jobs, edges, windows, pieces, npieces, table, arena, overflow};
        timed_launch(ctx, "coverage", algo_bytes * (double)n_bands[t] / total, [&] {
            hipLaunchKernelGGL(kernel, dim3((uint32_t)n_bands[t]), dim3(threads), 0, ctx->stream, a);
        });
        RVK_HIP_CHECK(hipGetLastError());
        return RVK_OK;
    };
    RVK_TRY(launch(k_coverage<(int)rvkr::kCoverageKeys[0]>, 0, kRowWaves * kWave));
    RVK_TRY(launch(k_coverage<(int)rvkr::kCoverageKeys[1]>, 1, kRowWaves * kWave));
    RVK_TRY(launch(k_coverage<(int)rvkr::kCoverageKeys[2]>, 2, kRowWaves * kWave));
    RVK_TRY(launch(k_coverage_many, 3, kWave));
    return RVK_OK;
}

rvk_status launch_draw_items(rvk_context *ctx, uint8_t *target, uint32_t w, uint32_t h, int32_t x0, int32_t y0,
                             int32_t x1, int32_t y1, const DrawItem *items, const DrawCull *cull, uint32_t nitems,
                             const uint16_t *table, const uint8_t *arena, const ShaderParams *shaders,
                             const uint32_t *hair_tiles, const uint32_t *hair_bins, const HairLine *hair_lines,
                             bool patterns, double algo_bytes) {
    if (nitems == 0 || x1 <= x0 || y1 <= y0 || x0 < 0 || y0 < 0) return RVK_OK;
    // the draw rect in whole coverage tiles (the tile grids are aligned to the target)
    const int32_t otx = x0 / rvkr::kTile, oty = y0 / rvkr::kTile;
    const uint32_t ntx = (uint32_t)(div_up((uint32_t)x1, (uint32_t)rvkr::kTile) - (uint32_t)otx);
    const uint32_t nty = (uint32_t)(div_up((uint32_t)y1, (uint32_t)rvkr::kTile) - (uint32_t)oty);
    const uint32_t blocks_x = div_up(ntx, (uint32_t)kWavesX), blocks_y = div_up(nty, (uint32_t)(TY / kWaveH));
    const DrawArgs a{items, cull, nitems, table, arena, shaders, hair_tiles, hair_bins, hair_lines};
    timed_launch(ctx, "draw_items", algo_bytes, [&] {
        if (patterns)
            hipLaunchKernelGGL(k_draw<true>, dim3(blocks_x * blocks_y), dim3(256), 0, ctx->stream, (uint32_t *)target,
                               w, h, otx, oty, blocks_x, a);
        else
            hipLaunchKernelGGL(k_draw<false>, dim3(blocks_x * blocks_y), dim3(256), 0, ctx->stream, (uint32_t *)target,
                               w, h, otx, oty, blocks_x, a);
    });
    RVK_HIP_CHECK(hipGetLastError());
    return RVK_OK;
}

}  // namespace rvk
