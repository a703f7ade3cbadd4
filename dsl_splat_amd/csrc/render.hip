// Front-to-back alpha blending on 16x16 tiles and its reverse traversal.
//
// gs3d/render.py:36-208 (forward) and :211-356 (backward).  One workgroup
// per tile.  A lane owns PIX pixels of the tile (1: one pixel, 256 threads;
// 2: a horizontal pair, 128 threads).  The tile's sorted Gaussians are staged
// in LDS in batches (centre, conic + opacity, exponent limit and the full
// blended channel vector), so the inner loop reads only LDS broadcasts.  A
// wavefront leaves the inner loop once its pixels are done, and the workgroup
// stops at the next batch once all pixels are.
//
// Exponent limit: a Gaussian with opacity o can only reach alpha >= 1/255
// where -power <= ln(255 o); beyond that bound plus a 1% margin (far above
// the few-ulp error of exp, log and the product) the blend rejects the
// Gaussian.  Decisions, and therefore every output, are identical to
// evaluating the exponential.
//
// Vector arithmetic bounds both directions.  Measured per SIMD with several
// wavefronts: 2.7 cycles for a float add, multiply or fused multiply-add, 4.5
// for a compare, select, conversion, ldexp or DPP add, 8.5 for a reciprocal or
// a permlane swap, and 23 for a two-operand select on vcc right behind
// another.  So the loops keep their tests as scalar lane masks, form the
// exponential from adds, multiplies and one shift, and add a rejected
// Gaussian's channels with weight zero instead of selecting each sum.
//
// Backward: only batches below the largest last contributor of the tile are
// visited; a wavefront sums its pixels' gradients before one atomic
// instruction adds them, one entry per lane, instead of one atomic per entry
// and pixel as in the reference.
//
// Channel windows: the reference specialises its kernels on any channel count
// D' (gs3d/render.py:36-38, :211-213).  A launch here blends a window of at
// most 64 channels [c0, c0 + CH) of the D'-channel vector; wider vectors run
// one launch per window.  Forward windows are independent (the blend weights
// do not depend on the channels); window 0 writes the transmittance and last
// contributors.  Backward: the geometry launch (window 0) owns the centre,
// conic and opacity gradients, which need the dot product of the Gaussian's
// full channel vector with the pixel's upstream gradient; its window holds at
// most 64 - 8 channels, so its gradient entries fit the 64 lanes of one
// wavefront sum, and channels beyond it enter the dot product from global
// memory.  Further windows add only their channels' feature gradients.
#include <type_traits>

#include "common.hpp"

#ifndef GS3D_FWD_PIX
#define GS3D_FWD_PIX 2
#endif
#ifndef GS3D_BWD_PIX
#define GS3D_BWD_PIX 2
#endif
// Pixels per lane for 9-36 channels.
#ifndef GS3D_WIDE_FWD_PIX
#define GS3D_WIDE_FWD_PIX 1
#endif
#ifndef GS3D_WIDE_BWD_PIX
#define GS3D_WIDE_BWD_PIX 1
#endif

namespace gs3d {

constexpr int kTile = 16;
constexpr int kTilePixels = kTile * kTile;

// Gaussians staged per batch.  Up to 8 channels a workgroup holds 2
// wavefronts and LDS bounds the resident workgroups: batches of 128 leave
// room for more of them (3M Gaussians, 4 x 1080p: backward 1.93 -> 1.86 ms,
// forward 1.11 -> 1.09 ms against 256; 64 and 96 were slower).  Wider
// vectors run 4 wavefronts per workgroup at one pixel per lane, where
// smaller batches only add staging rounds (32 channels: 128 was 3% slower
// than 256); the widest vectors take 128 to fit the LDS budget.
template <int CH>
struct Batch {
    static constexpr int size = CH <= 8 ? 128 : CH <= 36 ? 256 : 128;
};

// Channels of the geometry launch's window: with the 8 geometric entries
// (absolute gradients included) they fill one 64-entry wavefront sum.
constexpr int kGeomWindow = 56;
// Channels of a forward window and of a further backward window.
constexpr int kWindow = 64;

// Pixels per lane for a channel count (the widest vectors keep one pixel per
// lane to bound register use).
template <int CH, bool BWD>
struct PixFor {
    static constexpr int value = CH <= 8    ? (BWD ? GS3D_BWD_PIX : GS3D_FWD_PIX)
                                 : CH <= 36 ? (BWD ? GS3D_WIDE_BWD_PIX : GS3D_WIDE_FWD_PIX)
                                            : 1;
};

// The wavefronts of a tile each own a rectangle of its pixels, 16 x 8 at two
// pixels per lane and 8 x 8 at one.  A Gaussian touches a square of 8 x 8
// pixels less often than a strip of 16 x 4: a 256x256 frame's backward took
// 138 against 142 us, a 637x421 frame's with 9 channels 217 against 238.
template <int PIX>
struct TileWaves {
    static_assert(PIX == 1 || PIX == 2, "pixel_of lays 8 lanes along a row");
    static constexpr int count = kTilePixels / PIX / 64;
    static constexpr int cols = PIX == 1 ? 8 : 16;
    static constexpr int rows = 64 * PIX / cols;
    static constexpr int across = kTile / cols;
};

// Tile-local coordinates of pixel k of thread t: a lane owns PIX neighbours
// of a row, 8 lanes a row of the wavefront's rectangle.
template <int PIX>
GS3D_DEV void pixel_of(int t, int k, int& x, int& y) {
    const int w = t >> 6, lane = t & 63;
    x = (w % TileWaves<PIX>::across) * TileWaves<PIX>::cols + PIX * (lane & 7) + k;
    y = (w / TileWaves<PIX>::across) * TileWaves<PIX>::rows + (lane >> 3);
}

struct TileInfo {
    int view, x0, y0, first, last, tile;
};

// Workgroups go to the 8 XCDs in turn; within every run of 8 * GS3D_TILE_CHUNK
// workgroups, XCD x takes the x-th chunk of GS3D_TILE_CHUNK consecutive tiles
// so that neighbouring tiles, which share most of their Gaussians, meet in one
// L2 (the final partial run keeps the identity order).
#ifndef GS3D_TILE_CHUNK
#define GS3D_TILE_CHUNK 8
#endif
GS3D_DEV int tile_of_block(int b, int blocks) {
    constexpr int C = GS3D_TILE_CHUNK, R = 8 * C;
    if (C <= 1) return b;
    const int run = b / R;
    if ((run + 1) * R > blocks) return b;
    const int w = b - run * R;
    return run * R + (w & 7) * C + (w >> 3);
}

GS3D_DEV TileInfo tile_info(const gs3d_render_args& a, int tile) {
    const int gx = (a.width + kTile - 1) / kTile, gy = (a.height + kTile - 1) / kTile;
    const int per_view = gx * gy;
    TileInfo t;
    t.view = tile / per_view;
    const int local = tile - t.view * per_view;
    const int ty = local / gx, tx = local - ty * gx;
    t.x0 = tx * kTile;
    t.y0 = ty * kTile;
    t.first = a.ranges[2 * (int64_t)tile];
    t.last = a.ranges[2 * (int64_t)tile + 1];
    t.tile = tile;
    return t;
}

GS3D_DEV TileInfo tile_info(const gs3d_render_args& a) { return tile_info(a, tile_of_block(blockIdx.x, gridDim.x)); }

// The blends work with the negated exponent, -power: alpha = o e^power can
// only reach 1/255 where -power <= ln(255 o) + 0.01 (see the file comment).
// -inf rejects everything (o <= 0).  Beyond 86 the exponential is zero, so a
// finite opacity rejects there in any case; a NaN or infinite one accepts
// every pixel with -power >= 0 (min(0.99, NaN) = 0.99), and +inf says so.
GS3D_DEV float exponent_limit(float o) {
    if (o > 0.0f) return o < __builtin_inff() ? sel_min(__logf(255.0f * o) + 0.01f, 86.0f) : __builtin_inff();
    return o <= 0.0f ? -__builtin_inff() : __builtin_inff();
}

// -power of the blend, from the two products of dy: the negation of
// blend_power bit for bit (rounding is symmetric in the sign), except that a
// zero is always +0: accepts() compares bit patterns.
GS3D_DEV float blend_exponent(float a, float b, float dx, float dy, float c_dy_dy) {
    const float q = __builtin_fmaf(a * dx, dx, c_dy_dy);
    return __builtin_fmaf(0.5f, q, __builtin_fmaf(b * dx, dy, 0.0f));
}

// 0 <= x <= limit for a positive limit, in one compare: positive floats order
// as their bit patterns, negative numbers and NaNs lie above all of them.
GS3D_DEV bool accepts(float x, float limit) { return __float_as_uint(x) <= __float_as_uint(limit); }

// blend_exp(-x) for 0 <= x <= 86 without its range check: the same reduction
// and polynomial.  The integer k comes from adding 1.5 * 2^23 (the sum rounds
// t to the nearest integer, ties to even, as rint does) and stays in the low
// bits of that sum, whose shift into the exponent field is the exact scaling
// (every result is a normal number).  rndne, cvt and ldexp run at half the
// rate of an add on this part, and the check is a compare and a select more.
GS3D_DEV float blend_exp_neg(float x) {
    const float z = x * -1.44269502e+00f + 12582912.0f;
    const float k = z - 12582912.0f;
    float r = __builtin_fmaf(k, -6.93145752e-01f, -x);
    r = __builtin_fmaf(k, -1.42860677e-06f, r);
    float p = 1.98412701e-04f;
    p = __builtin_fmaf(p, r, 1.38888892e-03f);
    p = __builtin_fmaf(p, r, 8.33333377e-03f);
    p = __builtin_fmaf(p, r, 4.16666679e-02f);
    p = __builtin_fmaf(p, r, 1.66666672e-01f);
    p = __builtin_fmaf(p, r, 5.00000000e-01f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_fmaf(p, r, 1.0f);
    return __uint_as_float(__float_as_uint(p) + (__float_as_uint(z) << 23));
}

// An exponent beyond 86, accepted only because the opacity is not finite,
// kept in blend_exp_neg's range (alpha is 0.99 whatever the exponential is).
// Opaque, so that the rare case stays a branch instead of selects for
// everyone.
GS3D_DEV float clamp_exponent(float x) {
    asm volatile("v_min_f32 %0, 0x42ac0000, %0" : "+v"(x));
    return x;
}

// A workgroup barrier behind which every LDS operation before it is done.
// The wait is spelled out: at the head of a loop the compiler leaves it out
// (it relies on LDS operations of a workgroup running in order, which an
// atomic that is still on its way from another SIMD does not).
GS3D_DEV void block_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
}

// Lane masks of the whole wavefront as scalars, and a select by one.  Written
// out as the three-operand form: consecutive two-operand selects on vcc issue
// five times slower than others on this part (23 against 4.5 cycles in a loop
// of them).
GS3D_DEV uint64_t lanes(bool v) { return __builtin_amdgcn_ballot_w64(v); }
GS3D_DEV float select(uint64_t mask, float yes, float no) {
    float r;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(no), "v"(yes), "s"(mask));
    return r;
}
GS3D_DEV float select0(uint64_t mask, float yes) {
    float r;
    asm("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(r) : "v"(yes), "s"(mask));
    return r;
}
GS3D_DEV int select(uint64_t mask, int yes, int no) {
    int r;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(no), "v"(yes), "s"(mask));
    return r;
}

// Minimum over dx in [lo, hi] of Q = a dx^2 + 2 b dx dy + c dy^2 at a fixed
// dy (a > 0): Q at the clamped stationary point -b dy / a.  The reciprocal
// is approximate; moving the point by a relative 1e-7 changes Q by a second
// order amount, far inside the culling margin.
GS3D_DEV float edge_min(float a, float inv_a, float b, float c, float dy, float lo, float hi) {
    const float d = sel_clamp(-b * dy * inv_a, lo, hi);
    return (a * d + 2.0f * b * dy) * d + c * dy * dy;
}

// Bit w is set unless every pixel of wavefront w's rectangle is certain to
// reject the Gaussian: the ellipse {-power <= limit}, its quadratic form Q
// widened by 1% + 0.01, misses the rectangle of pixel centres -- first by its
// bounding box (widened by 0.01 px), then exactly: the rectangle is kept when
// the centre lies inside the rectangle or Q's minimum over one of the
// rectangle's four edges is within the widened bound.  Float32 evaluation of
// Q is off by at most about 8 * 2^-24 * (a + c) |d|^2, below 2e-4 Q for the
// conics culled here, and the blend's power evaluation by as little, both far
// inside the 1% margin.  Culling
// is attempted only where a*c <= 100*det (correlation below 0.995): there the
// float32 determinant is within 1.3e-5 relative of the exact one (its
// cancellation error is at most 2^-24 * 2ac <= 200 * 2^-24 * det), so the box
// stays wider than the exact ellipse's by far more than the float32 error of
// the blend's power evaluation.  More elongated conics, non-positive-definite
// ones, overflowing products and NaNs are never culled.  Rejected pairs change
// no output, so culling leaves every result identical.
template <int PIX>
GS3D_DEV uint32_t strip_mask(float2 xy, float4 con, float limit, int x0, int y0) {
    using W = TileWaves<PIX>;
    constexpr uint32_t all = (1u << W::count) - 1u;
    const float q = 2.0f * limit;  // -power <= limit  <=>  a dx^2 + 2 b dx dy + c dy^2 <= q
    if (!(q > 0.0f) && q == q) return 0u;  // nothing passes the limit
    const float a = con.x, b = con.y, c = con.z;
    const float ac = a * c;
    const float det = ac - b * b;
    if (!(a > 0.0f && c > 0.0f && det > 0.0f && ac < 1.0e30f && ac <= 100.0f * det && q < 1.0e30f)) return all;
    // Hardware reciprocal and square root (about one ulp each): the box is
    // widened by 1% + 0.01 px, orders of magnitude beyond their error.
    const float s = (q * 1.01f + 0.01f) * __builtin_amdgcn_rcpf(det);
    const float hx = __builtin_amdgcn_sqrtf(s * c) + 0.01f;
    const float hy = __builtin_amdgcn_sqrtf(s * a) + 0.01f;
    const float bound = q * 1.01f + 0.01f;
    const float inv_a = __builtin_amdgcn_rcpf(a), inv_c = __builtin_amdgcn_rcpf(c);
    uint32_t m = 0u;
#pragma unroll
    for (int w = 0; w < W::count; ++w) {
        const float x_lo = (float)(x0 + (w % W::across) * W::cols), x_hi = x_lo + (float)(W::cols - 1);
        const float y_lo = (float)(y0 + (w / W::across) * W::rows), y_hi = y_lo + (float)(W::rows - 1);
        if (xy.x + hx < x_lo || xy.x - hx > x_hi || xy.y + hy < y_lo || xy.y - hy > y_hi) continue;
        // Centre minus pixel over the rectangle.
        const float dx_lo = xy.x - x_hi, dx_hi = xy.x - x_lo;
        const float dy_lo = xy.y - y_hi, dy_hi = xy.y - y_lo;
        bool keep = dx_lo <= 0.0f && dx_hi >= 0.0f && dy_lo <= 0.0f && dy_hi >= 0.0f;  // centre inside
        if (!keep) {
            const float e0 = edge_min(a, inv_a, b, c, dy_lo, dx_lo, dx_hi);
            const float e1 = edge_min(a, inv_a, b, c, dy_hi, dx_lo, dx_hi);
            const float e2 = edge_min(c, inv_c, b, a, dx_lo, dy_lo, dy_hi);
            const float e3 = edge_min(c, inv_c, b, a, dx_hi, dy_lo, dy_hi);
            keep = !(sel_min(sel_min(e0, e1), sel_min(e2, e3)) > bound);
        }
        if (keep) m |= 1u << w;
    }
    return m;
}

// One staged Gaussian in LDS: conic + opacity, centre, exponent cutoff and
// the window's channels in one 16-byte-aligned record, so that the blend
// loops read all of it from one LDS address (with immediate offsets) instead
// of materialising one address per field from the scalar slot index.  The
// strip masks stay in their own array: the wavefronts read them per lane.
template <int CH>
struct alignas(16) StagedRec {
    float4 con;
    float2 xy;
    float limit;  // exponent_limit
    int entry;    // list position, 1-based (forward)
    float f[CH];
};

// Strip-mask bit of a Gaussian whose opacity (kStrange) is not finite (in the
// grouped backward: or beyond kHugeOpacity), one of whose staged channels
// (kStrangeColor) is not finite, or one of whose conic entries (kSharp) is
// beyond kMomentConic: the blend loops take their cases apart.
constexpr uint32_t kStrange = 1u << 31, kStrangeColor = 1u << 30, kSharp = 1u << 29;

// Largest conic entry whose centre gradient the backward takes from moments.
// They are formed about the middle of a lane's pixels, blended or not: beside
// a pixel within a standard deviation of the centre that loses about sqrt(a)
// * 2^-24 of the gradient, and overflows for entries near the end of the
// range.  Projection dilates covariances by 0.3 (entries below 3.34); sharper
// conics come from geometry made by hand and are summed pixel by pixel.
constexpr float kMomentConic = 4.0f;

// Beyond this opacity e^power of a blended pixel may be so small that its
// product with the pixel's gradient falls below the normal range; the grouped
// backward keeps it times kHugeScale there, and stages the opacity over it.
constexpr float kHugeOpacity = 0x1p64f, kHugeScale = 0x1p64f;

// Stage one Gaussian's centre, conic, cutoff, strip mask and the channels
// [c0, c0 + CH) of its channel vector (zero beyond D').  GROUPED, for the
// grouped backward: sharp conics are marked, and the record's entry holds 1, or
// 1 / kHugeScale where the opacity is staged times that.
template <int CH, int PIX, bool LAUNDER = false, bool GROUPED = false>
GS3D_DEV void stage_gaussian(const gs3d_render_args& a, const TileInfo& t, int32_t g, int slot, int entry, int c0,
                             StagedRec<CH>* s_g, uint32_t* s_mask) {
    const int view = t.view;
    const int64_t row = (int64_t)view * a.n + g;
    const float2 xy = reinterpret_cast<const float2*>(a.centers)[row];
    const float4 con = reinterpret_cast<const float4*>(a.conics)[row];
    // The channel vector [features | extra | 1]: its loads are issued with
    // the centre's and conic's, before the cutoff and strip mask wait for
    // those (compile-time channel slots, predicated on the counts).
    const int F = a.feat_channels, E = a.extra_channels;
    const float* f = a.features + view * a.feat_view_stride + (int64_t)g * a.feat_stride;
    const float* e = E > 0 ? a.extra + view * a.extra_view_stride + (int64_t)g * a.extra_stride : nullptr;
    float v[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int gc = c0 + c;
        float x = 0.0f;
        if (gc < F)
            x = f[gc];
        else if (gc < F + E)
            x = e[gc - F];
        else if (gc == F + E && a.one_tail)
            x = 1.0f;
        v[c] = x;
    }
    StagedRec<CH>& rec = s_g[slot];
    rec.con = con;
    rec.xy = xy;
    const float limit = exponent_limit(con.w);
    rec.limit = limit;
    const bool huge = GROUPED && con.w > kHugeOpacity && con.w < __builtin_inff();
    if constexpr (GROUPED) {
        const float scale = huge ? 1.0f / kHugeScale : 1.0f;
        rec.con.w = con.w * scale;
        rec.entry = __float_as_int(scale);
    } else {
        rec.entry = entry;
    }
    int x0 = t.x0, y0 = t.y0;
    if constexpr (LAUNDER) {
        // The tile origin passes through an opaque scalar move, so that the
        // strip edges' float conversions are redone here (a few VALU per
        // staged Gaussian) instead of being hoisted out of the batch loop
        // into VGPRs that stay live over the whole traversal.
        asm volatile("" : "+s"(x0), "+s"(y0));
    }
    uint32_t mask = strip_mask<PIX>(xy, con, limit, x0, y0);
    // The channels' magnitudes, largest first: a NaN survives the integer
    // maximum of the bit patterns.
    uint32_t top = 0u;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        rec.f[c] = v[c];
        top = max(top, __float_as_uint(v[c]) & 0x7FFFFFFFu);
    }
    if (top >= 0x7F800000u) mask |= kStrangeColor;
    if (limit == __builtin_inff() || huge) mask |= kStrange;
    if constexpr (GROUPED) {
        if (!(sel_max(sel_max(__builtin_fabsf(con.x), __builtin_fabsf(con.y)), __builtin_fabsf(con.z)) <= kMomentConic))
            mask |= kSharp;
    }
    s_mask[slot] = mask;
}

// 0.0f that the compiler cannot see through (a register written by an
// opaque move), so accumulators initialised from it are updated in place.
GS3D_DEV float opaque_zero() {
    float z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    return z;
}

// Two opaque zeros from one 64-bit move.
GS3D_DEV void opaque_zero2(float& a, float& b) {
    uint64_t z;
    asm volatile("v_mov_b64 %0, 0" : "=v"(z));
    a = __uint_as_float((uint32_t)z);
    b = __uint_as_float((uint32_t)(z >> 32));
}

// One staged Gaussian as the blend loops read it from LDS.  The loops load
// the next Gaussian of their wavefront before blending the current one, so
// the LDS latency overlaps the arithmetic.
template <int CH>
struct Staged {
    float2 xy;
    float4 con;
    float limit;
    int entry;
    float f[CH];
};

template <int CH>
GS3D_DEV Staged<CH> load_staged(int j, const StagedRec<CH>* s_g) {
    const StagedRec<CH>& rec = s_g[j];
    Staged<CH> g;
    g.xy = rec.xy;
    g.con = rec.con;
    g.limit = rec.limit;
    g.entry = rec.entry;
#pragma unroll
    for (int c = 0; c < CH; ++c) g.f[c] = rec.f[c];
    return g;
}

// Contribution statistics of one accepted Gaussian (statistics.py:46-70,
// observed at gs3d/render.py:109-115).  Each lane forms, for every request r
// of the launch (RB, the request count rounded up to 1, 2, 4 or 8), its
// pixels' part: the number of accepted pixels whose value is nonzero for a
// masked count, the sum of value * alpha * T over them for a weighted sum.
// A count request's pixel values are replaced by 0/1 masks when they are
// loaded, so both kinds are one multiply-add per pixel: value times
// (accepted ? alpha * T : 0) for a sum, mask times (accepted ? 1 : 0) for a
// count.  That product form is exact only for finite values (a rejected
// pixel's value times zero), so a wavefront with a non-finite value selects
// each term instead (wave-uniform choice).  One wavefront sum covers all
// requests together (permlane pairing and a DPP row butterfly, as in the
// backward), and each lane that holds a request's total (stat_lane) adds it
// to the Gaussian's LDS slot, where the tile's wavefronts meet; once every
// wavefront is past the batch, the thread that staged the Gaussian adds the
// slot's nonzero totals to the request rows with one global atomic each
// (flush_statistics): half the global atomics of one per wavefront.
// Counts are exact (at most 256 per tile, summed in float32 without
// rounding); sums differ from per-pixel atomics only in the order of the
// float additions, which atomics leave unspecified anyway.
template <int RB>
GS3D_DEV int stat_lane(const gs3d_render_stats_args& st, int lane) {
    int r = 0;
    if constexpr (RB == 1) {
        if (lane != 63) return -1;
    } else {
        constexpr int rows = (RB + 3) / 4;
        r = wave_sum_rows_value(lane);
        if ((lane & 15) >= rows || r >= RB) return -1;
    }
    return r < st.requests ? r : -1;
}

// Adds a staged Gaussian's per-request totals (slot[r]) to the request rows
// of view `view` (each row among the rows of its kind) and clears the slot.
template <int RB>
GS3D_DEV void flush_statistics(const gs3d_render_stats_args& st, int view, int n, int32_t g, float* slot) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        if (r >= st.requests) break;
        const float v = slot[r];
        slot[r] = 0.0f;
        if (v == 0.0f) continue;
        const uint32_t before = st.sum_mask & ((1u << r) - 1u);
        if ((st.sum_mask >> r) & 1u)
            atomicAdd(st.sums + view * st.sums_view_stride + (int64_t)__builtin_popcount(before) * n + g, v);
        else
            atomicAdd(st.counts + view * st.counts_view_stride + (int64_t)(r - __builtin_popcount(before)) * n + g,
                      (int)v);
    }
}

// KINDS: the requests' kinds as a compile-time sum mask (bit r set: request
// r is a weighted sum) for launches of one or two requests, -1 to read them
// from st.sum_mask.
template <int PIX, int RB, int KINDS>
GS3D_DEV void observe_statistics(const gs3d_render_stats_args& st, int dst_r, float* slot,
                                 const uint64_t (&acc)[PIX], const float (&w)[PIX], const float (&val)[PIX][RB],
                                 bool finite, int lane) {
    float e[RB];
    if (finite) {
        float one[PIX];
#pragma unroll
        for (int k = 0; k < PIX; ++k) one[k] = select0(acc[k], 1.0f);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            // wave-uniform; a compile-time constant for KINDS >= 0
            const bool is_sum = KINDS >= 0 ? ((KINDS >> r) & 1) != 0 : ((st.sum_mask >> r) & 1u) != 0;
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < PIX; ++k) v = __builtin_fmaf(val[k][r], is_sum ? w[k] : one[k], v);
            e[r] = v;
        }
    } else {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const bool is_sum = (st.sum_mask >> r) & 1u;
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < PIX; ++k) {
                const bool hit = ((acc[k] >> lane) & 1) && val[k][r] != 0.0f;
                v += hit ? (is_sum ? val[k][r] * w[k] : 1.0f) : 0.0f;
            }
            e[r] = v;
        }
    }
    float total;
    if constexpr (RB == 1) {
        total = wave_sum_to_lane63(e[0]);
    } else {
        constexpr int rows = (RB + 3) / 4;
        float sums[rows];
        wave_sum_rows<RB>(e, sums);
#pragma unroll
        for (int q = 0; q < rows; ++q) asm volatile("" : "+v"(sums[q]));
        total = sums[0];
#pragma unroll
        for (int q = 1; q < rows; ++q) total = ((lane & 15) == q) ? sums[q] : total;
    }
    if (dst_r >= 0 && total != 0.0f) atomicAdd(slot + dst_r, total);  // LDS
}

// Up to 4 channels the kernel is held to 80 VGPRs (6 wavefronts per SIMD
// instead of 5: 1.180 -> 1.130 ms on RGB), up to 8 to 96, up to 36 to 168 (3
// wavefronts), beyond to 256 (2: 64 slots left to themselves took 284 to 302
// registers and one wavefront, 60 channels at 1237x822 893 against 549 us, with
// two statistics 1075 against 643).  Wide kernels spill a few tens of registers
// at these bounds, most of them with statistics.  Lane masks, weights of zero and the exponential from adds
// (see the file comment): 3M Gaussians, 4 x 1920x1080, 1005 -> 790 us; 500K
// at 1280x720 169 -> 138 us; 34 channels at 1600x1200 688 -> 596 us.
//
// MODE: 0 plain; 1 with contribution statistics; 2 also counting (pixel,
// Gaussian) pairs into counts[0..2]: visited as the reference's loop visits
// them (list entries up to and including the one that terminates the pixel,
// the whole list otherwise), evaluated by this kernel (after strip culling,
// while the pixel is live) and accepted (blended).
//
// RB: statistics requests compiled in (MODE 1; the launch's request count
// rounded up to 1, 2, 4 or 8), so that only their pixel values take
// registers; KINDS: their kinds as a sum mask for one or two requests (the
// observer then needs no per-request selects), -1 otherwise.
//
// LISTS (MODE 0): 0 whole lists; 1 lists capped by gs3d_render_args.caps
// and/or stops reported (stop_out, redo flags); 2 a redo launch
// (gs3d_render_args.redo_pass), whose workgroups walk the tiles listed by the
// capped launch.  Only the instantiations that use them carry the stop
// tracking and the loop.
template <int CH, int PIX, int MODE, int RB = 1, int KINDS = -1, int LISTS = 0>
__global__ __launch_bounds__(kTilePixels / PIX) __attribute__((amdgpu_waves_per_eu(CH <= 4 ? 6 : CH <= 8 ? 5 : CH <= 36 ? 3 : 2))) void render_fwd_kernel(gs3d_render_args a, gs3d_render_stats_args st, int c0, unsigned long long* counts) {
    constexpr bool STATS = MODE == 1, COUNTS = MODE == 2;
    constexpr int NT = kTilePixels / PIX;
    constexpr int B = Batch<CH>::size;
    __shared__ StagedRec<CH> s_g[B];
    __shared__ uint32_t s_mask[B];
    __shared__ int s_live[TileWaves<PIX>::count];
    // Per staged Gaussian: the tile's totals of every statistics request.
    __shared__ float s_stat[STATS ? B * RB : 1];
    static_assert(LISTS == 0 || MODE == 0, "capped lists neither count pairs nor total statistics");
    // The blend of one tile: a normal launch blends the tile of its
    // workgroup, a redo launch walks the tiles that the capped launch listed.
    auto blend = [&](const TileInfo t) {
        // With caps the tile's list is read up to list_cap of its previous stop
        // (the id-write pass wrote that far); a redo reads whole lists.
        int last = t.last;
        bool capped = false;
        if constexpr (LISTS == 1) {
            if (a.caps) {
                const uint32_t cap = list_cap(a.caps[t.tile]);
                if ((uint32_t)(t.last - t.first) > cap) {
                    last = t.first + (int)cap;
                    capped = true;
                }
            }
        }
        const int D = a.feat_channels + a.extra_channels + (a.one_tail ? 1 : 0);
        const int lane = lane_id(), wave = threadIdx.x >> 6;
        if constexpr (STATS)
            for (int e = threadIdx.x; e < B * RB; e += NT) s_stat[e] = 0.0f;
        if (c0 == 0 && a.zero_out) {
            // The blend VJP's accumulation buffers, cleared by the first
            // window's launch: the stores drain while the blend computes.
            typedef float zero4 __attribute__((ext_vector_type(4)));
            const int64_t n4 = a.zero_count >> 2;
            zero4* z = reinterpret_cast<zero4*>(a.zero_out);
            const int64_t step = (int64_t)gridDim.x * NT;
            for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < n4; i += step)
                __builtin_nontemporal_store(zero4{0.0f, 0.0f, 0.0f, 0.0f}, z + i);
            if (blockIdx.x == 0 && threadIdx.x < (a.zero_count & 3)) a.zero_out[(n4 << 2) + threadIdx.x] = 0.0f;
        }
        // Pixels that have terminated or lie outside the image, as lane masks:
        // the tests' results meet in scalar registers, beside the vector work.
        uint64_t done[PIX];
        float fx[PIX], fy, T[PIX], color[PIX][CH];
        int px[PIX], py, last_contributor[PIX];
        bool outside[PIX];
        float val[PIX][STATS ? RB : 1];
        int visited[PIX];
        uint64_t evaluated = 0, accepted = 0;  // of the wavefront
#pragma unroll
        for (int k = 0; k < PIX; ++k) {
            int lx, ly;
            pixel_of<PIX>(threadIdx.x, k, lx, ly);
            px[k] = t.x0 + lx;
            py = t.y0 + ly;  // a lane's pixels share their row
            fx[k] = (float)px[k];
            fy = (float)py;
            outside[k] = !(px[k] < a.width && py < a.height);
            done[k] = lanes(outside[k]);
            visited[k] = outside[k] ? 0 : last - t.first;  // the whole list unless the pixel terminates
            T[k] = 1.0f;
            last_contributor[k] = 0;
#pragma unroll
            for (int c = 0; c < CH; ++c) color[k][c] = 0.0f;
            if constexpr (STATS) {
                const float* pv = st.pixel_values + t.view * st.pixel_view_stride + (int64_t)py * a.width + px[k];
                const int64_t plane = (int64_t)a.width * a.height;
#pragma unroll
                for (int r = 0; r < RB; ++r) {
                    const float v = (r < st.requests && !outside[k]) ? pv[r * plane] : 0.0f;
                    // Count requests keep a 0/1 mask (see observe_statistics).
                    val[k][r] = ((st.sum_mask >> r) & 1u) ? v : (v != 0.0f ? 1.0f : 0.0f);
                }
            }
        }
        // Each thread stages at most one Gaussian per batch (B <= NT); its index
        // for the next batch is loaded while the current batch blends (clamped
        // into the list, so the load is unconditional).
        static_assert(B <= NT, "one staged Gaussian per thread and batch");
        int32_t next_id = last > t.first ? a.ids[min(t.first + (int)threadIdx.x, last - 1)] : 0;
        int stat_r = -1;
        bool stat_finite = true;
        // The Gaussian this thread staged for the batch being blended, whose
        // statistics slot it flushes (-1: none).
        int32_t flush_id = -1;
        auto flush = [&]() {
            if constexpr (STATS) {
                if (flush_id >= 0) flush_statistics<RB>(st, t.view, a.n, flush_id, &s_stat[threadIdx.x * RB]);
                flush_id = -1;
            }
        };
        if constexpr (STATS) {
            stat_r = stat_lane<RB>(st, lane);
            bool finite = true;
#pragma unroll
            for (int k = 0; k < PIX; ++k)
#pragma unroll
                for (int r = 0; r < RB; ++r) finite = finite && __builtin_fabsf(val[k][r]) <= 3.0e38f;
            stat_finite = __ballot(!finite) == 0;
        }
        auto alive = [&]() {
            uint64_t all = done[0];
#pragma unroll
            for (int k = 1; k < PIX; ++k) all &= done[k];
            return all != ~0ull;
        };
        // A barrier that tells whether any wavefront has a live pixel.
        auto any_alive = [&]() {
            if (lane == 0) s_live[wave] = alive();
            block_barrier();
            int v = 0;
#pragma unroll
            for (int w = 0; w < TileWaves<PIX>::count; ++w) v |= s_live[w];
            return __builtin_amdgcn_readfirstlane(v) != 0;
        };
        int stop = -1;  // list entries read before every pixel terminated (-1: never)
        for (int begin = t.first; begin < last; begin += B) {
            const bool more_pixels = any_alive();
            flush();  // every wavefront is past the previous batch
            if (!more_pixels) {
                stop = begin - t.first;
                break;
            }
            if (threadIdx.x < B) {
                const int e = threadIdx.x;
                const int32_t g = next_id;
                if (begin + e < last) {
                    // The 4-channel plain blend fits its registers without the
                    // tile-origin laundering (and is fastest so).
                    stage_gaussian<CH, PIX, (STATS || CH > 4)>(a, t, g, e, begin - t.first + e + 1, c0, s_g, s_mask);
                    if constexpr (STATS) flush_id = g;
                }
                if (begin + B < last) next_id = a.ids[min(begin + B + e, last - 1)];
            }
            block_barrier();
            const int cnt = min(B, last - begin);
            bool live = alive();
            for (int c0 = 0; c0 < cnt && live; c0 += 64) {
                // This wavefront's Gaussians of the next 64, in list order.
                const uint32_t flags = s_mask[min(c0 + lane, B - 1)];
                uint64_t todo = lanes(c0 + lane < cnt && ((flags >> wave) & 1u));
                if (!todo) continue;
                // Some opacity is not finite (of any of the chunk's Gaussians).
                const bool strange = (lanes((flags & kStrange) != 0) & todo) != 0;
                const bool strange_color = (lanes((flags & kStrangeColor) != 0) & todo) != 0;
                // Blend one Gaussian (batch slot j) into this lane's pixels.
                // Tests are lane masks combined in scalar registers; a pixel
                // that rejects the Gaussian adds each channel with weight
                // zero, which leaves a finite sum as it was.  Channels that
                // are not all finite (FINITE false) are selected instead, so
                // that a rejected Gaussian's cannot reach the pixel.
                auto blend = [&](const Staged<CH>& g, int j, auto finite) {
                    constexpr bool FINITE = decltype(finite)::value;
                    const float dy = g.xy.y - fy;
                    const float c_dy_dy = (g.con.z * dy) * dy;
                    float x[PIX];
                    uint64_t in[PIX], any = 0;
#pragma unroll
                    for (int k = 0; k < PIX; ++k) {
                        x[k] = blend_exponent(g.con.x, g.con.y, g.xy.x - fx[k], dy, c_dy_dy);
                        in[k] = lanes(accepts(x[k], g.limit)) & ~done[k];
                        any |= in[k];
                        if constexpr (COUNTS) evaluated += __builtin_popcountll(~done[k]);
                    }
                    if (!any) return;
                    if (strange) {
#pragma unroll
                        for (int k = 0; k < PIX; ++k) x[k] = clamp_exponent(x[k]);
                    }
                    float w[PIX];
                    uint64_t upd[PIX];
#pragma unroll
                    for (int k = 0; k < PIX; ++k) {
                        const float alpha = sel_min(0.99f, g.con.w * blend_exp_neg(x[k]));
                        const float next_t = T[k] * (1.0f - alpha);
                        const uint64_t take = lanes(alpha >= 1.0f / 255.0f) & in[k];
                        const uint64_t low = lanes(next_t < 0.0001f);
                        const uint64_t term = take & low;
                        upd[k] = take & ~low;
                        done[k] |= term;
                        w[k] = select0(upd[k], alpha * T[k]);
                        T[k] = select(upd[k], next_t, T[k]);
                        if constexpr (COUNTS) {
                            visited[k] = select(term, g.entry, visited[k]);
                            accepted += __builtin_popcountll(upd[k]);
                        }
#pragma unroll
                        for (int c = 0; c < CH; ++c) {
                            const float sum = __builtin_fmaf(g.f[c], w[k], color[k][c]);
                            color[k][c] = FINITE ? sum : select(upd[k], sum, color[k][c]);
                        }
                        last_contributor[k] = select(upd[k], g.entry, last_contributor[k]);
                    }
                    if constexpr (STATS) {
                        uint64_t hit = 0;
#pragma unroll
                        for (int k = 0; k < PIX; ++k) hit |= upd[k];
                        if (hit)
                            observe_statistics<PIX, RB, KINDS>(st, stat_r, &s_stat[j * RB], upd, w, val, stat_finite, lane);
                    }
                };
                auto take = [&]() {
                    const int j = c0 + __builtin_ctzll(todo);
                    todo &= todo - 1;
                    return j;
                };
                auto at_use = [&](auto finite) {
                    while (todo) {
                        if (!alive()) {
                            live = false;
                            break;
                        }
                        const int j = take();
                        blend(load_staged<CH>(j, s_g), j, finite);
                    }
                };
                if (strange_color) {
                    at_use(std::false_type{});
                } else if constexpr ((STATS && (RB > 2 || CH > 4)) || CH > 16) {
                    // Loads at use: the pipelined form's extra registers would
                    // cost occupancy -- with statistics beyond two requests (their
                    // pixel values take 4 * PIX registers or more) or four
                    // channels (up to both, the pipelined form is held to 80
                    // VGPRs with up to seven spilled at two pixels per lane),
                    // and beyond 16 channels a wavefront per SIMD (36 channels:
                    // 0.83 -> 0.72 ms on the 32-feature workload; 64: 1078 -> 921
                    // us at 62 channels, 300K Gaussians, 1280x960).
                    at_use(std::true_type{});
                } else {
                    // Unrolled by two: the next Gaussian is loaded into the other
                    // buffer before the current one is blended.
                    int ja = take(), jb = 0;
                    Staged<CH> ga = load_staged<CH>(ja, s_g), gb;
                    while (true) {
                        if (!alive()) {
                            live = false;
                            break;
                        }
                        bool more = todo != 0;
                        if (more) {
                            jb = take();
                            gb = load_staged<CH>(jb, s_g);
                        }
                        blend(ga, ja, std::true_type{});
                        if (!more) break;
                        // Liveness is checked once per two Gaussians: a Gaussian
                        // blended after every pixel is done changes nothing (no
                        // pixel accepts it).
                        more = todo != 0;
                        if (more) {
                            ja = take();
                            ga = load_staged<CH>(ja, s_g);
                        }
                        blend(gb, jb, std::true_type{});
                        if (!more) break;
                    }
                }
            }
        }
        if constexpr (STATS) {
            // The last batch, when the loop ran to the end of the list.
            block_barrier();
            flush();
        }
        if constexpr (LISTS != 0) {
            if (stop < 0) {
                // The loop ran to the end of the list it had: all of it read.
                if (!any_alive()) stop = last - t.first;
            }
            if (threadIdx.x == 0 && c0 == 0) {
                // A capped tile with pixels still live needs its whole list:
                // flagged and listed for a redo (its outputs here are
                // incomplete).
                if (LISTS == 1 && a.redo) {
                    const bool redo = capped && stop < 0;
                    a.redo[t.tile] = redo ? 1 : 0;
                    if (redo) {
                        // The list holds one slot per tile (a count left
                        // uncleared cannot send the store out of it).
                        const int slot = atomicAdd(a.redo_list, 1);
                        if ((unsigned)slot < (unsigned)gridDim.x) a.redo_list[1 + slot] = t.tile;
                    }
                }
                if (a.stop_out) a.stop_out[t.tile] = stop;
            }
        }
        const float* bg = a.background ? a.background + t.view * a.background_view_stride : nullptr;
        const int F = a.feat_channels, E = a.extra_channels;
#pragma unroll
        for (int k = 0; k < PIX; ++k) {
            if (outside[k]) continue;
            const int64_t pix = ((int64_t)t.view * a.height + py) * a.width + px[k];
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int gc = c0 + c;
                if (gc >= D) continue;
                const float v = __builtin_fmaf(T[k], (bg && gc < F) ? bg[gc] : 0.0f, color[k][c]);
                if (gc < F)
                    a.image[pix * F + gc] = v;
                else if (gc < F + E)
                    a.image_extra[pix * E + (gc - F)] = v;
                else
                    a.image_alpha[pix] = v;
            }
            if (c0 == 0) {
                a.final_t[pix] = T[k];
                a.contributors[pix] = last_contributor[k];
            }
        }
        if constexpr (COUNTS) {
            uint64_t v = 0;
#pragma unroll
            for (int k = 0; k < PIX; ++k) v += (uint64_t)visited[k];
            const uint64_t e = evaluated, c = accepted;
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) v += (uint64_t)__shfl_xor((long long)v, d, 64);
            if (lane == 0) {
                atomicAdd(counts, (unsigned long long)v);
                atomicAdd(counts + 1, (unsigned long long)e);
                atomicAdd(counts + 2, (unsigned long long)c);
            }
        }
    };
    if constexpr (LISTS == 2) {
        // redo_list[0] tiles from redo_list[1], over a grid smaller than the
        // frame's; the next tile reuses the staging LDS.  Counts and tile
        // indices beyond the frame's tiles are ignored.
        const int tiles = a.views * ((a.width + kTile - 1) / kTile) * ((a.height + kTile - 1) / kTile);
        const int items = min(a.redo_list[0], tiles);
        for (int item = blockIdx.x; item < items; item += gridDim.x) {
            const int tile = a.redo_list[1 + item];
            if ((unsigned)tile >= (unsigned)tiles) continue;  // uniform: one value per workgroup
            blend(tile_info(a, tile));
            block_barrier();
        }
    } else {
        blend(tile_info(a));
    }
}

// Channels [c_begin, D) of Gaussian g's vector dotted with the upstream
// gradient of pixel (px, py) (geometry launch of a vector wider than its
// window: the channels beyond the window come from global memory).
GS3D_DEV float rest_dot(const gs3d_render_bwd_args& b, int view, int64_t g, float px, float py, int c_begin) {
    const gs3d_render_args& a = b.fwd;
    const int64_t pix = ((int64_t)view * a.height + (int)py) * a.width + (int)px;
    const int F = a.feat_channels, E = a.extra_channels;
    float dot = 0.0f;
    int c = c_begin;
    if (c < F) {
        const float* f = a.features + view * a.feat_view_stride + g * a.feat_stride;
        const float* u = b.upstream ? b.upstream + pix * b.upstream_stride : nullptr;
        for (; c < F; ++c) dot = __builtin_fmaf(f[c], u ? u[c] : 0.0f, dot);
    }
    if (c < F + E) {
        const float* f = a.extra + view * a.extra_view_stride + g * a.extra_stride;
        const float* u = b.upstream_extra ? b.upstream_extra + pix * b.upstream_extra_stride : nullptr;
        for (; c < F + E; ++c) dot = __builtin_fmaf(f[c - F], u ? u[c - F] : 0.0f, dot);
    }
    if (c == F + E && a.one_tail && b.upstream_alpha) dot += b.upstream_alpha[pix * b.upstream_alpha_stride];
    return dot;
}

// ---------------------------------------------------------------------------
// Backward, up to 44 channels: four Gaussians at a time
//
// The gradients of a Gaussian are sums over pixels that depend on a pixel
// through two numbers, the blend weight alpha T (colour gradients) and
// h = e^power dL/dalpha (everything else: with w = o h the centre gradient is
// -sum w (a dx + b dy, c dy + b dx), the conic's -1/2 sum w (dx dx, 2 dx dy,
// dy dy), the opacity's sum h).  So a lane keeps only those two per pixel, for
// four accepted Gaussians; eight or sixteen permlane swaps then exchange them
// such that the 16 lanes of row q hold Gaussian q, each lane with the pixels of
// four of the wavefront's row pairs.  There the sums over a lane's pixels are
// separable moments -- over its pixels h, h dy and h dy dy need no product
// with dx per pixel -- and one reduction over 16 lanes finishes four
// Gaussians, whose entries one atomic instruction adds.  Before, every
// Gaussian's ten products were formed per pixel and summed over 64 lanes by
// themselves, 40% of the kernel's vector time.
// ---------------------------------------------------------------------------

// Exchanges register r's row s of 16 lanes with register s's row r, for two
// sets of four registers.  In one block: the wait states that a swap needs
// after a vector write of its operands are spelled out once, and between the
// two levels the other set's swaps provide them.
GS3D_DEV void exchange_rows(float (&a)[4], float (&b)[4]) {
    asm volatile(
        "s_nop 1\n\t"
        "v_permlane32_swap_b32 %0, %2\n\t"
        "v_permlane32_swap_b32 %1, %3\n\t"
        "v_permlane32_swap_b32 %4, %6\n\t"
        "v_permlane32_swap_b32 %5, %7\n\t"
        "v_permlane16_swap_b32 %0, %1\n\t"
        "v_permlane16_swap_b32 %2, %3\n\t"
        "v_permlane16_swap_b32 %4, %5\n\t"
        "v_permlane16_swap_b32 %6, %7\n\t"
        "s_nop 1"
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
}

// Sums V values over each row of 16 lanes; for every i the total of value
// 4 * i + row_bank_value(lane) ends in v[4 * i] of every lane.  The first
// two levels write two values' sums into the two halves, then the four banks
// of four lanes, of one register (masked DPP adds): 21 instructions for ten
// values.  Each block starts with the wait states a DPP read needs.
template <int V>
GS3D_DEV void sum_rows_packed(float (&v)[V]) {
#pragma unroll
    for (int i = 0; i < V; i += 2) {
        if (i + 1 < V)
            asm volatile(
                "s_nop 1\n\t"
                "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
                "v_add_f32_dpp %0, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xc"
                : "+v"(v[i]) : "v"(v[i + 1 < V ? i + 1 : i]));
        else
            asm volatile("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf" : "+v"(v[i]));
    }
#pragma unroll
    for (int i = 0; i < V; i += 4) {
        if (i + 2 < V)
            asm volatile(
                "s_nop 1\n\t"
                "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
                "v_add_f32_dpp %0, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xa"
                : "+v"(v[i]) : "v"(v[i + 2 < V ? i + 2 : i]));
        else
            asm volatile("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf" : "+v"(v[i]));
    }
#pragma unroll
    for (int i = 0; i < V; i += 4)
        asm volatile(
            "s_nop 1\n\t"
            "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "s_nop 1\n\t"
            "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
            : "+v"(v[i]));
}

// Exchanges rows of 16 lanes among 1, 2 or 4 registers, register i's row q
// holding part i of Gaussian q, so that each Gaussian's parts lie in the rows
// of one register: all four rows of register q, rows 2 (q / 2) and on of
// register q % 2, or as they are.  An atomic instruction costs by the cache
// lines that its lanes touch, so a Gaussian's parts leave together: 100K
// Gaussians at 1920x1080, some covering much of the frame, 28 channels 2566 us
// part by part, 1655 gathered; 13 channels 1314 and 910.
GS3D_DEV void gather_entries(float (&)[1]) {}
GS3D_DEV void gather_entries(float (&a)[2]) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a[0]), "+v"(a[1]));
}
GS3D_DEV void gather_entries(float (&a)[4]) {
    asm volatile(
        "s_nop 1\n\t"
        "v_permlane32_swap_b32 %0, %2\n\t"
        "v_permlane32_swap_b32 %1, %3\n\t"
        "s_nop 1\n\t"
        "v_permlane16_swap_b32 %0, %1\n\t"
        "v_permlane16_swap_b32 %2, %3\n\t"
        "s_nop 1"
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
}

GS3D_DEV int row_bank_value(int lane) {
    const int bank = (lane >> 2) & 3;
    return 2 * (bank & 1) + (bank >> 1);
}

// a x + b y to about one rounding of its own value: the rounding error of
// b y, which dominates where the terms cancel, is added back.
GS3D_DEV float dot2_accurate(float a, float x, float b, float y) {
    const float p = b * y;
    const float e = __builtin_fmaf(b, y, -p);
    return __builtin_fmaf(a, x, p) + e;
}

// Upstream gradient of blended channel gc at pixel index pix.
GS3D_DEV float upstream_at(const gs3d_render_bwd_args& b, int64_t pix, int gc, int D) {
    // The channel's source (wave-uniform selects, no branch); channels
    // without one read final_t and take 0.
    const int F = b.fwd.feat_channels, E = b.fwd.extra_channels;
    const float* src = gc < F ? b.upstream : gc < F + E ? b.upstream_extra : b.upstream_alpha;
    const int64_t stride = gc < F ? b.upstream_stride : gc < F + E ? b.upstream_extra_stride : b.upstream_alpha_stride;
    const int off = gc < F ? gc : gc < F + E ? gc - F : 0;
    const bool has = gc < D && src != nullptr;
    const float u = has ? src[pix * stride + off] : b.fwd.final_t[pix];
    return has ? u : 0.0f;
}

// Gaussians staged per batch: the staged channels and the pixels' gradients
// share the LDS that resident workgroups leave.  9 to 16 channels hold three
// wavefronts per SIMD with 256 (43 KB); 128 would make it four, 3340 -> 2995 us
// for 13 channels of 1M Gaussians 4x1080p, and cost frames that have fewer
// wavefronts than that their staging rounds, 145 -> 158 us at 256x256.
template <int CH>
struct RowsBatch {
    static constexpr int size = CH <= 8 ? 128 : CH <= 16 ? 256 : CH <= 20 ? 128 : 64;
};

// D <= CH channels, of which at most NC have gradients (the constant alpha
// channel, last, has none).  Bound by vector instructions: at two pixels per
// lane about 90 per Gaussian undo it from the pixels and 35 are its share of a
// group's sums; without the atomics the kernel takes 1% less where Gaussians
// are small and 24% less where some cover thousands of tiles.  Against one
// Gaussian at a time: 1M Gaussians 4x1080p 1615 -> 1345 us (94 VGPRs, five
// wavefronts per SIMD), with 18 channels 6600 -> 2770, with 36 6910 -> 5080;
// 400K at 1237x822 283 -> 224, with 9 channels 448 -> 360.  The pixels'
// gradients for the second half lie in LDS: in registers (24 more) the kernel
// spilled or lost a wavefront per SIMD.
template <int CH, int NC, bool ABS, int PIX>
__global__ __launch_bounds__(kTilePixels / PIX) __attribute__((amdgpu_waves_per_eu(CH <= 4 ? 5 : CH <= 8 ? 4 : CH <= 16 ? 3 : CH <= 20 ? 4 : CH <= 36 ? 3 : 2))) void render_bwd_rows_kernel(gs3d_render_bwd_args b) {
    constexpr int NT = kTilePixels / PIX;
    constexpr int B = RowsBatch<CH>::size;
    constexpr int FB = ABS ? 8 : 6;
    constexpr int V = FB + NC;  // entries: centre xy, conic abc, opacity, [|centre| xy], channels
    // Rows of 16 lanes that hold a Gaussian's entries when they are added.
    constexpr int ROWS = V <= 16 ? 1 : V <= 32 ? 2 : 4;
    static_assert(B <= 256, "four batch slots are packed into one word");
    static_assert(B <= NT, "one staged Gaussian per thread and batch");
    static_assert(NC == CH || NC == CH - 1, "");
    __shared__ StagedRec<CH> s_g[B];
    __shared__ uint32_t s_mask[B];
    __shared__ int32_t s_id[B];
    __shared__ int s_max_last;
    // The wavefronts' upstream gradients by place after the exchange: [row
    // pair and pixel of the lane][lane of the row of 16].
    struct alignas(16) PixelGrad {
        float c[(NC + 3) / 4 * 4];  // the padding may be read, never used
    };
    __shared__ PixelGrad s_grad[TileWaves<PIX>::count][4 * PIX][16];
    const gs3d_render_args& a = b.fwd;
    const TileInfo t = tile_info(a);
    const int F = a.feat_channels, E = a.extra_channels;
    const int D = F + E + (a.one_tail ? 1 : 0);
    const int lane = lane_id(), wave = threadIdx.x >> 6, q = lane >> 4;
    // Per pixel: S = sum_c accum_c * grad_c, the colour accumulated behind
    // the current Gaussian dotted with the upstream gradient.  With
    // dot = sum_c f_c * grad_c the alpha gradient sum_c (f_c - accum_c) grad_c
    // (gs3d/render.py:300-312) is E = dot - S, and
    // accum_c = la last_c + (1 - la) accum_c becomes S = S + la E_last with
    // la and E_last those of the last accepted Gaussian: no per-channel state
    // besides grad.  bg_t = -T_final * sum_c bg_c grad_c is the background
    // term, divided by the transmittance factors as they are undone.
    float fx[PIX], fy, T[PIX], bg_t[PIX], last_alpha[PIX], S[PIX], last_e[PIX];
    float grad[PIX][CH];
    int last_contributor[PIX];
    bool inside[PIX];
    if (threadIdx.x == 0) s_max_last = 0;
    const float* bg = a.background ? a.background + t.view * a.background_view_stride : nullptr;
    int my_max = 0;
    int x_first, y_own;
    pixel_of<PIX>(threadIdx.x, 0, x_first, y_own);
    x_first += t.x0;
    y_own += t.y0;
    fy = (float)y_own;
    auto pixel_index = [&](int x, int y) {
        return ((int64_t)t.view * a.height + min(y, a.height - 1)) * a.width + min(x, a.width - 1);
    };
    // Per-pixel inputs: every load first, from the pixel clamped into the
    // image, then the pixels outside the image are cleared.  A load under a
    // per-lane condition would be a branch that waits for its data.
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        const int64_t pix = pixel_index(x_first + k, y_own);
        fx[k] = (float)(x_first + k);
        inside[k] = x_first + k < a.width && y_own < a.height;
        T[k] = a.final_t[pix];
        last_contributor[k] = a.contributors[pix];
#pragma unroll
        for (int c = 0; c < CH; ++c) grad[k][c] = upstream_at(b, pix, c, D);
    }
    bool finite = true;
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        bg_t[k] = last_alpha[k] = S[k] = last_e[k] = 0.0f;
        if (!inside[k]) {
            T[k] = 0.0f;
            last_contributor[k] = 0;
#pragma unroll
            for (int c = 0; c < CH; ++c) grad[k][c] = 0.0f;
        }
        PixelGrad& place = s_grad[wave][PIX * q + k][lane & 15];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            place.c[c] = grad[k][c];
            finite = finite && __builtin_fabsf(grad[k][c]) <= 3.4028235e38f;
        }
        float bg_grad = 0.0f;
        if (bg) {
#pragma unroll
            for (int c = 0; c < CH; ++c) bg_grad += (c < F ? bg[c] : 0.0f) * grad[k][c];
        }
        if (inside[k]) bg_t[k] = -T[k] * bg_grad;
        my_max = max(my_max, last_contributor[k]);
    }
    const bool all_finite = lanes(!finite) == 0;
    block_barrier();
    if (my_max > 0) atomicMax(&s_max_last, my_max);
    block_barrier();
    const int max_last = min(s_max_last, t.last - t.first);
    // The gradient entry this lane adds: entry k of Gaussian g lies at base +
    // g * step.  The entries of a Gaussian are added by one instruction (two
    // Gaussians share it up to 32 entries, four up to 16): lanes of row q hold
    // the 16 entries from 16 * (q % ROWS).
    const int k_low = 4 * (lane & 3) + row_bank_value(lane);
    float* dst_base = nullptr;
    uint32_t dst_step = 0;  // row strides below 2^31 (checked on the host)
    {
        const int k = 16 * (q % ROWS) + k_low;
        const int64_t row0 = (int64_t)t.view * a.n;
        if (k >= V) {
        } else if (k < 2) {
            dst_base = b.grad_centers + row0 * b.grad_centers_stride + k;
            dst_step = b.grad_centers_stride;
        } else if (k < 6) {
            dst_base = b.grad_conics + row0 * b.grad_conics_stride + (k - 2);
            dst_step = b.grad_conics_stride;
        } else if (ABS && k < 8) {
            dst_base = b.abs_centers + row0 * b.abs_stride + (k - 6);
            dst_step = b.abs_stride;
        } else {
            const int c = k - FB;
            if (c < F) {
                if (b.grad_features) {
                    dst_base = b.grad_features + t.view * b.grad_feat_view_stride + c;
                    dst_step = b.grad_feat_stride;
                }
            } else if (c < F + E && b.grad_extra) {
                dst_base = b.grad_extra + t.view * b.grad_extra_view_stride + (c - F);
                dst_step = b.grad_extra_stride;
            }
        }
    }
    // What entry k_low, the only one of the lane's with a factor, is multiplied
    // by: all but the opacity's by the opacity.
    const bool times_opacity = k_low < FB && k_low != 5, is_opacity = k_low == 5;
    const float entry_scale = k_low < 2 || k_low == 3 ? -1.0f : k_low == 2 || k_low == 4 ? -0.5f : 1.0f;
    // Largest last contributor among this wavefront's pixels (wave-uniform).
    int wave_last = my_max;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) wave_last = max(wave_last, __shfl_xor(wave_last, d, 64));
    // As in the forward: one staged Gaussian per thread and batch, its index
    // for the next batch loaded while the current one is traversed.
    int32_t next_id = max_last > 0 ? a.ids[t.first + max(max_last - 1 - (int)threadIdx.x, 0)] : 0;
    for (int top = max_last; top > 0; top -= B) {
        block_barrier();
        if (threadIdx.x < B) {
            const int e = threadIdx.x;
            const int p = top - 1 - e;
            const int32_t g = next_id;
            if (p >= 0) {
                s_id[e] = g;
                stage_gaussian<CH, PIX, true, true>(a, t, g, e, 0, 0, s_g, s_mask);
            }
            if (top > B) next_id = a.ids[t.first + max(p - B, 0)];
        }
        block_barrier();
        const int cnt = min(B, top);
        // Up to four blended Gaussians: values [pixel][slot], and their batch
        // slots, a byte each.
        float aT[PIX][4], h[PIX][4];
        uint32_t slots = 0;
        int used = 0;
        bool sharp = false;  // one of the batch's Gaussians so far is kSharp
        // The gradients of the Gaussians in the slots.
        auto finish = [&]() {
            // Row q of lanes: Gaussian q of the four, [pixel][row pair].
#pragma unroll
            for (int k = 0; k < PIX; ++k) exchange_rows(aT[k], h[k]);
            const int j = (slots >> (8 * q)) & 255;
            const float4 con = s_g[j].con;
            const float2 xy = s_g[j].xy;
            const float unscale = __int_as_float(s_g[j].entry);
            const int32_t id = s_id[j];
            float dx[PIX], dy[4];
#pragma unroll
            for (int k = 0; k < PIX; ++k) dx[k] = xy.x - fx[k];
#pragma unroll
            for (int r = 0; r < 4; ++r) dy[r] = (xy.y - (fy - (float)(2 * q))) - (float)(2 * r);
            float v[V];
            // Moments over the lane's pixels: per column k the sums of h
            // and h dy, per row pair P_r = sum_k h.
            float A[PIX], H[PIX], P[4], yy = 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                P[r] = PIX == 2 ? h[0][r] + h[PIX - 1][r] : h[0][r];
                const float py = P[r] * dy[r];
                yy = r ? __builtin_fmaf(py, dy[r], yy) : py * dy[r];
            }
#pragma unroll
            for (int k = 0; k < PIX; ++k) {
                A[k] = (h[k][0] + h[k][1]) + (h[k][2] + h[k][3]);
                H[k] = h[k][0] * dy[0];
#pragma unroll
                for (int r = 1; r < 4; ++r) H[k] = __builtin_fmaf(h[k][r], dy[r], H[k]);
            }
            const float mass = PIX == 2 ? A[0] + A[PIX - 1] : A[0];
            // The centre gradient from the moments about the middle of
            // the lane's pixels (column offsets of 1/2, rows of 1 and 3):
            // a dx + b dy may cancel, and is taken there to one rounding.
            const float mx = PIX == 2 ? 0.5f * (A[0] - A[PIX - 1]) : 0.0f;
            const float my = __builtin_fmaf(3.0f, P[0] - P[3], P[1] - P[2]);
            const float dxm = PIX == 2 ? dx[0] - 0.5f : dx[0], dym = dy[0] - 3.0f;
            const float ux = dot2_accurate(con.x, dxm, con.y, dym);
            const float uy = dot2_accurate(con.z, dym, con.y, dxm);
            v[0] = __builtin_fmaf(ux, mass, con.y * my);
            v[1] = __builtin_fmaf(uy, mass, con.z * my);
            if constexpr (PIX == 2) {
                v[0] = __builtin_fmaf(con.x, mx, v[0]);
                v[1] = __builtin_fmaf(con.y, mx, v[1]);
            }
            if constexpr (ABS) {
                v[6] = v[7] = 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float bdy = con.y * dy[r], cdy = con.z * dy[r];
#pragma unroll
                    for (int k = 0; k < PIX; ++k) {
                        const float px = __builtin_fmaf(con.x, dx[k], bdy), py = __builtin_fmaf(con.y, dx[k], cdy);
                        v[6] = __builtin_fmaf(__builtin_fabsf(h[k][r]), __builtin_fabsf(px), v[6]);
                        v[7] = __builtin_fmaf(__builtin_fabsf(h[k][r]), __builtin_fabsf(py), v[7]);
                    }
                }
            }
            v[2] = (A[0] * dx[0]) * dx[0];
            v[3] = H[0] * dx[0];
            if constexpr (PIX == 2) {
                v[2] = __builtin_fmaf(A[PIX - 1] * dx[PIX - 1], dx[PIX - 1], v[2]);
                v[3] = __builtin_fmaf(H[PIX - 1], dx[PIX - 1], v[3]);
            }
            v[4] = yy;
            v[5] = mass;
            // The colour sums, four pixels and four channels at a time, so that
            // no more gradients hold registers.  Beyond 8 channels the next
            // ones are on their way from LDS while the ones before are added
            // (42 channels of a 256x256 frame 272 -> 257 us); below, that would
            // spill, or cost a wavefront per SIMD (8 channels 240 -> 258 us at
            // 1237x822).  Choosing by all_finite per load had made a block of
            // each, waiting for LDS one by one: 36 channels of a 256x256 frame
            // 322 -> 232 us, of 1M Gaussians 4x1080p 6440 -> 5080 us.  A pixel
            // that did not blend the Gaussian has weight zero; a non-finite
            // gradient there must not reach it.
            auto colors = [&](auto finite) {
                constexpr bool FINITE = decltype(finite)::value;
                constexpr int STEPS = (NC + 3) / 4 * PIX;
                constexpr bool AHEAD = CH > 8;
                float4 u[2][4];
                auto load = [&](int step) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        u[step & 1][i] = *reinterpret_cast<const float4*>(
                            s_grad[wave][4 * (step % PIX) + i][lane & 15].c + 4 * (step / PIX));
                };
                if constexpr (AHEAD) load(0);
#pragma unroll
                for (int step = 0; step < STEPS; ++step) {
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (!AHEAD) load(step);
                    else if (step + 1 < STEPS) load(step + 1);
                    float sum[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int cc = 4 * (step / PIX) + c;
                        if (cc >= NC) continue;
                        sum[c] = step % PIX ? v[FB + (cc < NC ? cc : 0)] : 0.0f;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int p = 4 * (step % PIX) + i;
                            const float w = aT[p % PIX][p / PIX];
                            const float4 g4 = u[step & 1][i];
                            const float g1 = c == 0 ? g4.x : c == 1 ? g4.y : c == 2 ? g4.z : g4.w;
                            sum[c] = FINITE ? __builtin_fmaf(w, g1, sum[c]) : sum[c] + (w != 0.0f ? w * g1 : 0.0f);
                        }
                        v[FB + (cc < NC ? cc : 0)] = sum[c];
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            if (all_finite) colors(std::true_type{});
            else colors(std::false_type{});
            if (sharp) {
                // Their centre gradients again, pixel by pixel: a pixel that did
                // not blend the Gaussian (h = 0) adds nothing, whatever its
                // product with the conic.
                v[0] = v[1] = 0.0f;
                if constexpr (ABS) v[6] = v[7] = 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
#pragma unroll
                    for (int k = 0; k < PIX; ++k) {
                        const float hp = h[k][r];
                        const float px = __builtin_fmaf(con.x, dx[k], con.y * dy[r]);
                        const float py = __builtin_fmaf(con.z, dy[r], con.y * dx[k]);
                        const float tx = hp != 0.0f ? hp * px : 0.0f, ty = hp != 0.0f ? hp * py : 0.0f;
                        v[0] += tx;
                        v[1] += ty;
                        if constexpr (ABS) {
                            v[6] += __builtin_fabsf(tx);
                            v[7] += __builtin_fabsf(ty);
                        }
                    }
                }
            }
            sum_rows_packed<V>(v);
            float total[ROWS];
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                total[i] = 16 * i < V ? v[16 * i < V ? 16 * i : 0] : 0.0f;
#pragma unroll
                for (int m = 1; m < 4; ++m)
                    if (16 * i + 4 * m < V) total[i] = ((lane & 3) == m) ? v[16 * i + 4 * m < V ? 16 * i + 4 * m : 0] : total[i];
            }
            total[0] *= times_opacity ? entry_scale * con.w : is_opacity ? unscale : 1.0f;
            // Row q of register i: Gaussian q's entries from 16 i.  Gathered
            // so that a Gaussian's entries leave together.
            gather_entries(total);
            float ids[ROWS];
#pragma unroll
            for (int i = 0; i < ROWS; ++i)
                ids[i] = __int_as_float(ROWS == 4 ? __builtin_amdgcn_readlane(id, 16 * i) : id);
            if constexpr (ROWS == 2) gather_entries(ids);
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                const int gaussian = ROWS == 4 ? i : ROWS == 2 ? (q & 2) + i : q;
                // One 32 x 32 -> 64-bit multiply-add for the address (ids
                // are non-negative, strides below 2^31).
                if (dst_base && gaussian < used)
                    atomicAdd(dst_base + (uint64_t)__float_as_uint(ids[i]) * dst_step, total[i]);
            }
            used = 0;
            slots = 0;
        };
        for (int c0 = 0; c0 < cnt; c0 += 64) {
            // This wavefront's Gaussians of the next 64 that lie before its
            // pixels' last contributors, in traversal order.
            const int slot0 = c0 + lane;
            const uint32_t flags = s_mask[min(slot0, B - 1)];
            uint64_t todo = lanes(slot0 < cnt && top - 1 - slot0 < wave_last && ((flags >> wave) & 1u));
            const bool strange = (lanes((flags & kStrange) != 0) & todo) != 0;
            sharp |= (lanes((flags & kSharp) != 0) & todo) != 0;
            while (todo) {
                // One Gaussian undone from this lane's pixels: its weight and h.
                const int j = c0 + __builtin_ctzll(todo);
                todo &= todo - 1;
                const Staged<CH> g = load_staged<CH>(j, s_g);
                const int entry = top - j;  // list position, 1-based
                const float dy = g.xy.y - fy;
                const float c_dy_dy = (g.con.z * dy) * dy;
                float x[PIX];
                uint64_t in[PIX], any = 0;
#pragma unroll
                for (int k = 0; k < PIX; ++k) {
                    x[k] = blend_exponent(g.con.x, g.con.y, g.xy.x - fx[k], dy, c_dy_dy);
                    in[k] = lanes(accepts(x[k], g.limit)) & lanes(entry <= last_contributor[k]);
                    any |= in[k];
                }
                if (!any) continue;
                float G[PIX], alpha[PIX], weight[PIX], hv[PIX];
                if (strange) {
#pragma unroll
                    for (int k = 0; k < PIX; ++k) {
                        G[k] = blend_exp(-x[k]);
                        if (__int_as_float(g.entry) != 1.0f) G[k] *= kHugeScale;
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < PIX; ++k) G[k] = blend_exp_neg(x[k]);
                }
                any = 0;
#pragma unroll
                for (int k = 0; k < PIX; ++k) {
                    alpha[k] = sel_min(0.99f, g.con.w * G[k]);
                    in[k] &= lanes(alpha[k] >= 1.0f / 255.0f);
                    any |= in[k];
                }
                if (!any) continue;
#pragma unroll
                for (int k = 0; k < PIX; ++k) {
                    // Gradients only need tolerance-level agreement: one hardware
                    // reciprocal (1 - alpha >= 0.01) and fused multiply-adds.
                    const float inv = __builtin_amdgcn_rcpf(1.0f - alpha[k]);
                    // Channel slots at or beyond D hold zero features and
                    // zero upstream gradients; a last slot without a
                    // gradient is the constant channel or one of those.
                    float dot = NC < CH ? grad[k][CH - 1] : g.f[CH - 1] * grad[k][CH - 1];
#pragma unroll
                    for (int c = 0; c + 1 < CH; ++c) dot = __builtin_fmaf(g.f[c], grad[k][c], dot);
                    // A branch: the pixel's state then changes in place.
                    if (__builtin_amdgcn_inverse_ballot_w64(in[k])) {
                        T[k] = T[k] * inv;
                        S[k] = __builtin_fmaf(last_alpha[k], last_e[k], S[k]);
                        last_e[k] = dot - S[k];
                        last_alpha[k] = alpha[k];
                    }
                    weight[k] = alpha[k] * T[k];
                    hv[k] = G[k] * __builtin_fmaf(last_e[k], T[k], bg_t[k] * inv);
                }
                // Into the next slot (a wave-uniform branch).
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (used == s) {
#pragma unroll
                        for (int k = 0; k < PIX; ++k) {
                            aT[k][s] = select0(in[k], weight[k]);
                            h[k][s] = select0(in[k], hv[k]);
                        }
                    }
                slots |= (uint32_t)j << (8 * used);
                if (++used == 4) finish();
            }
        }
        if (used) {
            // The slots past the last one.
#pragma unroll
            for (int s = 1; s < 4; ++s)
                if (used <= s) {
#pragma unroll
                    for (int k = 0; k < PIX; ++k) aT[k][s] = h[k][s] = 0.0f;
                }
            finish();
        }
    }
}

// The backward of wider vectors, one Gaussian at a time: every lane
// accumulates its pixels' contributions to the current Gaussian and the
// wavefront sums all entries together (wave_sum_rows).
//
// GEOM: the geometry launch (window 0, c0 = 0): centre, conic and opacity
// gradients (+ absolute centre gradients with ABS) and the window's feature
// gradients; channels from CH on, if any, enter the alpha gradient through
// rest_dot.  !GEOM: a further window [c0, c0 + CH), feature gradients only.
template <int CH, bool ABS, int PIX, bool GEOM>
__global__ __launch_bounds__(kTilePixels / PIX) __attribute__((amdgpu_waves_per_eu(1))) void render_bwd_kernel(gs3d_render_bwd_args b, int c0) {
    constexpr int NT = kTilePixels / PIX;
    constexpr int B = Batch<CH>::size;
    // Gradient entries per Gaussian: [centre xy, conic abc, opacity, |centre| xy]
    // for the geometry launch, then the window's channels; one wavefront sum
    // covers at most 64.
    constexpr int FB = GEOM ? (ABS ? 8 : 6) : 0;
    constexpr int NV = FB + CH;
    static_assert(NV <= 64, "one wavefront sum holds at most 64 gradient entries");
    constexpr int R = (NV + 3) / 4;
    __shared__ StagedRec<CH> s_g[B];
    __shared__ uint32_t s_mask[B];
    __shared__ int32_t s_id[B];
    __shared__ int s_max_last;
    const gs3d_render_args& a = b.fwd;
    const TileInfo t = tile_info(a);
    const int D = a.feat_channels + a.extra_channels + (a.one_tail ? 1 : 0);
    const int Dg = D - (a.one_tail ? 1 : 0);
    static_assert(!GEOM || CH == kGeomWindow, "narrower vectors run the grouped backward");
    const bool rest = GEOM && D > CH;  // channels beyond the window; wave-uniform
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    // Per pixel: S = sum_c accum_c * grad_c, the colour accumulated behind
    // the current Gaussian dotted with the upstream gradient.  With
    // dot = sum_c f_c * grad_c the alpha gradient sum_c (f_c - accum_c) grad_c
    // (gs3d/render.py:300-312) is E = dot - S, and
    // accum_c = la last_c + (1 - la) accum_c becomes S = S + la E_last with
    // la and E_last those of the last accepted Gaussian: no per-channel state
    // besides grad.  bg_t = -T_final * sum_c bg_c grad_c is the background
    // term, divided by the transmittance factors as they are undone.
    float fx[PIX], fy[PIX], T[PIX], bg_t[PIX], last_alpha[PIX], S[PIX], last_e[PIX];
    float grad[PIX][CH];
    int last_contributor[PIX];
    bool inside[PIX];
    if (threadIdx.x == 0) s_max_last = 0;
    const float* bg = a.background ? a.background + t.view * a.background_view_stride : nullptr;
    int my_max = 0;
    // Per-pixel inputs: every load first, from the pixel clamped into the
    // image (the branches below depend only on the channel, so all lanes
    // load together), then the pixels outside the image are cleared.  A load
    // under a per-lane condition would be a branch that waits for its data.
    const int F = a.feat_channels, E = a.extra_channels;
    int64_t pix[PIX];
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        int lx, ly;
        pixel_of<PIX>(threadIdx.x, k, lx, ly);
        const int x = t.x0 + lx, y = t.y0 + ly;
        fx[k] = (float)x;
        fy[k] = (float)y;
        inside[k] = x < a.width && y < a.height;
        pix[k] = ((int64_t)t.view * a.height + min(y, a.height - 1)) * a.width + min(x, a.width - 1);
        T[k] = a.final_t[pix[k]];
        last_contributor[k] = a.contributors[pix[k]];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            // The channel's source (wave-uniform selects, no branch); channels
            // without one read final_t and take 0.
            const int gc = c0 + c;
            const float* src = gc < F ? b.upstream : gc < F + E ? b.upstream_extra : b.upstream_alpha;
            const int64_t stride = gc < F ? b.upstream_stride
                                          : gc < F + E ? b.upstream_extra_stride : b.upstream_alpha_stride;
            const int off = gc < F ? gc : gc < F + E ? gc - F : 0;
            const bool has = gc < D && src != nullptr;
            const float u = has ? src[pix[k] * stride + off] : a.final_t[pix[k]];
            grad[k][c] = has ? u : 0.0f;
        }
    }
#pragma unroll
    for (int k = 0; k < PIX; ++k) {
        bg_t[k] = last_alpha[k] = S[k] = last_e[k] = 0.0f;
        if (!inside[k]) {
            T[k] = 0.0f;
            last_contributor[k] = 0;
#pragma unroll
            for (int c = 0; c < CH; ++c) grad[k][c] = 0.0f;
            continue;
        }
        if (GEOM) {
            float bg_grad = 0.0f;
            if (bg) {
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    const int gc = c0 + c;
                    bg_grad += (gc < D && gc < F ? bg[gc] : 0.0f) * grad[k][c];
                }
                // Background channels beyond the window.
                if (b.upstream)
                    for (int gc = CH; gc < F; ++gc) bg_grad += bg[gc] * b.upstream[pix[k] * b.upstream_stride + gc];
            }
            bg_t[k] = -T[k] * bg_grad;
        }
        my_max = max(my_max, last_contributor[k]);
    }
    block_barrier();
    if (my_max > 0) atomicMax(&s_max_last, my_max);
    block_barrier();
    const int max_last = min(s_max_last, t.last - t.first);
    // Gradient entry this lane adds after the wavefront sums (see
    // wave_sum_rows): entry k of Gaussian g lives at dst_base + g * dst_step.
    float* dst_base = nullptr;
    uint32_t dst_step = 0;  // row strides below 2^31 (checked on the host)
    float dst_scale = 1.0f;
    {
        const int k = wave_sum_rows_value(lane);
        if (GEOM) {
            if (k < 2 || k == 3) dst_scale = -1.0f;
            if (k == 2 || k == 4) dst_scale = -0.5f;
        }
        const int64_t row0 = (int64_t)t.view * a.n;
        if ((lane & 15) >= R || k >= NV) {
        } else if (GEOM && k < 2) {
            dst_base = b.grad_centers + row0 * b.grad_centers_stride + k;
            dst_step = b.grad_centers_stride;
        } else if (GEOM && k < 6) {
            dst_base = b.grad_conics + row0 * b.grad_conics_stride + (k - 2);
            dst_step = b.grad_conics_stride;
        } else if (GEOM && ABS && k < 8) {
            dst_base = b.abs_centers + row0 * b.abs_stride + (k - 6);
            dst_step = b.abs_stride;
        } else {
            const int c = c0 + k - FB;
            if (c < a.feat_channels) {
                if (b.grad_features) {
                    dst_base = b.grad_features + t.view * b.grad_feat_view_stride + c;
                    dst_step = b.grad_feat_stride;
                }
            } else if (c < Dg && b.grad_extra) {
                dst_base = b.grad_extra + t.view * b.grad_extra_view_stride + (c - a.feat_channels);
                dst_step = b.grad_extra_stride;
            }
        }
    }
    // Largest last contributor among this wavefront's pixels (wave-uniform).
    const int lane_last = my_max;
    int wave_last = my_max;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) wave_last = max(wave_last, __shfl_xor(wave_last, d, 64));
    // As in the forward: one staged Gaussian per thread and batch, its index
    // for the next batch loaded while the current one is traversed.
    static_assert(B <= NT, "one staged Gaussian per thread and batch");
    int32_t next_id = max_last > 0 ? a.ids[t.first + max(max_last - 1 - (int)threadIdx.x, 0)] : 0;
    for (int top = max_last; top > 0; top -= B) {
        block_barrier();
        if (threadIdx.x < B) {
            const int e = threadIdx.x;
            const int p = top - 1 - e;
            const int32_t g = next_id;
            if (p >= 0) {
                s_id[e] = g;
                // Tile origin laundered (see stage_gaussian).
                stage_gaussian<CH, PIX, true>(a, t, g, e, p + 1, c0, s_g, s_mask);
            }
            if (top > B) next_id = a.ids[t.first + max(p - B, 0)];
        }
        block_barrier();
        const int cnt = min(B, top);
        for (int c0b = 0; c0b < cnt; c0b += 64) {
          // This wavefront's Gaussians of the next 64 that lie before its
          // pixels' last contributors, in traversal order.
          const int e = c0b + lane;
          uint64_t todo = __ballot(e < cnt && top - 1 - e < wave_last && ((s_mask[min(e, B - 1)] >> wave) & 1u));
          while (todo) {
            const int j = c0b + __builtin_ctzll(todo);
            todo &= todo - 1;
            const int pos = top - 1 - j;
            // Pixels outside the image have last contributor 0.
            if (__ballot(pos < lane_last) == 0) continue;
            const float2 xy = s_g[j].xy;
            const float4 con = s_g[j].con;
            const float limit = s_g[j].limit;
            const float* f = s_g[j].f;
            // Accumulators start from an opaque zero: a literal zero would be
            // folded into each accumulator's first FMA, and every path that
            // skips a pixel would then re-materialise the zeros.  vals holds,
            // in gradient-entry order, sum w (a dx + b dy), sum w (c dy + b dx),
            // sum w dx dx, sum w dx dy, sum w dy dy with w = o G dL/dalpha,
            // then sum G dL/dalpha, the absolute centre terms and the feature
            // terms; the constant factors (-1, -1/2) are applied per lane
            // after the wavefront sum.
            float vals[NV];
#pragma unroll
            for (int i = 0; i + 1 < NV; i += 2) opaque_zero2(vals[i], vals[i + 1]);
            if constexpr (NV % 2) vals[NV - 1] = opaque_zero();
            bool accepted = false;
#pragma unroll
            for (int k = 0; k < PIX; ++k) {
                if (!(pos < last_contributor[k])) continue;
                const float dx = xy.x - fx[k], dy = xy.y - fy[k];
                const float power = blend_power(con.x, con.y, con.z, dx, dy);
                if (!(power <= 0.0f) || !(power >= -limit)) continue;
                const float G = blend_exp(power);
                const float og = con.w * G;
                const float alpha = sel_min(0.99f, og);
                if (!(alpha >= 1.0f / 255.0f)) continue;
                accepted = true;
                // Gradients only need tolerance-level agreement: one hardware
                // reciprocal (1 - alpha >= 0.01) and fused multiply-adds.
                const float inv = __builtin_amdgcn_rcpf(1.0f - alpha);
                T[k] = T[k] * inv;
                const float aT = alpha * T[k];
                // Every compiled channel slot is processed: slots at or beyond
                // D hold zero features and zero upstream gradients (no
                // contribution), and the constant alpha channel's entry has no
                // destination, so no per-channel branch is needed.
#pragma unroll
                for (int c = 0; c < CH; ++c) vals[FB + c] = __builtin_fmaf(aT, grad[k][c], vals[FB + c]);
                if constexpr (GEOM) {
                    float dot = 0.0f;
#pragma unroll
                    for (int c = 0; c < CH; ++c) dot = __builtin_fmaf(f[c], grad[k][c], dot);
                    if (rest) dot += rest_dot(b, t.view, s_id[j], fx[k], fy[k], CH);
                    const float la = last_alpha[k];
                    S[k] = __builtin_fmaf(la, last_e[k], S[k]);
                    last_e[k] = dot - S[k];
                    const float grad_alpha = __builtin_fmaf(last_e[k], T[k], bg_t[k] * inv);
                    last_alpha[k] = alpha;
                    // dL/dG = o dL/dalpha; the centre gradient is
                    // -w (a dx + b dy, c dy + b dx) and the conic gradient
                    // -w (dx dx / 2, dx dy, dy dy / 2).
                    const float w = og * grad_alpha;
                    const float ux = __builtin_fmaf(con.x, dx, con.y * dy);
                    const float uy = __builtin_fmaf(con.z, dy, con.y * dx);
                    if (ABS) {
                        const float cx = w * ux, cy = w * uy;
                        vals[0] += cx;
                        vals[1] += cy;
                        vals[6] += __builtin_fabsf(cx);
                        vals[7] += __builtin_fabsf(cy);
                    } else {
                        vals[0] = __builtin_fmaf(w, ux, vals[0]);
                        vals[1] = __builtin_fmaf(w, uy, vals[1]);
                    }
                    const float wx = w * dx, wy = w * dy;
                    vals[2] = __builtin_fmaf(wx, dx, vals[2]);
                    vals[3] = __builtin_fmaf(wx, dy, vals[3]);
                    vals[4] = __builtin_fmaf(wy, dy, vals[4]);
                    vals[5] = __builtin_fmaf(G, grad_alpha, vals[5]);
                }
            }
            if (__ballot(accepted) == 0) continue;
            // Wavefront sums of all gradient entries at once; one atomic
            // instruction, each active lane adding one entry.
            float sums[R];
            wave_sum_rows<NV>(vals, sums);
            // Finish the sums on every lane, ahead of the branch: the last
            // row step then stays one DPP add.
#pragma unroll
            for (int r = 0; r < R; ++r) asm volatile("" : "+v"(sums[r]));
            if (dst_base) {
                const int slot = lane & 15;
                float v = sums[0];
#pragma unroll
                for (int r = 1; r < R; ++r) v = (slot == r) ? sums[r] : v;
                // One 32 x 32 -> 64-bit multiply-add for the address (ids
                // are non-negative, strides below 2^31): 1829 against 1865
                // us for the 3M-Gaussian blend VJP.
                atomicAdd(dst_base + (uint64_t)(uint32_t)s_id[j] * dst_step, v * dst_scale);
            }
          }
        }
    }
}

// Grids of fewer tiles than this (all views) run the narrow-channel blends
// at one pixel per lane: four wavefronts per tile instead of two, so that a
// small frame still spreads over the SIMDs.  Each tile's list is walked
// serially; at two pixels per lane a few thousand tiles make little more than
// one full set of resident wavefronts (6 per SIMD, 6144 on the chip), and the
// longest lists set the time.  Forward at one against two pixels per lane:
// 300K Gaussians at 1152x960 (4320 tiles) 115 against 132 us, at 1600x1200
// (7500 tiles) 152 against 152.
//
// The backward adds a Gaussian's gradients once per wavefront, so there one
// pixel per lane means twice the atomics, and these are the bound where large
// Gaussians are many.  From kSmallGridBwd tiles it is taken only if the
// frame's lists are known to hold few entries per Gaussian (and view).  One
// against two pixels per lane, 4 channels: 1152x960 with 13 entries per Gaussian
// 196 against 222 us, with 38 147 against 166, with 103 420 against 253;
// 1440x1040 with 19 220 against 254, with 52 171 against 168, with 146 567
// against 315.
#ifndef GS3D_SMALL_GRID
#define GS3D_SMALL_GRID 6144
#endif
constexpr unsigned kSmallGrid = GS3D_SMALL_GRID, kSmallGridBwd = 4096;
constexpr int64_t kEntriesPerGaussian = 40;

// ids_count: the lists' entries in all, or negative if not known.
inline bool small_grid_bwd(const gs3d_render_args& a, unsigned blocks, int64_t ids_count) {
    if (blocks < kSmallGridBwd) return true;
    return blocks < kSmallGrid && ids_count >= 0 && ids_count <= kEntriesPerGaussian * a.n * a.views;
}

// Workgroups of a redo launch (gs3d_render_args.redo_pass).
constexpr unsigned kRedoGrid = 512;

template <int CH, int PIX>
int launch_fwd_pix(const gs3d_render_args& a, const gs3d_render_stats_args* st, unsigned long long* counts,
                   unsigned blocks, int c0, hipStream_t s) {
    const dim3 grid(blocks), block(kTilePixels / PIX);
    if (st) {
        const uint32_t kinds = st->sum_mask;
        if (st->requests <= 1) {
            if (kinds & 1u)
                hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, 1, 1>), grid, block, 0, s, a, *st, c0, nullptr);
            else
                hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, 1, 0>), grid, block, 0, s, a, *st, c0, nullptr);
        } else if (st->requests <= 2) {
            switch (kinds & 3u) {
                case 0: hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, 2, 0>), grid, block, 0, s, a, *st, c0, nullptr); break;
                case 1: hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, 2, 1>), grid, block, 0, s, a, *st, c0, nullptr); break;
                case 2: hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, 2, 2>), grid, block, 0, s, a, *st, c0, nullptr); break;
                default: hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, 2, 3>), grid, block, 0, s, a, *st, c0, nullptr); break;
            }
        } else if (st->requests <= 4)
            hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, 4>), grid, block, 0, s, a, *st, c0, nullptr);
        else
            hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 1, GS3D_MAX_STATISTICS>), grid, block, 0, s, a, *st, c0,
                               nullptr);
        return launch_status("gs3d_render_fwd_stats");
    }
    const gs3d_render_stats_args none = {};
    if (a.redo_pass) {
        // The workgroups walk the listed tiles (usually none).
        hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 0, 1, -1, 2>), dim3(min(blocks, kRedoGrid)), block, 0, s, a,
                           none, c0, nullptr);
        return launch_status("gs3d_render_fwd");
    }
    if (a.caps || a.stop_out) {
        hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 0, 1, -1, 1>), grid, block, 0, s, a, none, c0, nullptr);
        return launch_status("gs3d_render_fwd");
    }
    if (counts) {
        hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 2>), grid, block, 0, s, a, none, c0, counts);
        return launch_status("gs3d_render_pair_counts");
    }
    hipLaunchKernelGGL((render_fwd_kernel<CH, PIX, 0>), grid, block, 0, s, a, none, c0, nullptr);
    return launch_status("gs3d_render_fwd");
}

template <int CH>
int launch_fwd(const gs3d_render_args& a, const gs3d_render_stats_args* st, unsigned long long* counts,
               unsigned blocks, int c0, hipStream_t s) {
    constexpr int PIX = PixFor<CH, false>::value;
    if constexpr (PIX > 1) {
        if (blocks < kSmallGrid) return launch_fwd_pix<CH, 1>(a, st, counts, blocks, c0, s);
    }
    return launch_fwd_pix<CH, PIX>(a, st, counts, blocks, c0, s);
}

// One forward window of `width` channels starting at c0.  Every slot of a
// kernel's width costs a multiply-add per accepted pixel, 4 bytes of LDS per
// staged Gaussian and registers, so the lines lie where a wider kernel holds
// fewer wavefronts per SIMD: up to 20 slots four (110 registers forward, 128
// backward), 36 three (168), beyond two.  44 is the line of the grouped
// backward (59 of 64 KB LDS, 225 registers); the kernels of 64 and 56 slots are
// what is left.  17 to 20 channels in 36 slots against 20, and 37 to 44 in 64
// and 56 against 44, forward and backward in us:
//   300K Gaussians 1280x960   17: 264 + 515, 207 + 320     20: 282 + 516, 230 + 330
//                             37: 503 + 1255, 434 + 788    44: 525 + 1282, 465 + 826
//   10K Gaussians 256x256     17: 105 + 234, 88 + 159      44: 145 + 379, 123 + 257
//   100K, some very large,    17: 414 + 976, 348 + 856     44: 794 + 2143, 716 + 2120
//   1920x1080
// What still rides in wider slots: 21 channels 278 + 518, 45 channels 525 + 1290
// at 1280x960.
inline int launch_fwd_window(const gs3d_render_args& a, const gs3d_render_stats_args* st, unsigned long long* counts,
                             unsigned blocks, int c0, int width, hipStream_t s) {
    if (width <= 4) return launch_fwd<4>(a, st, counts, blocks, c0, s);
    if (width <= 8) return launch_fwd<8>(a, st, counts, blocks, c0, s);
    if (width <= 16) return launch_fwd<16>(a, st, counts, blocks, c0, s);
    if (width <= 20) return launch_fwd<20>(a, st, counts, blocks, c0, s);
    if (width <= 36) return launch_fwd<36>(a, st, counts, blocks, c0, s);
    if (width <= 44) return launch_fwd<44>(a, st, counts, blocks, c0, s);
    return launch_fwd<kWindow>(a, st, counts, blocks, c0, s);
}

template <int CH, int NC, int PIX>
int launch_bwd_rows(const gs3d_render_bwd_args& b, unsigned blocks, hipStream_t s) {
    const dim3 grid(blocks), block(kTilePixels / PIX);
    if (b.abs_centers)
        hipLaunchKernelGGL((render_bwd_rows_kernel<CH, NC, true, PIX>), grid, block, 0, s, b);
    else
        hipLaunchKernelGGL((render_bwd_rows_kernel<CH, NC, false, PIX>), grid, block, 0, s, b);
    return launch_status("gs3d_render_bwd");
}

// All gradients of a vector of at most 44 channels.
template <int CH>
int launch_bwd_rows(const gs3d_render_bwd_args& b, unsigned blocks, bool small, int gradient_channels, hipStream_t s) {
    constexpr int PIX = PixFor<CH, true>::value;
    auto run = [&](auto nc) {
        constexpr int NC = decltype(nc)::value;
        if constexpr (PIX > 1) {
            if (small) return launch_bwd_rows<CH, NC, 1>(b, blocks, s);
        }
        return launch_bwd_rows<CH, NC, PIX>(b, blocks, s);
    };
    return gradient_channels < CH ? run(std::integral_constant<int, CH - 1>{}) : run(std::integral_constant<int, CH>{});
}

template <int CH, bool GEOM, int PIX = PixFor<CH, true>::value>
int launch_bwd(const gs3d_render_bwd_args& b, unsigned blocks, bool small, int c0, hipStream_t s) {
    if constexpr (PIX > 1) {
        if (small) return launch_bwd<CH, GEOM, 1>(b, blocks, small, c0, s);
    }
    const dim3 grid(blocks), block(kTilePixels / PIX);
    if constexpr (GEOM) {
        if (b.abs_centers) {
            hipLaunchKernelGGL((render_bwd_kernel<CH, true, PIX, true>), grid, block, 0, s, b, c0);
            return launch_status("gs3d_render_bwd");
        }
    }
    hipLaunchKernelGGL((render_bwd_kernel<CH, false, PIX, GEOM>), grid, block, 0, s, b, c0);
    return launch_status("gs3d_render_bwd");
}

inline int check_render_args(const gs3d_render_args& a) {
    if (a.width <= 0 || a.height <= 0 || a.views < 0 || a.n < 0) return GS3D_ERR_ARGUMENT;
    if (a.feat_channels < 0 || a.extra_channels < 0 || (a.extra_channels > 0 && !a.extra)) return GS3D_ERR_ARGUMENT;
    if (a.views > 0 && !a.ranges) return GS3D_ERR_ARGUMENT;
    if (a.views > 0 && a.n > 0 && (!a.centers || !a.conics || (a.feat_channels > 0 && !a.features)))
        return GS3D_ERR_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(a.centers) & 7) || (reinterpret_cast<uintptr_t>(a.conics) & 15))
        return GS3D_ERR_ARGUMENT;
    const int D = a.feat_channels + a.extra_channels + (a.one_tail ? 1 : 0);
    if (D <= 0) return GS3D_ERR_ARGUMENT;
    return GS3D_OK;
}

inline unsigned render_blocks(const gs3d_render_args& a) {
    const int64_t per_view = (int64_t)((a.width + kTile - 1) / kTile) * ((a.height + kTile - 1) / kTile);
    return (unsigned)(per_view * a.views);
}

}  // namespace gs3d

namespace gs3d {

int render_fwd(const gs3d_render_args* args, const gs3d_render_stats_args* st, unsigned long long* counts,
               void* stream) {
    if (!args) return GS3D_ERR_ARGUMENT;
    const gs3d_render_args& a = *args;
    int status = check_render_args(a);
    if (status != GS3D_OK) return status;
    if (a.zero_count < 0 || (a.zero_count > 0 && (!a.zero_out || (reinterpret_cast<uintptr_t>(a.zero_out) & 15))))
        return GS3D_ERR_ARGUMENT;
    // Capped lists: overflowing tiles must be reported; a redo launch skips
    // tiles, so it cannot clear a buffer, count pairs or total statistics
    // (nor can a capped launch, whose redone tiles would total twice).
    if (a.caps && !a.redo_pass && (!a.redo || !a.redo_list)) return GS3D_ERR_ARGUMENT;
    if (a.redo_pass && (!a.redo_list || a.zero_out)) return GS3D_ERR_ARGUMENT;
    if ((a.caps || a.redo_pass || a.stop_out) && (st || counts)) return GS3D_ERR_ARGUMENT;
    if (a.views == 0) return GS3D_OK;
    if ((a.feat_channels > 0 && !a.image) || (a.extra_channels > 0 && !a.image_extra) ||
        (a.one_tail && !a.image_alpha) || !a.final_t || !a.contributors)
        return GS3D_ERR_ARGUMENT;
    const int D = a.feat_channels + a.extra_channels + (a.one_tail ? 1 : 0);
    const unsigned blocks = render_blocks(a);
    hipStream_t s = as_stream(stream);
    // Windows of up to 64 channels; the statistics ride on window 0.
    for (int c0 = 0; c0 < D; c0 += kWindow) {
        status = launch_fwd_window(a, c0 == 0 ? st : nullptr, c0 == 0 ? counts : nullptr, blocks, c0,
                                   min(kWindow, D - c0), s);
        if (status != GS3D_OK) return status;
    }
    return GS3D_OK;
}

}  // namespace gs3d

extern "C" int gs3d_render_fwd(const gs3d_render_args* args, void* stream) {
    return gs3d::render_fwd(args, nullptr, nullptr, stream);
}

extern "C" int gs3d_render_pair_counts(const gs3d_render_args* args, uint64_t* counts, void* stream) {
    if (!counts || (reinterpret_cast<uintptr_t>(counts) & 7)) return GS3D_ERR_ARGUMENT;
    return gs3d::render_fwd(args, nullptr, reinterpret_cast<unsigned long long*>(counts), stream);
}

extern "C" int gs3d_render_fwd_stats(const gs3d_render_args* args, const gs3d_render_stats_args* stats,
                                     void* stream) {
    if (!args || !stats) return GS3D_ERR_ARGUMENT;
    const gs3d_render_stats_args& st = *stats;
    if (st.requests < 1 || st.requests > GS3D_MAX_STATISTICS) return GS3D_ERR_ARGUMENT;
    const uint32_t used = (1u << st.requests) - 1u;
    if (st.sum_mask & ~used) return GS3D_ERR_ARGUMENT;
    const bool any_sum = st.sum_mask != 0, any_count = st.sum_mask != used;
    if (!st.pixel_values || (any_sum && !st.sums) || (any_count && !st.counts)) return GS3D_ERR_ARGUMENT;
    if (st.pixel_view_stride < 0 || st.counts_view_stride < 0 || st.sums_view_stride < 0) return GS3D_ERR_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(st.pixel_values) | reinterpret_cast<uintptr_t>(st.counts) |
         reinterpret_cast<uintptr_t>(st.sums)) & 3)
        return GS3D_ERR_ARGUMENT;
    return gs3d::render_fwd(args, stats, nullptr, stream);
}

extern "C" int gs3d_render_bwd(const gs3d_render_bwd_args* args, void* stream) {
    return gs3d_render_bwd_lists(args, -1, stream);
}

extern "C" int gs3d_render_bwd_lists(const gs3d_render_bwd_args* args, int64_t ids_count, void* stream) {
    if (!args) return GS3D_ERR_ARGUMENT;
    const gs3d_render_bwd_args& b = *args;
    const gs3d_render_args& a = b.fwd;
    int status = gs3d::check_render_args(a);
    if (status != GS3D_OK) return status;
    if (a.views == 0) return GS3D_OK;
    if (!a.final_t || !a.contributors || !b.grad_centers || !b.grad_conics) return GS3D_ERR_ARGUMENT;
    if (b.grad_centers_stride < 2 || b.grad_conics_stride < 4 || (b.abs_centers && b.abs_stride < 2))
        return GS3D_ERR_ARGUMENT;
    // Gradient row strides feed 32-bit multipliers in the kernel.
    for (int64_t stride : {b.grad_centers_stride, b.grad_conics_stride, b.abs_stride, b.grad_feat_stride,
                           b.grad_extra_stride})
        if (stride < 0 || stride > INT32_MAX) return GS3D_ERR_ARGUMENT;
    if ((b.upstream && b.upstream_stride < a.feat_channels) ||
        (b.upstream_extra && b.upstream_extra_stride < a.extra_channels) ||
        (b.upstream_alpha && b.upstream_alpha_stride < 1))
        return GS3D_ERR_ARGUMENT;
    using namespace gs3d;
    const int D = a.feat_channels + a.extra_channels + (a.one_tail ? 1 : 0);
    const int Dg = D - (a.one_tail ? 1 : 0);
    const unsigned blocks = render_blocks(a);
    const bool small = small_grid_bwd(a, blocks, ids_count);
    hipStream_t s = as_stream(stream);
    // Geometry launch over the first window (channels beyond it enter its
    // alpha gradient from global memory), then the feature gradients of the
    // further windows that hold channels with a destination.
    if (D <= 4) status = launch_bwd_rows<4>(b, blocks, small, Dg, s);
    else if (D <= 8) status = launch_bwd_rows<8>(b, blocks, small, Dg, s);
    else if (D <= 16) status = launch_bwd_rows<16>(b, blocks, small, Dg, s);
    else if (D <= 20) status = launch_bwd_rows<20>(b, blocks, small, Dg, s);
    else if (D <= 36) status = launch_bwd_rows<36>(b, blocks, small, Dg, s);
    else if (D <= 44) status = launch_bwd_rows<44>(b, blocks, small, Dg, s);
    else status = launch_bwd<kGeomWindow, true>(b, blocks, small, 0, s);
    if (status != GS3D_OK || (!b.grad_features && !b.grad_extra)) return status;
    for (int c0 = kGeomWindow; c0 < Dg; c0 += kWindow) {
        const int width = min(kWindow, D - c0);
        if (width <= 4) status = launch_bwd<4, false>(b, blocks, small, c0, s);
        else if (width <= 8) status = launch_bwd<8, false>(b, blocks, small, c0, s);
        else if (width <= 16) status = launch_bwd<16, false>(b, blocks, small, c0, s);
        else if (width <= 36) status = launch_bwd<36, false>(b, blocks, small, c0, s);
        else status = launch_bwd<kWindow, false>(b, blocks, small, c0, s);
        if (status != GS3D_OK) return status;
    }
    return GS3D_OK;
}
