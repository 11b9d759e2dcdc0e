// Pieces shared by the inference, training-forward, max-weight and backward blend kernels.
#pragma once

#include <type_traits>

#include "common.h"

namespace htgs {

// ---------------------------------------------------------------------------------------------
// tile-relative form.  With px = px0 - dx VPMT4, py = py0 - dy VPMT4, where px0 / py0 are
// the reference's planes (R/include/hybrid_blend/kernels/inference.cuh:137-141) through the tile centre and
// (dx, dy) is the pixel's offset from it,
//     d = cross(px.n, py.n)     = A  + dy B  + dx C
//     m = px.w py.n - px.n py.w = Am + dy Bm + dx Cm            (the dx dy terms cancel)
// so |m|^2, |d|^2 and MT3.n . cross(d, m) are quadratics in (dx, dy).  The lane that stages an instance
// computes the 18 coefficients once; every pixel then needs 5 fused multiply-adds per quadratic.
// LDS layout per instance, coefficient order (1, dx, dy, dx^2, dx dy, dy^2):
//     q[0] = n0 nx ny nxx   q[1] = nxy nyy d0 dx   q[2] = dy dxx dxy dyy      (n = |m|^2 / cut-off)
//     q[3] = z0 zx zy zxx   q[4] = zxy zyy MT3.w opacity   q[5] = r g b (primitive index bits)
// ---------------------------------------------------------------------------------------------
template <int N>
struct TileStage {
    float4 q[6][N];
};

__device__ __forceinline__ void cross3(const float *a, const float *b, float *o)
{
    o[0] = __builtin_fmaf(a[1], b[2], -(a[2] * b[1]));
    o[1] = __builtin_fmaf(a[2], b[0], -(a[0] * b[2]));
    o[2] = __builtin_fmaf(a[0], b[1], -(a[1] * b[0]));
}
__device__ __forceinline__ float dotf(const float *a, const float *b)
{
    return __builtin_fmaf(a[2], b[2], __builtin_fmaf(a[1], b[1], a[0] * b[0]));
}

// the six vectors of the tile-relative form and what they are built from
struct TileGeometry {
    float a[3], aw, b[3], bw, v[3], vw;        // px0 = (a, aw), py0 = (b, bw), VPMT4 = (v, vw)
    float A[3], B[3], C[3], Am[3], Bm[3], Cm[3];
};
__device__ __forceinline__ void tile_geometry(const float4 &r1, const float4 &r2, const float4 &r4, float cx, float cy, TileGeometry &g)
{
    const float V1[4] = { r1.x, r1.y, r1.z, r1.w }, V2[4] = { r2.x, r2.y, r2.z, r2.w }, V4[4] = { r4.x, r4.y, r4.z, r4.w };
    float px0[4], py0[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        px0[k] = __builtin_fmaf(-V4[k], cx, V1[k]);
        py0[k] = __builtin_fmaf(-V4[k], cy, V2[k]);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) { g.a[k] = px0[k]; g.b[k] = py0[k]; g.v[k] = V4[k]; }
    g.aw = px0[3]; g.bw = py0[3]; g.vw = V4[3];
    cross3(px0, py0, g.A);
    cross3(V4, px0, g.B);
    cross3(py0, V4, g.C);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        g.Am[k] = __builtin_fmaf(px0[3], py0[k], -(px0[k] * py0[3]));
        g.Bm[k] = __builtin_fmaf(px0[k], V4[3], -(px0[3] * V4[k]));
        g.Cm[k] = __builtin_fmaf(V4[k], py0[3], -(V4[3] * py0[k]));
    }
}
// coefficients (1, dx, dy, dx^2, dx dy, dy^2) of |m|^2 / cut-off and of |d|^2
template <int MODE>
__device__ __forceinline__ void tile_quadratics(const TileGeometry &g, float (&n)[6], float (&d)[6])
{
    constexpr float kc = ModeCfg<MODE>::cutoff_rcp;
    n[0] = dotf(g.Am, g.Am) * kc; n[1] = (2.0f * dotf(g.Am, g.Cm)) * kc; n[2] = (2.0f * dotf(g.Am, g.Bm)) * kc;
    n[3] = dotf(g.Cm, g.Cm) * kc; n[4] = (2.0f * dotf(g.Bm, g.Cm)) * kc; n[5] = dotf(g.Bm, g.Bm) * kc;
    d[0] = dotf(g.A, g.A); d[1] = 2.0f * dotf(g.A, g.C); d[2] = 2.0f * dotf(g.A, g.B);
    d[3] = dotf(g.C, g.C); d[4] = 2.0f * dotf(g.B, g.C); d[5] = dotf(g.B, g.B);
}

// True when no pixel of the tile can pass both the cut-off and the alpha test of an instance, given the
// coefficients of |m|^2 / cut-off (n) and |d|^2 (d) and the opacity.  The cut-off is 2 ln(1 / min_alpha) in every
// mode, so opacity * exp(-rho^2 / 2) >= min_alpha is n / d <= 1 + log2(opacity) / log2(1 / min_alpha) =: r, and both
// tests together are  Q = n - min(r, 1) d <= 0.  Q is a quadratic of the pixel offset; per pixel row its least value
// over the row's pixels is at the pixel next to the vertex (or at a row end), so one evaluation per row gives the
// least Q over the tile.  The margin (1e-5 of the sum of the magnitudes of all terms, with r raised by 1e-5) is an
// order of magnitude above the rounding of the per-pixel evaluation, of 2^x and of this routine; non-finite
// coefficients never report a miss.
template <int MODE>
__device__ __forceinline__ bool tile_misses(const float (&n)[6], const float (&d)[6], float opacity)
{
    constexpr int rows = ModeCfg<MODE>::tile;
    constexpr float h = 0.5f * (float)(rows - 1);
    float r = __builtin_fmaf(__builtin_amdgcn_logf(opacity), -1.0f / ModeCfg<MODE>::exp2_scale, 1.0f);
    r = r < 1.0f ? r : 1.0f;                       // (also a NaN opacity: the cut-off alone decides)
    r = r > -1.0f ? r : -1.0f;
    r += 1e-5f;
    float q[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) q[i] = __builtin_fmaf(-r, d[i], n[i]);
    const float s0 = __builtin_fabsf(n[0]) + __builtin_fabsf(d[0]);
    const float s1 = (__builtin_fabsf(n[1]) + __builtin_fabsf(d[1])) + (__builtin_fabsf(n[2]) + __builtin_fabsf(d[2]));
    const float s2 = ((__builtin_fabsf(n[3]) + __builtin_fabsf(d[3])) + (__builtin_fabsf(n[4]) + __builtin_fabsf(d[4]))) +
                     (__builtin_fabsf(n[5]) + __builtin_fabsf(d[5]));
    const float margin = 1e-5f * __builtin_fmaf(h * h, s2, __builtin_fmaf(h, s1, s0));
    const bool convex = q[3] > 0.0f;
    const float to_vertex = -0.5f * __builtin_amdgcn_rcpf(q[3]);
    float least = __FLT_MAX__;
#pragma nounroll
    for (int row = 0; row < rows; ++row) {           // (kept a loop: unrolled, the rows crowd the callers' K-buffers out of registers)
        const float y = (float)row - h;
        const float b = __builtin_fmaf(q[4], y, q[1]);
        const float c = __builtin_fmaf(y, __builtin_fmaf(q[5], y, q[2]), q[0]);
        float xv = __builtin_rintf(__builtin_fmaf(b, to_vertex, 0.5f)) - 0.5f;
        xv = __builtin_fminf(__builtin_fmaxf(xv, -h), h);
        least = __builtin_fminf(least, __builtin_fmaf(xv, __builtin_fmaf(q[3], xv, b), c));
    }
    return convex && least > margin;                 // (a quadratic that is not convex along the rows is never left out)
}

// The same bound per 4x4 quadrant of the tile: a clear bit says that no pixel of that quadrant can pass.  For an 8x8 tile bit q =
// 2 (row >= 4) + (column >= 4); for the 16x16 tile of ALPHA_BLEND_GLOBAL_ORDERING bit 4 s + q stands for quadrant q, numbered so, of the
// 8x8 sub-tile s = 2 (row >= 8) + (column >= 8).  Per pixel row the least value of Q over a quadrant's four pixels is at the
// one nearest to the vertex, so one evaluation per quadrant and row does.
// A row is some twenty instructions of every staged batch (all of it: 50 of the 1300 us of a frame of 3 M Gaussians at
// 1920x1080, HYBRID_BLEND), so: the columns are counted from half a pixel left of the centre, which makes them whole numbers and the
// nearest one the sum of the vertex and 1.5 2^23; a row's two coefficients follow from the row before by addition,
// started afresh every four rows (some 1e-6 of the sum of the magnitudes, within the margin); the minimum is taken without
// the quieting of NaNs that fminf brings (a coefficient that is not a number makes the margin one, and nothing is left out).
// Whole passes: GLOBAL_ORDERING, 3 M at 1920x1080, 787 -> 778 us, HYBRID 1312 -> 1301, OIT 334 k at 1237x821 159.2 -> 158.3.
template <int MODE>
__device__ __forceinline__ uint32_t tile_quadrant_hits(const float (&n)[6], const float (&d)[6], float opacity)
{
    constexpr int kBands = ModeCfg<MODE>::tile / 4;
    constexpr float h = 0.5f * (float)(ModeCfg<MODE>::tile - 1);
    constexpr int kUnroll = kBands == 2 ? 2 : 4;         // (all four rows of an 8x8 tile's band crowd the callers' K-buffers out of registers)
    float r = __builtin_fmaf(__builtin_amdgcn_logf(opacity), -1.0f / ModeCfg<MODE>::exp2_scale, 1.0f);
    r = r < 1.0f ? r : 1.0f;
    r = r > -1.0f ? r : -1.0f;
    r += 1e-5f;
    float q[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) q[i] = __builtin_fmaf(-r, d[i], n[i]);
    const float s0 = __builtin_fabsf(n[0]) + __builtin_fabsf(d[0]);
    const float s1 = (__builtin_fabsf(n[1]) + __builtin_fabsf(d[1])) + (__builtin_fabsf(n[2]) + __builtin_fabsf(d[2]));
    const float s2 = ((__builtin_fabsf(n[3]) + __builtin_fabsf(d[3])) + (__builtin_fabsf(n[4]) + __builtin_fabsf(d[4]))) +
                     (__builtin_fabsf(n[5]) + __builtin_fabsf(d[5]));
    const float margin = 1e-5f * __builtin_fmaf(h * h, s2, __builtin_fmaf(h, s1, s0));
    if (!(q[3] > 0.0f)) return (1u << (kBands * kBands)) - 1u;       // (not convex along the rows, or not a number: kept everywhere)
    const float to_vertex = -0.5f * __builtin_amdgcn_rcpf(q[3]);
    // about (-1/2, 0): Q = q3 u^2 + (q1 + q4 y) u + q0 + q2 y + q5 y^2 at the whole numbers u = x + 1/2
    q[0] = __builtin_fmaf(0.25f, q[3], __builtin_fmaf(-0.5f, q[1], q[0]));
    q[1] -= q[3];
    q[2] = __builtin_fmaf(-0.5f, q[4], q[2]);
    const float twice = q[5] + q[5];
    uint32_t bits = 0;
    float y = -h;
#pragma nounroll
    for (int band = 0; band < kBands; ++band) {          // four pixel rows: one row of quadrants
        float b = __builtin_fmaf(q[4], y, q[1]);
        float step = __builtin_fmaf(q[5], y, q[2]);
        float c = __builtin_fmaf(y, step, q[0]);
        step = __builtin_fmaf(q[5], y + 1.0f, step);     // c(y + 1) - c(y) = q2 + q5 (2 y + 1)
        float least[kBands];
#pragma unroll
        for (int k = 0; k < kBands; ++k) least[k] = __FLT_MAX__;
#pragma unroll kUnroll
        for (int row = 0; row < 4; ++row) {
            const float u = __builtin_fmaf(b, to_vertex, 12582912.0f) - 12582912.0f;
#pragma unroll
            for (int k = 0; k < kBands; ++k) {
                const float lo = (float)(4 * k) - h + 0.5f;
                const float uk = __builtin_amdgcn_fmed3f(u, lo, lo + 3.0f);
                const float value = __builtin_fmaf(uk, __builtin_fmaf(q[3], uk, b), c);
                asm("v_min_f32 %0, %0, %1" : "+v"(least[k]) : "v"(value));
            }
            b += q[4];
            c += step;
            step += twice;
        }
        y += 4.0f;
#pragma unroll
        for (int k = 0; k < kBands; ++k)
            if (!(least[k] > margin)) bits |= 1u << (kBands == 2 ? 2 * band + k : 4 * (2 * (band >> 1) + (k >> 1)) + 2 * (band & 1) + (k & 1));
    }
    return bits;
}

// A depth that no fragment of an instance is nearer than, as the walk computes it.  A fragment's point is u = cross(d, m) / |d|^2 of the Gaussian's
// unit space, |u| = |m| / |d| within the cut-off and within the radius at which alpha falls to the mode's least (r of the squared cut-off), and
// its depth is MT3.n u + MT3.w: no nearer than MT3.w - |MT3.n| |m| / |d|, whatever the vectors A .. Cm have been rounded to.  The walk's |m|^2, |d|^2
// and MT3.n cross(d, m) are quadratics, whose rounding is some 3e-6 at most of M^2, D^2 and |MT3.n| D M, where M = |Am| + h |Bm| + h |Cm| and D likewise
// (h: half the tile): M^2 <= 3 (n0 + h^2 (n3 + n5)) cut-offs, D^2 <= 3 (d0 + h^2 (d3 + d5)).  With km = 1e-5 of the former sum over the tile's
// least |d|^2 and kd = 1e-5 of the latter, a fragment that passes has |u| below cut-off^1/2 (((1 + kd) (r + km))^1/2 + (kd km)^1/2); the
// twentieth that is added covers kd up to 1e-3.  An instance beyond that, or with a quantity that is not a number, is not bounded.  What cancels is
// discs and needles far thinner than a pixel and a thousand times as wide: without km and kd 36 of 24 M of all shapes, evaluated in 32 bits, had a
// fragment nearer than the bound, by up to half of its depth; with them none had.  (FIRST_K 1 M at 1280x720 308.4 -> 306.5 us.)
template <int MODE>
__device__ __forceinline__ float nearest_depth(const float (&n)[6], const float (&d)[6], const float4 &mt3, float opacity)
{
    constexpr float h = 0.5f * (float)(ModeCfg<MODE>::tile - 1);
    float r = __builtin_fmaf(__builtin_amdgcn_logf(opacity), -1.0f / ModeCfg<MODE>::exp2_scale, 1.0f);
    r = r < 1.0f ? r : 1.0f;
    r = r > 0.0f ? r : 0.0f;
    const float d_least = __builtin_fmaf(-h * h, __builtin_fabsf(d[4]), __builtin_fmaf(-h, __builtin_fabsf(d[1]) + __builtin_fabsf(d[2]), d[0]));
    const float d_sum = __builtin_fmaf(h * h, d[3] + d[5], d[0]), n_sum = __builtin_fmaf(h * h, n[3] + n[5], n[0]);
    const float within = (r + 1e-4f) + 1e-5f * (n_sum * __builtin_amdgcn_rcpf(d_least));
    const float reach = 1.05f * __builtin_amdgcn_sqrtf(ModeCfg<MODE>::cutoff_sq * within * __builtin_fmaf(mt3.z, mt3.z, __builtin_fmaf(mt3.y, mt3.y, mt3.x * mt3.x)));
    const float depth = mt3.w - __builtin_fmaf(1e-5f, __builtin_fabsf(mt3.w), reach);
    return d_sum < 100.0f * d_least ? depth : -__FLT_MAX__;
}

// Stages instance `fetch` of the sorted list in slot `slot` (the same arithmetic as tile_geometry / tile_quadratics,
// written out so that every row is stored as soon as it is complete: the kernels that call this hold a K-buffer in
// registers).  Returns whether the slot holds an instance that can reach a pixel of the tile: always true for a
// loaded slot unless CULL asks for tile_misses -- for walks that apply the cut-off and the alpha threshold
// (kCullAlpha), or the cut-off alone (kCullCutoff: the test with opacity 1).  What that leaves out contributes to
// no pixel, so a walk over the hits alone gives the results of the full walk bit for bit.
// the pixel's offset from the tile centre (exact)
struct PixelTerms {
    float X, Y;
};
__device__ __forceinline__ PixelTerms pixel_terms(uint32_t local_x, uint32_t local_y, int tile)
{
    PixelTerms p;
    p.X = (float)local_x - 0.5f * (float)(tile - 1);
    p.Y = (float)local_y - 0.5f * (float)(tile - 1);
    return p;
}
__device__ __forceinline__ float tile_centre(uint32_t first_pixel, int tile) { return (float)first_pixel + 0.5f * (float)(tile - 1); }

__device__ __forceinline__ float quad_eval(float c0, float cx, float cy, float cxx, float cxy, float cyy, const PixelTerms &p)
{
    const float tx = __builtin_fmaf(cxy, p.Y, __builtin_fmaf(cxx, p.X, cx));
    const float ty = __builtin_fmaf(cyy, p.Y, cy);
    return __builtin_fmaf(p.Y, ty, __builtin_fmaf(p.X, tx, c0));
}

// lane -> pixel of the quadrant walk (below): lanes 16 q .. 16 q + 15 hold the 4x4 pixels of quadrant q
__device__ __forceinline__ void quadrant_pixel(uint32_t lane, uint32_t &local_x, uint32_t &local_y)
{
    local_x = ((lane >> 4) & 1) * 4 + (lane & 3);
    local_y = (lane >> 5) * 4 + ((lane >> 2) & 3);
}

// the same for the banked layout (quadrant q = lanes 4 q .. 4 q + 3 of every row of sixteen lanes; the row is the pixel row)
__device__ __forceinline__ void banked_quadrant_pixel(uint32_t lane, uint32_t &local_x, uint32_t &local_y)
{
    const uint32_t q = (lane >> 2) & 3u;
    local_x = (q & 1u) * 4u + (lane & 3u);
    local_y = (q >> 1) * 4u + (lane >> 4);
}

// kCullPixels: a slot counts for a quadrant when the instance passes the cut-off -- with the walk's own arithmetic -- at
// one of the pixels named by pixel_lanes (a wave-uniform mask over the lanes of the quadrant walk) that lie in it.
// kCullScaled: kCullAlpha for a least alpha of the walk's own, as opacity times cull_scale = the mode's least alpha over it.
enum { kCullNone = 0, kCullAlpha = 1, kCullCutoff = 2, kCullPixels = 3, kCullScaled = 4 };

// With QUADRANTS the result has one bit per 4x4 quadrant of the tile (tile_quadrant_hits) instead of one for the tile.
// REC4: 16-byte words per record of prim (five; eight in training frames).
// UNIT: the opacity is staged held to at most 1 (the image-only fast path, whose fragments then need no clamp of their own).
// POS: the last word of the slot holds the instance's place in the list (fetch) instead of the Gaussian's index.
// GIVEN: the caller has read inst[fetch] already (`given`).
// nearest: receives a depth that no fragment of the instance is nearer than (nearest_depth).
template <int MODE, int N, bool DEPTH, int CULL = kCullNone, bool QUADRANTS = false, int REC4 = HTGS_PRIM_FLOATS / 4, bool UNIT = false, bool POS = false,
          bool GIVEN = false>
__device__ __forceinline__ uint32_t tile_stage_load(TileStage<N> &st, const float4 *__restrict__ prim, const uint32_t *__restrict__ inst,
                                                    uint32_t fetch, uint32_t last, int slot, float cx, float cy, uint64_t pixel_lanes = 0, uint32_t given = 0, float cull_scale = 1.0f,
                                                    float *nearest = nullptr);

// (PixelTerms is complete by the time the template is instantiated)
template <int MODE, int N, bool DEPTH, int CULL, bool QUADRANTS, int REC4, bool UNIT, bool POS, bool GIVEN>
__device__ __forceinline__ uint32_t tile_stage_load(TileStage<N> &st, const float4 *__restrict__ prim, const uint32_t *__restrict__ inst,
                                                    uint32_t fetch, uint32_t last, int slot, float cx, float cy, uint64_t pixel_lanes, uint32_t given, float cull_scale,
                                                    float *nearest)
{
    if (fetch >= last) return 0;
    const uint32_t g = GIVEN ? given : inst[fetch];
    const float4 *rec = prim + (size_t)g * REC4;
    // (with CULL the record's colour row is fetched when it is needed, behind a compiler fence: it comes from a cache
    // line the other rows have just brought in, and four registers less at the peak keep the callers' K-buffers out
    // of scratch memory inside the batch loop)
    const float4 r1 = rec[0], r2 = rec[1], r4 = rec[2], r3 = rec[3];
    float4 col;
    if (CULL == kCullNone) col = rec[4];
    const float V1[4] = { r1.x, r1.y, r1.z, r1.w }, V2[4] = { r2.x, r2.y, r2.z, r2.w }, V4[4] = { r4.x, r4.y, r4.z, r4.w };
    float px0[4], py0[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        px0[k] = __builtin_fmaf(-V4[k], cx, V1[k]);
        py0[k] = __builtin_fmaf(-V4[k], cy, V2[k]);
    }
    float A[3], B[3], C[3], Am[3], Bm[3], Cm[3];
    cross3(px0, py0, A);
    cross3(V4, px0, B);
    cross3(py0, V4, C);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        Am[k] = __builtin_fmaf(px0[3], py0[k], -(px0[k] * py0[3]));
        Bm[k] = __builtin_fmaf(px0[k], V4[3], -(px0[3] * V4[k]));
        Cm[k] = __builtin_fmaf(V4[k], py0[3], -(V4[3] * py0[k]));
    }
    float zxy = 0.0f, zyy = 0.0f;
    if (DEPTH) {
        const float MT3[3] = { r3.x, r3.y, r3.z };
        float PA[3], PB[3], PC[3];
        cross3(MT3, A, PA);
        cross3(MT3, B, PB);
        cross3(MT3, C, PC);
        st.q[3][slot] = make_float4(dotf(PA, Am), dotf(PA, Cm) + dotf(PC, Am), dotf(PA, Bm) + dotf(PB, Am), dotf(PC, Cm));
        zxy = dotf(PB, Cm) + dotf(PC, Bm);
        zyy = dotf(PB, Bm);
    }
    constexpr float kc = ModeCfg<MODE>::cutoff_rcp;
    const float n[6] = { dotf(Am, Am) * kc, (2.0f * dotf(Am, Cm)) * kc, (2.0f * dotf(Am, Bm)) * kc,
                         dotf(Cm, Cm) * kc, (2.0f * dotf(Bm, Cm)) * kc, dotf(Bm, Bm) * kc };
    const float d[6] = { dotf(A, A), 2.0f * dotf(A, C), 2.0f * dotf(A, B), dotf(C, C), 2.0f * dotf(B, C), dotf(B, B) };
    st.q[0][slot] = make_float4(n[0], n[1], n[2], n[3]);
    st.q[1][slot] = make_float4(n[4], n[5], d[0], d[1]);
    st.q[2][slot] = make_float4(d[2], d[3], d[4], d[5]);
    if (CULL != kCullNone) {
        asm volatile("" ::: "memory");
        col = rec[4];
    }
    if (nearest != nullptr) *nearest = nearest_depth<MODE>(n, d, r3, col.w);
    if (UNIT) col.w = col.w < 1.0f ? col.w : 1.0f;
    st.q[4][slot] = make_float4(zxy, zyy, r3.w, col.w);
    st.q[5][slot] = make_float4(col.x, col.y, col.z, bits_to_float(POS ? fetch : g));
    if constexpr (CULL == kCullNone) return QUADRANTS ? 0xfu : 1u;
    else if constexpr (CULL == kCullPixels) {
        static_assert(QUADRANTS, "per quadrant");
        uint32_t bits = 0;
        for (uint64_t m = pixel_lanes; m != 0; m &= m - 1) {      // (wave-uniform)
            const uint32_t p = (uint32_t)__builtin_ctzll(m);
            uint32_t local_x, local_y;
            quadrant_pixel(p, local_x, local_y);
            const PixelTerms pt = pixel_terms(local_x, local_y, 8);
            const float num = quad_eval(n[0], n[1], n[2], n[3], n[4], n[5], pt), den = quad_eval(d[0], d[1], d[2], d[3], d[4], d[5], pt);
            if (!(num > den)) bits |= 1u << (p >> 4);
        }
        return bits;
    }
    else if constexpr (QUADRANTS) return tile_quadrant_hits<MODE>(n, d, CULL == kCullCutoff ? 1.0f : CULL == kCullScaled ? col.w * cull_scale : col.w);
    else return (uint32_t)!tile_misses<MODE>(n, d, CULL == kCullCutoff ? 1.0f : col.w);
}

struct TileFrag {
    float num, den, den_rcp, alpha;
};

// The per-pixel loops address the staged instance through one VGPR that holds the LDS byte address of q[0][j] and
// is advanced by an opaque add (the compiler would otherwise rebuild the address from the scalar loop counter
// before every read).
struct __attribute__((aligned(16))) Float4Pod { float x, y, z, w; };
typedef __attribute__((address_space(3))) const Float4Pod lds_float4;
typedef __attribute__((address_space(3))) const float lds_float;
template <int N>
__device__ __forceinline__ uint32_t stage_address(const TileStage<N> &st) { return (uint32_t)(uintptr_t)(lds_float4 *)&st.q[0][0]; }
__device__ __forceinline__ void stage_advance(uint32_t &addr) { asm volatile("v_add_u32 %0, 16, %0" : "+v"(addr)); }
// Quadrant walk.  Lanes 16 q .. 16 q + 15 hold the 4x4 pixels of quadrant q of the tile and walk the hits of that
// quadrant, in list order, in lock step with the other three quadrants: a turn of the loop serves up to four instances,
// one per quadrant, and a batch takes as many turns as its busiest quadrant has hits (an instance reaches 1.9 of the four
// quadrants on average, so this is well under the number of instances that reach the tile).  Every pixel still sees its
// fragments in list order.  The four hit masks are wave-uniform (scalar registers).
constexpr uint32_t kNoHit = 0xfffffff0u;           // 16 * s_ff1(0): the address a quadrant without a hit left gets
struct QuadrantHits {
    uint64_t h[4];
};
__device__ __forceinline__ QuadrantHits quadrant_ballot(uint32_t bits)
{
    QuadrantHits w;
#pragma unroll
    for (int q = 0; q < 4; ++q) w.h[q] = __ballot((bits >> q) & 1);
    return w;
}
__device__ __forceinline__ bool quadrant_pending(const QuadrantHits &w) { return (w.h[0] | w.h[1] | w.h[2] | w.h[3]) != 0; }
// LDS address, relative to the stage, of the q[0] entry of the lane's quadrant's next hit, or kNoHit.  Per quadrant two
// scalar instructions: s_ff1 gives the slot (-1 for an empty mask, which the shift turns into kNoHit) and s_bitset0
// clears that bit (bit 63 of an empty mask).  A quadrant is one row of sixteen lanes to the data-parallel primitives, so
// its lanes take the slot by a move with that row's mask: no exec writes, and the scalar unit, which the four SIMDs of a
// compute unit share, is left to the loop's branches.
// BANKED: a quadrant is not a row of sixteen lanes but lanes 4 q .. 4 q + 3 of each of the four rows (bank q of the
// data-parallel primitives), which is the layout in which sums over a quadrant's lanes fold across the rows.
template <bool BANKED = false>
__device__ __forceinline__ uint32_t quadrant_next_hit(QuadrantHits &w)
{
    uint32_t a0, a1, a2, a3, addr, t;
    // (two statements: one with scalar results only, which the compiler then knows to be wave-uniform)
    asm volatile("s_ff1_i32_b64 %[a0], %[h0]\n\ts_ff1_i32_b64 %[a1], %[h1]\n\ts_ff1_i32_b64 %[a2], %[h2]\n\ts_ff1_i32_b64 %[a3], %[h3]\n\t"
                 "s_bitset0_b64 %[h0], %[a0]\n\ts_bitset0_b64 %[h1], %[a1]\n\ts_bitset0_b64 %[h2], %[a2]\n\ts_bitset0_b64 %[h3], %[a3]"
                 : [a0] "=&s"(a0), [a1] "=&s"(a1), [a2] "=&s"(a2), [a3] "=&s"(a3),
                   [h0] "+s"(w.h[0]), [h1] "+s"(w.h[1]), [h2] "+s"(w.h[2]), [h3] "+s"(w.h[3]));
    if constexpr (BANKED)
        asm volatile("v_mov_b32 %[addr], %[a0]\n\t"
                     "v_mov_b32 %[t], %[a1]\n\t"
                     "s_nop 1\n\t"
                     "v_mov_b32_dpp %[addr], %[t] quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0x2\n\t"
                     "v_mov_b32 %[t], %[a2]\n\t"
                     "s_nop 1\n\t"
                     "v_mov_b32_dpp %[addr], %[t] quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0x4\n\t"
                     "v_mov_b32 %[t], %[a3]\n\t"
                     "s_nop 1\n\t"
                     "v_mov_b32_dpp %[addr], %[t] quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0x8\n\t"
                     "v_lshlrev_b32 %[addr], 4, %[addr]"
                     : [addr] "=&v"(addr), [t] "=&v"(t)
                     : [a0] "s"(a0), [a1] "s"(a1), [a2] "s"(a2), [a3] "s"(a3));
    else
        asm volatile("v_mov_b32 %[addr], %[a0]\n\t"
                     "v_mov_b32 %[t], %[a1]\n\t"
                     "s_nop 1\n\t"
                     "v_mov_b32_dpp %[addr], %[t] quad_perm:[0,1,2,3] row_mask:0x2 bank_mask:0xf\n\t"
                     "v_mov_b32 %[t], %[a2]\n\t"
                     "s_nop 1\n\t"
                     "v_mov_b32_dpp %[addr], %[t] quad_perm:[0,1,2,3] row_mask:0x4 bank_mask:0xf\n\t"
                     "v_mov_b32 %[t], %[a3]\n\t"
                     "s_nop 1\n\t"
                     "v_mov_b32_dpp %[addr], %[t] quad_perm:[0,1,2,3] row_mask:0x8 bank_mask:0xf\n\t"
                     "v_lshlrev_b32 %[addr], 4, %[addr]"
                     : [addr] "=&v"(addr), [t] "=&v"(t)
                     : [a0] "s"(a0), [a1] "s"(a1), [a2] "s"(a2), [a3] "s"(a3));
    return addr;
}
// Quadrant lists: the same walk with the scalar bit scans taken out of the loop.  After a batch is staged, the slots that
// reach quadrant q are written, in list order, to a short list in LDS (their LDS addresses), padded up to the length of
// the longest of the four lists with the address of a slot that no fragment passes (entry 0 of every row of a stage with
// kStageSlots entries per row: a cut-off quadratic above its |d|^2, opacity 0).  A turn of the loop is then one LDS read
// per lane -- entry `turn` of its quadrant's list -- instead of eight scalar and nine vector instructions that pick the
// next set bit of four masks and hand it to the quadrant's lanes, and a quadrant that has run out of hits evaluates the
// dummy slot, which fails the walk's own test, instead of being masked off: one exec level less.
constexpr int kStageSlots = 65;
typedef TileStage<kStageSlots> TileStageQ;
struct __attribute__((aligned(8))) QuadrantLists {
    uint32_t a[4][64];
    uint32_t beyond[2];         // (the walks read one entry or one pair of entries ahead)
};
typedef __attribute__((address_space(3))) const uint32_t lds_u32;
typedef __attribute__((address_space(3))) const uint64_t lds_u64;
// (one lane) the slot that fails every test: |m|^2 / cut-off = 1 everywhere, |d|^2 = 1/2, opacity 0
__device__ __forceinline__ void stage_dummy_init(TileStageQ &st, uint32_t lane)
{
    if (lane == 0) {
        st.q[0][0] = make_float4(1.0f, 0.0f, 0.0f, 0.0f);
        st.q[1][0] = make_float4(0.0f, 0.0f, 0.5f, 0.0f);
        st.q[2][0] = st.q[3][0] = st.q[4][0] = st.q[5][0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}
// LDS address of the q[0] entry of staged slot `slot` (0 .. 63)
__device__ __forceinline__ uint32_t stage_slot_address(const TileStageQ &st, uint32_t slot) { return stage_address(st) + 16u * (slot + 1u); }
// Called by the wave after tile_stage_load (bits: the lane's slot's quadrant bits): writes the four lists and returns the
// number of turns, the length of the longest (wave-uniform).  Every lane writes one entry per list: a slot that reaches
// the quadrant its address at the number of such slots before it, the others the dummy address behind all of them.
__device__ __forceinline__ uint32_t quadrant_lists_build(QuadrantLists &ql, uint32_t bits, uint32_t lane, const TileStageQ &st)
{
    const uint32_t dummy = stage_address(st), mine = stage_slot_address(st, lane);
    uint32_t most = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool hit = (bits >> q) & 1u;
        const uint64_t h = __ballot(hit);
        const uint32_t count = (uint32_t)__popcll(h);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(h >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)h, 0u));
        ql.a[q][hit ? below : count + (lane - below)] = hit ? mine : dummy;
        most = most > count ? most : count;
    }
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)most);
}
// turn(addr) is called n_turns times, by all lanes: addr = the LDS address of the q[0] entry of the slot the lane's quadrant
// (lanes 16 q .. 16 q + 15) evaluates in this turn.
template <typename Turn>
__device__ __forceinline__ void quadrant_list_walk(const QuadrantLists &ql, uint32_t n_turns, uint32_t lane, Turn &&turn)
{
    // (the entry of the next turn is read while this turn's slot is evaluated: one LDS round trip per turn, not two)
    uint32_t p = (uint32_t)(uintptr_t)(lds_u32 *)&ql.a[lane >> 4][0];
    uint32_t addr = *(lds_u32 *)(uintptr_t)p;
    // (two turns per round of the loop, the entry that was read ahead changing registers, so that no turn moves it)
    uint32_t t = 0;
    for (; t + 1 < n_turns; t += 2) {
        asm volatile("v_add_u32 %0, 4, %0" : "+v"(p));
        const uint32_t next = *(lds_u32 *)(uintptr_t)p;
        turn(addr);
        asm volatile("v_add_u32 %0, 4, %0" : "+v"(p));
        addr = *(lds_u32 *)(uintptr_t)p;
        turn(next);
    }
    if (t < n_turns) turn(addr);
}
// The same walk two turns at a time: turns(one, two) with the addresses of two turns in a row.  What the two fragments are is
// worked out side by side, so that the waits of one -- for LDS, for a compare that a branch depends on -- are filled by the
// other.  An odd number of turns ends with a turn of dummy slots (every list has 64 entries, the dummy's behind the hits).
// A wave that runs alone issues an instruction every 2.5 ns, waits 24 ns for a row from LDS and 14 ns between a compare and
// the branch on it; five waves a SIMD cover most of that but not all.  One turn -> two at a time, whole passes: HYBRID K = 16, 3 M
// Gaussians at 1920x1080 1373 -> 1306 us, FIRST_K 1 M at 1280x720 351 -> 334, OIT 334 k at 1237x821 163.8 -> 159.8 (3 M at 1920x1080,
// one wave a tile, is bound by the reads of LDS and gains nothing: blend 800 -> 801).  Cores of 32 have
// no registers left for a second fragment and keep the walk above, like the walks with three registers a slot.
template <typename Turns>
__device__ __forceinline__ void quadrant_list_walk_pairs(const QuadrantLists &ql, uint32_t n_turns, uint32_t lane, Turns &&turns)
{
    uint32_t p = (uint32_t)(uintptr_t)(lds_u32 *)&ql.a[lane >> 4][0];
    uint64_t at = *(lds_u64 *)(uintptr_t)p;
    for (uint32_t t = 0; t < n_turns; t += 2) {
        asm volatile("v_add_u32 %0, 8, %0" : "+v"(p));
        const uint64_t next = *(lds_u64 *)(uintptr_t)p;
        turns((uint32_t)at, (uint32_t)(at >> 32));
        at = next;
    }
}
// The walk over instances [first, last) of a tile's list (whole batches of 64 from `first` on, `step` apart) by one wave, lanes =
// pixels by quadrants: every batch is staged (tile_stage_load with the CULL asked for), its quadrant lists are built and
// turn(addr) is called for every turn.  SOLO: the wave is the whole workgroup (its barriers are the workgroup's).
// AHEAD: a lane reads the list entry of the next batch before it walks this one (one register more through the walk; the
// entry is then there when the batch is staged, and the records' fetch does not wait for it).
// PAIRS: two turns at a time, turn(one, two).
// last_depth(): the depth from which on a fragment is of no use to the lane's pixel any more (AllDepths: none is); an instance that is
// nowhere nearer than that for all pixels of a quadrant is left out of the quadrant's list.
// step: from one batch of the wave's to the next, and how many instances each has (waves that share a list: blend_waves.h).
struct AllDepths {};
struct ListStep {
    uint32_t step, batch;
    __device__ __forceinline__ ListStep(uint32_t s, uint32_t b = 64u) : step(s), batch(b) {}
    __device__ __forceinline__ uint32_t at(uint32_t base, uint32_t last, uint32_t lane) const { return batch >= 64u || lane < batch ? base + lane : last; }
};
// the largest of the values of each quadrant's sixteen lanes, the same in all lanes
struct QuadrantDepths { float q[4]; };
__device__ __forceinline__ QuadrantDepths quadrant_most(float v)
{
    float m = v;
    const auto step = [&m](float o) { m = m > o ? m : o; };
    step(bits_to_float((uint32_t)__builtin_amdgcn_update_dpp((int)float_to_bits(m), (int)float_to_bits(m), 0x121, 0xf, 0xf, false)));      // row_ror:1
    step(bits_to_float((uint32_t)__builtin_amdgcn_update_dpp((int)float_to_bits(m), (int)float_to_bits(m), 0x122, 0xf, 0xf, false)));      // row_ror:2
    step(bits_to_float((uint32_t)__builtin_amdgcn_update_dpp((int)float_to_bits(m), (int)float_to_bits(m), 0x124, 0xf, 0xf, false)));      // row_ror:4
    step(bits_to_float((uint32_t)__builtin_amdgcn_update_dpp((int)float_to_bits(m), (int)float_to_bits(m), 0x128, 0xf, 0xf, false)));      // row_ror:8
    QuadrantDepths most;
#pragma unroll
    for (int q = 0; q < 4; ++q) most.q[q] = bits_to_float((uint32_t)__builtin_amdgcn_readlane((int)float_to_bits(m), 16 * q));
    return most;
}
template <int MODE, bool DEPTH, int CULL, bool SOLO, int REC4 = HTGS_PRIM_FLOATS / 4, bool UNIT = false, bool POS = false, bool AHEAD = false, bool PAIRS = false,
          typename Turn, typename Last = AllDepths>
__device__ __forceinline__ void tile_list_walk(TileStageQ &st, QuadrantLists &ql, const float4 *__restrict__ prim, const uint32_t *__restrict__ inst,
                                               uint32_t first, uint32_t last, uint32_t lane, float cx, float cy, Turn &&turn, uint64_t pixel_lanes = 0,
                                               float cull_scale = 1.0f, ListStep step = 64u, Last &&last_depth = Last())
{
    constexpr bool kNear = !std::is_same<typename std::decay<Last>::type, AllDepths>::value;
    stage_dummy_init(st, lane);
    uint32_t listed = 0;
    const auto list_entry = [&](uint32_t base) { const uint32_t at = step.at(base, last, lane); return at < last ? inst[at] : 0u; };
    if (AHEAD) listed = list_entry(first);
    for (uint32_t base = first; base < last; base += step.step) {
        if (SOLO) __syncthreads(); else wave_lds_sync();
        float nearest = -__FLT_MAX__;
        uint32_t bits = tile_stage_load<MODE, kStageSlots, DEPTH, CULL, true, REC4, UNIT, POS, AHEAD>(st, prim, inst, step.at(base, last, lane), last, lane + 1, cx, cy, pixel_lanes,
                                                                                                     listed, cull_scale, kNear ? &nearest : nullptr);
        if constexpr (kNear) {
            const QuadrantDepths most = quadrant_most(last_depth());
#pragma unroll
            for (int q = 0; q < 4; ++q) bits &= nearest > most.q[q] ? ~(1u << q) : ~0u;
        }
        if (AHEAD) listed = list_entry(base + step.step);
        const uint32_t n_turns = quadrant_lists_build(ql, bits, lane, st);
        if (SOLO) __syncthreads(); else wave_lds_sync();
        // lanes outside the image run along (their results are never stored): the loop stays wave-uniform
        if constexpr (PAIRS) quadrant_list_walk_pairs(ql, n_turns, lane, turn);
        else quadrant_list_walk(ql, n_turns, lane, turn);
    }
}
// The per-pixel records of the training pass are kept tile by tile: the 64 pixels of an 8x8 tile, row-major, are
// contiguous, so a tile's workgroup writes and reads whole lines whatever order the tiles are taken in.  A record plane
// has 64 entries per tile of the launch (gridDim.x tiles, the pixels beyond the image included).
__device__ __forceinline__ size_t record_pixel(uint32_t tile, uint32_t x, uint32_t y) { return (size_t)tile * 64u + (y & 7u) * 8u + (x & 7u); }
__device__ __forceinline__ size_t record_plane() { return (size_t)gridDim.x * 64u; }
// the tile a workgroup takes: the launch's blocks go through htgs_frame.tile_order (longest lists first) if there is one
__device__ __forceinline__ uint32_t block_tile(const uint32_t *__restrict__ tile_order) { return tile_order ? tile_order[blockIdx.x] : blockIdx.x; }
// pixel of a lane in an 8x8 tile that is walked by quadrants
struct TilePixel {
    uint32_t x, y;
    bool inside;
    PixelTerms pt;
    float cx, cy;
};
template <int N, int ROW>
__device__ __forceinline__ float4 stage_row(uint32_t addr)
{
    lds_float4 *p = (lds_float4 *)(uintptr_t)(addr + ROW * N * 16);
    return make_float4(p->x, p->y, p->z, p->w);
}
template <int N>
__device__ __forceinline__ float stage_opacity(uint32_t addr) { return *(lds_float *)(uintptr_t)(addr + 4 * N * 16 + 12); }
template <int N>
__device__ __forceinline__ uint32_t stage_index(uint32_t addr) { return float_to_bits(*(lds_float *)(uintptr_t)(addr + 5 * N * 16 + 12)); }

// |m|^2 <= cutoff |d|^2 ?  (inference.cuh:147)
template <int N>
__device__ __forceinline__ bool tile_frag_cutoff(uint32_t addr, const PixelTerms &p, TileFrag &o)
{
    const float4 q0 = stage_row<N, 0>(addr), q1 = stage_row<N, 1>(addr), q2 = stage_row<N, 2>(addr);
    o.num = quad_eval(q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, p);
    o.den = quad_eval(q1.z, q1.w, q2.x, q2.y, q2.z, q2.w, p);
    return !(o.num > o.den);
}

// camera-space depth of the point of maximum contribution (inference.cuh:151-152); needs o.den_rcp
template <int N>
__device__ __forceinline__ float tile_frag_depth(uint32_t addr, const PixelTerms &p, const TileFrag &o)
{
    const float4 q3 = stage_row<N, 3>(addr), q4 = stage_row<N, 4>(addr);
    return __builtin_fmaf(quad_eval(q3.x, q3.y, q3.z, q3.w, q4.x, q4.y, p), o.den_rcp, q4.z);
}

// The image-only fast path (FAST) takes the hardware's reciprocal and 2^x (v_rcp_f32, v_exp_f32: one ulp, a quarter of
// the instruction slots); every other kernel uses the exactly reproducible routines.
template <bool FAST>
__device__ __forceinline__ float frag_rcp(float x) { return FAST ? __builtin_amdgcn_rcpf(x) : rcp_exact(x); }

// alpha of the fragment, false below the mode's threshold; needs o.den_rcp
template <int MODE, bool FAST = false>
__device__ __forceinline__ bool tile_frag_alpha(float opacity, TileFrag &o)
{
    const float t = (o.num * ModeCfg<MODE>::exp2_scale) * o.den_rcp;
    const float G = FAST ? __builtin_amdgcn_exp2f(t) : d_exp2(t);
    const float a = opacity * G;
    o.alpha = a < kMaxFragmentAlpha ? a : kMaxFragmentAlpha;
    return !(o.alpha < ModeCfg<MODE>::min_alpha);
}

// The exact fragment in one piece: whether it passes the cut-off and the alpha threshold; o is complete.  1 / |d|^2 is the refined
// reciprocal, and the alpha is worked out with it before anything asks whether a lane's |d|^2 is outside that form's range
// (rcp_exact's test): the branch then does not wait for its compare.
template <int MODE, int N>
__device__ __forceinline__ bool tile_frag_exact(uint32_t addr, const PixelTerms &p, TileFrag &o)
{
    const bool in_reach = tile_frag_cutoff<N>(addr, p, o);
    const float opacity = stage_opacity<N>(addr);
    const uint64_t leaves = __ballot(!rcp_in_range(o.den));
    o.den_rcp = rcp_refined(o.den);
    bool passes = tile_frag_alpha<MODE, false>(opacity, o);
    if (__builtin_expect(leaves != 0, 0)) {
        o.den_rcp = 1.0f / o.den;
        passes = tile_frag_alpha<MODE, false>(opacity, o);
    }
    return passes && in_reach;
}
// two of them (quadrant_list_walk_pairs)
template <int MODE, int N>
__device__ __forceinline__ void tile_frag_exact_pair(uint32_t one, uint32_t two, const PixelTerms &p, TileFrag &o, TileFrag &t, bool &one_passes, bool &two_passes)
{
    const bool o_reach = tile_frag_cutoff<N>(one, p, o), t_reach = tile_frag_cutoff<N>(two, p, t);
    const float o_opacity = stage_opacity<N>(one), t_opacity = stage_opacity<N>(two);
    const uint64_t leaves = __ballot(!rcp_in_range(o.den)) | __ballot(!rcp_in_range(t.den));
    o.den_rcp = rcp_refined(o.den);
    t.den_rcp = rcp_refined(t.den);
    one_passes = tile_frag_alpha<MODE, false>(o_opacity, o);
    two_passes = tile_frag_alpha<MODE, false>(t_opacity, t);
    if (__builtin_expect(leaves != 0, 0)) {
        o.den_rcp = 1.0f / o.den;
        t.den_rcp = 1.0f / t.den;
        one_passes = tile_frag_alpha<MODE, false>(o_opacity, o);
        two_passes = tile_frag_alpha<MODE, false>(t_opacity, t);
    }
    one_passes = one_passes && o_reach;
    two_passes = two_passes && t_reach;
}

// The image-only fast path's fragment: with the opacity staged at no more than 1 (UNIT) alpha = opacity * G needs no clamp, and a
// fragment beyond the cut-off has G below the alpha threshold (the cut-off is where G equals it), so the alpha test alone
// decides; a vanishing or non-finite |d|^2 gives alpha 0 or NaN, which fails it.  Needs o.num, o.den.
template <int MODE, int N>
__device__ __forceinline__ bool tile_frag_fast(uint32_t addr, const PixelTerms &p, TileFrag &o)
{
    tile_frag_cutoff<N>(addr, p, o);
    o.den_rcp = __builtin_amdgcn_rcpf(o.den);
    o.alpha = stage_opacity<N>(addr) * __builtin_amdgcn_exp2f((o.num * ModeCfg<MODE>::exp2_scale) * o.den_rcp);
    return o.alpha >= ModeCfg<MODE>::min_alpha;
}

// Sorted insertion into a K-slot buffer (depth, alpha, index per slot) walks the slots front to back carrying the
// displaced entry (the reference's exchange walk); the slots are taken four at a time and the whole wave skips a group
// that no active lane can change (the carried depth is not below the group's last slot).  One slot: v_cmpx narrows
// exec to the lanes whose carried depth is below the slot's, three moves through a scratch register exchange each
// of the three registers (a wave64 v_mov_b32 holds the vector ALU for two cycles, v_swap_b32 for eight,
// v_cndmask_b32 for four), and exec is restored.  On return (depth, alpha, index) is what the walk pushed out.
constexpr int kInsertGroup = 4;
template <typename IndexT>
__device__ __forceinline__ void exchange_step(float &D, float &A, IndexT &I, float &d, float &a, IndexT &x, uint64_t all)
{
    static_assert(sizeof(IndexT) == 4, "one register");
    float t;
    asm volatile("v_cmpx_lt_f32 vcc, %[D], %[d]\n\t"
                 "v_mov_b32 %[t], %[d]\n\tv_mov_b32 %[d], %[D]\n\tv_mov_b32 %[D], %[t]\n\t"
                 "v_mov_b32 %[t], %[a]\n\tv_mov_b32 %[a], %[A]\n\tv_mov_b32 %[A], %[t]\n\t"
                 "v_mov_b32 %[t], %[x]\n\tv_mov_b32 %[x], %[I]\n\tv_mov_b32 %[I], %[t]\n\t"
                 "s_mov_b64 exec, %[all]"
                 : [D] "+v"(D), [A] "+v"(A), [I] "+v"(I), [d] "+v"(d), [a] "+v"(a), [x] "+v"(x), [t] "=&v"(t)
                 : [all] "s"(all)
                 : "vcc");
}
// four slots in one statement: exec is saved once and restored after every slot
#define HTGS_EXCHANGE_SLOT(n)                                                                                            \
    "v_cmpx_lt_f32 vcc, %[d], %[D" #n "]\n\t"                                                                           \
    "v_mov_b32 %[t], %[D" #n "]\n\tv_mov_b32 %[D" #n "], %[d]\n\tv_mov_b32 %[d], %[t]\n\t"                              \
    "v_mov_b32 %[t], %[A" #n "]\n\tv_mov_b32 %[A" #n "], %[a]\n\tv_mov_b32 %[a], %[t]\n\t"                              \
    "v_mov_b32 %[t], %[I" #n "]\n\tv_mov_b32 %[I" #n "], %[x]\n\tv_mov_b32 %[x], %[t]\n\t"                              \
    "s_mov_b64 exec, %[all]\n\t"
template <typename IndexT>
__device__ __forceinline__ void exchange_step4(float &d, float &a, IndexT &x, float &D0, float &A0, IndexT &I0, float &D1, float &A1, IndexT &I1,
                                               float &D2, float &A2, IndexT &I2, float &D3, float &A3, IndexT &I3)
{
    static_assert(sizeof(IndexT) == 4, "one register");
    float t;
    uint64_t all;
    asm volatile("s_mov_b64 %[all], exec\n\t" HTGS_EXCHANGE_SLOT(0) HTGS_EXCHANGE_SLOT(1) HTGS_EXCHANGE_SLOT(2) HTGS_EXCHANGE_SLOT(3)
                 : [d] "+v"(d), [a] "+v"(a), [x] "+v"(x), [D0] "+v"(D0), [A0] "+v"(A0), [I0] "+v"(I0), [D1] "+v"(D1), [A1] "+v"(A1), [I1] "+v"(I1),
                   [D2] "+v"(D2), [A2] "+v"(A2), [I2] "+v"(I2), [D3] "+v"(D3), [A3] "+v"(A3), [I3] "+v"(I3), [t] "=&v"(t), [all] "=&s"(all)
                 :
                 : "vcc");
}
#undef HTGS_EXCHANGE_SLOT
template <int K, typename IndexT>
__device__ __forceinline__ void core_exchange_walk(float &depth, float &alpha, IndexT &index, float (&cd)[K], float (&ca)[K], IndexT (&ci)[K])
{
    const uint64_t all = __ballot(true);               // the lanes that called
#pragma unroll
    for (int g0 = 0; g0 < K; g0 += kInsertGroup) {
        if (K > kInsertGroup && !__any(depth < cd[g0 + kInsertGroup - 1 < K ? g0 + kInsertGroup - 1 : K - 1])) continue;
        if constexpr (K % kInsertGroup == 0 && kInsertGroup == 4) {
            exchange_step4(depth, alpha, index, cd[g0], ca[g0], ci[g0], cd[g0 + 1], ca[g0 + 1], ci[g0 + 1], cd[g0 + 2], ca[g0 + 2], ci[g0 + 2],
                           cd[g0 + 3], ca[g0 + 3], ci[g0 + 3]);
        } else {
#pragma unroll
            for (int i = g0; i < g0 + kInsertGroup && i < K; ++i) exchange_step(depth, alpha, index, cd[i], ca[i], ci[i], all);
        }
    }
}

// The image-only fast path, and the shared walks of blend_hybrid_long_kernel, insert by shifting instead: the entry that moves down the core alternates between two register
// triples, so that a slot costs two moves per register (slot -> the other triple, this triple -> slot) instead of an
// exchange through a scratch register.  Both triples start out as the fragment; a lane joins at the first slot that is
// not nearer than its fragment and from there on moves every slot down by one (<=: once it has joined, the entry it carries
// is the previous slot's, which is never deeper than the next slot's).  This is the stable insertion, not the reference's
// exchange walk: where two stored fragments have exactly the same depth the two differ in which of them ends up in front,
// which the fast path does not promise to reproduce.  On return (depth, alpha, index) is what was pushed out.
#define HTGS_QUICK_SLOT(n, R, W)                                                                                         \
    "v_cmpx_le_f32 vcc, %[d" #R "], %[D" #n "]\n\t"                                                                     \
    "v_mov_b32 %[d" #W "], %[D" #n "]\n\tv_mov_b32 %[D" #n "], %[d" #R "]\n\t"                                         \
    "v_mov_b32 %[a" #W "], %[A" #n "]\n\tv_mov_b32 %[A" #n "], %[a" #R "]\n\t"                                         \
    "v_mov_b32 %[x" #W "], %[I" #n "]\n\tv_mov_b32 %[I" #n "], %[x" #R "]\n\t"                                         \
    "s_mov_b64 exec, %[all]\n\t"
template <typename IndexT>
__device__ __forceinline__ void quick_step4(float &d0, float &a0, IndexT &x0, float &d1, float &a1, IndexT &x1, float &D0, float &A0, IndexT &I0,
                                            float &D1, float &A1, IndexT &I1, float &D2, float &A2, IndexT &I2, float &D3, float &A3, IndexT &I3)
{
    static_assert(sizeof(IndexT) == 4, "one register");
    uint64_t all;
    asm volatile("s_mov_b64 %[all], exec\n\t" HTGS_QUICK_SLOT(0, 0, 1) HTGS_QUICK_SLOT(1, 1, 0) HTGS_QUICK_SLOT(2, 0, 1) HTGS_QUICK_SLOT(3, 1, 0)
                 : [d0] "+v"(d0), [a0] "+v"(a0), [x0] "+v"(x0), [d1] "+v"(d1), [a1] "+v"(a1), [x1] "+v"(x1), [D0] "+v"(D0), [A0] "+v"(A0),
                   [I0] "+v"(I0), [D1] "+v"(D1), [A1] "+v"(A1), [I1] "+v"(I1), [D2] "+v"(D2), [A2] "+v"(A2), [I2] "+v"(I2), [D3] "+v"(D3),
                   [A3] "+v"(A3), [I3] "+v"(I3), [all] "=&s"(all)
                 :
                 : "vcc");
}
#undef HTGS_QUICK_SLOT
template <int K, typename IndexT>
__device__ __forceinline__ void core_quick_walk(float &depth, float &alpha, IndexT &index, float (&cd)[K], float (&ca)[K], IndexT (&ci)[K])
{
    if constexpr (K % 4 != 0) core_exchange_walk<K>(depth, alpha, index, cd, ca, ci);
    else {
        float d1 = depth, a1 = alpha;
        IndexT x1 = index;
#pragma unroll
        for (int g0 = 0; g0 < K; g0 += 4) {
            // (a group that no lane's entry is nearer than the end of: nothing moves there; a group is an even number of
            // slots, so the entry is back in the first triple at every group's start)
            if (K > 4 && !__any(depth < cd[g0 + 3])) continue;
            quick_step4(depth, alpha, index, d1, a1, x1, cd[g0], ca[g0], ci[g0], cd[g0 + 1], ca[g0 + 1], ci[g0 + 1], cd[g0 + 2], ca[g0 + 2], ci[g0 + 2],
                        cd[g0 + 3], ca[g0 + 3], ci[g0 + 3]);
        }
    }
}

__device__ __forceinline__ TilePixel quadrant_tile_pixel(uint32_t tile, uint32_t grid_w, uint32_t lane, uint32_t width, uint32_t height)
{
    TilePixel p;
    const uint32_t x0 = (tile % grid_w) * 8, y0 = (tile / grid_w) * 8;
    uint32_t local_x, local_y;
    quadrant_pixel(lane, local_x, local_y);
    p.x = x0 + local_x;
    p.y = y0 + local_y;
    p.inside = p.x < width && p.y < height;
    p.pt = pixel_terms(local_x, local_y, 8);
    // (the same in every lane: held in scalar registers, two vector registers less in kernels that count them)
    p.cx = bits_to_float((uint32_t)__builtin_amdgcn_readfirstlane((int)float_to_bits(tile_centre(x0, 8))));
    p.cy = bits_to_float((uint32_t)__builtin_amdgcn_readfirstlane((int)float_to_bits(tile_centre(y0, 8))));
    return p;
}

// The 16x16 tile of ALPHA_BLEND_GLOBAL_ORDERING: 256 threads, wave w holds the 8x8 sub-tile 2 (row >= 8) + (column >= 8)
// = w, laid out for the quadrant walk.
__device__ __forceinline__ void subtile_pixel(uint32_t thread, uint32_t &local_x, uint32_t &local_y)
{
    quadrant_pixel(thread & 63u, local_x, local_y);
    local_x += 8u * ((thread >> 6) & 1u);
    local_y += 8u * (thread >> 7);
}
// One batch of 256 staged instances (reach[slot]: the sixteen quadrant bits tile_stage_load returned for it): the wave
// walks the hits of its own four quadrants, 64 slots at a time, and stops early once all_done() says so (wave-uniform).  Two turns
// at a time, for the reason given at quadrant_list_walk_pairs: turns(one, one_listed, two, two_listed); a quadrant without a hit left
// gets the part's first slot, not listed.
template <typename Done, typename Turns>
__device__ __forceinline__ void subtile_walk(const uint16_t *reach, uint32_t stage_base, uint32_t n_staged, uint32_t wave, uint32_t lane,
                                             Done &&all_done, Turns &&turns)
{
    for (uint32_t part = 0; part < 4 && 64u * part < n_staged; ++part) {
        if (all_done()) break;
        QuadrantHits hits = quadrant_ballot(((uint32_t)reach[64u * part + lane] >> (4u * wave)) & 0xfu);
        const uint32_t part_base = stage_base + 64u * 16u * part;
        while (quadrant_pending(hits)) {
            const uint32_t one = quadrant_next_hit(hits), two = quadrant_next_hit(hits);
            turns(one != kNoHit ? one + part_base : part_base, one != kNoHit, two != kNoHit ? two + part_base : part_base, two != kNoHit);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Lists in bins of depth (htgs_frame.depth_bins): a tile's list is up to kDepthBins runs, each by Gaussian index.  What the
// reference's insertion leaves where fragments are exactly equally deep depends on their order by index over the whole list.
// ---------------------------------------------------------------------------------------------
// The finished core's entries [i], [i + 1] of equal depth, in the order the reference's insertion leaves them in: an entry that
// comes nearer than both hops the first over the second, so they are by index if an even number of the nearer entries has a
// higher index than both, and the other way round if an odd number has.  (All nearer fragments are in the core as long as
// the two are.)  True where more than two are equally deep: that order takes a walk by index.
template <int K, typename IndexT>
__device__ __forceinline__ bool settle_equal_pairs(float (&cd)[K], float (&ca)[K], IndexT (&ci)[K])
{
    static_assert(sizeof(IndexT) == 4, "an index or its bit pattern");
    bool more = false;
#pragma unroll
    for (int i = 0; i + 1 < K; ++i) {
        const bool equal = ca[i + 1] > 0.0f && cd[i] == cd[i + 1];
        if (!__any(equal)) continue;
        if (i + 2 < K) more = more || (equal && ca[i + 2 < K ? i + 2 : i] > 0.0f && cd[i + 1] == cd[i + 2 < K ? i + 2 : i]);
        uint32_t a, b;
        __builtin_memcpy(&a, &ci[i], 4);
        __builtin_memcpy(&b, &ci[i + 1], 4);
        const uint32_t high = a > b ? a : b;
        bool odd = false;
#pragma unroll
        for (int j = 0; j < i; ++j) {
            uint32_t x;
            __builtin_memcpy(&x, &ci[j], 4);
            odd = odd != (x > high);
        }
        if (equal && (a > b) != odd) {
            const float t = ca[i]; ca[i] = ca[i + 1]; ca[i + 1] = t;
            const IndexT x = ci[i]; ci[i] = ci[i + 1]; ci[i + 1] = x;
        }
    }
    return more;
}

// What a walk notes of equal depths at the end of a pixel's core: the least depth at which a fragment stayed out of the core, or left it,
// that is exactly as deep as the entry that is last then (the core's last depth never grows, so the latest such depth is the least); that
// fragment's index, with kMoreTied if it was not the only one as deep.
constexpr uint32_t kMoreTied = 1u << 31;
struct CoreTie {
    float depth;
    uint32_t other;
    __device__ __forceinline__ void init() { depth = __FLT_MAX__; other = 0u; }
    // the lanes with `met` note it; a wave without one branches over it, on the compare's own result
    __device__ __forceinline__ void note(bool met, float at, uint32_t index)
    {
        if (__ballot(met) == 0ull) return;
        asm volatile("");
        other = met ? index | (depth == at ? kMoreTied : 0u) : other;
        depth = met ? at : depth;
    }
    // another wave's note of the same pixel
    __device__ __forceinline__ void join(const CoreTie &t)
    {
        other = t.depth < depth ? t.other : t.depth == depth ? other | kMoreTied : other;
        depth = t.depth < depth ? t.depth : depth;
    }
    // (nothing stays out of a core that is not full)
    __device__ __forceinline__ bool at_end(float last_depth) const { return depth < __FLT_MAX__ && depth <= last_depth; }
};
// Whether what stayed out of a core, or left it, is as deep as the entry that is last now.  (An empty slot, whose depth is the largest float, is not:
// the last entry's depth is held below it, which takes one instruction where a second test takes three.)
__device__ __forceinline__ bool meets_core_end(float depth, float last_depth)
{
    float last;
    asm("v_min_f32 %0, 0x7f7ffffe, %1" : "=v"(last) : "v"(last_depth));
    return depth == last;
}
// two entries of the finished core are exactly as deep as each other, or one that is not in it is as deep as its last
template <int K>
__device__ __forceinline__ bool core_tied(const float (&cd)[K], const float (&ca)[K], const CoreTie &tie)
{
    bool tied = tie.at_end(cd[K - 1]);
#pragma unroll
    for (int i = 0; i + 1 < K; ++i) tied = tied || (ca[i + 1] > 0.0f && cd[i] == cd[i + 1]);
    return tied;
}
// Depth and alpha of Gaussian `other` at the pixels of the lanes that have noted one, by the walk's own arithmetic.
struct TieFragment { float depth, alpha; };
template <int MODE, int REC4>
__device__ __forceinline__ TieFragment tie_fragment(TileStageQ &st, const float4 *__restrict__ prim, uint32_t lane, const PixelTerms &pt, float cx, float cy, bool noted,
                                                    uint32_t other)
{
    wave_lds_sync();
    // (a slot for each lane, as in a batch of the walk)
    tile_stage_load<MODE, kStageSlots, true, kCullNone, true, REC4, false, false, true>(st, prim, nullptr, noted ? 0u : 1u, 1u, (int)lane + 1, cx, cy, 0, other);
    wave_lds_sync();
    const uint32_t addr = stage_slot_address(st, lane);
    TileFrag f;
    tile_frag_exact<MODE, kStageSlots>(addr, pt, f);
    return TieFragment{ tile_frag_depth<kStageSlots>(addr, pt, f), f.alpha };
}
// The finished core of every pixel of the wave with its entries of equal depth as the reference's insertion leaves them, from the core
// alone: pairs inside it are put in order (settle_equal_pairs), and where its last entry and one other fragment are equally deep, that
// fragment is evaluated at the pixel and takes the last entry's place if the order by index says so: of the two, the one
// with the lower index stays if an even number of the nearer entries has a higher index than both, the other one if an odd number
// has.  (The last arrival of the K + 1 decides: one of the two is turned away, any other hops the first over the second, which
// leaves.)  noted: a fragment met the last entry's depth; other: its index, more: it was not the only one (CoreTie).
// swapped(in, out): the tail has gained a fragment of the last entry's depth and lost another one.  True for the pixels that this does not settle: more than two of a depth, or a tail that cannot give up an opaque fragment.
// A pixel that is settled so costs the evaluation of one fragment; walking the tile's list for it took as long as a list of a
// third of its length, at the end of a launch as often as not (6 M Gaussians of the stress scene at 1600x1066: the launch with
// one wave per tile 1050 -> 730 us).
template <int MODE, int K, int REC4, typename IndexT, typename Swapped>
__device__ __forceinline__ bool settle_core(TileStageQ &st, const float4 *__restrict__ prim, uint32_t lane, const PixelTerms &pt, float cx, float cy, float (&cd)[K],
                                            float (&ca)[K], IndexT (&ci)[K], bool noted, uint32_t other, bool more, Swapped &&swapped)
{
    bool again = false, pairs = false;
#pragma unroll
    for (int i = 0; i + 1 < K; ++i) pairs = pairs || (ca[i + 1] > 0.0f && cd[i] == cd[i + 1]);
    if (__any(pairs)) again = settle_equal_pairs<K>(cd, ca, ci);
    if (!__any(noted)) return again;
    const TieFragment f = tie_fragment<MODE, REC4>(st, prim, lane, pt, cx, cy, noted, other);
    const bool meets = noted && f.depth == cd[K - 1];
    if (meets && (more || (K > 1 && cd[K - 1] == cd[K > 1 ? K - 2 : 0]) || (MODE == HTGS_MODE_HYBRID_BLEND && f.alpha > 0.99f))) again = true;
    uint32_t last;
    __builtin_memcpy(&last, &ci[K - 1], 4);
    const uint32_t high = last > other ? last : other;
    bool odd = false;
#pragma unroll
    for (int j = 0; j + 1 < K; ++j) {
        uint32_t x;
        __builtin_memcpy(&x, &ci[j], 4);
        odd = odd != (x > high);
    }
    if (meets && !again && (other > last) == odd) {
        swapped(ca[K - 1], f.alpha);
        ca[K - 1] = f.alpha;
        __builtin_memcpy(&ci[K - 1], &other, 4);
    }
    return again;
}
// (the lane and its pixel worked out afresh, so that nothing has to live through the pixels' finish for a rare second walk)
__device__ __forceinline__ uint32_t fresh_lane()
{
    uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    return lane;
}

// The tile's list [first, last) of inst by Gaussian index: spare, into whose stretch of the same place the runs are merged, or inst
// where the list is one run (a frame without bins).  Called by WAVES whole waves (WAVES = 1: by a wave, whatever else its workgroup
// does) of which each merges a range of the indices; more than one synchronises before it reads what the others wrote.  s_runs:
// 1 + kDepthBins words of LDS.  A step looks at the next eight entries of every run: what is not above the least of the runs' eighth
// entries is among the 64, and goes out in its order (28 to 64 entries a step; a list of 500 entries 20 us).
template <int WAVES>
__device__ __forceinline__ const uint32_t *list_in_index_order(const uint32_t *inst, uint32_t first, uint32_t last, uint32_t *spare, uint32_t *s_runs, uint32_t wave,
                                                               uint32_t lane)
{
    static_assert(kDepthBins * 8 == kWave, "eight lanes to a run");
    const auto sync = []() { if (WAVES > 1) __syncthreads(); else wave_lds_sync(); };
    sync();
    if (lane == 0 && wave == 0) s_runs[0] = 0u;
    sync();
    const uint32_t batches = (last - first + 63u) / 64u;
    for (uint32_t b = (uint32_t)((uint64_t)batches * wave / WAVES); b < (uint32_t)((uint64_t)batches * (wave + 1u) / WAVES); ++b) {
        const uint32_t at = first + 64u * b + lane;
        const bool begins = at < last && at > first && inst[at] < inst[at - 1u];
        for (uint64_t m = __ballot(begins); m != 0; m &= m - 1) {              // (wave-uniform)
            if (lane == 0) {
                const uint32_t k = atomicAdd(s_runs, 1u);
                if (k < (uint32_t)kDepthBins - 1u) s_runs[1u + k] = first + 64u * b + (uint32_t)__builtin_ctzll(m);
            }
        }
    }
    sync();
    const uint32_t more = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_runs[0]);
    if (more == 0u || more > (uint32_t)kDepthBins - 1u) return inst;
    // lane r: what is left of run r
    uint32_t at = last, end = last;
    if (lane == 0) at = first;
    uint32_t start = last;
    if (lane >= 1u && lane <= more) start = s_runs[lane];
    uint32_t rank = 0;
    for (uint32_t j = 1; j <= more; ++j) rank += s_runs[j] < start ? 1u : 0u;
    sync();
    if (lane >= 1u && lane <= more) s_runs[1u + rank] = start;                  // (every wave the same)
    sync();
    if (lane >= 1u && lane <= more) at = s_runs[lane];
    if (lane < more) end = s_runs[lane + 1u];
    uint32_t put = first;
    if (WAVES > 1) {
        uint32_t top = lane <= more ? inst[end - 1u] : 0u;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) { const uint32_t v = __shfl_xor(top, d, kWave); top = top > v ? top : v; }
        const uint64_t values = (uint64_t)top + 1u, bounds[2] = { values * wave / WAVES, values * (wave + 1u) / WAVES };
        uint32_t cut[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            uint32_t lo = at, hi = end;
            while (lo < hi) {
                const uint32_t mid = lo + (hi - lo) / 2u;
                if ((uint64_t)inst[mid] < bounds[k]) lo = mid + 1u; else hi = mid;
            }
            cut[k] = lo;
        }
        uint32_t below = cut[0] - at;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) below += __shfl_xor(below, d, kWave);
        put += below;
        at = cut[0]; end = cut[1];
    }
    uint32_t left = end - at;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) left += __shfl_xor(left, d, kWave);
    const uint32_t stop = (uint32_t)__builtin_amdgcn_readfirstlane((int)(put + left));
    put = (uint32_t)__builtin_amdgcn_readfirstlane((int)put);
    while (put < stop) {
        const uint32_t run = lane >> 3, k = lane & 7u;
        const uint32_t from = __shfl(at, (int)run, kWave) + k, to = __shfl(end, (int)run, kWave);
        const bool there = from < to;
        const uint32_t v = there ? inst[from] : 0xffffffffu;
        uint32_t limit = k == 7u && there ? v : 0xffffffffu;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) { const uint32_t o = __shfl_xor(limit, d, kWave); limit = limit < o ? limit : o; }
        const bool goes = there && v <= limit;
        const uint64_t going = __ballot(goes);
        uint32_t place = 0;
        for (uint64_t m = going; m != 0; m &= m - 1) place += (uint32_t)__builtin_amdgcn_readlane((int)v, __builtin_ctzll(m)) < v ? 1u : 0u;
        if (goes) spare[put + place] = v;
        if (lane < (uint32_t)kDepthBins) at += (uint32_t)__popcll(going >> (8u * lane) & 0xffull);
        put += (uint32_t)__popcll(going);
    }
    __threadfence_block();
    return spare;
}

}  // namespace htgs
