// The walks of the three modes with 8x8 tiles (HYBRID_BLEND, ALPHA_BLEND_FIRST_K, OIT_BLEND), the inference kernels with one
// wave per tile and the kernels for tiles with very long lists.  The latter are shared by the inference and the training
// forward pass: what is done with a pixel's finished core, tail or sums is a function object of the launch (Finish), and
// the size of a record of `prim` a template parameter (REC4, in 16-byte words).
// Restates blend_cu of R/include/hybrid_blend/kernels/inference.cuh:78-216,
// R/include/alpha_blend_first_k/kernels/inference.cuh:78-206 and R/include/oit_blend/kernels/inference.cuh:78-177.
#pragma once

#include <type_traits>

#include "blend_common.h"

namespace htgs {

__device__ __forceinline__ void store_pixel(float *__restrict__ image, float *__restrict__ depths, uint32_t w, uint32_t h,
                                            uint32_t x, uint32_t y, bool chw, float r, float g, float b, float depth)
{
    const size_t pix = (size_t)w * y + x, np = (size_t)w * h;
    r = saturate(r); g = saturate(g); b = saturate(b);
    if (chw) { image[pix] = r; image[np + pix] = g; image[2 * np + pix] = b; }
    else { image[3 * pix] = r; image[3 * pix + 1] = g; image[3 * pix + 2] = b; }
    if (depths) depths[pix] = depth;
}

// ---------------------------------------------------------------------------------------------
// HYBRID_BLEND: K nearest fragments with alpha >= 1/20 are alpha-blended in depth order, everything
// else is merged order-independently into one tail fragment behind them.
// ---------------------------------------------------------------------------------------------
// The tail of a pixel: colour sums (every fragment's alpha * colour; the final core's share is taken out when the pixel
// is composited), alpha sum, depth sum and transmittance of what is not in the core.
struct HybridTail {
    float T, c0, c1, c2, alpha, depth;
};
__device__ __forceinline__ void hybrid_tail_init(HybridTail &t) { t.T = 1.0f; t.c0 = t.c1 = t.c2 = t.alpha = t.depth = 0.0f; }
// what joins the tail: a fragment itself, the entry it pushed out of the core, or an empty slot (alpha 0)
template <bool FAST>
__device__ __forceinline__ void hybrid_tail_add(HybridTail &t, float depth, float alpha)
{
    t.alpha += alpha;
    if (!FAST) t.depth = __builtin_fmaf(depth, alpha, t.depth);      // (not used for the median depth)
    t.T *= 1.0f - alpha;
}
template <int K>
__device__ __forceinline__ void hybrid_core_init(float (&cd)[K], float (&ca)[K], float (&ci)[K])
{
#pragma unroll
    for (int i = 0; i < K; ++i) {
        cd[i] = __FLT_MAX__; ca[i] = 0.0f; ci[i] = 0.0f;
        asm volatile("" : "+v"(cd[i]), "+v"(ca[i]), "+v"(ci[i]));      // one register per slot, never a 16-wide tuple
    }
}

// The walk over instances [first, last) of a tile's list (whole batches of 64 from `first` on) by one wave: lanes =
// pixels, by quadrants.  A core slot holds depth, alpha and the Gaussian's index (an exchange moves three registers); the
// colours are fetched once, when the sorted core is blended.  Every fragment's alpha * colour goes into the tail sums
// when it is evaluated, and the share of the fragments that end up in the core is taken out again at the end, so an
// entry pushed out of the core needs no colour: its alpha and depth, which the tail also needs, are in the slot.
// SOLO: the wave is the whole workgroup (its barriers are the workgroup's).
// TIES: `tie` receives what stayed out of the core, or left it, exactly as deep as the entry that is last then.  (A candidate as
// deep as the last entry counts: another wave's share, or a list in bins of depth, may hold one that came before it by index.)
// PIXELS: only the pixels of the lanes in pixel_lanes are wanted; instances that do not reach one of them are left out
// (the other lanes' cores and tails come out incomplete).
// QUICK: insertion by shifting (core_quick_walk), for a caller that settles every pixel at which depths coincide afterwards, also
// where its wave has walked the whole list (6 M Gaussians of the stress scene at 1600x1066: 4940 -> 4865 us, training of 600 k of
// it 2406 -> 2370).
template <int K, bool FAST, bool SOLO, bool TIES = false, bool PIXELS = false, int REC4 = HTGS_PRIM_FLOATS / 4, bool QUICK = false>
__device__ __forceinline__ void hybrid_walk(TileStageQ &st, QuadrantLists &ql, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
                                            uint32_t first, uint32_t last, uint32_t lane, const PixelTerms &pt, float cx, float cy, float (&cd)[K],
                                            float (&ca)[K], float (&ci)[K], HybridTail &tail, CoreTie *tie = nullptr, uint64_t pixel_lanes = 0, ListStep step = 64u)
{
    constexpr int MODE = HTGS_MODE_HYBRID_BLEND;
    constexpr int N = kStageSlots;
    tile_list_walk<MODE, true, PIXELS ? kCullPixels : kCullAlpha, SOLO, REC4, FAST>(st, ql, prim, inst, first, last, lane, cx, cy, [&](uint32_t addr) {
        // cut-off and alpha threshold are tested together: the lanes of a quadrant that its instance does not
        // reach run along to the second test (one exec level less for the scalar unit to manage; the staging
        // cull leaves hardly a turn in which no lane passes, so there is nothing to skip)
        TileFrag f;
        bool fragment;
        if constexpr (FAST) fragment = tile_frag_fast<MODE, N>(addr, pt, f);
        else fragment = tile_frag_exact<MODE, N>(addr, pt, f);
        const float4 col = stage_row<N, 5>(addr);
        if (!fragment) return;
        float depth = tile_frag_depth<N>(addr, pt, f);
        float p3 = f.alpha;
        tail.c0 = __builtin_fmaf(p3, col.x, tail.c0);
        tail.c1 = __builtin_fmaf(p3, col.y, tail.c1);
        tail.c2 = __builtin_fmaf(p3, col.z, tail.c2);
        if ((TIES ? depth <= cd[K - 1] : depth < cd[K - 1]) && f.alpha >= kMinAlphaCore) {
            float pi = col.w;
            if constexpr ((FAST && !TIES) || QUICK) core_quick_walk<K>(depth, p3, pi, cd, ca, ci);
            else core_exchange_walk<K>(depth, p3, pi, cd, ca, ci);
            if (TIES) tie->note(meets_core_end(depth, cd[K - 1]), depth, float_to_bits(pi));
        }
        hybrid_tail_add<FAST>(tail, depth, p3);
    }, pixel_lanes, 1.0f, step);
}

// ---------------------------------------------------------------------------------------------
// HYBRID_BLEND's core as sorted 64-bit keys (the kernel with one wave per tile, inference).  A slot is one register pair:
// the high word holds the depth, the low word alpha as a fraction of 19 to 23 bits (rounded: an absolute error of 2^-20 at
// most, 2^-24 in the tiles with short lists; KeyFormat) above the instance's place in the tile's list (at most 13 bits: the
// lists this kernel walks are no longer than the threshold beyond which a tile goes to the other kernel, at most
// kPackedListMost).  Floats of one sign order like their bit patterns
// and so do the doubles made of (depth, low word): one step of the insertion is slot' = min(carried, slot), carried' =
// max(carried, slot), two instructions without exec masks or moves (a third of the exchange of three registers), and what
// is pushed out carries the alpha that the tail needs.  The Gaussian's index, which only the final core needs, is looked
// up from the place in the list when the pixel is composited.  Which of two fragments of equal depth comes first is
// decided by the low word here, not by the reference's insertion: the image-only fast path leaves it at that; with exact
// arithmetic the walk notes where it can matter (hybrid_key_walk), such pixels are settled from their cores (settle_core), and those
// with more than two fragments of a depth are walked again.
// ---------------------------------------------------------------------------------------------
typedef double CoreKey;
constexpr uint32_t kPackedListMost = 8192;
// How a tile's keys divide the low word (the same for every pixel of the tile: scalar registers).  The place takes the bits
// that the length of the tile's list asks for, nine at least, and alpha the other 19 to 23: a fraction of 23 bits is within
// 2^-24 of the float, so in the tiles with up to 512 instances a key holds its alpha almost as the float does.
struct KeyFormat {
    uint32_t shift, place_mask;     // bits of the place; 2^shift - 1
    float one, one_rcp;             // 2^(32 - shift) - 1, the fraction that stands for alpha = 1, and its reciprocal
};
__device__ __forceinline__ KeyFormat key_format(uint32_t list_length)      // 1 .. kPackedListMost
{
    KeyFormat f;
    f.shift = 32u - (uint32_t)__builtin_clz((list_length - 1u) | 0x1ffu);
    f.place_mask = (1u << f.shift) - 1u;
    f.one = (float)((1u << (32u - f.shift)) - 1u);
    f.one_rcp = 1.0f / f.one;
    return f;
}
__device__ __forceinline__ float key_depth(CoreKey k) { return bits_to_float((uint32_t)__double2hiint(k)); }
__device__ __forceinline__ uint32_t key_low(CoreKey k) { return (uint32_t)__double2loint(k); }
__device__ __forceinline__ CoreKey make_key(float depth, uint32_t low) { return __hiloint2double((int)float_to_bits(depth), (int)low); }
__device__ __forceinline__ uint32_t key_fraction(float alpha, const KeyFormat &f) { return (uint32_t)__builtin_fmaf(alpha, f.one, 0.5f); }      // alpha in [0, 1]
__device__ __forceinline__ uint32_t key_pack(float alpha, uint32_t place, const KeyFormat &f) { return key_fraction(alpha, f) << f.shift | place; }
__device__ __forceinline__ float key_alpha(uint32_t low, const KeyFormat &f) { return (float)(low >> f.shift) * f.one_rcp; }
// What a walk of keys notes of equal depths at the end of a pixel's core: the low words of the last two entries that stayed out of it, or left it,
// exactly as deep as the entry that was last then (0: an empty slot, or none).  Three vector instructions a fragment and no branch; how deep they
// are, and whether they are equally deep, is evaluated after the walk where there is one (noted_ties).  (With the depth and a flag noted behind
// a branch -> so, the launch alone: HYBRID 250 k Gaussians at 1280x720 120.1 -> 112.4 us, 200 k at 1920x1080 214.7 -> 210.1, FIRST_K 137.9 -> 134.9.)
struct KeyNotes {
    uint32_t latest, before;
    __device__ __forceinline__ void init() { latest = before = 0u; }
    __device__ __forceinline__ void note(bool met, uint32_t low)
    {
        before = met ? latest : before;
        latest = met ? low : latest;
    }
};
__device__ __forceinline__ void key_step(CoreKey &carried, CoreKey &slot)
{
    CoreKey out;
    asm("v_max_f64 %0, %2, %1\n\tv_min_f64 %1, %2, %1" : "=&v"(out), "+v"(slot) : "v"(carried));
    carried = out;
}
template <int K>
__device__ __forceinline__ void core_key_walk(CoreKey &carried, CoreKey (&core)[K])
{
#pragma unroll
    for (int g0 = 0; g0 < K; g0 += kInsertGroup) {
        const int g1 = g0 + kInsertGroup < K ? g0 + kInsertGroup : K;
        if (K > kInsertGroup && !__any(key_depth(carried) < key_depth(core[g1 - 1]))) continue;
#pragma unroll
        for (int i = g0; i < g1; ++i) key_step(carried, core[i]);
    }
}
// FAST or not is the arithmetic of a fragment alone.  Without FAST, `tie` receives what stayed out of the core, or left it, exactly as
// deep as the entry that is last then.
template <int K, bool FAST, bool SOLO, int REC4 = HTGS_PRIM_FLOATS / 4, bool AHEAD = false>
__device__ __forceinline__ void hybrid_key_walk(TileStageQ &st, QuadrantLists &ql, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
                                                uint32_t first, uint32_t last, uint32_t lane, const PixelTerms &pt, float cx, float cy,
                                                CoreKey (&core)[K], HybridTail &tail, KeyNotes &notes, const KeyFormat &fmt, uint32_t list_first, ListStep step = 64u)
{
    constexpr int MODE = HTGS_MODE_HYBRID_BLEND;
    constexpr int N = kStageSlots;
    constexpr bool PAIRS = K <= 16;
    // a fragment that passes the tests joins the pixel
    const auto joins = [&](const TileFrag &f, float depth, const float4 &col) {
        float p3 = f.alpha, leaving = p3;
        if ((FAST ? depth < key_depth(core[K - 1]) : depth <= key_depth(core[K - 1])) && p3 >= kMinAlphaCore) {
            // (a fragment that enters the core has the alpha that its key holds from here on: what the colour sums
            // receive now is what is taken out of them again for the entries of the finished core)
            // (the fast path's alpha is opacity * 2^t with the opacity held to 1 and t <= 0 up to the rounding of the staged
            // quadratic: held to 1 here, the fraction has no room for more; the exact path's is held to 1 when it is evaluated)
            if constexpr (FAST) p3 = p3 < 1.0f ? p3 : 1.0f;
            const uint32_t fraction = key_fraction(p3, fmt);
            p3 = (float)fraction * fmt.one_rcp;
            CoreKey carried = make_key(depth, fraction << fmt.shift | (float_to_bits(col.w) - list_first));
            core_key_walk<K>(carried, core);
            depth = key_depth(carried);
            leaving = key_alpha(key_low(carried), fmt);
            if constexpr (!FAST) notes.note(depth == key_depth(core[K - 1]), key_low(carried));
        }
        tail.c0 = __builtin_fmaf(p3, col.x, tail.c0);
        tail.c1 = __builtin_fmaf(p3, col.y, tail.c1);
        tail.c2 = __builtin_fmaf(p3, col.z, tail.c2);
        hybrid_tail_add<FAST>(tail, depth, leaving);
    };
    if constexpr (PAIRS) {
        tile_list_walk<MODE, true, kCullAlpha, SOLO, REC4, FAST, true, AHEAD, true>(st, ql, prim, inst, first, last, lane, cx, cy, [&](uint32_t one, uint32_t two) {
            TileFrag f1, f2;
            bool pass1, pass2;
            if constexpr (FAST) {
                pass1 = tile_frag_fast<MODE, N>(one, pt, f1);
                pass2 = tile_frag_fast<MODE, N>(two, pt, f2);
            } else tile_frag_exact_pair<MODE, N>(one, two, pt, f1, f2, pass1, pass2);
            // (for all lanes: hardly a turn has none that passes)
            const float depth1 = tile_frag_depth<N>(one, pt, f1), depth2 = tile_frag_depth<N>(two, pt, f2);
            const float4 col1 = stage_row<N, 5>(one), col2 = stage_row<N, 5>(two);
            if (pass1) joins(f1, depth1, col1);
            if (pass2) joins(f2, depth2, col2);
        }, 0, 1.0f, step);
    } else {
        tile_list_walk<MODE, true, kCullAlpha, SOLO, REC4, FAST, true, AHEAD>(st, ql, prim, inst, first, last, lane, cx, cy, [&](uint32_t addr) {
            TileFrag f;
            const bool fragment = FAST ? tile_frag_fast<MODE, N>(addr, pt, f) : tile_frag_exact<MODE, N>(addr, pt, f);
            const float4 col = stage_row<N, 5>(addr);
            if (fragment) joins(f, tile_frag_depth<N>(addr, pt, f), col);
        }, 0, 1.0f, step);
    }
}
// the finished keys as the three arrays the composite takes
template <int K>
__device__ __forceinline__ void key_core_unpack(const CoreKey (&core)[K], const uint32_t *__restrict__ inst, uint32_t first, uint32_t last, float (&cd)[K],
                                                float (&ca)[K], float (&ci)[K], const KeyFormat &fmt)
{
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const uint32_t low = key_low(core[i]), place = low & fmt.place_mask;
        cd[i] = key_depth(core[i]);
        ca[i] = key_alpha(low, fmt);
        ci[i] = ca[i] > 0.0f && first + place < last ? bits_to_float(inst[first + place]) : 0.0f;
    }
}

// The notes of a walk with the depth they are at; `other` is the place in the tile's list.  (The walk's last depth never grows: the latest note is the
// least deep.)
template <int MODE, int REC4>
__device__ __forceinline__ CoreTie noted_ties(TileStageQ &st, const float4 *__restrict__ prim, const uint32_t *__restrict__ inst, uint32_t first, uint32_t last, uint32_t lane,
                                              const TilePixel &px, const KeyNotes &notes, const KeyFormat &fmt)
{
    CoreTie tie;
    tie.init();
    const uint32_t place = notes.latest & fmt.place_mask, place_before = notes.before & fmt.place_mask;
    const bool noted = px.inside && notes.latest >> fmt.shift != 0u && first + place < last;
    if (!__any(noted)) return tie;
    const float depth = tie_fragment<MODE, REC4>(st, prim, lane, px.pt, px.cx, px.cy, noted, noted ? inst[first + place] : 0u).depth;
    const bool twice = noted && notes.before >> fmt.shift != 0u && first + place_before < last;
    bool more = false;
    if (__any(twice))
        more = tie_fragment<MODE, REC4>(st, prim, lane, px.pt, px.cx, px.cy, twice, twice ? inst[first + place_before] : 0u).depth == depth && twice;
    if (noted) {
        tie.depth = depth;
        tie.other = place | (more ? kMoreTied : 0u);
    }
    return tie;
}
// settle_core of a core of keys, before it is unpacked: nearly every wave has no two equal depths that matter and is through after a compare for each
// slot, and where one has, the keys, the indices that the pairs and the parity take and then the staged record are not all held at once.
// (From the unpacked core, with the tail and the record beside it, the kernels with K = 16 spilled 43 and 57 registers instead of 30 and
// 31, also for the waves without a tie, and K = 32 took 291 us for 300 k Gaussians at 1280x720 instead of 274.)
template <int MODE, int K, int REC4, typename Swapped>
__device__ __forceinline__ bool settle_keys(TileStageQ &st, const float4 *__restrict__ prim, const uint32_t *__restrict__ inst, uint32_t first, uint32_t last, uint32_t lane,
                                            const TilePixel &px, CoreKey (&core)[K], const CoreTie &tie, const KeyFormat &fmt, Swapped &&swapped)
{
    const auto equal = [&](int i) { return key_low(core[i + 1]) >> fmt.shift != 0u && key_depth(core[i]) == key_depth(core[i + 1]); };
    const auto held = [&](uint32_t place, bool is) { return is && first + place < last ? inst[first + place] : 0u; };
    const uint32_t place = tie.other & ~kMoreTied;
    const bool noted = px.inside && tie.at_end(key_depth(core[K - 1])) && first + place < last;
    bool pairs = false;
#pragma unroll
    for (int i = 0; i + 1 < K; ++i) pairs = pairs || equal(i);
    pairs = pairs && px.inside;
    if (!__any(pairs || noted)) return false;
    bool again = false, stays;
    const uint32_t other = held(place, noted);
    {
        uint32_t x[K];
#pragma unroll
        for (int i = 0; i < K; ++i) x[i] = held(key_low(core[i]) & fmt.place_mask, key_low(core[i]) >> fmt.shift != 0u);
        const auto odd_above = [&](int n, uint32_t high) {
            bool odd = false;
#pragma unroll
            for (int j = 0; j < K; ++j)
                if (j < n) odd = odd != (x[j] > high);
            return odd;
        };
#pragma unroll
        for (int i = 0; i + 1 < K; ++i) {
            const bool here = pairs && equal(i);
            if (!__any(here)) continue;
            if (i + 2 < K) again = again || (here && equal(i + 2 < K ? i + 1 : i));
            if (here && (x[i] > x[i + 1]) != odd_above(i, x[i] > x[i + 1] ? x[i] : x[i + 1])) {
                const uint32_t low = key_low(core[i]), y = x[i];
                core[i] = make_key(key_depth(core[i]), key_low(core[i + 1])); x[i] = x[i + 1];
                core[i + 1] = make_key(key_depth(core[i + 1]), low); x[i + 1] = y;
            }
        }
        stays = (other > x[K - 1]) != odd_above(K - 1, other > x[K - 1] ? other : x[K - 1]);
    }
    if (!__any(noted)) return again;
    const TieFragment f = tie_fragment<MODE, REC4>(st, prim, lane, px.pt, px.cx, px.cy, noted, other);
    const bool meets = noted && f.depth == key_depth(core[K - 1]);
    if (meets && ((tie.other & kMoreTied) != 0u || (K > 1 && key_depth(core[K - 1]) == key_depth(core[K > 1 ? K - 2 : 0])) || (MODE == HTGS_MODE_HYBRID_BLEND && f.alpha > 0.99f)))
        again = true;
    if (meets && !again && !stays) {
        const uint32_t fraction = key_fraction(f.alpha, fmt);
        swapped(key_alpha(key_low(core[K - 1]), fmt), (float)fraction * fmt.one_rcp);
        core[K - 1] = make_key(key_depth(core[K - 1]), fraction << fmt.shift | place);
    }
    return again;
}
// a fragment of the tail's takes the place of another one of the same depth
__device__ __forceinline__ auto tail_swap(HybridTail &t, float depth)
{
    return [&t, depth](float in, float out) {
        t.alpha += in - out;
        t.depth = __builtin_fmaf(depth, in - out, t.depth);
        t.T *= (1.0f - in) / (1.0f - out);
    };
}
// settle_core of the walks by insertion
template <int MODE, int K, int REC4, typename IndexT, typename Swapped>
__device__ __forceinline__ bool settle_exact_core(TileStageQ &st, const float4 *__restrict__ prim, uint32_t lane, const TilePixel &px, float (&cd)[K], float (&ca)[K],
                                                  IndexT (&ci)[K], const CoreTie &tie, Swapped &&swapped)
{
    return settle_core<MODE, K, REC4>(st, prim, lane, px.pt, px.cx, px.cy, cd, ca, ci, px.inside && tie.at_end(cd[K - 1]), tie.other & ~kMoreTied,
                                      (tie.other & kMoreTied) != 0u, swapped);
}

// core + tail -> pixel (R/include/hybrid_blend/kernels/inference.cuh:172-213)
template <int K, int REC4 = HTGS_PRIM_FLOATS / 4>
__device__ __forceinline__ void hybrid_composite(const float4 *__restrict__ prim, float (&cd)[K], float (&ca)[K], float (&ci)[K], HybridTail &tail,
                                                 float *__restrict__ image, float *__restrict__ depths, uint32_t width, uint32_t height,
                                                 uint32_t x, uint32_t y, int chw, int median)
{
    constexpr int MODE = HTGS_MODE_HYBRID_BLEND;
    float tail0 = tail.c0, tail1 = tail.c1, tail2 = tail.c2;
    const float tail3 = tail.alpha, depth_tail = tail.depth, T_tail = tail.T;
    float r = 0.0f, g = 0.0f, b = 0.0f, depth_pixel = 0.0f, T_core = 1.0f;
    float4 cc[K];
#pragma unroll
    for (int i = 0; i < K; ++i)
        cc[i] = ca[i] > 0.0f ? prim[(size_t)float_to_bits(ci[i]) * REC4 + 4] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int i = 0; i < K; ++i) {                      // the core's share of the colour sums
        tail0 = __builtin_fmaf(-ca[i], cc[i].x, tail0);
        tail1 = __builtin_fmaf(-ca[i], cc[i].y, tail1);
        tail2 = __builtin_fmaf(-ca[i], cc[i].z, tail2);
    }
    tail0 = clamp_pos(tail0); tail1 = clamp_pos(tail1); tail2 = clamp_pos(tail2);   // colours are >= 0, so is the exact difference
#pragma unroll
    for (int i = 0; i < K; ++i) {
        if (T_core >= kTransmittanceThreshold) {
            const float w = T_core * ca[i];
            r = __builtin_fmaf(w, cc[i].x, r);
            g = __builtin_fmaf(w, cc[i].y, g);
            b = __builtin_fmaf(w, cc[i].z, b);
            if (median) depth_pixel = (T_core > 0.5f && cd[i] < __FLT_MAX__) ? cd[i] : depth_pixel;
            else depth_pixel = __builtin_fmaf(w, cd[i], depth_pixel);
            T_core *= 1.0f - ca[i];
        }
    }
    float total_alpha = 0.0f;
    if (!median) total_alpha = 1.0f - T_core;
    if (T_core >= kTransmittanceThreshold && tail3 >= ModeCfg<MODE>::min_alpha) {
        const float weight_tail = T_core * (1.0f - T_tail);
        const float wn = weight_tail * (1.0f / tail3);
        r = __builtin_fmaf(wn, tail0, r);
        g = __builtin_fmaf(wn, tail1, g);
        b = __builtin_fmaf(wn, tail2, b);
        if (!median) { depth_pixel = __builtin_fmaf(wn, depth_tail, depth_pixel); total_alpha += weight_tail; }
    }
    if (!median) depth_pixel = total_alpha > 0.0f ? depth_pixel / total_alpha : 0.0f;
    store_pixel(image, depths, width, height, x, y, chw, r, g, b, depth_pixel);
}

// what the inference kernels do with a pixel's finished core and tail: composite and store
struct HybridImage {
    float *image, *depths;
    uint32_t width, height;
    int chw, median;
    template <int K>
    __device__ __forceinline__ void operator()(const float4 *__restrict__ prim, uint32_t, const TilePixel &px, float (&cd)[K], float (&ca)[K], float (&ci)[K],
                                               HybridTail &tail) const
    {
        hybrid_composite<K>(prim, cd, ca, ci, tail, image, depths, width, height, px.x, px.y, chw, median);
    }
};

// One tile by one wave with the core as keys; finish(prim, tile, px, cd, ca, ci, tail) is called once per pixel inside the
// image.  Without FAST, the pixels at which fragments of exactly equal depth met where they decide the core (a pixel or
// two in a tile in a hundred) are settled from it, and where more than two are as deep as each other walked again afterwards, over
// the instances that reach one of them, with the reference's insertion.
template <int K, bool FAST, int REC4, typename Finish>
__device__ __forceinline__ void hybrid_tile_by_keys(TileStageQ &st, QuadrantLists &ql, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
                                                    uint32_t tile, uint32_t first, uint32_t last, uint32_t lane, const TilePixel &px, uint32_t grid_w,
                                                    uint32_t width, uint32_t height, uint32_t *__restrict__ spare, const Finish &finish)
{
    HybridTail tail;
    hybrid_tail_init(tail);
    float cd[K], ca[K], ci[K];                 // ci: the index's bit pattern
    CoreKey core[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        core[i] = make_key(__FLT_MAX__, 0u);
        asm volatile("" : "+v"(core[i]));      // one register pair per slot, never a wide tuple
    }
    KeyNotes notes;
    notes.init();
    const KeyFormat fmt = key_format(last > first ? last - first : 1u);
    hybrid_key_walk<K, FAST, true, REC4, true>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, core, tail, notes, fmt, first);
    if constexpr (FAST) {
        if (!px.inside) return;
        key_core_unpack<K>(core, inst, first, last, cd, ca, ci, fmt);
        finish(prim, tile, px, cd, ca, ci, tail);
    } else {
        const CoreTie tie = noted_ties<HTGS_MODE_HYBRID_BLEND, REC4>(st, prim, inst, first, last, lane, px, notes, fmt);
        const bool again = settle_keys<HTGS_MODE_HYBRID_BLEND, K, REC4>(st, prim, inst, first, last, lane, px, core, tie, fmt, tail_swap(tail, key_depth(core[K - 1])));
        const uint64_t again_lanes = __ballot(again);
        key_core_unpack<K>(core, inst, first, last, cd, ca, ci, fmt);
        if (px.inside && !again) finish(prim, tile, px, cd, ca, ci, tail);
        if (again_lanes == 0) return;
        // (the lane and its pixel are worked out afresh, so that nothing the first walk keeps in registers has to
        // live through the pixels' finish for the sake of this rare second walk)
        uint32_t lane_again = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(lane_again));
        const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
        const uint32_t *const list = spare != nullptr ? list_in_index_order<1>(inst, first, last, spare, ql.a[0], 0u, lane_again) : inst;
        hybrid_tail_init(tail);
        hybrid_core_init<K>(cd, ca, ci);
        hybrid_walk<K, false, true, false, true, REC4>(st, ql, list, prim, first, last, lane_again, px_again.pt, px_again.cx, px_again.cy, cd, ca, ci, tail, nullptr,
                                                       again_lanes);
        if ((again_lanes >> lane_again & 1ull) != 0) finish(prim, tile, px_again, cd, ca, ci, tail);
    }
}

// ---------------------------------------------------------------------------------------------
// Several waves share a list, every WAVES-th batch of it each: what each has walked is merged pairwise.  Two sorted cores are merged without
// insertions: the nearer of entry i of one and entry K - 1 - i of the other are the K nearest of both (what is farther
// joins the tail), in an order that log2 K rounds of compare and exchange sort -- K = 16: 48 exchanges of 28 cycles (8 for
// keys), where inserting sixteen entries one by one takes 9000 cycles.  Which entry of exactly equal depth stays is not the
// reference's choice then: the merges note what was left out exactly as deep as the last entry that stays, as the walks do.
// ---------------------------------------------------------------------------------------------
// LDS of a workgroup whose waves walk shares and then hand them on, ROWS rows of 64 lanes a share: the merge buffers, one
// per pair of waves, lie over the stages.
template <int WAVES, uint32_t ROWS> constexpr size_t shared_walk_lds()
{
    constexpr size_t stages = WAVES * (sizeof(TileStageQ) + ((sizeof(QuadrantLists) + 15) & ~(size_t)15)), buffers = (WAVES / 2) * (size_t)ROWS * 64 * 4;
    return stages > buffers ? stages : buffers;
}
__device__ __forceinline__ TileStageQ &wave_stage(unsigned char *lds, uint32_t wave) { return reinterpret_cast<TileStageQ *>(lds)[wave]; }
template <int WAVES>
__device__ __forceinline__ QuadrantLists &wave_lists(unsigned char *lds, uint32_t wave)
{
    return *reinterpret_cast<QuadrantLists *>(lds + WAVES * sizeof(TileStageQ) + wave * ((sizeof(QuadrantLists) + 15) & ~(size_t)15));
}

// sorts a bitonic sequence of K keys
template <int K>
__device__ __forceinline__ void sort_bitonic(CoreKey (&core)[K])
{
#pragma unroll
    for (int half = K / 2; half > 0; half /= 2) {
#pragma unroll
        for (int i = 0; i < K; ++i)
            if ((i & half) == 0) {
                CoreKey lo, hi;
                asm("v_min_f64 %0, %2, %3\n\tv_max_f64 %1, %2, %3" : "=&v"(lo), "=&v"(hi) : "v"(core[i]), "v"(core[i + half]));
                core[i] = lo;
                core[i + half] = hi;
            }
    }
}
// The least deep of the entries that a merge of two cores pushes out, and the next (an empty slot has the largest depth): four instructions for
// each.  (With the flag worked out on the way, eight, and a row more of what
// a part of a list leaves: long lists of the weights of 600 k Gaussians of the stress scene at 309x378, FIRST_K K = 32 467 -> 451 us, HYBRID K = 16 313 -> 309.)
struct LeastPushed {
    float least = __FLT_MAX__, next = __FLT_MAX__;
    uint32_t index = 0u;
    __device__ __forceinline__ void add(float depth, uint32_t x)
    {
        index = depth < least ? x : index;
        next = __builtin_amdgcn_fmed3f(depth, least, next);
        least = depth < least ? depth : least;
        asm volatile("" : "+v"(index), "+v"(next), "+v"(least));      // (now, not for all entries at the end: that took a hundred scalar registers)
    }
    __device__ __forceinline__ void join(CoreTie &tie, float last_depth) const
    {
        if (least == last_depth) tie.join(CoreTie{ least, index | (next == least ? kMoreTied : 0u) });
    }
};
// A core of keys joins the running one; pushed(key) is called with every entry that is in neither's K nearest.  tie: see above.
template <int K, bool TIES, typename Pushed>
__device__ __forceinline__ void merge_key_cores(const float *from, CoreKey (&core)[K], CoreTie &tie, const KeyFormat &fmt, Pushed &&pushed)
{
    LeastPushed left;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const CoreKey other = __hiloint2double((int)float_to_bits(from[(2 * (K - 1 - i)) * 64]), (int)float_to_bits(from[(2 * (K - 1 - i) + 1) * 64]));
        CoreKey lo, hi;
        asm("v_min_f64 %0, %2, %3\n\tv_max_f64 %1, %2, %3" : "=&v"(lo), "=&v"(hi) : "v"(core[i]), "v"(other));
        core[i] = lo;
        if (TIES) left.add(key_depth(hi), key_low(hi) & fmt.place_mask);
        pushed(hi);
    }
    sort_bitonic<K>(core);
    if (TIES) left.join(tie, key_depth(core[K - 1]));
}
// the same for cores of three registers a slot (an empty slot has alpha 0 and the largest depth)
template <typename IndexT>
__device__ __forceinline__ void order_entries(float &d0, float &a0, IndexT &i0, float &d1, float &a1, IndexT &i1)
{
    const bool swap = d1 < d0;
    const float d = swap ? d1 : d0, a = swap ? a1 : a0;
    const IndexT x = swap ? i1 : i0;
    d1 = swap ? d0 : d1; a1 = swap ? a0 : a1; i1 = swap ? i0 : i1;
    d0 = d; a0 = a; i0 = x;
}
template <int K, bool TIES, typename IndexT, typename Pushed>
__device__ __forceinline__ void merge_cores(const float *from, float (&cd)[K], float (&ca)[K], IndexT (&ci)[K], CoreTie &tie, Pushed &&pushed)
{
    LeastPushed left;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        float d = from[(3 * (K - 1 - i)) * 64], a = from[(3 * (K - 1 - i) + 1) * 64];
        IndexT x;
        const float bits = from[(3 * (K - 1 - i) + 2) * 64];
        __builtin_memcpy(&x, &bits, 4);
        order_entries(cd[i], ca[i], ci[i], d, a, x);
        if (TIES) {
            uint32_t index;
            __builtin_memcpy(&index, &x, 4);
            left.add(d, index);
        }
        pushed(d, a);
        asm volatile("" : "+v"(cd[i]), "+v"(ca[i]), "+v"(ci[i]));
    }
#pragma unroll
    for (int half = K / 2; half > 0; half /= 2) {
#pragma unroll
        for (int i = 0; i < K; ++i)
            if ((i & half) == 0) order_entries(cd[i], ca[i], ci[i], cd[i + half], ca[i + half], ci[i + half]);
    }
    if (TIES) left.join(tie, cd[K - 1]);
}
template <int K, typename IndexT>
__device__ __forceinline__ void give_core(float *to, const float (&cd)[K], const float (&ca)[K], const IndexT (&ci)[K])
{
#pragma unroll
    for (int i = 0; i < K; ++i) {
        float bits;
        __builtin_memcpy(&bits, &ci[i], 4);
        to[(3 * i) * 64] = cd[i]; to[(3 * i + 1) * 64] = ca[i]; to[(3 * i + 2) * 64] = bits;
    }
}
template <int K>
__device__ __forceinline__ void give_key_core(float *to, const CoreKey (&core)[K])
{
#pragma unroll
    for (int i = 0; i < K; ++i) {
        to[(2 * i) * 64] = key_depth(core[i]);
        to[(2 * i + 1) * 64] = bits_to_float(key_low(core[i]));
    }
}
template <int ROW>
__device__ __forceinline__ void give_tail(float *to, const HybridTail &t)
{
    to[ROW * 64] = t.T; to[(ROW + 1) * 64] = t.c0; to[(ROW + 2) * 64] = t.c1; to[(ROW + 3) * 64] = t.c2; to[(ROW + 4) * 64] = t.alpha; to[(ROW + 5) * 64] = t.depth;
}
template <int ROW>
__device__ __forceinline__ void take_tail(const float *from, HybridTail &t)
{
    t.T *= from[ROW * 64];
    t.c0 += from[(ROW + 1) * 64]; t.c1 += from[(ROW + 2) * 64]; t.c2 += from[(ROW + 3) * 64]; t.alpha += from[(ROW + 4) * 64]; t.depth += from[(ROW + 5) * 64];
}
// A note in one row: it is of use if it is as deep as the core's last entry, whose depth is in the core (from row LAST on).
constexpr uint32_t kNoTie = ~0u;
template <int ROW>
__device__ __forceinline__ void give_tie(float *to, const CoreTie &tie, float last_depth) { to[ROW * 64] = bits_to_float(tie.at_end(last_depth) ? tie.other : kNoTie); }
template <int ROW, int LAST>
__device__ __forceinline__ void take_tie(const float *from, CoreTie &tie)
{
    const uint32_t other = float_to_bits(from[ROW * 64]);
    tie.join(CoreTie{ other != kNoTie ? from[LAST * 64] : __FLT_MAX__, other });
}
// ---------------------------------------------------------------------------------------------
// Tiles with very long lists (HYBRID_BLEND, ALPHA_BLEND_FIRST_K and OIT_BLEND, which walk all of a list): the kernel
// with one wave per tile puts a tile whose list is longer than long_threshold on a list instead of walking it, if the
// caller provided that list, and a second launch of workgroups of several waves takes those: one wave walks one tile at some
// 200 ns per instance once it has a SIMD to itself, so a single list of 300 000 instances would otherwise hold the
// launch for 70 ms.
// long_tiles[0] = entries on the list, [1..3] = work counters, [4] = workgroups done, all zeroed with the
// ranges and again by the last workgroup of the second launch; [5] = the threshold, if it was chosen on the device
// (ListThreshold); [6], [7] = tiles with pixels settled from their cores or by a second look / walked again in one piece (upper half: of these,
// after a second look that ran out of room) since the ranges were made (for the tests); then 2 n_tiles words for the entries (tile | part << 20 |
// (parts - 1) << 25: a tile is on the list once per part, and the parts beyond the first of all tiles together are held
// to n_tiles, so the list cannot overflow) and n_tiles words that count a tile's finished parts.
// ---------------------------------------------------------------------------------------------
constexpr uint32_t kLongHeader = 8, kLongRounds = 3, kLongParts = 32;
constexpr int kLongWavesHeld = 16;        // waves that a compute unit holds of these kernels
// calls launch(std::integral_constant<int, long_waves_of(f)>) for a core of K entries
template <int K, typename Launch>
inline void with_long_waves(const htgs_frame *f, Launch &&launch)
{
    if constexpr (K <= 16) {
        if (long_waves_of(f) == 16u) { launch(std::integral_constant<int, 16>{}); return; }
    }
    launch(std::integral_constant<int, 8>{});
}
constexpr unsigned long_grid(int waves) { return 256u * (unsigned)(kLongWavesHeld / waves); }

// What a workgroup leaves of its part of a list, in 64-lane rows: HYBRID's core, tail and what met at its end.
template <int K> constexpr uint32_t long_part_words() { return (3u * K + 7u) * 64u; }
// The parts a list of this length is walked in by separate workgroups (1: by one).  A part is at least part_least
// long (least_part), long enough that what the parts leave behind (part_words each) fits into the list's own stretch of
// the spare value buffer, and at least as long as the frame's average list (part_floor = instances / tiles, rounded
// up): the parts beyond the first of all tiles together then cannot exceed the number of tiles, which is what the list
// of entries has room for, and how a list is split is a function of its length and of the frame alone -- no budget
// shared between workgroups, nothing that depends on the order in which they run.
__device__ __forceinline__ uint32_t long_parts(uint32_t length, uint32_t part_least, uint32_t part_words, uint32_t part_floor)
{
    uint32_t least = part_least > part_words ? part_least : part_words;
    least = least > part_floor ? least : part_floor;
    const uint32_t parts = length / least;
    return parts < 1u ? 1u : parts > kLongParts ? kLongParts : parts;
}
// With htgs_frame.long_counters every die has work counters of its own.  An atomic on a line that another die's cache holds
// takes 0.1 us and the next one waits for it: with one counter for all, a list of 2000 entries cost three rounds of 2000 such
// atomics (weights of 2.9 M Gaussians at 1416x701, OIT: 1430 us of a kernel that has next to nothing to walk; now 270).
// (one lane of the tile's wave) enters the tile; part_floor = 0: in one part
__device__ __forceinline__ void long_tile_enter(uint32_t *__restrict__ long_tiles, uint32_t tile, uint32_t n_tiles, uint32_t length,
                                                uint32_t part_least, uint32_t part_words, uint32_t part_floor, uint32_t long_threshold, uint32_t *counters)
{
    const uint32_t parts = part_floor != 0u ? long_parts(length, part_least, part_words, part_floor) : 1u;
    if (parts > 1u) long_tiles[kLongHeader + 2u * n_tiles + tile] = 0u;
    if (counters != nullptr) {
        // (no part is longer than this; its class and the ones below it, which the other parts may be of)
        const uint32_t longest = length / parts + 128u;
        if (longest > 16u * long_threshold) counters[kDieRounds] = 1u;
        if (longest > 4u * long_threshold) counters[kDieRounds + 1u] = 1u;
    }
    const uint32_t at = kLongHeader + atomicAdd(long_tiles, parts);
    for (uint32_t part = 0; part < parts; ++part) long_tiles[at + part] = tile | part << 20 | (parts - 1u) << 25;
}
// An entry of the list: part `part` of `parts` of the tile's list [tile_first, tile_last) is [first, last), whole batches of 64.
struct LongEntry {
    uint32_t tile, part, parts, tile_first, tile_last, first, last;
};
// The workgroups take the entries off the list one by one, the longest first: the list is gone through kLongRounds times
// (a counter per round, `round` starts at 0), and a round takes the entries of its length class only -- more than 16, more
// than 4 and up to 4 times the threshold.  The lists differ in length by orders of magnitude, and the launch ends when the
// workgroup with the longest one does.  With counters every die's workgroups go through every eighth entry, and a round
// whose class no entry is of is left out.  Called by all threads of the workgroup (barriers inside); false: the list is
// through.  The last workgroup to find that clears the list's header and the counters, so that the list is empty again for
// the next blend of this frame (htgs_blend called again without htgs_extract_ranges).
__device__ __forceinline__ bool long_tile_take(const uint32_t *long_tiles, const uint32_t *__restrict__ ranges, uint32_t long_threshold,
                                               uint32_t *counters, uint32_t &round, uint32_t *s_next, LongEntry &e)
{
    const uint32_t n_long = long_tiles[0];
    // (a launch of fewer workgroups than dies: as many shares of the list as workgroups)
    const uint32_t shares = counters == nullptr ? 1u : gridDim.x < kDies ? gridDim.x : kDies, share = blockIdx.x % shares;
    uint32_t *const line = counters != nullptr ? counters + kDieLine * share : const_cast<uint32_t *>(long_tiles) + 1;
    for (;;) {
        if (counters != nullptr)
            while (round + 1u < kLongRounds && counters[kDieRounds + round] == 0u) ++round;
        __syncthreads();
        if (threadIdx.x == 0) *s_next = atomicAdd(line + round, 1u);
        __syncthreads();
        const uint32_t j = shares * (uint32_t)__builtin_amdgcn_readfirstlane((int)*s_next) + share;     // (the same in every lane: what follows stays in scalar registers)
        if (j >= n_long) {
            if (++round < kLongRounds) continue;
            if (threadIdx.x == 0) {
                uint32_t *header = const_cast<uint32_t *>(long_tiles);
                __threadfence();
                bool last = atomicAdd(line + kLongRounds, 1u) == (gridDim.x - share + shares - 1u) / shares - 1u;
                if (last && counters != nullptr) last = atomicAdd(counters + kDieRounds + kLongRounds, 1u) == shares - 1u;
                if (last) {
#pragma unroll
                    for (uint32_t k = 0; k < 5; ++k) header[k] = 0u;
                    if (counters != nullptr)
                        for (uint32_t d = 0; d <= kDies; ++d)
#pragma unroll
                            for (uint32_t k = 0; k <= kLongRounds; ++k) counters[kDieLine * d + k] = 0u;
                }
            }
            return false;
        }
        const uint32_t entry = long_tiles[kLongHeader + j];
        e.tile = entry & 0xfffffu; e.part = entry >> 20 & 31u; e.parts = (entry >> 25) + 1u;
        e.tile_first = ranges[2 * e.tile]; e.tile_last = ranges[2 * e.tile + 1];
        const uint32_t tile_batches = (e.tile_last - e.tile_first + 63u) / 64u;
        e.first = e.tile_first + 64u * (uint32_t)((uint64_t)tile_batches * e.part / e.parts);
        e.last = e.tile_first + 64u * (uint32_t)((uint64_t)tile_batches * (e.part + 1u) / e.parts);
        e.last = e.last < e.tile_last ? e.last : e.tile_last;
        const uint32_t length = e.last - e.first;
        const uint32_t length_class = length > 16u * long_threshold ? 0u : length > 4u * long_threshold ? 1u : 2u;
        if (length_class == round) return true;
    }
}
// share of wave `wave` of [first, last): whole batches of 64
__device__ __forceinline__ void long_wave_share(uint32_t first, uint32_t last, uint32_t wave, uint32_t &share_first, uint32_t &share_last,
                                                uint32_t waves)
{
    const uint32_t n_batches = (last - first + 63u) / 64u;
    share_first = first + 64u * (uint32_t)((uint64_t)n_batches * wave / waves);
    share_last = first + 64u * (uint32_t)((uint64_t)n_batches * (wave + 1) / waves);
    share_last = share_last < last ? share_last : last;
}
// One of several parts is done and the first wave has written what it left (and called __threadfence()): whether the
// other parts are there already, so that this workgroup ends the tile.  Called by all threads; the first wave calls
// __threadfence() again before it reads the other parts.
__device__ __forceinline__ bool long_part_done(const uint32_t *long_tiles, uint32_t n_tiles, const LongEntry &e, uint32_t *s_whole)
{
    if (threadIdx.x == 0) *s_whole = atomicAdd(const_cast<uint32_t *>(long_tiles) + kLongHeader + 2u * n_tiles + e.tile, 1u) == e.parts - 1u;
    __syncthreads();
    return *s_whole != 0;
}

// One wave per tile; the tiles with very long lists are left to blend_hybrid_long_kernel.
// KEYS (with long_tiles and a threshold of no more than kPackedListMost): the core as sorted 64-bit keys, hybrid_tile_by_keys.
// (K = 32: two registers a slot leave room for four waves per SIMD instead of three -- cfg2 442 -> 488 FPS)
template <int K, bool FAST, bool KEYS = false>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(K <= 16 ? 5 : KEYS ? 4 : 3))) blend_hybrid_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
    float *__restrict__ image, float *__restrict__ depths, uint32_t width, uint32_t height, uint32_t grid_w, int chw, int median,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare)
{
    __shared__ TileStageQ st;
    __shared__ QuadrantLists ql;
    const uint32_t tile = block_tile(tile_order);
    const uint32_t lane = threadIdx.x;
    const uint32_t first = ranges[2 * tile], last = ranges[2 * tile + 1];
    const uint32_t long_threshold = threshold.get(long_tiles);
    if (long_tiles != nullptr && last - first > long_threshold) {
        if (lane == 0) long_tile_enter(long_tiles, tile, gridDim.x, last - first, threshold.least_part(long_threshold), long_part_words<K>(), part_floor.get(gridDim.x), long_threshold, threshold.counters);
        return;
    }
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    if constexpr (KEYS) {
        hybrid_tile_by_keys<K, FAST, HTGS_PRIM_FLOATS / 4>(st, ql, inst, prim, tile, first, last, lane, px, grid_w, width, height, spare,
                                                           HybridImage{ image, depths, width, height, chw, median });
    } else {
        HybridTail tail;
        hybrid_tail_init(tail);
        float cd[K], ca[K], ci[K];                 // ci: the index's bit pattern
        hybrid_core_init<K>(cd, ca, ci);
        hybrid_walk<K, FAST, true>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, cd, ca, ci, tail);
        if (!px.inside) return;
        hybrid_composite<K>(prim, cd, ca, ci, tail, image, depths, width, height, px.x, px.y, chw, median);
    }
}

__device__ __forceinline__ float wave_total(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ float wave_product(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v *= __shfl_xor(v, o);
    return v;
}
// (out of line: the kernels for long lists have no scalar registers left for it)
template <int WAVES>
__device__ __attribute__((noinline)) const uint32_t *list_in_index_order_by(const uint32_t *inst, uint32_t first, uint32_t last, uint32_t *spare, uint32_t *s_runs, uint32_t wave,
                                                                            uint32_t lane)
{
    return list_in_index_order<WAVES>(inst, first, last, spare, s_runs, wave, lane);
}
constexpr int kAgainPixels = 2;       // pixels a pass of pixels_again takes at once
constexpr int kAgainMost = 8;         // pixels of a tile beyond which they are walked again in one piece instead
constexpr uint32_t kAgainEntries = 1024;        // entries of pixels_again, of all waves, beyond which so are they
// The entries of pixels_again by Gaussian index, or as they are listed (one wave): returns their offsets in `entries`, listed[w] of them
// from from(w) on, in LDS.
template <int WAVES, bool BY_INDEX, typename From>
__device__ __forceinline__ const uint32_t *entries_in_order(const uint32_t *entries, const uint32_t *listed, uint32_t *lds, uint32_t lane, uint32_t &total, From &&from)
{
    uint32_t *const index = lds, *const at = lds + kAgainEntries, *const ordered = lds + 2u * kAgainEntries;
    total = 0;
#pragma nounroll
    for (uint32_t w = 0; w < (uint32_t)WAVES; ++w) {
        const uint32_t n = listed[w], start = from(w);
        for (uint32_t e = lane; e < n; e += 64u) {
            at[total + e] = start + 4u * e;
            index[total + e] = entries[start + 4u * e + 3u];
        }
        total += n;
    }
    wave_lds_sync();
    if (!BY_INDEX) return at;
    for (uint32_t e = lane; e < total; e += 64u) {
        const uint32_t mine = index[e];
        uint32_t rank = 0;
        for (uint32_t j = 0; j < total; ++j) rank += index[j] < mine || (index[j] == mine && j < e) ? 1u : 0u;
        ordered[rank] = at[e];
    }
    wave_lds_sync();
    return ordered;
}

// The second look at the pixels of pixel_lanes, whose cores the merge could not settle: lanes = instances.  Every wave
// goes through its share [first, last) of the tile's list once per kAgainPixels pixels and evaluates each instance at these
// pixels with the walk's own arithmetic.  A fragment that cannot be in the pixel's final core -- farther than the merged
// core's last entry (last_depth[pixel]: which depths the K nearest have is certain, which fragments of equal depth they
// are is not), or too faint for the core -- joins the pixel's tail in sums[][j] (this wave's sums and product, to be combined
// over the waves; the colour sums take every fragment); the others, the few that decide the core, are put down in list
// order at `out` as (pixel, depth, alpha, index) for the walk's insertion to be replayed on them alone.  Returns their
// number, or ~0u when `room` entries were not enough.  pass_done(pixels) is called, by the whole workgroup, after each pass.
// ALPHA_BLEND_FIRST_K has no tail: its fragments that are not farther than the core's last entry are put down, no sums.
template <int MODE, bool FAST, int REC4, typename PassDone>
__device__ __forceinline__ uint32_t pixels_again(TileStage<64> &st, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t first,
                                                        uint32_t last, uint32_t lane, float cx, float cy, uint64_t pixel_lanes,
                                                        const float *last_depth, float (*sums)[6], uint32_t *__restrict__ out, uint32_t room,
                                                        PassDone pass_done)
{
    constexpr bool kTail = MODE == HTGS_MODE_HYBRID_BLEND;
    uint32_t n_out = 0;
    bool fits = true;
    for (uint64_t todo = pixel_lanes; todo != 0;) {
        uint32_t pixel[kAgainPixels];
        PixelTerms pt[kAgainPixels];
        float farthest[kAgainPixels];
        HybridTail acc[kAgainPixels];
#pragma unroll
        for (int j = 0; j < kAgainPixels; ++j) {
            pixel[j] = todo != 0 ? (uint32_t)__builtin_ctzll(todo) : 64u;
            todo &= todo - 1;                                       // (0 stays 0)
            uint32_t local_x, local_y;
            quadrant_pixel(pixel[j] & 63u, local_x, local_y);
            pt[j] = pixel_terms(local_x, local_y, 8);
            farthest[j] = last_depth[pixel[j] & 63u];
            hybrid_tail_init(acc[j]);
        }
        for (uint32_t base = first; base < last; base += 64) {
            wave_lds_sync();
            tile_stage_load<MODE, 64, true, kCullNone, true, REC4>(st, prim, inst, base + lane, last, lane, cx, cy);
            wave_lds_sync();
            const bool loaded = base + lane < last;
            const uint32_t addr = stage_address(st) + 16u * lane;
#pragma unroll
            for (int j = 0; j < kAgainPixels; ++j) {
                if (pixel[j] >= 64u) continue;                      // (wave-uniform)
                TileFrag f;
                const bool in_reach = tile_frag_cutoff<64>(addr, pt[j], f);
                f.den_rcp = frag_rcp<FAST>(f.den);
                const float4 col = stage_row<64, 5>(addr);
                const bool fragment = tile_frag_alpha<MODE, FAST>(stage_opacity<64>(addr), f) && in_reach && loaded;
                const float depth = tile_frag_depth<64>(addr, pt[j], f);
                bool decides = false;
                if (fragment) {
                    if (kTail) {
                        acc[j].c0 = __builtin_fmaf(f.alpha, col.x, acc[j].c0);
                        acc[j].c1 = __builtin_fmaf(f.alpha, col.y, acc[j].c1);
                        acc[j].c2 = __builtin_fmaf(f.alpha, col.z, acc[j].c2);
                    }
                    decides = depth <= farthest[j] && (!kTail || f.alpha >= kMinAlphaCore);
                    if (kTail && !decides) hybrid_tail_add<false>(acc[j], depth, f.alpha);
                }
                const uint64_t deciding = __ballot(decides);
                if (deciding != 0) {
                    const uint32_t at = n_out + (uint32_t)__popcll(deciding & ((1ull << lane) - 1ull));
                    n_out += (uint32_t)__popcll(deciding);
                    fits = fits && n_out <= room;
                    if (decides && fits) {
                        out[4 * at] = pixel[j]; out[4 * at + 1] = float_to_bits(depth); out[4 * at + 2] = float_to_bits(f.alpha);
                        out[4 * at + 3] = float_to_bits(col.w);
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; kTail && j < kAgainPixels; ++j) {
            const float T = wave_product(acc[j].T), c0 = wave_total(acc[j].c0), c1 = wave_total(acc[j].c1), c2 = wave_total(acc[j].c2),
                        alpha = wave_total(acc[j].alpha), depth = wave_total(acc[j].depth);
            if (lane == 0) { sums[j][0] = T; sums[j][1] = c0; sums[j][2] = c1; sums[j][3] = c2; sums[j][4] = alpha; sums[j][5] = depth; }
        }
        pass_done(pixel);
    }
    return fits ? n_out : ~0u;
}

// A core, a tail and a tie (3K + 7 rows of 64 lanes at from[]) join the running ones: they cover the stretch of the
// list that follows.
template <int K, bool FAST>
__device__ __forceinline__ void hybrid_merge(const float *from, uint32_t lane, float (&cd)[K], float (&ca)[K], float (&ci)[K], HybridTail &tail,
                                             CoreTie &tie)
{
    take_tie<3 * K + 6, 3 * (K - 1)>(from + lane, tie);
    merge_cores<K, !FAST>(from + lane, cd, ca, ci, tie, [&](float depth, float alpha) { hybrid_tail_add<FAST>(tail, depth, alpha); });
    take_tail<3 * K>(from + lane, tail);
}
template <int K>
__device__ __forceinline__ void hybrid_put(float *to, uint32_t lane, const float (&cd)[K], const float (&ca)[K], const float (&ci)[K], const HybridTail &tail, const CoreTie &tie)
{
    give_core<K>(to + lane, cd, ca, ci);
    give_tail<3 * K>(to + lane, tail);
    give_tie<3 * K + 6>(to + lane, tie, cd[K - 1]);
}
// The waves' shares, merged pairwise into the first wave's: put(buffer) by the wave that hands its share on, merge(buffer) by
// the one that takes it (all threads of the workgroup call this).
template <int WAVES, uint32_t ROWS, typename Put, typename Merge>
__device__ __forceinline__ void merge_all_shares(unsigned char *lds, uint32_t wave, Put &&put, Merge &&merge)
{
    for (uint32_t step = 1; step < (uint32_t)WAVES; step *= 2) {
        float *buffer = reinterpret_cast<float *>(lds) + (size_t)(wave / (2u * step)) * ROWS * 64u;
        __syncthreads();
        if ((wave & (2u * step - 1u)) == step) put(buffer);
        __syncthreads();
        if ((wave & (2u * step - 1u)) == 0u) merge(buffer);
    }
    __syncthreads();                                       // (the stages are free again)
}
// The long tiles: a workgroup of WAVES waves takes a tile, every wave walks a share of the list (every WAVES-th batch of 64)
// into a core and a tail of its own, and the shares are then merged pairwise into the first wave's, through LDS: the nearer
// entries of both cores stay (what does not, of either, joins the tail), the tails add up.  Nothing of this is in list order.  The pixel gets the K nearest fragments of the whole list and
// everything else in its tail, as in a single walk; what differs from the single walk is the order in which the tail's
// sums are added (rounding) and which of two stored fragments of exactly equal depth is kept when a nearer one arrives.
// binned: the lists are in bins of depth (htgs_frame.depth_bins) and are put in order by index before one is walked again; the others
// are as they are and not searched for runs.
// finish(prim, tile, px, cd, ca, ci, tail) is called by the lanes of the first wave whose pixels lie inside the image, once
// per pixel, with the pixel's finished core and tail.
template <int K, int WAVES, bool FAST, int REC4, typename Finish>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(K > 16 ? 2 : kLongWavesHeld / 4))) blend_hybrid_long_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, const uint32_t *long_tiles,
    uint32_t width, uint32_t height, uint32_t grid_w, uint32_t *__restrict__ shortlist, int binned, ListThreshold threshold, const Finish finish)
{
    constexpr int kWaves = WAVES;
    constexpr uint32_t kRows = 3 * K + 7;             // a wave's core, tail and tie
    __shared__ __attribute__((aligned(16))) unsigned char lds[shared_walk_lds<kWaves, kRows>()];
    static_assert(shared_walk_lds<kWaves, kRows>() >= 3u * kAgainEntries * sizeof(uint32_t), "entries_in_order lies over it");
    __shared__ uint32_t s_next;
    __shared__ uint32_t s_redo[2];                    // the pixels (lanes) to walk again
    __shared__ uint32_t s_short[kWaves];          // how many instances of each share reach one of them
    __shared__ uint32_t s_runs[1 + kDepthBins];
    __shared__ uint32_t s_whole;                      // this workgroup finished the last part of its tile
    __shared__ float s_last_depth[64];                // depth of the merged core's last entry
    __shared__ float s_sums[kWaves][kAgainPixels][6], s_tails[64][6];   // tails of the pixels looked at again: per wave, whole
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (long_tiles[0] == 0) return;                   // (the ordinary frame)
    const uint32_t long_threshold = threshold.get(long_tiles);
    const uint32_t n_tiles = grid_w * ((height + 7u) / 8u);
    uint32_t round = 0;
    LongEntry entry;
    while (long_tile_take(long_tiles, ranges, long_threshold, threshold.counters, round, &s_next, entry)) {
        // (the same in every lane; said so, they live in scalar registers through the walks that follow)
        const auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
        const uint32_t tile = uniform(entry.tile), part = uniform(entry.part), parts = uniform(entry.parts), tile_first = uniform(entry.tile_first),
                       tile_last = uniform(entry.tile_last);
        uint32_t first = uniform(entry.first), last = uniform(entry.last);
        const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
        uint32_t n_batches = (last - first + 63u) / 64u;
        uint32_t seg_first, seg_last;
        long_wave_share(first, last, wave, seg_first, seg_last, kWaves);
        constexpr bool kTies = !FAST;
        HybridTail tail;
        hybrid_tail_init(tail);
        float cd[K], ca[K], ci[K];
        hybrid_core_init<K>(cd, ca, ci);
        CoreTie tie;                                    // fragments of equal depth at the end of a core
        tie.init();
        hybrid_walk<K, FAST, false, kTies, false, REC4, true>(wave_stage(lds, wave), wave_lists<kWaves>(lds, wave), inst, prim, first + 64u * wave, last, lane, px.pt, px.cx, px.cy, cd, ca, ci, tail, &tie,
                                                              0, 64u * kWaves);
        merge_all_shares<kWaves, kRows>(lds, wave, [&](float *to) { hybrid_put<K>(to, lane, cd, ca, ci, tail, tie); },
                                        [&](const float *from) { hybrid_merge<K, FAST>(from, lane, cd, ca, ci, tail, tie); });
        if (parts > 1u) {
            // One of several parts: what it came to goes to the tile's stretch of the spare value buffer (which is as long as the
            // list and unused until pixels are walked again), and the workgroup that finds the other parts there already
            // merges them all, one after the other, and goes on with the whole tile.
            float *const left = reinterpret_cast<float *>(shortlist + tile_first);
            if (wave == 0) {
                hybrid_put<K>(left + (size_t)part * long_part_words<K>(), lane, cd, ca, ci, tail, tie);
                __threadfence();
            }
            if (!long_part_done(long_tiles, n_tiles, entry, &s_whole)) continue;
            if (wave == 0) {
                __threadfence();
                hybrid_tail_init(tail);
                hybrid_core_init<K>(cd, ca, ci);
                tie.init();
                for (uint32_t other = 0; other < parts; ++other)
                    hybrid_merge<K, FAST>(left + (size_t)other * long_part_words<K>(), lane, cd, ca, ci, tail, tie);
            }
            first = tile_first; last = tile_last; n_batches = (last - first + 63u) / 64u;
            long_wave_share(first, last, wave, seg_first, seg_last, kWaves);
            __syncthreads();                               // (the parts are read before the shortlist overwrites them)
        }
        if (kTies) {
            // Equal depths matter where they can change the final core: a tie no deeper than its last entry (both
            // fragments of a deeper tie end in the tail either way), or two equal depths next to each other in it.
            // There the merged walk and the single walk can keep different fragments, or keep them in another order: the
            // reference's insertion lets a displaced entry hop over a stored one of exactly equal depth.  Where no more than two are
            // as deep as each other, what that insertion leaves follows from the core alone (settle_core; the second look cost up to 800 of the
            // 3400 us of this kernel with 6 M Gaussians of the stress scene at 1600x1066).  The other pixels are looked at again by all
            // waves, or walked again in one piece by the first one, over the instances that reach one of them; every wave picks those out of
            // its share first (into the tile's own stretch of the shortlist), since the walk of one wave alone is bound by the
            // latency of staging.
            bool redo = false;
            if (wave == 0) {
                const bool met = core_tied<K>(cd, ca, tie);
                if (__any(met)) {
                    redo = settle_exact_core<HTGS_MODE_HYBRID_BLEND, K, REC4>(wave_stage(lds, 0), prim, lane, px, cd, ca, ci, tie, tail_swap(tail, cd[K - 1])) && px.inside;
                    if (lane == 0 && !__any(redo)) atomicAdd(const_cast<uint32_t *>(long_tiles) + 6, 1u);
                }
                const uint64_t lanes = __ballot(redo);
                if (lane == 0) { s_redo[0] = (uint32_t)lanes; s_redo[1] = (uint32_t)(lanes >> 32); }
            }
            __syncthreads();
            const uint64_t redo_lanes = (uint64_t)s_redo[0] | (uint64_t)s_redo[1] << 32;
            if (redo_lanes != 0) {
                bool others_done = false;                       // the pixels that need no second look are composited
                if (shortlist != nullptr && __popcll(redo_lanes) <= kAgainMost) {
                    // All waves look at these pixels again, lanes = instances (pixels_again), into the tile's stretch of
                    // the shortlist, four words per fragment that decides a core: a wave has a quarter as many entries as
                    // its share has instances, which is ample unless depths coincide by the hundred -- then, and when the
                    // pixels are many (a pass over the list serves kAgainPixels of them), the other way below is taken.
                    others_done = true;
                    if (wave == 0) {
                        s_last_depth[lane] = cd[K - 1];
                        if (px.inside && !redo) finish(prim, tile, px, cd, ca, ci, tail);
                    }
                    __syncthreads();
                    const uint32_t listed = pixels_again<HTGS_MODE_HYBRID_BLEND, false, REC4>(
                        reinterpret_cast<TileStage<64> &>(wave_stage(lds, wave)), inst, prim, seg_first, seg_last, lane, px.cx, px.cy, redo_lanes, s_last_depth, s_sums[wave], shortlist + seg_first,
                        (seg_last - seg_first) / 4u, [&](const uint32_t (&pixel)[kAgainPixels]) {
                            __syncthreads();
                            if (wave == 0 && lane < (uint32_t)kAgainPixels) {      // the waves' sums of a pixel, wave after wave (contiguous shares here)
                                uint32_t mine = pixel[0];
#pragma unroll
                                for (int j = 1; j < kAgainPixels; ++j) mine = lane == (uint32_t)j ? pixel[j] : mine;
                                if (mine < 64u) {
                                    float T = 1.0f, sum[5] = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
                                    for (int w = 0; w < kWaves; ++w) {
                                        T *= s_sums[w][lane][0];
#pragma unroll
                                        for (int k = 0; k < 5; ++k) sum[k] += s_sums[w][lane][1 + k];
                                    }
                                    s_tails[mine][0] = T;
#pragma unroll
                                    for (int k = 0; k < 5; ++k) s_tails[mine][1 + k] = sum[k];
                                }
                            }
                            __syncthreads();
                        });
                    if (lane == 0) s_short[wave] = listed;
                    __syncthreads();
                    bool settled = true;
                    uint32_t entries = 0;
#pragma nounroll
                    for (int w = 0; w < kWaves; ++w) {
                        settled = settled && s_short[w] != ~0u;
                        entries += s_short[w];
                    }
                    settled = settled && entries <= kAgainEntries;
                    __syncthreads();                            // (s_short is written again below)
                    if (settled) {
                        if (wave == 0) {
                            // The walk's insertion, on the fragments that decide the cores alone, by index; every pixel's lane
                            // takes its own.
                            hybrid_core_init<K>(cd, ca, ci);
                            tail.T = s_tails[lane][0]; tail.c0 = s_tails[lane][1]; tail.c1 = s_tails[lane][2]; tail.c2 = s_tails[lane][3];
                            tail.alpha = s_tails[lane][4]; tail.depth = s_tails[lane][5];
                            uint32_t total;
                            const uint32_t *const ordered = entries_in_order<kWaves, true>(shortlist, s_short, reinterpret_cast<uint32_t *>(lds), lane, total,
                                [&](uint32_t w) { return first + 64u * (uint32_t)((uint64_t)n_batches * w / kWaves); });
                            for (uint32_t e = 0; e < total; ++e) {
                                const uint32_t *const entry = shortlist + ordered[e];
                                float depth = bits_to_float(entry[1]), alpha = bits_to_float(entry[2]), index = bits_to_float(entry[3]);
                                if (lane == entry[0]) {
                                    if (depth < cd[K - 1]) core_exchange_walk<K>(depth, alpha, index, cd, ca, ci);
                                    hybrid_tail_add<false>(tail, depth, alpha);
                                }
                            }
                            if (px.inside && redo) finish(prim, tile, px, cd, ca, ci, tail);
                        }
                        if (threadIdx.x == 0) atomicAdd(const_cast<uint32_t *>(long_tiles) + 6, 1u);
                        continue;
                    }
                }
                if (threadIdx.x == 0) atomicAdd(const_cast<uint32_t *>(long_tiles) + 7, others_done ? 0x10001u : 1u);
                const uint32_t *const list = binned && shortlist != nullptr ? list_in_index_order_by<kWaves>(inst, first, last, shortlist, s_runs, wave, lane) : inst;
                __syncthreads();
                if (shortlist != nullptr) {
                    uint32_t kept = 0;
                    // (in place where the list by index is in the shortlist: a wave's picks never get ahead of what it has read)
                    for (uint32_t base = seg_first; base < seg_last; base += 64) {
                        const uint32_t fetch = base + lane;
                        const uint32_t g = fetch < seg_last ? list[fetch] : 0u;
                        const bool reaches = tile_stage_load<HTGS_MODE_HYBRID_BLEND, 64, true, kCullPixels, true, REC4, false, false, true>(reinterpret_cast<TileStage<64> &>(wave_stage(lds, wave)), prim, list, fetch, seg_last, lane,
                                                                                                               px.cx, px.cy, redo_lanes, g) != 0;
                        const uint64_t keep = __ballot(reaches);
                        if (reaches) shortlist[seg_first + kept + (uint32_t)__popcll(keep & ((1ull << lane) - 1ull))] = g;
                        kept += (uint32_t)__popcll(keep);
                    }
                    if (lane == 0) s_short[wave] = kept;
                    __syncthreads();
                }
                if (wave == 0) {
                    if (!others_done && px.inside && !redo)
                        finish(prim, tile, px, cd, ca, ci, tail);
                    hybrid_tail_init(tail);
                    hybrid_core_init<K>(cd, ca, ci);
                    if (shortlist != nullptr) {
                        for (uint32_t s = 0; s < (uint32_t)kWaves; ++s) {
                            const uint32_t from = first + 64u * (uint32_t)((uint64_t)n_batches * s / kWaves);
                            hybrid_walk<K, FAST, false, false, true, REC4>(wave_stage(lds, 0), wave_lists<kWaves>(lds, 0), shortlist, prim, from, from + s_short[s], lane, px.pt, px.cx, px.cy, cd, ca, ci,
                                                                     tail, nullptr, redo_lanes);
                        }
                    } else {
                        hybrid_walk<K, FAST, false, false, true, REC4>(wave_stage(lds, 0), wave_lists<kWaves>(lds, 0), inst, prim, first, last, lane, px.pt, px.cx, px.cy, cd, ca, ci, tail, nullptr, redo_lanes);
                    }
                    if (px.inside && redo) finish(prim, tile, px, cd, ca, ci, tail);
                }
                continue;
            }
        }
        if (wave == 0 && px.inside) finish(prim, tile, px, cd, ca, ci, tail);
    }
}

// ---------------------------------------------------------------------------------------------
// ALPHA_BLEND_FIRST_K: the K nearest fragments with alpha >= 1/20, alpha-blended; no tail.
// ---------------------------------------------------------------------------------------------
template <int K>
__device__ __forceinline__ void first_k_core_init(float (&cd)[K], float (&ca)[K], uint32_t (&ci)[K])
{
#pragma unroll
    for (int i = 0; i < K; ++i) {
        ca[i] = 0.0f; cd[i] = __FLT_MAX__; ci[i] = 0xffffffffu;
        asm volatile("" : "+v"(cd[i]), "+v"(ca[i]), "+v"(ci[i]));      // one register per slot
    }
}
// Waves that share a list know more together than each from its own core: if every wave has k fragments of a pixel with k times WAVES no less than K,
// the K nearest of all are no deeper than the deepest of those waves' k-th.  Every wave leaves its own in LDS before it stages a batch
// and takes what the others have left, whatever they have walked until then: a depth that only grows nearer with time, behind
// which there is nothing to be found for the pixel.
template <int WAVES, int K>
struct SharedDepth {
    static constexpr int kSlot = (K + WAVES - 1) / WAVES - 1;
    float (*s_depth)[64];                  // LDS, [WAVES][64]
    uint32_t wave, lane;
    __device__ __forceinline__ void init() const { s_depth[wave][lane] = __FLT_MAX__; }      // (and a barrier of the workgroup)
    __device__ __forceinline__ float operator()(float own) const
    {
        typedef __attribute__((address_space(3))) volatile float lds_shared;
        lds_shared *const all = (lds_shared *)&s_depth[0][lane];
        all[64u * wave] = own;
        float most = own;
#pragma unroll
        for (uint32_t w = 0; w < (uint32_t)WAVES; ++w) {
            const float v = all[64u * w];
            most = w != wave && v > most ? v : most;
        }
        return most;
    }
};
struct NoSharedDepth {
    static constexpr int kSlot = 0;
    __device__ __forceinline__ float operator()(float) const { return __FLT_MAX__; }
};
// The walk over instances [first, last) of a tile's list by one wave (SOLO: the wave is the whole workgroup).  TIES (the
// walks whose pixels are settled afterwards): `tie` notes the entries that stayed out of the core, or left it, exactly as deep as the
// entry that is now last (CoreTie).
// PIXELS: only the pixels of the lanes in pixel_lanes are wanted; instances that do not reach one of them are left out.
template <int K, bool FAST, bool SOLO, bool TIES = false, int REC4 = HTGS_PRIM_FLOATS / 4, bool PIXELS = false, typename Shared = NoSharedDepth>
__device__ __forceinline__ void first_k_walk(TileStageQ &st, QuadrantLists &ql, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
                                             uint32_t first, uint32_t last, uint32_t lane, const PixelTerms &pt, float cx, float cy, float (&cd)[K],
                                             float (&ca)[K], uint32_t (&ci)[K], CoreTie *tie = nullptr, uint64_t pixel_lanes = 0, ListStep step = 64u,
                                             const Shared &shared = Shared())
{
    constexpr int MODE = HTGS_MODE_ALPHA_BLEND_FIRST_K;
    constexpr int N = kStageSlots;
    tile_list_walk<MODE, true, PIXELS ? kCullPixels : kCullAlpha, SOLO, REC4>(st, ql, prim, inst, first, last, lane, cx, cy, [&](uint32_t addr) {
        TileFrag f;
        const bool in_reach = tile_frag_cutoff<N>(addr, pt, f);
        f.den_rcp = frag_rcp<FAST>(f.den);
        float depth = tile_frag_depth<N>(addr, pt, f);
        if (!(in_reach && (TIES ? depth <= cd[K - 1] : depth < cd[K - 1]))) return;          // depth test before the exponential (:151)
        if (!tile_frag_alpha<MODE, FAST>(stage_opacity<N>(addr), f)) return;
        float alpha = f.alpha;
        uint32_t idx = stage_index<N>(addr);
        core_exchange_walk<K>(depth, alpha, idx, cd, ca, ci);
        if (TIES) tie->note(meets_core_end(depth, cd[K - 1]), depth, idx);
    }, pixel_lanes, 1.0f, step, [&]() {
        const float of_all = shared(cd[Shared::kSlot]);
        return cd[K - 1] < of_all ? cd[K - 1] : of_all;
    });
}
// The same walk with the core as sorted 64-bit keys (above HYBRID_BLEND's: depth | alpha as a fraction | place in the list),
// exact arithmetic; `notes` as in hybrid_key_walk.
template <int K, bool SOLO, int REC4 = HTGS_PRIM_FLOATS / 4, typename Shared = NoSharedDepth>
__device__ __forceinline__ void first_k_key_walk(TileStageQ &st, QuadrantLists &ql, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
                                                 uint32_t first, uint32_t last, uint32_t lane, const PixelTerms &pt, float cx, float cy,
                                                 CoreKey (&core)[K], KeyNotes &notes, const KeyFormat &fmt, uint32_t list_first, ListStep step = 64u,
                                                 const Shared &shared = Shared())
{
    constexpr int MODE = HTGS_MODE_ALPHA_BLEND_FIRST_K;
    constexpr int N = kStageSlots;
    tile_list_walk<MODE, true, kCullAlpha, SOLO, REC4, false, true, true, true>(st, ql, prim, inst, first, last, lane, cx, cy, [&](uint32_t one, uint32_t two) {
        TileFrag f1, f2;
        const bool reach1 = tile_frag_cutoff<N>(one, pt, f1), reach2 = tile_frag_cutoff<N>(two, pt, f2);
        const uint64_t leaves = __ballot(!rcp_in_range(f1.den)) | __ballot(!rcp_in_range(f2.den));      // (tile_frag_exact)
        f1.den_rcp = rcp_refined(f1.den);
        f2.den_rcp = rcp_refined(f2.den);
        float depth1 = tile_frag_depth<N>(one, pt, f1), depth2 = tile_frag_depth<N>(two, pt, f2);
        if (__builtin_expect(leaves != 0, 0)) {
            f1.den_rcp = 1.0f / f1.den;
            f2.den_rcp = 1.0f / f2.den;
            depth1 = tile_frag_depth<N>(one, pt, f1);
            depth2 = tile_frag_depth<N>(two, pt, f2);
        }
        const auto joins = [&](uint32_t addr, TileFrag &f, bool in_reach, float depth) {
            if (!(in_reach && depth <= key_depth(core[K - 1]))) return;         // depth test before the exponential (:151)
            if (!tile_frag_alpha<MODE, false>(stage_opacity<N>(addr), f)) return;
            CoreKey carried = make_key(depth, key_pack(f.alpha, stage_index<N>(addr) - list_first, fmt));      // (the slot's last word is the place in the list)
            core_key_walk<K>(carried, core);
            depth = key_depth(carried);
            notes.note(depth == key_depth(core[K - 1]), key_low(carried));
        };
        joins(one, f1, reach1, depth1);
        joins(two, f2, reach2, depth2);
    }, 0, 1.0f, step, [&]() {
        const float of_all = shared(key_depth(core[Shared::kSlot])), own = key_depth(core[K - 1]);
        return own < of_all ? own : of_all;
    });
}
// the finished keys as the three arrays the composite takes (an empty slot has the index 0xffffffff)
template <int K>
__device__ __forceinline__ void first_k_core_unpack(const CoreKey (&core)[K], const uint32_t *__restrict__ inst, uint32_t first, uint32_t last, float (&cd)[K],
                                                    float (&ca)[K], uint32_t (&ci)[K], const KeyFormat &fmt)
{
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const uint32_t low = key_low(core[i]), place = low & fmt.place_mask;
        cd[i] = key_depth(core[i]);
        ca[i] = key_alpha(low, fmt);
        ci[i] = low >> fmt.shift != 0u && first + place < last ? inst[first + place] : 0xffffffffu;
    }
}
template <int K, int REC4 = HTGS_PRIM_FLOATS / 4>
__device__ __forceinline__ void first_k_composite(const float4 *__restrict__ prim, const float (&cd)[K], const float (&ca)[K], const uint32_t (&ci)[K],
                                                  float *__restrict__ image, float *__restrict__ depths, uint32_t width, uint32_t height, uint32_t x,
                                                  uint32_t y, int chw, int median)
{
    float r = 0.0f, g = 0.0f, b = 0.0f, depth_pixel = 0.0f, T = 1.0f;
    bool open = true;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        open = open && T >= kTransmittanceThreshold && ci[i] != 0xffffffffu;
        if (open) {
            const float wgt = T * ca[i];
            const float4 col = prim[(size_t)ci[i] * REC4 + 4];
            r = __builtin_fmaf(wgt, col.x, r);
            g = __builtin_fmaf(wgt, col.y, g);
            b = __builtin_fmaf(wgt, col.z, b);
            if (median) depth_pixel = T > 0.5f ? cd[i] : depth_pixel;
            else depth_pixel = __builtin_fmaf(wgt, cd[i], depth_pixel);
            T *= 1.0f - ca[i];
        }
    }
    if (!median) depth_pixel = T < 1.0f ? depth_pixel / (1.0f - T) : 0.0f;
    store_pixel(image, depths, width, height, x, y, chw, r, g, b, depth_pixel);
}
struct FirstKImage {
    float *image, *depths;
    uint32_t width, height;
    int chw, median;
    template <int K>
    __device__ __forceinline__ void operator()(const float4 *__restrict__ prim, uint32_t, const TilePixel &px, const float (&cd)[K], const float (&ca)[K],
                                               const uint32_t (&ci)[K]) const
    {
        first_k_composite<K>(prim, cd, ca, ci, image, depths, width, height, px.x, px.y, chw, median);
    }
};
// what a workgroup leaves of its part of a list: the core and what met at its end
template <int K> constexpr uint32_t first_k_part_words() { return (3u * K + 1u) * 64u; }
// KEYS (exact arithmetic, with long_tiles and a threshold of no more than kPackedListMost): the core as sorted 64-bit keys;
// the pixels at which fragments of exactly equal depth met where they decide the core are settled as in hybrid_tile_by_keys: from the
// core, or by another walk with the reference's insertion over the instances that reach one of them.
template <int K, bool FAST, bool KEYS = false>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(K <= 16 ? 5 : 2))) blend_first_k_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
    float *__restrict__ image, float *__restrict__ depths, uint32_t width, uint32_t height, uint32_t grid_w, int chw, int median,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare)
{
    static_assert(!(KEYS && FAST), "the keys of this mode are for the exact path");
    __shared__ TileStageQ st;
    __shared__ QuadrantLists ql;
    const uint32_t tile = block_tile(tile_order);
    const uint32_t lane = threadIdx.x;
    const uint32_t first = ranges[2 * tile], last = ranges[2 * tile + 1];
    const uint32_t long_threshold = threshold.get(long_tiles);
    if (long_tiles != nullptr && last - first > long_threshold) {
        if (lane == 0) long_tile_enter(long_tiles, tile, gridDim.x, last - first, threshold.least_part(long_threshold), first_k_part_words<K>(), part_floor.get(gridDim.x), long_threshold, threshold.counters);
        return;
    }
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    float ca[K], cd[K];
    uint32_t ci[K];
    if constexpr (KEYS) {
        CoreKey core[K];
#pragma unroll
        for (int i = 0; i < K; ++i) {
            core[i] = make_key(__FLT_MAX__, 0u);
            asm volatile("" : "+v"(core[i]));      // one register pair per slot, never a wide tuple
        }
        KeyNotes notes;
        notes.init();
        const KeyFormat fmt = key_format(last > first ? last - first : 1u);
        first_k_key_walk<K, true>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, core, notes, fmt, first);
        const CoreTie tie = noted_ties<HTGS_MODE_ALPHA_BLEND_FIRST_K, HTGS_PRIM_FLOATS / 4>(st, prim, inst, first, last, lane, px, notes, fmt);
        const bool again = settle_keys<HTGS_MODE_ALPHA_BLEND_FIRST_K, K, HTGS_PRIM_FLOATS / 4>(st, prim, inst, first, last, lane, px, core, tie, fmt, [](float, float) {});
        const uint64_t again_lanes = __ballot(again);
        first_k_core_unpack<K>(core, inst, first, last, cd, ca, ci, fmt);
        if (px.inside && !again) first_k_composite<K>(prim, cd, ca, ci, image, depths, width, height, px.x, px.y, chw, median);
        if (again_lanes == 0) return;
        // (the lane and its pixel are worked out afresh: nothing of the first walk has to live through the composite for this)
        uint32_t lane_again = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(lane_again));
        const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
        const uint32_t *const list = spare != nullptr ? list_in_index_order<1>(inst, first, last, spare, ql.a[0], 0u, lane_again) : inst;
        first_k_core_init<K>(cd, ca, ci);
        first_k_walk<K, false, true, false, HTGS_PRIM_FLOATS / 4, true>(st, ql, list, prim, first, last, lane_again, px_again.pt, px_again.cx, px_again.cy, cd, ca, ci,
                                                                         nullptr, again_lanes);
        if ((again_lanes >> lane_again & 1ull) != 0)
            first_k_composite<K>(prim, cd, ca, ci, image, depths, width, height, px_again.x, px_again.y, chw, median);
    } else {
        first_k_core_init<K>(cd, ca, ci);
        first_k_walk<K, FAST, true>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, cd, ca, ci);
        if (!px.inside) return;
        first_k_composite<K>(prim, cd, ca, ci, image, depths, width, height, px.x, px.y, chw, median);
    }
}

// A core and a tie (3K + 1 rows of 64 lanes at from[]) join the running ones: they cover the stretch of the list
// that follows.
template <int K>
__device__ __forceinline__ void first_k_merge(const float *from, uint32_t lane, float (&cd)[K], float (&ca)[K], uint32_t (&ci)[K], CoreTie &tie)
{
    take_tie<3 * K, 3 * (K - 1)>(from + lane, tie);
    merge_cores<K, true>(from + lane, cd, ca, ci, tie, [](float, float) {});
}
template <int K>
__device__ __forceinline__ void first_k_put(float *to, uint32_t lane, const float (&cd)[K], const float (&ca)[K], const uint32_t (&ci)[K], const CoreTie &tie)
{
    give_core<K>(to + lane, cd, ca, ci);
    give_tie<3 * K>(to + lane, tie, cd[K - 1]);
}

// The tiles with very long lists, as in blend_hybrid_long_kernel: every wave of the workgroup walks a share of the list
// into a core of its own, the cores are merged (and so are those of the parts of a list that several
// workgroups walked, through the tile's stretch of the spare value buffer `spare`), and the pixels at which fragments of
// exactly equal depth met where they can change the final core are settled from it where no more than two are of a depth (exact
// arithmetic); the others get a second look (pixels_again) with the insertion replayed by index on the fragments that are not farther than the merged core's last entry -- or, when they are many or the room
// for those fragments does not do, the first wave walks the whole list again for them.
// binned, finish(prim, tile, px, cd, ca, ci): as for blend_hybrid_long_kernel, with the pixel's finished core.
template <int K, int WAVES, bool FAST, int REC4, typename Finish>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(K > 16 ? 2 : kLongWavesHeld / 4))) blend_first_k_long_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, const uint32_t *long_tiles,
    uint32_t width, uint32_t height, uint32_t grid_w, uint32_t *__restrict__ spare, int binned, ListThreshold threshold, const Finish finish)
{
    constexpr int kWaves = WAVES;
    constexpr uint32_t kRows = 3 * K + 1;
    __shared__ __attribute__((aligned(16))) unsigned char lds[shared_walk_lds<kWaves, kRows>()];
    static_assert(shared_walk_lds<kWaves, kRows>() >= 3u * kAgainEntries * sizeof(uint32_t), "entries_in_order lies over it");
    __shared__ uint32_t s_next, s_whole, s_redo[2], s_listed[kWaves], s_runs[1 + kDepthBins];
    __shared__ float s_depth[kWaves][64];
    __shared__ float s_last_depth[64];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (long_tiles[0] == 0) return;                   // (the ordinary frame)
    const uint32_t long_threshold = threshold.get(long_tiles);
    const uint32_t n_tiles = grid_w * ((height + 7u) / 8u);
    constexpr bool kTies = true;                      // (the fast variant too: a tie decides which fragment a pixel shows)
    uint32_t round = 0;
    LongEntry entry;
    while (long_tile_take(long_tiles, ranges, long_threshold, threshold.counters, round, &s_next, entry)) {
        // (the same in every lane; said so, they live in scalar registers through the walks that follow)
        const auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
        const LongEntry e = { uniform(entry.tile), uniform(entry.part), uniform(entry.parts), uniform(entry.tile_first), uniform(entry.tile_last),
                              uniform(entry.first), uniform(entry.last) };
        const TilePixel px = quadrant_tile_pixel(e.tile, grid_w, lane, width, height);
        uint32_t share_first, share_last;
        long_wave_share(e.first, e.last, wave, share_first, share_last, kWaves);
        float ca[K], cd[K];
        uint32_t ci[K];
        first_k_core_init<K>(cd, ca, ci);
        CoreTie tie;
        tie.init();
        const SharedDepth<kWaves, K> shared = { s_depth, wave, lane };
        shared.init();
        __syncthreads();
        first_k_walk<K, FAST, false, kTies, REC4, false>(wave_stage(lds, wave), wave_lists<kWaves>(lds, wave), inst, prim, e.first + 64u * wave, e.last, lane, px.pt, px.cx, px.cy, cd, ca, ci, &tie,
                                                       0, 64u * kWaves, shared);
        merge_all_shares<kWaves, kRows>(lds, wave, [&](float *to) { first_k_put<K>(to, lane, cd, ca, ci, tie); },
                                        [&](const float *from) { first_k_merge<K>(from, lane, cd, ca, ci, tie); });
        if (e.parts > 1u) {
            float *const left = reinterpret_cast<float *>(spare + e.tile_first);
            if (wave == 0) {
                first_k_put<K>(left + (size_t)e.part * first_k_part_words<K>(), lane, cd, ca, ci, tie);
                __threadfence();
            }
            if (!long_part_done(long_tiles, n_tiles, e, &s_whole)) continue;
            if (wave == 0) {
                __threadfence();
                first_k_core_init<K>(cd, ca, ci);
                tie.init();
                for (uint32_t other = 0; other < e.parts; ++other)
                    first_k_merge<K>(left + (size_t)other * first_k_part_words<K>(), lane, cd, ca, ci, tie);
            }
            long_wave_share(e.tile_first, e.tile_last, wave, share_first, share_last, kWaves);
            __syncthreads();                               // (the parts are read before the second look overwrites them)
        }
        if (kTies) {
            bool redo = false;
            if (wave == 0) {
                redo = core_tied<K>(cd, ca, tie);                      // (as in blend_hybrid_long_kernel)
                if constexpr (!FAST) {
                    if (__any(redo)) {
                        redo = settle_exact_core<HTGS_MODE_ALPHA_BLEND_FIRST_K, K, REC4>(wave_stage(lds, 0), prim, lane, px, cd, ca, ci, tie, [](float, float) {}) && px.inside;
                        if (lane == 0 && !__any(redo)) atomicAdd(const_cast<uint32_t *>(long_tiles) + 6, 1u);
                    }
                }
                const uint64_t lanes = __ballot(redo);
                if (lane == 0) { s_redo[0] = (uint32_t)lanes; s_redo[1] = (uint32_t)(lanes >> 32); }
                s_last_depth[lane] = cd[K - 1];
                if (lanes != 0 && px.inside && !redo) finish(prim, e.tile, px, cd, ca, ci);
            }
            __syncthreads();
            const uint64_t redo_lanes = (uint64_t)s_redo[0] | (uint64_t)s_redo[1] << 32;
            if (redo_lanes != 0) {
                bool settled = false, looked = false;
                if (spare != nullptr && __popcll(redo_lanes) <= kAgainMost) {
                    looked = true;
                    const uint32_t listed = pixels_again<HTGS_MODE_ALPHA_BLEND_FIRST_K, FAST, REC4>(
                        reinterpret_cast<TileStage<64> &>(wave_stage(lds, wave)), inst, prim, share_first, share_last, lane, px.cx, px.cy, redo_lanes, s_last_depth, nullptr, spare + share_first,
                        (share_last - share_first) / 4u, [](const uint32_t (&)[kAgainPixels]) {});
                    if (lane == 0) s_listed[wave] = listed;
                    __syncthreads();
                    settled = true;
                    uint32_t entries = 0;
#pragma nounroll
                    for (int w = 0; w < kWaves; ++w) {
                        settled = settled && s_listed[w] != ~0u;
                        entries += s_listed[w];
                    }
                    settled = settled && entries <= kAgainEntries;
                }
                if (threadIdx.x == 0) atomicAdd(const_cast<uint32_t *>(long_tiles) + (settled ? 6 : 7), settled || !looked ? 1u : 0x10001u);
                const uint32_t *list = inst;
                if (!FAST && !settled && binned && spare != nullptr) {       // (the fast variant takes the list's own order)
                    list = list_in_index_order_by<kWaves>(inst, e.tile_first, e.tile_last, spare, s_runs, wave, lane);
                    __syncthreads();
                }
                if (wave == 0) {
                    first_k_core_init<K>(cd, ca, ci);
                    if (settled) {
                        uint32_t total;
                        const uint32_t *const ordered = entries_in_order<kWaves, !FAST>(spare, s_listed, reinterpret_cast<uint32_t *>(lds), lane, total, [&](uint32_t w) {
                            uint32_t from, to;
                            long_wave_share(e.tile_first, e.tile_last, w, from, to, kWaves);
                            return from;
                        });
                        for (uint32_t k = 0; k < total; ++k) {
                            const uint32_t *const candidate = spare + ordered[k];
                            float depth = bits_to_float(candidate[1]), alpha = bits_to_float(candidate[2]);
                            uint32_t index = candidate[3];
                            if (lane == candidate[0] && depth < cd[K - 1]) core_exchange_walk<K>(depth, alpha, index, cd, ca, ci);
                        }
                    } else {
                        first_k_walk<K, FAST, false, false, REC4>(wave_stage(lds, 0), wave_lists<kWaves>(lds, 0), list, prim, e.tile_first, e.tile_last, lane, px.pt, px.cx, px.cy, cd, ca, ci);
                    }
                    if (px.inside && redo) finish(prim, e.tile, px, cd, ca, ci);
                }
                continue;
            }
        }
        if (wave == 0 && px.inside) finish(prim, e.tile, px, cd, ca, ci);
    }
}

// ---------------------------------------------------------------------------------------------
// OIT_BLEND: weighted-sum order-independent transparency over all fragments.
// ---------------------------------------------------------------------------------------------
// what a pixel has summed up: alpha * (colour, depth), alpha, and the transmittance
struct OitSums {
    float a0, a1, a2, a3, alpha, T;
};
// The walk over instances [first, last) of a tile's list by one wave (SOLO: the wave is the whole workgroup).
// DEPTH: the depth sum is wanted (the training pass has no use for it)
template <bool FAST, bool SOLO, int REC4 = HTGS_PRIM_FLOATS / 4, bool DEPTH = !FAST>
__device__ __forceinline__ void oit_walk(TileStageQ &st, QuadrantLists &ql, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t first,
                                         uint32_t last, uint32_t lane, const PixelTerms &pt, float cx, float cy, OitSums &sum, ListStep step = 64u)
{
    constexpr int MODE = HTGS_MODE_OIT_BLEND;
    constexpr int N = kStageSlots;
    tile_list_walk<MODE, DEPTH, kCullAlpha, SOLO, REC4, FAST, false, false, true>(st, ql, prim, inst, first, last, lane, cx, cy, [&](uint32_t one, uint32_t two) {
        TileFrag f1, f2;
        bool pass1, pass2;
        if constexpr (FAST) {
            pass1 = tile_frag_fast<MODE, N>(one, pt, f1);
            pass2 = tile_frag_fast<MODE, N>(two, pt, f2);
        } else tile_frag_exact_pair<MODE, N>(one, two, pt, f1, f2, pass1, pass2);
        const float4 col1 = stage_row<N, 5>(one), col2 = stage_row<N, 5>(two);
        const float depth1 = DEPTH ? tile_frag_depth<N>(one, pt, f1) : 0.0f, depth2 = DEPTH ? tile_frag_depth<N>(two, pt, f2) : 0.0f;
        const auto joins = [&](const TileFrag &f, float depth, const float4 &col) {
            sum.a0 = __builtin_fmaf(f.alpha, col.x, sum.a0);
            sum.a1 = __builtin_fmaf(f.alpha, col.y, sum.a1);
            sum.a2 = __builtin_fmaf(f.alpha, col.z, sum.a2);
            if (DEPTH) sum.a3 = __builtin_fmaf(f.alpha, depth, sum.a3);
            sum.alpha += f.alpha;
            sum.T *= 1.0f - f.alpha;
        };
        if (pass1) joins(f1, depth1, col1);
        if (pass2) joins(f2, depth2, col2);
    }, 0, 1.0f, step);
}
__device__ __forceinline__ void oit_composite(const OitSums &sum, float *__restrict__ image, float *__restrict__ depths, uint32_t width, uint32_t height,
                                              uint32_t x, uint32_t y, int chw)
{
    float r = 0.0f, g = 0.0f, b = 0.0f, d = 0.0f;
    if (sum.alpha >= ModeCfg<HTGS_MODE_OIT_BLEND>::min_alpha) {
        const float alpha = 1.0f - sum.T;
        const float s = alpha * (1.0f / sum.alpha);
        r = s * sum.a0; g = s * sum.a1; b = s * sum.a2;
        d = (s * sum.a3) / alpha;
    }
    store_pixel(image, depths, width, height, x, y, chw, r, g, b, d);
}
struct OitImage {
    float *image, *depths;
    uint32_t width, height;
    int chw;
    __device__ __forceinline__ void operator()(uint32_t, const TilePixel &px, const OitSums &sum) const
    {
        oit_composite(sum, image, depths, width, height, px.x, px.y, chw);
    }
};
constexpr uint32_t kOitPartWords = 6u * 64u;
template <bool FAST>
__global__ void __launch_bounds__(64) blend_oit_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
    float *__restrict__ image, float *__restrict__ depths, uint32_t width, uint32_t height, uint32_t grid_w, int chw,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order)
{
    __shared__ TileStageQ st;
    __shared__ QuadrantLists ql;
    const uint32_t tile = block_tile(tile_order);
    const uint32_t lane = threadIdx.x;
    const uint32_t first = ranges[2 * tile], last = ranges[2 * tile + 1];
    const uint32_t long_threshold = threshold.get(long_tiles);
    if (long_tiles != nullptr && last - first > long_threshold) {
        if (lane == 0) long_tile_enter(long_tiles, tile, gridDim.x, last - first, threshold.least_part(long_threshold), kOitPartWords, part_floor.get(gridDim.x), long_threshold, threshold.counters);
        return;
    }
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    OitSums sum = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f };
    oit_walk<FAST, true>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, sum);
    if (!px.inside) return;
    oit_composite(sum, image, depths, width, height, px.x, px.y, chw);
}

// The tiles with very long lists: every wave of the workgroup walks a share of the list, the sums add up in the order of
// the shares (the transmittances multiply), and so do those of the parts of a list that several workgroups walked
// (`left`: the spare value buffer, where the parts of a tile leave their sums in the tile's own stretch).  The pixel's
// result is that of the single walk up to the order of its sums.
// finish(tile, px, sum): as for blend_hybrid_long_kernel, with the pixel's finished sums.
template <int WAVES, bool FAST, int REC4, typename Finish, bool DEPTH = !FAST>
__global__ void __launch_bounds__(64 * WAVES) blend_oit_long_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, const uint32_t *long_tiles,
    uint32_t width, uint32_t height, uint32_t grid_w, uint32_t *__restrict__ left, ListThreshold threshold, const Finish finish)
{
    __shared__ TileStageQ st[WAVES];
    __shared__ QuadrantLists ql[WAVES];
    __shared__ float s_sums[WAVES][6][64];
    __shared__ uint32_t s_next, s_whole;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (long_tiles[0] == 0) return;                   // (the ordinary frame)
    const uint32_t long_threshold = threshold.get(long_tiles);
    const uint32_t n_tiles = grid_w * ((height + 7u) / 8u);
    uint32_t round = 0;
    LongEntry entry;
    while (long_tile_take(long_tiles, ranges, long_threshold, threshold.counters, round, &s_next, entry)) {
        const TilePixel px = quadrant_tile_pixel(entry.tile, grid_w, lane, width, height);
        OitSums sum = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f };
        oit_walk<FAST, false, REC4, DEPTH>(st[wave], ql[wave], inst, prim, entry.first + 64u * wave, entry.last, lane, px.pt, px.cx, px.cy, sum, 64u * WAVES);
        s_sums[wave][0][lane] = sum.a0; s_sums[wave][1][lane] = sum.a1; s_sums[wave][2][lane] = sum.a2; s_sums[wave][3][lane] = sum.a3;
        s_sums[wave][4][lane] = sum.alpha; s_sums[wave][5][lane] = sum.T;
        __syncthreads();
        if (wave == 0) {
            for (int w = 1; w < WAVES; ++w) {
                sum.a0 += s_sums[w][0][lane]; sum.a1 += s_sums[w][1][lane]; sum.a2 += s_sums[w][2][lane]; sum.a3 += s_sums[w][3][lane];
                sum.alpha += s_sums[w][4][lane]; sum.T *= s_sums[w][5][lane];
            }
        }
        if (entry.parts > 1u) {
            float *const parts = reinterpret_cast<float *>(left + entry.tile_first);
            if (wave == 0) {
                float *mine = parts + (size_t)entry.part * kOitPartWords + lane;
                mine[0] = sum.a0; mine[64] = sum.a1; mine[128] = sum.a2; mine[192] = sum.a3; mine[256] = sum.alpha; mine[320] = sum.T;
                __threadfence();
            }
            if (!long_part_done(long_tiles, n_tiles, entry, &s_whole)) continue;
            if (wave == 0) {
                __threadfence();
                sum = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f };
                for (uint32_t part = 0; part < entry.parts; ++part) {
                    const float *its = parts + (size_t)part * kOitPartWords + lane;
                    sum.a0 += its[0]; sum.a1 += its[64]; sum.a2 += its[128]; sum.a3 += its[192]; sum.alpha += its[256]; sum.T *= its[320];
                }
            }
        }
        if (wave == 0 && px.inside) finish(entry.tile, px, sum);
    }
}


// The launches of the kernels for very long lists, after the one that has put the tiles on the list
template <int K, bool FAST, int REC4, typename Finish>
static void launch_hybrid_long(const htgs_frame *f, int sel, uint32_t grid_w, const Finish &finish)
{
    if (!may_have_long_lists(f)) return;
    with_long_waves<K>(f, [&](auto waves) {
        constexpr int WAVES = decltype(waves)::value;
        hipLaunchKernelGGL((blend_hybrid_long_kernel<K, WAVES, FAST, REC4, Finish>), dim3(long_grid(WAVES)), dim3(64 * WAVES), 0, (hipStream_t)f->stream, f->ranges, f->vals[sel],
                           (const float4 *)f->prim, f->long_tiles, (uint32_t)f->width, (uint32_t)f->height, grid_w, f->vals[sel ^ 1], frame_depth_binned(f) ? 1 : 0, list_threshold(f), finish);
    });
}
template <int K, bool FAST, int REC4, typename Finish>
static void launch_first_k_long(const htgs_frame *f, int sel, uint32_t grid_w, const Finish &finish)
{
    if (!may_have_long_lists(f)) return;
    with_long_waves<K>(f, [&](auto waves) {
        constexpr int WAVES = decltype(waves)::value;
        hipLaunchKernelGGL((blend_first_k_long_kernel<K, WAVES, FAST, REC4, Finish>), dim3(long_grid(WAVES)), dim3(64 * WAVES), 0, (hipStream_t)f->stream, f->ranges, f->vals[sel],
                           (const float4 *)f->prim, f->long_tiles, (uint32_t)f->width, (uint32_t)f->height, grid_w, f->vals[sel ^ 1], frame_depth_binned(f) ? 1 : 0, list_threshold(f), finish);
    });
}
template <bool FAST, int REC4, bool DEPTH, typename Finish>
static void launch_oit_long(const htgs_frame *f, int sel, uint32_t grid_w, const Finish &finish)
{
    if (!may_have_long_lists(f)) return;
    with_long_waves<1>(f, [&](auto waves) {
        constexpr int WAVES = decltype(waves)::value;
        hipLaunchKernelGGL((blend_oit_long_kernel<WAVES, FAST, REC4, Finish, DEPTH>), dim3(long_grid(WAVES)), dim3(64 * WAVES), 0, (hipStream_t)f->stream, f->ranges, f->vals[sel],
                           (const float4 *)f->prim, f->long_tiles, (uint32_t)f->width, (uint32_t)f->height, grid_w, f->vals[sel ^ 1], list_threshold(f), finish);
    });
}

}  // namespace htgs
