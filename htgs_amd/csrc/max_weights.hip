// Per-Gaussian maximum blending weight of a view (used by the reference's importance-based pruning).
// Restates update_max_weights_cu of R/include/hybrid_blend/kernels/update_max_weights.cuh:59-212,
// R/include/alpha_blend_first_k/kernels/update_max_weights.cuh:59-161,
// R/include/alpha_blend_global_ordering/kernels/update_max_weights.cuh:59-131 and
// R/include/oit_blend/kernels/update_max_weights.cuh:58-165.  The maximum is taken on the bit patterns of the
// (non-negative) weights with integer atomicMax, which makes the result independent of the order of arrival.
#include "blend_long.h"

namespace htgs {

__device__ __forceinline__ void raise_max(uint32_t *__restrict__ max_weights, uint32_t g, float w)
{
    if (g == 0xffffffffu) return;
    const uint32_t bits = float_to_bits(w);
    if (max_weights[g] < bits) atomicMax(max_weights + g, bits);
}

// The second walk's staging cull (kCullScaled): a fragment counts if alpha * tail weight reaches the threshold, so none below
// threshold / (largest tail weight of the tile's pixels) does -- behind a core of some transparency that is a good part of
// the tail, and in most tiles all of it (1 M Gaussians at 1080p, threshold 0.02: the kernel 494 -> 370 us).  An eighth per
// cent is left for rounding; a threshold of 0 leaves the cut-off alone.
template <int MODE>
__device__ __forceinline__ float tail_cull_scale(float tail_weight, float weight_threshold)
{
    float most = tail_weight;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = __builtin_fmaxf(most, __shfl_xor(most, o));
    return most * (1.00125f * ModeCfg<MODE>::min_alpha) / weight_threshold;
}

// HYBRID_BLEND (TAIL = true, CORE = true), ALPHA_BLEND_FIRST_K (CORE only), OIT_BLEND (TAIL only, K unused)
// BINNED: the lists are in bins of depth.  A list by index is settled by the insertion itself: its walk looks for no equal depths, which costs a turn
// of two Gaussians twelve vector and fourteen scalar instructions (the launch alone: HYBRID 100 k at 1280x720
// 110.6 -> 102.8 us, FIRST_K 70 k at 1920x1080 105.3 -> 100.6).
template <int K, int MODE, bool BINNED>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(K <= 16 ? 5 : 2))) max_weights_tile_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
    uint32_t *__restrict__ max_weights, uint32_t width, uint32_t height, uint32_t grid_w, float weight_threshold, const uint32_t *__restrict__ tile_order,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, uint32_t *__restrict__ spare)
{
    constexpr bool kCore = MODE != HTGS_MODE_OIT_BLEND;
    constexpr bool kTail = MODE != HTGS_MODE_ALPHA_BLEND_FIRST_K;
    constexpr int KS = kCore ? K : 1;
    __shared__ TileStageQ st;
    __shared__ QuadrantLists ql;
    const uint32_t tile = block_tile(tile_order);
    const uint32_t lane = threadIdx.x;
    {
        // a tile with a very long list is left to the kernels that share a list between waves and workgroups
        const uint32_t length = ranges[2 * tile + 1] - ranges[2 * tile];
        const uint32_t long_threshold = threshold.get(long_tiles);
        if (long_tiles != nullptr && length > long_threshold) {
            constexpr uint32_t part_words = MODE == HTGS_MODE_HYBRID_BLEND ? long_part_words<KS>() : MODE == HTGS_MODE_OIT_BLEND ? kOitPartWords : first_k_part_words<KS>();
            if (lane == 0) long_tile_enter(long_tiles, tile, gridDim.x, length, threshold.least_part(long_threshold), part_words, part_floor.get(gridDim.x), long_threshold, threshold.counters);
            return;
        }
    }
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    const bool inside = px.inside;
    const PixelTerms pt = px.pt;
    const float cx = px.cx, cy = px.cy;

    float alpha_sum, T_tail;
    CoreTie tie;
    tie.init();
    float ca[KS], cd[KS];
    uint32_t ci[KS];
    const uint32_t first = ranges[2 * tile], last = ranges[2 * tile + 1];
    // the walk by the reference's insertion; AGAIN: over a list by index, for the pixels of pixel_lanes
    const auto walk = [&](auto again, const uint32_t *list, uint64_t pixel_lanes) {
        constexpr bool AGAIN = decltype(again)::value, NOTES = BINNED && !AGAIN;
        alpha_sum = 0.0f; T_tail = 1.0f;
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            ca[i] = 0.0f; cd[i] = __FLT_MAX__; ci[i] = 0xffffffffu;
            asm volatile("" : "+v"(cd[i]), "+v"(ca[i]), "+v"(ci[i]));      // one register per slot
        }
        const auto turn = [&](uint32_t addr) {
            // (TIES of hybrid_walk and first_k_walk)
            const auto enters = [&](float depth) { return NOTES ? depth <= cd[KS - 1] : depth < cd[KS - 1]; };
            TileFrag f;
            bool in_reach = tile_frag_cutoff<kStageSlots>(addr, pt, f);
            f.den_rcp = rcp_exact(f.den);
            float depth = 0.0f;
            if (MODE == HTGS_MODE_ALPHA_BLEND_FIRST_K) {
                depth = tile_frag_depth<kStageSlots>(addr, pt, f);
                in_reach = in_reach && enters(depth);
            }
            if (!(tile_frag_alpha<MODE>(stage_opacity<kStageSlots>(addr), f) && in_reach)) return;
            float alpha = f.alpha;
            if (MODE == HTGS_MODE_HYBRID_BLEND) depth = tile_frag_depth<kStageSlots>(addr, pt, f);
            if (kCore && (MODE == HTGS_MODE_ALPHA_BLEND_FIRST_K || (enters(depth) && alpha >= kMinAlphaCore))) {
                uint32_t idx = stage_index<kStageSlots>(addr);
                core_exchange_walk<KS>(depth, alpha, idx, cd, ca, ci);
                if (NOTES && alpha > 0.0f && depth == cd[KS - 1]) tie.note(true, depth, idx);
            }
            if (kTail) { alpha_sum += alpha; T_tail *= 1.0f - alpha; }
        };
        constexpr int CULL = AGAIN ? kCullPixels : kCullAlpha;
        if constexpr (kTail) tile_list_walk<MODE, kCore, CULL, true>(st, ql, prim, list, first, last, lane, cx, cy, turn, pixel_lanes);
        else tile_list_walk<MODE, kCore, CULL, true>(st, ql, prim, list, first, last, lane, cx, cy, turn, pixel_lanes, 1.0f, 64u, [&]() { return cd[KS - 1]; });
    };
    // the core's weights; returns the weight of a tail fragment per unit of alpha
    const auto weigh = [&]() {
        float T_core = 1.0f;
        if (kCore) {
#pragma unroll
            for (int i = 0; i < KS; ++i) {
                const float w = T_core * ca[i];
                T_core *= 1.0f - ca[i];
                if (T_core < kTransmittanceThreshold) T_core = 0.0f;
                if (!(w < weight_threshold)) raise_max(max_weights, ci[i], w);
            }
        }
        return kTail && alpha_sum >= weight_threshold ? (T_core * (1.0f - T_tail)) * (1.0f / alpha_sum) : 0.0f;
    };
    walk(std::false_type{}, inst, 0);
    float tail_weight = 0.0f;
    bool again = false;
    if constexpr (kCore && BINNED)
        again = settle_exact_core<MODE, KS, HTGS_PRIM_FLOATS / 4>(st, prim, lane, px, cd, ca, ci, tie, [&](float in, float out) {
            if (kTail) { alpha_sum += in - out; T_tail *= (1.0f - in) / (1.0f - out); }
        }) && inside;
    if (inside && !again) tail_weight = weigh();
    if constexpr (kCore && BINNED) {
        const uint64_t again_lanes = __ballot(again);
        if (again_lanes != 0) {
            walk(std::true_type{}, list_in_index_order<1>(inst, first, last, spare, ql.a[0], 0u, lane), again_lanes);
            if (again) tail_weight = weigh();
        }
    }
    if (!kTail) return;
    const bool active = inside && tail_weight >= weight_threshold;
    if (!__any(active)) return;
    // second walk over the tile's list: alpha * tail weight for every fragment that passes the cut-off (no alpha
    // threshold here, R/include/hybrid_blend/kernels/update_max_weights.cuh:197-204)
    tile_list_walk<MODE, false, kCullScaled, true>(st, ql, prim, inst, first, last, lane, cx, cy, [&](uint32_t addr) {
        TileFrag f;
        if (!active || !tile_frag_cutoff<kStageSlots>(addr, pt, f)) return;
        const float G = d_exp2((f.num * ModeCfg<MODE>::exp2_scale) * rcp_exact(f.den));
        const float a = stage_opacity<kStageSlots>(addr) * G;
        const float w = (a < kMaxFragmentAlpha ? a : kMaxFragmentAlpha) * tail_weight;
        if (!(w < weight_threshold)) raise_max(max_weights, stage_index<kStageSlots>(addr), w);
    }, 0, tail_cull_scale<MODE>(active ? tail_weight : 0.0f, weight_threshold));
}

__global__ void __launch_bounds__(256) max_weights_global_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
    uint32_t *__restrict__ max_weights, uint32_t width, uint32_t height, uint32_t grid_w, float weight_threshold, const uint32_t *__restrict__ tile_order)
{
    constexpr int MODE = HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING;
    __shared__ TileStage<256> st;
    __shared__ uint16_t s_reach[256];                  // per staged slot: the quadrants of the tile it can reach
    const uint32_t tile = block_tile(tile_order);
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const uint32_t x0 = (tile % grid_w) * 16, y0 = (tile / grid_w) * 16;
    uint32_t local_x, local_y;
    subtile_pixel(t, local_x, local_y);                // a wave = an 8x8 sub-tile, walked by quadrants
    const uint32_t x = x0 + local_x, y = y0 + local_y;
    const bool inside = x < width && y < height;
    const PixelTerms pt = pixel_terms(local_x, local_y, 16);
    const float cx = tile_centre(x0, 16), cy = tile_centre(y0, 16);
    float T = 1.0f;
    bool done = !inside;
    const uint32_t first = ranges[2 * tile], last = ranges[2 * tile + 1];
    for (uint32_t base = first; base < last; base += 256) {
        if (__syncthreads_count(done) == 256) break;
        s_reach[t] = (uint16_t)tile_stage_load<MODE, 256, false, kCullAlpha, true>(st, prim, inst, base + t, last, t, cx, cy);
        __syncthreads();
        const uint32_t stage_base = __builtin_amdgcn_readfirstlane(stage_address(st));
        subtile_walk(s_reach, stage_base, last - base < 256u ? last - base : 256u, wave, lane,
                     [&]() { return __ballot(!done) == 0; },
                     [&](uint32_t one, bool one_listed, uint32_t two, bool two_listed) {
            TileFrag f1, f2;
            bool pass1, pass2;
            tile_frag_exact_pair<MODE, 256>(one, two, pt, f1, f2, pass1, pass2);
            const auto joins = [&](uint32_t addr, const TileFrag &f) {
                const float w = T * f.alpha;
                T *= 1.0f - f.alpha;
                done = T < kTransmittanceThreshold;
                if (!(w < weight_threshold)) raise_max(max_weights, stage_index<256>(addr), w);
            };
            if (pass1 && one_listed && !done) joins(one, f1);
            if (pass2 && two_listed && !done) joins(two, f2);
        });
    }
}

// What the pass does with a pixel's finished core and tail when the tile's list was walked by the kernels for very long
// lists: the weights of the core's entries, and the weight of a tail fragment per unit of alpha into tail_weights[64 tile +
// lane] (0: no tail fragment of this pixel can reach the threshold) for the second walk (max_weights_tail_long_kernel).
struct MaxWeightsHybrid {
    uint32_t *max_weights;
    float *tail_weights;
    float weight_threshold;
    template <int K>
    __device__ __forceinline__ void operator()(const float4 *__restrict__, uint32_t tile, const TilePixel &, float (&)[K], float (&ca)[K], float (&ci)[K],
                                               HybridTail &tail) const
    {
        float T_core = 1.0f;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const float w = T_core * ca[i];
            T_core *= 1.0f - ca[i];
            if (T_core < kTransmittanceThreshold) T_core = 0.0f;
            if (ca[i] > 0.0f && !(w < weight_threshold)) raise_max(max_weights, float_to_bits(ci[i]), w);
        }
        float tail_weight = 0.0f;
        if (tail.alpha >= weight_threshold) tail_weight = (T_core * (1.0f - tail.T)) * (1.0f / tail.alpha);
        tail_weights[64u * (size_t)tile + (threadIdx.x & 63u)] = tail_weight >= weight_threshold ? tail_weight : 0.0f;
    }
};
struct MaxWeightsFirstK {
    uint32_t *max_weights;
    float weight_threshold;
    template <int K>
    __device__ __forceinline__ void operator()(const float4 *__restrict__, uint32_t, const TilePixel &, const float (&)[K], const float (&ca)[K],
                                               const uint32_t (&ci)[K]) const
    {
        float T_core = 1.0f;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const float w = T_core * ca[i];
            T_core *= 1.0f - ca[i];
            if (T_core < kTransmittanceThreshold) T_core = 0.0f;
            if (!(w < weight_threshold)) raise_max(max_weights, ci[i], w);
        }
    }
};
struct MaxWeightsOit {
    float *tail_weights;
    float weight_threshold;
    __device__ __forceinline__ void operator()(uint32_t tile, const TilePixel &, const OitSums &sum) const
    {
        float tail_weight = 0.0f;
        if (sum.alpha >= weight_threshold) tail_weight = (1.0f * (1.0f - sum.T)) * (1.0f / sum.alpha);
        tail_weights[64u * (size_t)tile + (threadIdx.x & 63u)] = tail_weight >= weight_threshold ? tail_weight : 0.0f;
    }
};

// After the kernels for very long lists have left the tail weights of such tiles: the tiles are entered on the list again,
// in parts, for the second walk.
__global__ void __launch_bounds__(256) max_weights_tail_enter_kernel(const uint32_t *__restrict__ ranges, uint32_t *__restrict__ long_tiles, uint32_t n_tiles,
                                                                    ListThreshold threshold, PartFloor part_floor)
{
    const uint32_t tile = blockIdx.x * 256 + threadIdx.x;
    if (tile >= n_tiles) return;
    const uint32_t length = ranges[2 * tile + 1] - ranges[2 * tile];
    const uint32_t long_threshold = threshold.get(long_tiles);
    if (length > long_threshold) long_tile_enter(long_tiles, tile, n_tiles, length, long_threshold, 0u, part_floor.get(n_tiles), long_threshold, threshold.counters);   // (parts of one threshold's length)
}
// The second walk (alpha * tail weight for every fragment that passes the cut-off) over the parts of the very long lists:
// a workgroup of four waves per part, every wave a share of it; the maximum is order independent, nothing to merge.
constexpr int kTailWaves = 4;
template <int MODE>
__global__ void __launch_bounds__(64 * kTailWaves) max_weights_tail_long_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, const uint32_t *long_tiles,
    uint32_t *__restrict__ max_weights, const float *__restrict__ tail_weights, uint32_t width, uint32_t height, uint32_t grid_w, float weight_threshold,
    ListThreshold threshold)
{
    __shared__ TileStageQ st[kTailWaves];
    __shared__ QuadrantLists ql[kTailWaves];
    __shared__ uint32_t s_next;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (long_tiles[0] == 0) return;                   // (the ordinary frame)
    const uint32_t long_threshold = threshold.get(long_tiles);
    uint32_t round = 0;
    LongEntry e;
    while (long_tile_take(long_tiles, ranges, long_threshold, threshold.counters, round, &s_next, e)) {
        const TilePixel px = quadrant_tile_pixel(e.tile, grid_w, lane, width, height);
        const PixelTerms pt = px.pt;
        const float tail_weight = px.inside ? tail_weights[64u * (size_t)e.tile + lane] : 0.0f;
        const bool active = tail_weight > 0.0f;
        if (__syncthreads_or(active) == 0) continue;
        uint32_t share_first, share_last;
        long_wave_share(e.first, e.last, wave, share_first, share_last, kTailWaves);
        tile_list_walk<MODE, false, kCullScaled, false>(st[wave], ql[wave], prim, inst, share_first, share_last, lane, px.cx, px.cy, [&](uint32_t addr) {
            TileFrag f;
            if (!active || !tile_frag_cutoff<kStageSlots>(addr, pt, f)) return;
            const float G = d_exp2((f.num * ModeCfg<MODE>::exp2_scale) * rcp_exact(f.den));
            const float a = stage_opacity<kStageSlots>(addr) * G;
            const float w = (a < kMaxFragmentAlpha ? a : kMaxFragmentAlpha) * tail_weight;
            if (!(w < weight_threshold)) raise_max(max_weights, stage_index<kStageSlots>(addr), w);
        }, 0, tail_cull_scale<MODE>(tail_weight, weight_threshold));
    }
}

// (lists are not split when there is no spare value buffer for what the parts leave behind)
static PartFloor part_floor_of(const htgs_frame *f, int sel, bool needs_spare)
{
    return PartFloor{ instance_count(f), needs_spare && f->vals[sel ^ 1] == nullptr ? 0u : 1u };
}
// the tiles with very long lists are taken by the kernels that share a list only when the caller provided the list for such
// tiles and, in the modes with a tail, the per-pixel scratch for the tail weights between the two walks
template <int MODE>
static bool shares_long_lists(const htgs_frame *f) { return f->long_tiles != nullptr && (MODE == HTGS_MODE_ALPHA_BLEND_FIRST_K || f->pixel_scratch != nullptr); }

template <int K, int MODE>
static void launch_tile(const htgs_frame *f, int sel, uint32_t *max_weights, float thr, uint32_t grid_w, uint32_t n_tiles)
{
    hipStream_t s = (hipStream_t)f->stream;
    const ListThreshold threshold = list_threshold(f);
    const bool shared = shares_long_lists<MODE>(f);
    const uint32_t w = (uint32_t)f->width, h = (uint32_t)f->height;
    const auto launch = [&](auto binned) {
        hipLaunchKernelGGL((max_weights_tile_kernel<K, MODE, decltype(binned)::value>), dim3(n_tiles), dim3(64), 0, s, f->ranges, f->vals[sel], (const float4 *)f->prim,
                           max_weights, w, h, grid_w, thr, f->tile_order, shared ? f->long_tiles : nullptr, threshold, part_floor_of(f, sel, true), binned_spare(f, sel));
    };
    if constexpr (MODE != HTGS_MODE_OIT_BLEND) {
        if (frame_depth_binned(f)) launch(std::true_type{});
        else launch(std::false_type{});
    } else launch(std::false_type{});
    if (!shared || !may_have_long_lists(f)) return;
    constexpr int REC4 = HTGS_PRIM_FLOATS / 4;
    if constexpr (MODE == HTGS_MODE_HYBRID_BLEND)
        launch_hybrid_long<K, false, REC4>(f, sel, grid_w, MaxWeightsHybrid{ max_weights, f->pixel_scratch, thr });
    else if constexpr (MODE == HTGS_MODE_ALPHA_BLEND_FIRST_K)
        launch_first_k_long<K, false, REC4>(f, sel, grid_w, MaxWeightsFirstK{ max_weights, thr });
    else
        launch_oit_long<false, REC4, false>(f, sel, grid_w, MaxWeightsOit{ f->pixel_scratch, thr });
    if constexpr (MODE != HTGS_MODE_ALPHA_BLEND_FIRST_K) {
        hipLaunchKernelGGL(max_weights_tail_enter_kernel, dim3((n_tiles + 255) / 256), dim3(256), 0, s, f->ranges, f->long_tiles, n_tiles, threshold,
                           part_floor_of(f, sel, false));
        hipLaunchKernelGGL(max_weights_tail_long_kernel<MODE>, dim3(1024), dim3(64 * kTailWaves), 0, s, f->ranges, f->vals[sel], (const float4 *)f->prim, f->long_tiles,
                           max_weights, f->pixel_scratch, w, h, grid_w, thr, threshold);
    }
}

template <int MODE>
static void dispatch_tile(const htgs_frame *f, int sel, uint32_t *mw, float thr, uint32_t grid_w, uint32_t n_tiles)
{
    switch (htgs_effective_k(f->K)) {
        case 32: launch_tile<32, MODE>(f, sel, mw, thr, grid_w, n_tiles); break;
        case 16: launch_tile<16, MODE>(f, sel, mw, thr, grid_w, n_tiles); break;
        case 8: launch_tile<8, MODE>(f, sel, mw, thr, grid_w, n_tiles); break;
        case 4: launch_tile<4, MODE>(f, sel, mw, thr, grid_w, n_tiles); break;
        case 2: launch_tile<2, MODE>(f, sel, mw, thr, grid_w, n_tiles); break;
        default: launch_tile<1, MODE>(f, sel, mw, thr, grid_w, n_tiles); break;
    }
}

}  // namespace htgs

using namespace htgs;

extern "C" int htgs_max_weights_front(const htgs_frame *f)
{
    if (!f) return fail(HTGS_ERR_ARGUMENT, "htgs_max_weights_front: null frame");
    htgs_frame t = *f;
    t.scale_modifier = 1.0f;      // update_max_weights.cuh:46: the scale modifier is not applied
    t.sh_0 = nullptr;             // no colours
    t.sh_rest = nullptr;
    t.active_sh_bases = 1;
    t.total_sh_bases = 0;
    t.clamp_info = nullptr;
    int rc = htgs_preprocess(&t);
    if (rc != HTGS_OK) return rc;
    return htgs_scan_offsets(&t);
}

extern "C" int htgs_max_weights_blend(const htgs_frame *f, int selector, float *max_weights, float weight_threshold)
{
    if (!f) return fail(HTGS_ERR_ARGUMENT, "htgs_max_weights_blend: null frame");
    if (f->mode < 0 || f->mode > 3) return fail(HTGS_ERR_MODE, "unsupported rasterizer mode");
    if (selector < 0 || selector > 1 || f->width <= 0 || f->height <= 0) return fail(HTGS_ERR_ARGUMENT, "htgs_max_weights_blend: bad argument");
    if (frame_prim_floats(f) != HTGS_PRIM_FLOATS) return fail(HTGS_ERR_ARGUMENT, "htgs_max_weights_blend: reads records of HTGS_PRIM_FLOATS floats (prim_floats)");
    if (f->n_instances == 0 || f->n_primitives == 0) return HTGS_OK;
    if (!f->ranges || !f->vals[selector] || !f->prim || !max_weights || (frame_depth_binned(f) && !f->vals[selector ^ 1]))
        return fail(HTGS_ERR_ARGUMENT, "htgs_max_weights_blend: null pointer");
    const int tile = tile_size(f->mode);
    const uint32_t grid_w = div_up(f->width, tile), grid_h = div_up(f->height, tile);
    const uint32_t n_tiles = grid_w * grid_h;
    uint32_t *mw = reinterpret_cast<uint32_t *>(max_weights);
    switch (f->mode) {
        case HTGS_MODE_HYBRID_BLEND: dispatch_tile<HTGS_MODE_HYBRID_BLEND>(f, selector, mw, weight_threshold, grid_w, n_tiles); break;
        case HTGS_MODE_ALPHA_BLEND_FIRST_K: dispatch_tile<HTGS_MODE_ALPHA_BLEND_FIRST_K>(f, selector, mw, weight_threshold, grid_w, n_tiles); break;
        case HTGS_MODE_OIT_BLEND: launch_tile<1, HTGS_MODE_OIT_BLEND>(f, selector, mw, weight_threshold, grid_w, n_tiles); break;
        default:
            hipLaunchKernelGGL(max_weights_global_kernel, dim3(n_tiles), dim3(256), 0, (hipStream_t)f->stream, f->ranges, f->vals[selector],
                               (const float4 *)f->prim, mw, (uint32_t)f->width, (uint32_t)f->height, grid_w, weight_threshold, f->tile_order);
            break;
    }
    return check_launch("max_weights");
}

extern "C" int htgs_max_weights_back(const htgs_frame *f, float *max_weights, float weight_threshold)
{
    int selector = 0;
    int rc = htgs_create_instances(f);
    if (rc != HTGS_OK) return rc;
    rc = htgs_sort_instances(f, &selector);
    if (rc != HTGS_OK) return rc;
    rc = htgs_extract_ranges(f, selector);
    if (rc != HTGS_OK) return rc;
    return htgs_max_weights_blend(f, selector, max_weights, weight_threshold);
}
