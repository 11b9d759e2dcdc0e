// Training forward blend of the four modes: unclamped [3,H,W] image plus the per-pixel records that the
// backward pass needs.  Restates blend_cu of R/include/hybrid_blend/kernels/forward.cuh:78-235,
// R/include/alpha_blend_first_k/kernels/forward.cuh:78-215,
// R/include/alpha_blend_global_ordering/kernels/forward.cuh:78-156 and
// R/include/oit_blend/kernels/forward.cuh:76-165.
//
// Records are pixel-minor ([slot][pixel]) so that a wave writes 64 consecutive words.  Where the reference
// leaves a record unwritten (tail with an alpha sum below 1/255, skipped core slots) zeros are stored, so that
// backward never reads indeterminate memory.
#include "blend_records.h"

namespace htgs {

// One wave per tile: the walk of the inference kernel (slots hold depth, alpha and index; colours are fetched at the end and
// the core's share of the colour sums is taken out there), exact arithmetic, 128-byte records.  A tile whose list is
// longer than long_threshold is left to blend_hybrid_long_kernel if the caller provided the list for such tiles.
// (A core of sixteen with three registers a slot does not fit the 96 registers of five waves per SIMD: 120 bytes a lane in scratch
// memory, some of it inside the walk.  Four waves without them: training step of 1 M Gaussians at 1920x1080, HYBRID K = 16, 1734 ->
// 1686 us, FIRST_K 1180 -> 1169, 300 k at 1280x720 481 -> 456.  Where five waves fit, as for the cores of up to eight, four cost 6 %.)
// BINNED: the lists are in bins of depth (a list by index is settled by the insertion itself, and nothing is looked for: max_weights_tile_kernel).
template <int K, bool BINNED>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(K <= 8 ? 5 : K <= 16 ? 4 : 3))) blend_hybrid_forward_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare, const HybridRecords finish)
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
    HybridTail tail;
    hybrid_tail_init(tail);
    float cd[K], ca[K], ci[K];                 // ci: the index's bit pattern
    hybrid_core_init<K>(cd, ca, ci);
    CoreTie tie;
    tie.init();
    hybrid_walk<K, false, true, BINNED, false, HTGS_PRIM_FLOATS_TRAIN / 4>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, cd, ca, ci, tail, &tie);
    const bool again = BINNED && settle_exact_core<HTGS_MODE_HYBRID_BLEND, K, HTGS_PRIM_FLOATS_TRAIN / 4>(st, prim, lane, px, cd, ca, ci, tie, tail_swap(tail, cd[K - 1])) && px.inside;
    const uint64_t again_lanes = __ballot(again);
    if (px.inside && !again) finish(prim, tile, px, cd, ca, ci, tail);
    if (again_lanes == 0) return;
    const uint32_t lane_again = fresh_lane();
    const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
    const uint32_t *const list = list_in_index_order<1>(inst, first, last, spare, ql.a[0], 0u, lane_again);
    hybrid_tail_init(tail);
    hybrid_core_init<K>(cd, ca, ci);
    hybrid_walk<K, false, true, false, true, HTGS_PRIM_FLOATS_TRAIN / 4>(st, ql, list, prim, first, last, lane_again, px_again.pt, px_again.cx, px_again.cy, cd, ca, ci, tail,
                                                                        nullptr, again_lanes);
    if ((again_lanes >> lane_again & 1ull) != 0) finish(prim, tile, px_again, cd, ca, ci, tail);
}

template <int K, bool BINNED>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(K <= 8 ? 5 : K <= 16 ? 4 : 2))) blend_first_k_forward_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare, const FirstKRecords finish)
{
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
    first_k_core_init<K>(cd, ca, ci);
    CoreTie tie;
    tie.init();
    first_k_walk<K, false, true, BINNED, HTGS_PRIM_FLOATS_TRAIN / 4>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, cd, ca, ci, &tie);
    const bool again = BINNED && settle_exact_core<HTGS_MODE_ALPHA_BLEND_FIRST_K, K, HTGS_PRIM_FLOATS_TRAIN / 4>(st, prim, lane, px, cd, ca, ci, tie, [](float, float) {}) && px.inside;
    const uint64_t again_lanes = __ballot(again);
    if (px.inside && !again) finish(prim, tile, px, cd, ca, ci);
    if (again_lanes == 0) return;
    const uint32_t lane_again = fresh_lane();
    const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
    const uint32_t *const list = list_in_index_order<1>(inst, first, last, spare, ql.a[0], 0u, lane_again);
    first_k_core_init<K>(cd, ca, ci);
    first_k_walk<K, false, true, false, HTGS_PRIM_FLOATS_TRAIN / 4, true>(st, ql, list, prim, first, last, lane_again, px_again.pt, px_again.cx, px_again.cy, cd, ca, ci,
                                                                         nullptr, again_lanes);
    if ((again_lanes >> lane_again & 1ull) != 0) finish(prim, tile, px_again, cd, ca, ci);
}

__global__ void __launch_bounds__(64) blend_oit_forward_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, const OitRecords finish)
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
    oit_walk<false, true, HTGS_PRIM_FLOATS_TRAIN / 4, false>(st, ql, inst, prim, first, last, lane, px.pt, px.cx, px.cy, sum);
    if (!px.inside) return;
    finish(tile, px, sum);
}

__global__ void __launch_bounds__(256) blend_global_forward_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim,
    float *__restrict__ image, uint32_t width, uint32_t height, uint32_t grid_w, const uint32_t *__restrict__ tile_order)
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
    float r = 0.0f, g = 0.0f, b = 0.0f, T = 1.0f;
    bool done = !inside;

    const uint32_t first = ranges[2 * tile], last = ranges[2 * tile + 1];
    for (uint32_t base = first; base < last; base += 256) {
        if (__syncthreads_count(done) == 256) break;
        s_reach[t] = (uint16_t)tile_stage_load<MODE, 256, false, kCullAlpha, true, HTGS_PRIM_FLOATS_TRAIN / 4>(st, prim, inst, base + t, last, t, cx, cy);
        __syncthreads();
        const uint32_t stage_base = __builtin_amdgcn_readfirstlane(stage_address(st));
        subtile_walk(s_reach, stage_base, last - base < 256u ? last - base : 256u, wave, lane,
                     [&]() { return __ballot(!done) == 0; },
                     [&](uint32_t one, bool one_listed, uint32_t two, bool two_listed) {
            TileFrag f1, f2;
            bool pass1, pass2;
            tile_frag_exact_pair<MODE, 256>(one, two, pt, f1, f2, pass1, pass2);
            const auto joins = [&](uint32_t addr, const TileFrag &f) {
                const float4 col = stage_row<256, 5>(addr);
                const float bw = T * f.alpha;
                r = __builtin_fmaf(bw, col.x, r);
                g = __builtin_fmaf(bw, col.y, g);
                b = __builtin_fmaf(bw, col.z, b);
                T *= 1.0f - f.alpha;
                done = T < kTransmittanceThreshold;
            };
            if (pass1 && one_listed && !done) joins(one, f1);
            if (pass2 && two_listed && !done) joins(two, f2);
        });
    }
    if (!inside) return;
    const size_t pix = (size_t)width * y + x, np = (size_t)width * height;
    image[pix] = r; image[np + pix] = g; image[2 * np + pix] = b;
}

// (lists are not split without a spare value buffer to leave the parts' results in)
static PartFloor forward_part_floor(const htgs_frame *f, int sel) { return PartFloor{ instance_count(f), f->vals[sel ^ 1] != nullptr ? 1u : 0u }; }

template <int K>
static void launch_hybrid_forward(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    constexpr int REC4 = HTGS_PRIM_FLOATS_TRAIN / 4;
    const HybridRecords finish = { f->image, f->core_idx, (float4 *)f->core_info, f->tail_info, (uint32_t)f->width, (uint32_t)f->height, (size_t)n_tiles * 64u };
    const auto kernel = frame_depth_binned(f) ? blend_hybrid_forward_kernel<K, true> : blend_hybrid_forward_kernel<K, false>;
    hipLaunchKernelGGL(kernel, dim3(n_tiles), dim3(64), 0, (hipStream_t)f->stream, f->ranges, f->vals[sel], (const float4 *)f->prim,
                       (uint32_t)f->width, (uint32_t)f->height, grid_w, f->long_tiles, list_threshold(f), forward_part_floor(f, sel), f->tile_order, binned_spare(f, sel), finish);
    launch_hybrid_long<K, false, REC4>(f, sel, grid_w, finish);
}
template <int K>
static void launch_first_k_forward(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    constexpr int REC4 = HTGS_PRIM_FLOATS_TRAIN / 4;
    const FirstKRecords finish = { f->image, f->core_idx, (float4 *)f->core_info, (uint32_t)f->width, (uint32_t)f->height, (size_t)n_tiles * 64u };
    const auto kernel = frame_depth_binned(f) ? blend_first_k_forward_kernel<K, true> : blend_first_k_forward_kernel<K, false>;
    hipLaunchKernelGGL(kernel, dim3(n_tiles), dim3(64), 0, (hipStream_t)f->stream, f->ranges, f->vals[sel], (const float4 *)f->prim,
                       (uint32_t)f->width, (uint32_t)f->height, grid_w, f->long_tiles, list_threshold(f), forward_part_floor(f, sel), f->tile_order, binned_spare(f, sel), finish);
    launch_first_k_long<K, false, REC4>(f, sel, grid_w, finish);
}
static void launch_oit_forward(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    constexpr int REC4 = HTGS_PRIM_FLOATS_TRAIN / 4;
    const OitRecords finish = { f->image, f->tail_info, (uint32_t)f->width, (uint32_t)f->height, (size_t)n_tiles * 64u };
    hipLaunchKernelGGL(blend_oit_forward_kernel, dim3(n_tiles), dim3(64), 0, (hipStream_t)f->stream, f->ranges, f->vals[sel], (const float4 *)f->prim,
                       (uint32_t)f->width, (uint32_t)f->height, grid_w, f->long_tiles, list_threshold(f), forward_part_floor(f, sel), f->tile_order, finish);
    launch_oit_long<false, REC4, false>(f, sel, grid_w, finish);
}

}  // namespace htgs

using namespace htgs;

extern "C" int htgs_blend_forward(const htgs_frame *f, int selector)
{
    if (!f) return fail(HTGS_ERR_ARGUMENT, "htgs_blend_forward: null frame");
    if (f->mode < 0 || f->mode > 3) return fail(HTGS_ERR_MODE, "unsupported rasterizer mode");
    if (selector < 0 || selector > 1 || f->width <= 0 || f->height <= 0) return fail(HTGS_ERR_ARGUMENT, "htgs_blend_forward: bad argument");
    if (frame_depth_ordered(f)) return fail(HTGS_ERR_ARGUMENT, "htgs_blend_forward: depth_order is for the inference entry points");
    if (f->prim_floats != HTGS_PRIM_FLOATS_TRAIN) return fail(HTGS_ERR_ARGUMENT, "htgs_blend_forward: the training kernels read records of HTGS_PRIM_FLOATS_TRAIN floats (prim_floats)");
    const bool needs_core = f->mode == HTGS_MODE_HYBRID_BLEND || f->mode == HTGS_MODE_ALPHA_BLEND_FIRST_K;
    const bool needs_tail = f->mode == HTGS_MODE_HYBRID_BLEND || f->mode == HTGS_MODE_OIT_BLEND;
    if (!f->ranges || !f->image || (f->n_instances > 0 && (!f->vals[selector] || !f->prim || (frame_depth_binned(f) && !f->vals[selector ^ 1]))) ||
        (needs_core && (!f->core_idx || !f->core_info)) || (needs_tail && !f->tail_info))
        return fail(HTGS_ERR_ARGUMENT, "htgs_blend_forward: null pointer");
    const int tile = tile_size(f->mode);
    const uint32_t grid_w = div_up(f->width, tile), grid_h = div_up(f->height, tile);
    const uint32_t n_tiles = grid_w * grid_h;
    hipStream_t s = (hipStream_t)f->stream;
    const int K = htgs_effective_k(f->K);
    if (blend_forward_waves(f, selector, grid_w, n_tiles)) return check_launch("blend_forward");
    switch (f->mode) {
        case HTGS_MODE_HYBRID_BLEND:
            switch (K) {
                case 32: launch_hybrid_forward<32>(f, selector, grid_w, n_tiles); break;
                case 16: launch_hybrid_forward<16>(f, selector, grid_w, n_tiles); break;
                case 8: launch_hybrid_forward<8>(f, selector, grid_w, n_tiles); break;
                case 4: launch_hybrid_forward<4>(f, selector, grid_w, n_tiles); break;
                case 2: launch_hybrid_forward<2>(f, selector, grid_w, n_tiles); break;
                default: launch_hybrid_forward<1>(f, selector, grid_w, n_tiles); break;
            }
            break;
        case HTGS_MODE_ALPHA_BLEND_FIRST_K:
            switch (K) {
                case 32: launch_first_k_forward<32>(f, selector, grid_w, n_tiles); break;
                case 16: launch_first_k_forward<16>(f, selector, grid_w, n_tiles); break;
                case 8: launch_first_k_forward<8>(f, selector, grid_w, n_tiles); break;
                case 4: launch_first_k_forward<4>(f, selector, grid_w, n_tiles); break;
                case 2: launch_first_k_forward<2>(f, selector, grid_w, n_tiles); break;
                default: launch_first_k_forward<1>(f, selector, grid_w, n_tiles); break;
            }
            break;
        case HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING:
            hipLaunchKernelGGL(blend_global_forward_kernel, dim3(n_tiles), dim3(256), 0, s, f->ranges, f->vals[selector],
                               (const float4 *)f->prim, f->image, (uint32_t)f->width, (uint32_t)f->height, grid_w, f->tile_order);
            break;
        default:
            launch_oit_forward(f, selector, grid_w, n_tiles);
            break;
    }
    return check_launch("blend_forward");
}
