// Small grids: several waves per tile.
//
// The kernels with one wave per tile are bound by the issue rate of their instructions as long as every SIMD has five waves
// to choose from.  A grid of a few thousand tiles leaves it one or two, and then a launch lasts as long as its longest
// list: one wave takes 0.25 us for a turn of the walk, whose instructions depend on one another, and most of the device is
// idle beside it.  Here a workgroup of WAVES waves takes a tile: every wave walks a share of the list (every
// WAVES-th batch) into a core and a tail of its own, and the shares are merged pairwise through LDS.
// As in the kernels for very long lists, which entry of exactly equal depth stays is not the reference's choice then, so the
// walks and the merges note the entries as deep as the last one of the core, such pixels are settled from their cores (settle_core), and
// those with more than two fragments of a depth are walked again in one piece by the reference's insertion.  Sums come out in another order than in a single walk (rounding).
// Tiles x waves, one -> four waves: 10 k Gaussians at 256x256, K = 4: 38 -> 25 us; training pass of 20 k at 400x304, K = 16: 81 -> 36 us.
// From some number of tiles on, the workgroup's LDS, which is held until its first wave has finished the pixels, and the merging
// cost more than the shorter lists give (1920x1080 HYBRID 965 -> 1137 us); htgs_run's lines are in run.hip (waves_of).
#pragma once

#include "blend_long.h"

namespace htgs {

// The share of wave `wave` of a list: every WAVES-th batch from its own on.  (In a list in bins of depth the nearer Gaussians, which
// reach more of a tile, come first: contiguous shares would leave the first wave with the most work.)  The batches are as large as
// they come out if every wave has the same number of them, 64 at most.  Waves without a batch are the last ones.
// Small frames have lists of less than a batch, which one wave walked alone, and a list of 70 was 64 and 6.  Below the least share another
// wave's core costs more to merge than its turns take.  Whole passes, batches of 64 -> shares of 32 and more -> of 8 and 16 as here: HYBRID
// K = 4 10 k at 256x256 46.1 -> 43.9 -> 42.5 us, OIT 334 k at 1237x821 151.0 -> 148.7 -> 148.3, training of
// 20 k at 660x834, HYBRID K = 4, 232 -> 222 -> 219, of 244 k at 1694x265, K = 16, 317 -> 311.6 -> 310.
// FIRST_K's waves know from one another how deep they have to look (SharedDepth), and merge more than they
// spare below twice that (K = 4, 108 k at 451x862: 86.3 -> 85.4 -> 85.9).
constexpr uint32_t least_share(int K, bool tail) { return K > 16 ? 64u : (K <= 4 ? 8u : 16u) * (tail ? 1u : 2u); }
struct TileShare {
    uint32_t first, per;                   // per: where the next wave's begins
};
template <int WAVES, uint32_t LEAST>
__device__ __forceinline__ TileShare tile_share(uint32_t first, uint32_t last, uint32_t wave)
{
    const uint32_t n = last - first, rounds = n > 64u * WAVES ? (n + 64u * WAVES - 1u) / (64u * WAVES) : 1u;
    const uint32_t batch = (n + rounds * WAVES - 1u) / (rounds * WAVES), per = batch > LEAST ? batch : LEAST;
    return TileShare{ first + per * wave, per };
}
// The pairwise merging: give(buffer) is called by the wave that hands its share over, take(buffer) by the one that receives
// it (all lanes; buffer: 64-lane rows, one buffer per pair of waves); false: the wave is done.  The buffers lie over the stages,
// which nobody reads any more.
template <int WAVES, uint32_t ROWS, typename Give, typename Take>
__device__ __forceinline__ bool merge_shares(unsigned char *lds, const TileShare &share, uint32_t first, uint32_t last, uint32_t wave, Give &&give, Take &&take)
{
    float *buffers = reinterpret_cast<float *>(lds);
    // (every wave goes through the same barriers: which shares are empty is the same for all of them)
    for (uint32_t step = 1; step < (uint32_t)WAVES; step *= 2) {
        if (first + share.per * step >= last) break;
        float *buffer = buffers + (size_t)(wave / (2u * step)) * ROWS * 64u;
        const bool other = (wave & (2u * step - 1u)) == step, mine = (wave & (2u * step - 1u)) == 0u;
        __syncthreads();
        if (other && first + share.per * wave < last) give(buffer);
        __syncthreads();
        if (mine && first + share.per * (wave + step) < last) take(buffer);
    }
    return wave == 0;
}
// The tile a workgroup takes; false: its list is very long and goes to the kernels for those.
__device__ __forceinline__ bool tile_of_waves(const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ long_tiles,
                                              const ListThreshold &threshold, const PartFloor &part_floor, uint32_t part_words, uint32_t &tile, uint32_t &first, uint32_t &last)
{
    tile = block_tile(tile_order);
    first = ranges[2 * tile]; last = ranges[2 * tile + 1];
    const uint32_t long_threshold = threshold.get(long_tiles);
    if (long_tiles == nullptr || last - first <= long_threshold) return true;
    if (threadIdx.x == 0) long_tile_enter(long_tiles, tile, gridDim.x, last - first, threshold.least_part(long_threshold), part_words, part_floor.get(gridDim.x),
                                          long_threshold, threshold.counters);
    return false;
}

// HYBRID_BLEND, the core as keys (inference)
template <int WAVES, int K, bool FAST, typename Finish>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(K > 16 && !FAST ? 3 : K > 16 || (K == 16 && !FAST && WAVES == 4) ? 4 : 5))) blend_hybrid_waves_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare, const Finish finish)
{
    constexpr uint32_t kRows = 2 * K + 7;
    __shared__ __attribute__((aligned(16))) unsigned char lds[shared_walk_lds<WAVES, kRows>()];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    uint32_t tile, first, last;
    if (!tile_of_waves(ranges, tile_order, long_tiles, threshold, part_floor, long_part_words<K>(), tile, first, last)) return;
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    const TileShare share = tile_share<WAVES, least_share(K, true)>(first, last, wave);
    HybridTail tail;
    hybrid_tail_init(tail);
    CoreKey core[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        core[i] = make_key(__FLT_MAX__, 0u);
        asm volatile("" : "+v"(core[i]));
    }
    KeyNotes notes;
    notes.init();
    const KeyFormat fmt = key_format(last > first ? last - first : 1u);
    // (places count from the tile's first instance, as in the single walk)
    hybrid_key_walk<K, FAST, false, HTGS_PRIM_FLOATS / 4, true>(wave_stage(lds, wave), wave_lists<WAVES>(lds, wave), inst, prim, share.first, last, lane, px.pt, px.cx, px.cy,
                                                                core, tail, notes, fmt, first, ListStep(share.per * WAVES, share.per));
    CoreTie tie;
    if constexpr (FAST) tie.init();
    else tie = noted_ties<HTGS_MODE_HYBRID_BLEND, HTGS_PRIM_FLOATS / 4>(wave_stage(lds, wave), prim, inst, first, last, lane, px, notes, fmt);
    if (!merge_shares<WAVES, kRows>(lds, share, first, last, wave,
            [&](float *to) { give_key_core<K>(to + lane, core); give_tail<2 * K>(to + lane, tail); if (!FAST) give_tie<2 * K + 6>(to + lane, tie, key_depth(core[K - 1])); },
            [&](const float *from) {
                if (!FAST) take_tie<2 * K + 6, 2 * (K - 1)>(from + lane, tie);
                merge_key_cores<K, !FAST>(from + lane, core, tie, fmt, [&](CoreKey out) { hybrid_tail_add<FAST>(tail, key_depth(out), key_alpha(key_low(out), fmt)); });
                take_tail<2 * K>(from + lane, tail);
            })) return;
    float cd[K], ca[K], ci[K];
    if constexpr (FAST) {
        if (!px.inside) return;
        key_core_unpack<K>(core, inst, first, last, cd, ca, ci, fmt);
        finish(prim, tile, px, cd, ca, ci, tail);
    } else {
        wave_lds_sync();
        const bool again = settle_keys<HTGS_MODE_HYBRID_BLEND, K, HTGS_PRIM_FLOATS / 4>(wave_stage(lds, 0), prim, inst, first, last, lane, px, core, tie, fmt, tail_swap(tail, key_depth(core[K - 1])));
        const uint64_t again_lanes = __ballot(again);
        key_core_unpack<K>(core, inst, first, last, cd, ca, ci, fmt);
        if (px.inside && !again) finish(prim, tile, px, cd, ca, ci, tail);
        if (again_lanes == 0) return;
        const uint32_t lane_again = fresh_lane();
        const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
        const uint32_t *const list = spare != nullptr ? list_in_index_order<1>(inst, first, last, spare, wave_lists<WAVES>(lds, 0).a[0], 0u, lane_again) : inst;
        hybrid_tail_init(tail);
        hybrid_core_init<K>(cd, ca, ci);
        wave_lds_sync();
        hybrid_walk<K, false, false, false, true>(wave_stage(lds, 0), wave_lists<WAVES>(lds, 0), list, prim, first, last, lane_again, px_again.pt, px_again.cx, px_again.cy, cd, ca,
                                                  ci, tail, nullptr, again_lanes);
        if ((again_lanes >> lane_again & 1ull) != 0) finish(prim, tile, px_again, cd, ca, ci, tail);
    }
}
// HYBRID_BLEND, three registers a slot (the training pass)
template <int WAVES, int K, int REC4, typename Finish>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(K <= 16 ? 4 : 3))) blend_hybrid_waves_exact_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare, const Finish finish)
{
    constexpr uint32_t kRows = 3 * K + 7;
    __shared__ __attribute__((aligned(16))) unsigned char lds[shared_walk_lds<WAVES, kRows>()];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    uint32_t tile, first, last;
    if (!tile_of_waves(ranges, tile_order, long_tiles, threshold, part_floor, long_part_words<K>(), tile, first, last)) return;
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    const TileShare share = tile_share<WAVES, least_share(K, true)>(first, last, wave);
    HybridTail tail;
    hybrid_tail_init(tail);
    float cd[K], ca[K], ci[K];
    hybrid_core_init<K>(cd, ca, ci);
    CoreTie tie;
    tie.init();
    hybrid_walk<K, false, false, true, false, REC4>(wave_stage(lds, wave), wave_lists<WAVES>(lds, wave), inst, prim, share.first, last, lane, px.pt, px.cx, px.cy, cd, ca, ci,
                                                    tail, &tie, 0, ListStep(share.per * WAVES, share.per));
    if (!merge_shares<WAVES, kRows>(lds, share, first, last, wave,
            [&](float *to) { hybrid_put<K>(to, lane, cd, ca, ci, tail, tie); },
            [&](const float *from) { hybrid_merge<K, false>(from, lane, cd, ca, ci, tail, tie); })) return;
    // (a list by index that one wave walked is settled: the insertion was the reference's)
    wave_lds_sync();
    const bool again = (first + share.per < last || spare != nullptr) &&
                       settle_exact_core<HTGS_MODE_HYBRID_BLEND, K, REC4>(wave_stage(lds, 0), prim, lane, px, cd, ca, ci, tie, tail_swap(tail, cd[K - 1])) && px.inside;
    const uint64_t again_lanes = __ballot(again);
    if (px.inside && !again) finish(prim, tile, px, cd, ca, ci, tail);
    if (again_lanes == 0) return;
    const uint32_t lane_again = fresh_lane();
    const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
    const uint32_t *const list = spare != nullptr ? list_in_index_order<1>(inst, first, last, spare, wave_lists<WAVES>(lds, 0).a[0], 0u, lane_again) : inst;
    hybrid_tail_init(tail);
    hybrid_core_init<K>(cd, ca, ci);
    wave_lds_sync();
    hybrid_walk<K, false, false, false, true, REC4>(wave_stage(lds, 0), wave_lists<WAVES>(lds, 0), list, prim, first, last, lane_again, px_again.pt, px_again.cx, px_again.cy, cd, ca,
                                                    ci, tail, nullptr, again_lanes);
    if ((again_lanes >> lane_again & 1ull) != 0) finish(prim, tile, px_again, cd, ca, ci, tail);
}
// ALPHA_BLEND_FIRST_K, the core as keys (inference, exact arithmetic)
template <int WAVES, int K, typename Finish>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(K <= 16 ? 5 : 3))) blend_first_k_waves_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare, const Finish finish)
{
    constexpr uint32_t kRows = 2 * K + 1;
    __shared__ __attribute__((aligned(16))) unsigned char lds[shared_walk_lds<WAVES, kRows>()];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    uint32_t tile, first, last;
    if (!tile_of_waves(ranges, tile_order, long_tiles, threshold, part_floor, first_k_part_words<K>(), tile, first, last)) return;
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    const TileShare share = tile_share<WAVES, least_share(K, false)>(first, last, wave);
    CoreKey core[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        core[i] = make_key(__FLT_MAX__, 0u);
        asm volatile("" : "+v"(core[i]));
    }
    KeyNotes notes;
    notes.init();
    const KeyFormat fmt = key_format(last > first ? last - first : 1u);
    __shared__ float s_depth[WAVES][64];
    const SharedDepth<WAVES, K> shared = { s_depth, wave, lane };
    shared.init();
    __syncthreads();
    first_k_key_walk<K, false>(wave_stage(lds, wave), wave_lists<WAVES>(lds, wave), inst, prim, share.first, last, lane, px.pt, px.cx, px.cy, core, notes, fmt, first, ListStep(share.per * WAVES, share.per), shared);
    CoreTie tie = noted_ties<HTGS_MODE_ALPHA_BLEND_FIRST_K, HTGS_PRIM_FLOATS / 4>(wave_stage(lds, wave), prim, inst, first, last, lane, px, notes, fmt);
    if (!merge_shares<WAVES, kRows>(lds, share, first, last, wave,
            [&](float *to) { give_key_core<K>(to + lane, core); give_tie<2 * K>(to + lane, tie, key_depth(core[K - 1])); },
            [&](const float *from) {
                take_tie<2 * K, 2 * (K - 1)>(from + lane, tie);
                merge_key_cores<K, true>(from + lane, core, tie, fmt, [](CoreKey) {});
            })) return;
    float cd[K], ca[K];
    uint32_t ci[K];
    wave_lds_sync();
    const bool again = settle_keys<HTGS_MODE_ALPHA_BLEND_FIRST_K, K, HTGS_PRIM_FLOATS / 4>(wave_stage(lds, 0), prim, inst, first, last, lane, px, core, tie, fmt, [](float, float) {});
    const uint64_t again_lanes = __ballot(again);
    first_k_core_unpack<K>(core, inst, first, last, cd, ca, ci, fmt);
    if (px.inside && !again) finish(prim, tile, px, cd, ca, ci);
    if (again_lanes == 0) return;
    const uint32_t lane_again = fresh_lane();
    const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
    const uint32_t *const list = spare != nullptr ? list_in_index_order<1>(inst, first, last, spare, wave_lists<WAVES>(lds, 0).a[0], 0u, lane_again) : inst;
    first_k_core_init<K>(cd, ca, ci);
    wave_lds_sync();
    first_k_walk<K, false, false, false, HTGS_PRIM_FLOATS / 4, true>(wave_stage(lds, 0), wave_lists<WAVES>(lds, 0), list, prim, first, last, lane_again, px_again.pt, px_again.cx,
                                                                     px_again.cy, cd, ca, ci, nullptr, again_lanes);
    if ((again_lanes >> lane_again & 1ull) != 0) finish(prim, tile, px_again, cd, ca, ci);
}
// ALPHA_BLEND_FIRST_K, three registers a slot: the training pass, and the image-only path (FAST)
template <int WAVES, int K, bool FAST, int REC4, typename Finish>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(K <= 16 ? 4 : 3))) blend_first_k_waves_exact_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare, const Finish finish)
{
    constexpr uint32_t kRows = 3 * K + 1;
    __shared__ __attribute__((aligned(16))) unsigned char lds[shared_walk_lds<WAVES, kRows>()];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    uint32_t tile, first, last;
    if (!tile_of_waves(ranges, tile_order, long_tiles, threshold, part_floor, first_k_part_words<K>(), tile, first, last)) return;
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    const TileShare share = tile_share<WAVES, least_share(K, false)>(first, last, wave);
    float cd[K], ca[K];
    uint32_t ci[K];
    first_k_core_init<K>(cd, ca, ci);
    CoreTie tie;
    tie.init();
    __shared__ float s_depth[WAVES][64];
    const SharedDepth<WAVES, K> shared = { s_depth, wave, lane };
    shared.init();
    __syncthreads();
    first_k_walk<K, FAST, false, true, REC4, false>(wave_stage(lds, wave), wave_lists<WAVES>(lds, wave), inst, prim, share.first, last, lane, px.pt, px.cx, px.cy, cd, ca, ci, &tie, 0, ListStep(share.per * WAVES, share.per), shared);
    if (!merge_shares<WAVES, kRows>(lds, share, first, last, wave,
            [&](float *to) { first_k_put<K>(to, lane, cd, ca, ci, tie); },
            [&](const float *from) { first_k_merge<K>(from, lane, cd, ca, ci, tie); })) return;
    wave_lds_sync();
    bool again;
    if constexpr (FAST) again = px.inside && first + share.per < last && core_tied<K>(cd, ca, tie);       // (in the list's own order)
    else again = (first + share.per < last || spare != nullptr) &&
                 settle_exact_core<HTGS_MODE_ALPHA_BLEND_FIRST_K, K, REC4>(wave_stage(lds, 0), prim, lane, px, cd, ca, ci, tie, [](float, float) {}) && px.inside;
    const uint64_t again_lanes = __ballot(again);
    if (px.inside && !again) finish(prim, tile, px, cd, ca, ci);
    if (again_lanes == 0) return;
    const uint32_t lane_again = fresh_lane();
    const TilePixel px_again = quadrant_tile_pixel(tile, grid_w, lane_again, width, height);
    const uint32_t *const list = !FAST && spare != nullptr ? list_in_index_order<1>(inst, first, last, spare, wave_lists<WAVES>(lds, 0).a[0], 0u, lane_again) : inst;
    first_k_core_init<K>(cd, ca, ci);
    wave_lds_sync();
    first_k_walk<K, FAST, false, false, REC4, true>(wave_stage(lds, 0), wave_lists<WAVES>(lds, 0), list, prim, first, last, lane_again, px_again.pt, px_again.cx, px_again.cy, cd, ca,
                                                    ci, nullptr, again_lanes);
    if ((again_lanes >> lane_again & 1ull) != 0) finish(prim, tile, px_again, cd, ca, ci);
}
// OIT_BLEND
template <int WAVES, bool FAST, int REC4, typename Finish, bool DEPTH = !FAST>
__global__ void __launch_bounds__(64 * WAVES) blend_oit_waves_kernel(
    const uint32_t *__restrict__ ranges, const uint32_t *__restrict__ inst, const float4 *__restrict__ prim, uint32_t width, uint32_t height, uint32_t grid_w,
    uint32_t *__restrict__ long_tiles, ListThreshold threshold, PartFloor part_floor, const uint32_t *__restrict__ tile_order, uint32_t *__restrict__ spare, const Finish finish)
{
    constexpr uint32_t kRows = 6;
    __shared__ __attribute__((aligned(16))) unsigned char lds[shared_walk_lds<WAVES, kRows>()];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    uint32_t tile, first, last;
    if (!tile_of_waves(ranges, tile_order, long_tiles, threshold, part_floor, kOitPartWords, tile, first, last)) return;
    const TilePixel px = quadrant_tile_pixel(tile, grid_w, lane, width, height);
    const TileShare share = tile_share<WAVES, least_share(1, true)>(first, last, wave);
    OitSums sum = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 1.0f };
    oit_walk<FAST, false, REC4, DEPTH>(wave_stage(lds, wave), wave_lists<WAVES>(lds, wave), inst, prim, share.first, last, lane, px.pt, px.cx, px.cy, sum, ListStep(share.per * WAVES, share.per));
    if (!merge_shares<WAVES, kRows>(lds, share, first, last, wave,
            [&](float *to) {
                to += lane;
                to[0] = sum.a0; to[64] = sum.a1; to[128] = sum.a2; to[192] = sum.a3; to[256] = sum.alpha; to[320] = sum.T;
            },
            [&](const float *from) {
                from += lane;
                sum.a0 += from[0]; sum.a1 += from[64]; sum.a2 += from[128]; sum.a3 += from[192]; sum.alpha += from[256]; sum.T *= from[320];
            })) return;
    if (px.inside) finish(tile, px, sum);
}

// the host side of the two launches (inference, training)
inline bool takes_waves(const htgs_frame *f)
{
    return (f->waves_per_tile == 2 || f->waves_per_tile == 4) && f->long_tiles && most_threshold(f) <= kPackedListMost && f->mode != HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING;
}
template <int WAVES, typename Main, typename Finish>
static void launch_waves(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles, Main main, const Finish &finish)
{
    hipStream_t s = (hipStream_t)f->stream;
    const PartFloor floor = { instance_count(f), f->vals[sel ^ 1] != nullptr ? 1u : 0u };
    hipLaunchKernelGGL(main, dim3(n_tiles), dim3(64 * WAVES), 0, s, f->ranges, f->vals[sel], (const float4 *)f->prim, (uint32_t)f->width, (uint32_t)f->height, grid_w,
                       f->long_tiles, list_threshold(f), floor, f->tile_order, binned_spare(f, sel), finish);
}
// calls launch(std::integral_constant<int, K>{}) for the core size K that f asks for
template <typename Launch>
inline void with_core_size(const htgs_frame *f, Launch &&launch)
{
    switch (htgs_effective_k(f->K)) {
        case 32: launch(std::integral_constant<int, 32>{}); break;
        case 16: launch(std::integral_constant<int, 16>{}); break;
        case 8: launch(std::integral_constant<int, 8>{}); break;
        case 4: launch(std::integral_constant<int, 4>{}); break;
        case 2: launch(std::integral_constant<int, 2>{}); break;
        default: launch(std::integral_constant<int, 1>{}); break;
    }
}

}  // namespace htgs
