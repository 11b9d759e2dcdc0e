// Training forward blend of small grids: several waves per tile (blend_waves.h).
#include "blend_records.h"
#include "blend_waves.h"

namespace htgs {

template <int WAVES, typename Main, typename Finish>
static void launch_waves(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles, Main main, const Finish &finish)
{
    hipStream_t s = (hipStream_t)f->stream;
    const PartFloor floor = { instance_count(f), f->vals[sel ^ 1] != nullptr ? 1u : 0u };
    hipLaunchKernelGGL(main, dim3(n_tiles), dim3(64 * WAVES), 0, s, f->ranges, f->vals[sel], (const float4 *)f->prim, (uint32_t)f->width, (uint32_t)f->height, grid_w,
                       f->long_tiles, list_threshold(f), floor, f->tile_order, finish);
}
template <int WAVES, int K>
static void launch_k(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    constexpr int REC4 = HTGS_PRIM_FLOATS_TRAIN / 4;
    const uint32_t w = (uint32_t)f->width, h = (uint32_t)f->height;
    if (f->mode == HTGS_MODE_HYBRID_BLEND) {
        const HybridRecords finish = { f->image, f->core_idx, (float4 *)f->core_info, f->tail_info, w, h, (size_t)n_tiles * 64u };
        launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_hybrid_waves_exact_kernel<WAVES, K, REC4, HybridRecords>, finish);
        launch_hybrid_long<K, false, REC4>(f, sel, grid_w, finish);
    } else {
        const FirstKRecords finish = { f->image, f->core_idx, (float4 *)f->core_info, w, h, (size_t)n_tiles * 64u };
        launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_first_k_waves_exact_kernel<WAVES, K, false, REC4, FirstKRecords>, finish);
        launch_first_k_long<K, false, REC4>(f, sel, grid_w, finish);
    }
}

template <int WAVES>
static void launch_mode(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    if (f->mode == HTGS_MODE_OIT_BLEND) {
        constexpr int REC4 = HTGS_PRIM_FLOATS_TRAIN / 4;
        const OitRecords finish = { f->image, f->tail_info, (uint32_t)f->width, (uint32_t)f->height, (size_t)n_tiles * 64u };
        launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_oit_waves_kernel<WAVES, false, REC4, OitRecords, false>, finish);
        launch_oit_long<false, REC4, false>(f, sel, grid_w, finish);
        return;
    }
    switch (htgs_effective_k(f->K)) {
        case 32: launch_k<WAVES, 32>(f, sel, grid_w, n_tiles); break;
        case 16: launch_k<WAVES, 16>(f, sel, grid_w, n_tiles); break;
        case 8: launch_k<WAVES, 8>(f, sel, grid_w, n_tiles); break;
        case 4: launch_k<WAVES, 4>(f, sel, grid_w, n_tiles); break;
        case 2: launch_k<WAVES, 2>(f, sel, grid_w, n_tiles); break;
        default: launch_k<WAVES, 1>(f, sel, grid_w, n_tiles); break;
    }
}

bool blend_forward_waves(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    if ((f->waves_per_tile != 2 && f->waves_per_tile != 4) || !f->long_tiles || most_threshold(f) > kPackedListMost || f->mode == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING) return false;
    if (f->waves_per_tile == 4) launch_mode<4>(f, sel, grid_w, n_tiles);
    else launch_mode<2>(f, sel, grid_w, n_tiles);
    return true;
}

}  // namespace htgs
