// Inference blend of small grids: several waves per tile (blend_waves.h).
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
    constexpr int REC4 = HTGS_PRIM_FLOATS / 4;
    const uint32_t w = (uint32_t)f->width, h = (uint32_t)f->height;
    if (f->mode == HTGS_MODE_HYBRID_BLEND) {
        const HybridImage finish = { f->image, f->fast_math ? nullptr : f->depth, w, h, f->to_chw, f->use_median_depth };
        if (f->fast_math) {
            launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_hybrid_waves_kernel<WAVES, K, true, HybridImage>, finish);
            launch_hybrid_long<K, true, REC4>(f, sel, grid_w, finish);
        } else {
            launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_hybrid_waves_kernel<WAVES, K, false, HybridImage>, finish);
            launch_hybrid_long<K, false, REC4>(f, sel, grid_w, finish);
        }
    } else {
        const FirstKImage finish = { f->image, f->fast_math ? nullptr : f->depth, w, h, f->to_chw, f->use_median_depth };
        if (f->fast_math) {
            launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_first_k_waves_exact_kernel<WAVES, K, true, REC4, FirstKImage>, finish);
            launch_first_k_long<K, true, REC4>(f, sel, grid_w, finish);
        } else {
            launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_first_k_waves_kernel<WAVES, K, FirstKImage>, finish);
            launch_first_k_long<K, false, REC4>(f, sel, grid_w, finish);
        }
    }
}

template <int WAVES>
static void launch_mode(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    if (f->mode == HTGS_MODE_OIT_BLEND) {
        constexpr int REC4 = HTGS_PRIM_FLOATS / 4;
        const OitImage finish = { f->image, f->fast_math ? nullptr : f->depth, (uint32_t)f->width, (uint32_t)f->height, f->to_chw };
        if (f->fast_math) {
            launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_oit_waves_kernel<WAVES, true, REC4, OitImage>, finish);
            launch_oit_long<true, REC4, false>(f, sel, grid_w, finish);
        } else {
            launch_waves<WAVES>(f, sel, grid_w, n_tiles, blend_oit_waves_kernel<WAVES, false, REC4, OitImage>, finish);
            launch_oit_long<false, REC4, true>(f, sel, grid_w, finish);
        }
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

bool blend_waves(const htgs_frame *f, int sel, uint32_t grid_w, uint32_t n_tiles)
{
    if ((f->waves_per_tile != 2 && f->waves_per_tile != 4) || !f->long_tiles || most_threshold(f) > kPackedListMost || f->mode == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING) return false;
    if (f->waves_per_tile == 4) launch_mode<4>(f, sel, grid_w, n_tiles);
    else launch_mode<2>(f, sel, grid_w, n_tiles);
    return true;
}

}  // namespace htgs
