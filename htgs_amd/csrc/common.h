// Shared host/device declarations of the gfx950 rasterizer.
//
// Rounding convention.  The whole library is compiled with -ffp-contract=off, so a fused
// multiply-add exists exactly where __builtin_fmaf is written.  The per-Gaussian stage uses none
// (operand order of the reference source, R/include/kernel_utils.cuh).  The per-pixel stage evaluates
// the reference's ray / Gaussian expressions in the tile-relative form (TileFrag, blend_common.h), in which |m|^2, |d|^2 and
// MT3.(d x m) are quadratics of the pixel offset from the tile centre.  log and 2^x are the
// polynomial routines below, sqrt and division are correctly rounded
// (-fhip-fp32-correctly-rounded-divide-sqrt; rcp_exact is the same quotient, cheaper).  The
// CPU oracle of the tests follows the same convention, which is what makes tile counts, sort
// order and every per-fragment accept/reject decision reproducible bit for bit.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/htgs_amd.h"

namespace htgs {

constexpr int kWave = 64;

// R/include/<mode>/config.h
constexpr float kTransmittanceThreshold = 1e-4f;
constexpr float kMaxFragmentAlpha = 1.0f;
constexpr float kOneMinusAlphaEps = 1e-8f;
constexpr float kMinAlphaCore = 1.0f / 20.0f;

template <int MODE> struct ModeCfg {
    static constexpr int tile = MODE == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING ? 16 : 8;
    static constexpr float min_alpha_rcp = MODE == HTGS_MODE_ALPHA_BLEND_FIRST_K ? 20.0f : 255.0f;
    static constexpr float min_alpha = 1.0f / min_alpha_rcp;
    static constexpr float cutoff_sq = MODE == HTGS_MODE_ALPHA_BLEND_FIRST_K ? 5.99146454711f : 11.0825270903f;
    // tile-relative form: |m|^2 is staged divided by the cut-off (2 ln 20 resp. 2 ln 255), so the cut-off test is
    // num > den and exp(-rho^2 / 2) = 2^(-log2(20 or 255) num / den)
    static constexpr float cutoff_rcp = 1.0f / cutoff_sq;
    static constexpr float exp2_scale = MODE == HTGS_MODE_ALPHA_BLEND_FIRST_K ? -4.32192809488736235f : -7.99435343685885794f;
};

inline int tile_size(int mode) { return mode == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING ? 16 : 8; }
inline int div_up(int a, int b) { return (a + b - 1) / b; }
// floats per record of f->prim; -1 for a value that no entry point takes
inline int frame_prim_floats(const htgs_frame *f)
{
    return f->prim_floats == 0 || f->prim_floats == HTGS_PRIM_FLOATS ? HTGS_PRIM_FLOATS : f->prim_floats == HTGS_PRIM_FLOATS_TRAIN ? HTGS_PRIM_FLOATS_TRAIN : -1;
}

// The Gaussians are sorted by depth before the instances are made (htgs_frame.depth_order): ALPHA_BLEND_GLOBAL_ORDERING,
// whose lists must be in depth order, and, for callers of the stages that ask for it, the image-only fast path of the two modes with a
// sorted core, whose lists may be in any order (coarse keys, one pass; htgs_run has bins of depth there instead)
inline bool frame_coarse_depth_ordered(const htgs_frame *f)
{
    return f->depth_order != nullptr && f->fast_math && (f->mode == HTGS_MODE_HYBRID_BLEND || f->mode == HTGS_MODE_ALPHA_BLEND_FIRST_K);
}
inline bool frame_depth_ordered(const htgs_frame *f)
{
    return (f->mode == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING && f->depth_order != nullptr) || frame_coarse_depth_ordered(f);
}
// the parts of depth_order, n4 = N rounded up to a multiple of four words each: depth keys and Gaussian indices (two
// buffers each for the sort, which leaves its result in the first ones after four passes; htgs_preprocess writes the
// pairs), the counts and the tile rectangles (or touch entries) in depth order, scratch of the sort
struct DepthOrder {
    uint32_t *keys[2], *vals[2], *counts;
    uint16_t *bounds;
    uint32_t *touch;
    uint32_t *sort_tmp;
};
inline DepthOrder depth_order_parts(const htgs_frame *f)
{
    const size_t n4 = ((size_t)(f->n_primitives > 0 ? f->n_primitives : 0) + 3) & ~(size_t)3;
    DepthOrder d;
    d.keys[0] = f->depth_order; d.keys[1] = f->depth_order + n4;
    d.vals[0] = f->depth_order + 2 * n4; d.vals[1] = f->depth_order + 3 * n4;
    d.counts = f->depth_order + 4 * n4; d.bounds = reinterpret_cast<uint16_t *>(f->depth_order + 5 * n4); d.touch = f->depth_order + 5 * n4; d.sort_tmp = f->depth_order + 9 * n4;
    return d;
}
// The keys that sort the Gaussians by depth: the bit pattern of the centre's camera-space depth (for positive depths the
// patterns order like the depths; these are the low 32 bits of the reference's tile | depth keys) less that of the near
// plane, which no Gaussian that is not culled lies in front of, `culled` for a culled Gaussian (behind all others).  With
// the far plane as the upper bound the keys of the usual cameras have 27 bits: three passes of 9-bit digits.
// Coarse keys (frame_coarse_depth_ordered): the same keys shifted down until eight bits are left, one pass.
struct DepthKeys {
    uint32_t base, culled;
    int end_bit, digit_bits, passes, shift;
};
constexpr int kCoarseDepthBits = 8;
inline DepthKeys depth_key_range(const htgs_frame *f)
{
    DepthKeys k = { 0u, 0xffffffffu, 32, 8, 4, 0 };
    const float near_plane = f->near_plane, far_plane = f->far_plane;
    if (near_plane > 0.0f && far_plane >= near_plane && far_plane < __builtin_huge_valf()) {
        uint32_t lo, hi;
        __builtin_memcpy(&lo, &near_plane, 4);
        __builtin_memcpy(&hi, &far_plane, 4);
        k.base = lo;
        k.culled = hi - lo + 1u;
        k.end_bit = 1;
        while (k.end_bit < 32 && (k.culled >> k.end_bit) != 0u) ++k.end_bit;
        const int passes8 = (k.end_bit + 7) / 8, passes9 = (k.end_bit + 8) / 9;
        k.digit_bits = passes9 < passes8 ? 9 : 8;
        k.passes = passes9 < passes8 ? passes9 : passes8;
    }
    if (frame_coarse_depth_ordered(f)) {
        // (culled, the largest key, must fit the bits that are left)
        while (k.end_bit - k.shift > kCoarseDepthBits || ((k.culled - 1u) >> k.shift) + 1u >= (1u << kCoarseDepthBits)) ++k.shift;
        k.culled = ((k.culled - 1u) >> k.shift) + 1u;
        k.end_bit = kCoarseDepthBits; k.digit_bits = kCoarseDepthBits; k.passes = 1;
    }
    return k;
}
// The Gaussians are put into bins of depth, and the instances made bin by bin (htgs_frame.depth_bins).  The parts of
// depth_bins: the depths at which the bins after the first begin, the instances of each bin, a counter of the scan, the instances
// of every bin in every block of kCountBlock Gaussians (bin by bin, `stride` words each), the ones before each of these (the scan's
// result, apart from what it reads: it may be called again), the bin of every Gaussian.
constexpr int kDepthBins = 8;
inline bool frame_depth_binned(const htgs_frame *f)
{
    return f->depth_bins != nullptr && f->touch != nullptr && !frame_depth_ordered(f) && (f->mode == HTGS_MODE_HYBRID_BLEND || f->mode == HTGS_MODE_ALPHA_BLEND_FIRST_K);
}
struct DepthBins {
    float *limits;                         // [kDepthBins - 1]
    unsigned long long *totals;            // [kDepthBins]
    uint32_t *done, *sums, *before;        // [1], [kDepthBins][stride] twice
    uint8_t *of;                           // [N]
    uint32_t stride;
};
// where the blend stages put a tile's list by index when they need it so; nullptr: every list is
inline uint32_t *binned_spare(const htgs_frame *f, int selector) { return frame_depth_binned(f) ? f->vals[selector ^ 1] : nullptr; }
constexpr size_t kDepthBinsHeader = 32;    // words: limits from 0, totals from 8, done at 24
inline uint32_t depth_bins_stride(int n) { return ((uint32_t)div_up(n > 0 ? n : 1, 256) + 3u) & ~3u; }
inline DepthBins depth_bin_parts(const htgs_frame *f)
{
    DepthBins b;
    b.stride = depth_bins_stride(f->n_primitives);
    b.limits = reinterpret_cast<float *>(f->depth_bins);
    b.totals = reinterpret_cast<unsigned long long *>(f->depth_bins + 8);
    b.done = f->depth_bins + 24;
    b.sums = f->depth_bins + kDepthBinsHeader;
    b.before = b.sums + (size_t)kDepthBins * b.stride;
    b.of = reinterpret_cast<uint8_t *>(b.before + (size_t)kDepthBins * b.stride);
    return b;
}
// stable sort of n (32-bit key, value) pairs by the low end_bit key bits, digit_bits (8 or 9) a pass (radix_sort.hip);
// the result is in keys / vals[*selector]
int sort_u32_pairs(void *stream, uint32_t *const keys[2], uint32_t *const vals[2], uint32_t *sort_tmp, uint64_t n, int end_bit, int digit_bits,
                   int *selector);
// the same in one pass over keys of at most eight bits whose values are 0 .. n - 1 in this order, from keys / vals[0] to
// keys / vals[1]; the tile rectangles (four 16-bit bounds per value) are written in sorted order as well, with the number
// of tiles each covers (0 for the key `culled`); touch_in / touch_out in their place if they are given
int sort_u32_pairs_with_rectangles(void *stream, uint32_t *const keys[2], uint32_t *const vals[2], uint32_t *sort_tmp, uint64_t n, int bits,
                                   const uint16_t *rectangles_in, uint16_t *rectangles_out, const uint32_t *touch_in, uint32_t *touch_out,
                                   uint32_t *counts_out, uint32_t culled);

// The number of (tile, Gaussian) instances as a kernel sees it.  live = nullptr: `most` is the number, the host knows it
// (the stage-by-stage entry points).  Otherwise the kernels were queued before the host knew: they read the number the scan
// left on the device, and a number beyond `most`, which the buffers and the launches were sized for, counts as 0 -- every
// list is empty and the host, which learns the number meanwhile, queues the stages again (htgs_run).
struct InstanceCount {
    const uint32_t *live;
    uint32_t most;
    __device__ __forceinline__ uint32_t get() const
    {
        if (live == nullptr) return most;
        const uint32_t n = *live;
        return n <= most ? n : 0u;
    }
};
inline InstanceCount instance_count(const htgs_frame *f) { return InstanceCount{ f->n_instances_live, (uint32_t)f->n_instances }; }
// The least length of a part of a very long list: the frame's average list, rounded up (0: lists are not split)
struct PartFloor {
    InstanceCount count;
    uint32_t split;
    __device__ __forceinline__ uint32_t get(uint32_t n_tiles) const
    {
        if (split == 0u) return 0u;
        const uint32_t n = count.get(), floor = n / n_tiles + (n % n_tiles != 0u ? 1u : 0u);
        return floor < 1u ? 1u : floor;
    }
};

// What htgs_run's first queueing of a frame spares the later stages: the per-Gaussian stage also leaves the sums of its
// blocks' counts (scan_tmp) and clears the ranges, the tile order's bins and the header of long_tiles.  Nothing of it holds
// for a frame whose lists are made a second time.
constexpr int kCountBlock = 256;                 // Gaussians per block sum
struct FrameStart {
    uint32_t *block_sums;                        // [ceil(N / kCountBlock)] or nullptr
    uint32_t *clear[5];                          // ranges, order bins, long_tiles header and the bins of its threshold, long_counters
    uint32_t clear_words[5];
};
int preprocess_and_start(const htgs_frame *f, const FrameStart &start);                 // preprocess.hip
// The scan for htgs_run, which also writes tag << 32 | total to host memory.  with_sums: scan_tmp holds FrameStart's sums.
// Returns in *fused whether the scan was left to create_instances_fused (up to 2^21 Gaussians).
int scan_offsets_publish(const htgs_frame *f, unsigned long long *host_total, uint32_t tag, bool with_sums, bool *fused);    // instances.hip
int create_instances_fused(const htgs_frame *f, unsigned long long *host_total, uint32_t tag);
// (cleared: the ranges, bins and header are zero already; ranged: the sort has written the ranges)
int extract_ranges_of(const htgs_frame *f, int selector, bool cleared, bool ranged);
int sort_instances_of(const htgs_frame *f, int *selector, bool *ranged);                // radix_sort.hip
// words of scan_tmp for N Gaussians' block sums
inline size_t block_sum_words(int n) { return (size_t)div_up(n > 0 ? n : 1, kCountBlock); }

// The length beyond which a list is shared between the waves and workgroups of the kernels for long lists.  A tile's waves
// walk such a list while the launch ends, and the launch lasts as long as the longest of them or as all lists together
// take on the waves that the device holds, whichever is more; what is left to the kernels for long lists costs a launch of its
// own, and more for each instance, since the shares have to be merged.  The tile order's stage knows the lists' lengths and
// leaves the threshold of least cost in long_tiles[kChosenThreshold] (choose_threshold in instances.hip), in instances walked by
// a wave beside nineteen others on its compute unit (0.35 us each, HYBRID_BLEND with K = 16):
//   max(lists up to T / kWavesHeld, (kListAlways + kListPerWave / waves of a tile) T) + (none longer: 0; else kLongLaunch + kLongShare times the rest / kWavesHeld)
// (kLongWeights for the weights of a tail, whose walk of a whole list spares most tiles the second one: 3 M at 1024x768, HYBRID
// K = 16, 1170 us with 512, 827 with none on the long way).  Fitted to the times of all four modes, K of 4 to 32, images, training
// passes and weights, one, two and four waves a tile, 28 views of clusters of 1 to 3 M Gaussians at 640x480 to 1920x1080 and 25
// of the stress scene of 20 k to 6 M at 400x300 to 1600x1066: over the thresholds from 512 to 8192 the chosen one is 0.8 % behind
// the best on average, 1.3 on the stress scene.  A rule that weighs a list only against the lists up to it (within 1.5 times
// those over the waves) is as good on the stress scene and 18 % behind on the clusters, where it puts thousands of ordinary
// lists on the long way: blend of 1 M at 1366x768, HYBRID K = 16, 543 us with its 512, 340 with none there; fixed at 8192 the stress scene
// takes 2 to 4 times as long (6 M at 1600x1066 5.0 against 3.8 ms).
constexpr uint32_t kLongListDefault = 8192, kLeastThreshold = 512, kChosenThreshold = 5;
constexpr float kWavesHeld = 5120.0f;                               // (256 compute units, twenty waves each)
constexpr float kListAlways = 0.1f, kListPerWave = 0.6f, kLongLaunch = 600.0f, kLongShare = 1.5f, kLongWeights = 2.5f;
// Without a tile order (kUnorderedTiles tiles at most, all of them on the device at once) the lists' lengths are not known: this
// many times the instances over the waves held, for each of a tile's waves; more for the weights of a tail, whose two walks spare
// most tiles with long lists the second.
constexpr float kThresholdShare = 1.5f, kWeightsShare = 2.5f;
// words of htgs_frame.long_counters: a line for each of the eight dies that the workgroups' indices go round (a work counter for
// each of the long-list kernels' rounds and the workgroups that are done), then, for all of them, a word per round but the
// last, set if the list may hold an entry for it, the dies that are done, and the share of a long list that a wave should get
// (0: not chosen)
constexpr uint32_t kDies = 8, kDieLine = 32, kDieRounds = kDies * kDieLine, kChosenShare = kDieRounds + 8;
static_assert(HTGS_LONG_COUNTERS == kDieRounds + kDieLine, "a line per die and one for all");
// What a wave of the long-list kernels gets of a list at least: half of what it would walk of all long lists if they were
// shared evenly (longer shares spread badly, shorter ones cost more merges: 6 M Gaussians of the stress scene 5000 us with a
// half, 5060 with all of it, 5560 with a quarter of the threshold), between two batches and the threshold.
constexpr float kPartShare = 0.5f, kLongWavesOnDevice = 4096.0f;
constexpr uint32_t kLeastShare = 128;
struct ListThreshold {
    uint32_t fixed;                        // 0: chosen on the device
    InstanceCount count;
    float share;                           // threshold_share, where nothing was chosen
    uint32_t part_waves;                   // of a workgroup that walks a part of a long list
    uint32_t *counters;                    // htgs_frame.long_counters
    __device__ __forceinline__ uint32_t get(const uint32_t *long_tiles) const
    {
        if (fixed != 0u || long_tiles == nullptr) return fixed;
        const uint32_t chosen = long_tiles[kChosenThreshold];
        if (chosen != 0u) return chosen;
        const float t = share / kWavesHeld * (float)count.get();
        return t < 2.0f * kLeastThreshold ? 2u * kLeastThreshold : t < (float)kLongListDefault ? (uint32_t)t : kLongListDefault;
    }
    // the least length of such a part
    __device__ __forceinline__ uint32_t least_part(uint32_t long_threshold) const
    {
        const uint32_t share = fixed == 0u && counters != nullptr ? counters[kChosenShare] : 0u;
        return share != 0u ? share * part_waves : part_waves / 4u * long_threshold;
    }
    // The backward pass's parts, which one workgroup walks each: of a threshold's length, and shorter where the long lists are
    // few (20 k Gaussians of the stress scene at 400x300: a quarter of it 331 us a training step, all of it 370; 600 k at
    // 700x500, OIT: 692 and 670).
    __device__ __forceinline__ uint32_t least_backward_part(uint32_t long_threshold) const
    {
        const uint32_t share = fixed == 0u && counters != nullptr ? 2u * counters[kChosenShare] : 0u;
        return share == 0u || share > long_threshold ? long_threshold : share > long_threshold / 4u ? share : long_threshold / 4u;
    }
};
inline bool chooses_threshold(const htgs_frame *f) { return f->long_list_threshold < 0 && f->long_tiles != nullptr; }
// The waves of a workgroup of the long-list kernels, of which a compute unit holds sixteen.  Sixteen to a workgroup shorten a
// list most, but then a compute unit stands still while a workgroup merges its shares and takes its next part; two
// workgroups of eight fill in for each other.  Where the lists are few the first counts, where they are many the
// second: stress scene, K = 16, 16 waves -> 8: 300 k Gaussians at 1600x1000 602 -> 640 us, at 1024x768 425 -> 465, 600 k at
// 1600x1000 932 -> 825, 1 M at 700x500 644 -> 588, 6 M at 1600x1066 5600 -> 5000.  The sums of OIT_BLEND are merged at once
// (2.6 M Gaussians at 640x403: 796 -> 713 us) and a core of 32 leaves registers for eight waves only.  All that is for a
// threshold chosen from the lists; beyond a fixed one, 8192 or the caller's, lists are few and very long, and sixteen it is (stress
// scene, 1 M at 1600x1066, threshold 8192, eight -> sixteen: OIT image 1947 -> 1741 us, weights 1610 -> 1417, FIRST_K training
// 1806 -> 1577, HYBRID 2454 -> 2311).
constexpr int kManyGaussians = 1 << 19;
inline uint32_t long_waves_of(const htgs_frame *f)
{
    if (f->mode != HTGS_MODE_OIT_BLEND && htgs_effective_k(f->K) > 16) return 8u;
    if (!chooses_threshold(f)) return 16u;
    return f->mode == HTGS_MODE_OIT_BLEND || f->n_primitives > kManyGaussians ? 8u : 16u;
}
// kThresholdShare times the waves that a tile has (pixel_scratch: max weights)
inline float threshold_share(const htgs_frame *f)
{
    return f->pixel_scratch != nullptr ? kWeightsShare : kThresholdShare * (f->waves_per_tile > 1 ? (float)f->waves_per_tile : 1.0f);
}
inline ListThreshold list_threshold(const htgs_frame *f)
{
    const uint32_t fixed = f->long_list_threshold > 0 ? (uint32_t)f->long_list_threshold : chooses_threshold(f) ? 0u : kLongListDefault;
    return ListThreshold{ fixed, instance_count(f), threshold_share(f), long_waves_of(f), f->long_counters };
}
// the longest list that the kernels with one workgroup per tile can meet
inline uint32_t most_threshold(const htgs_frame *f) { return chooses_threshold(f) || f->long_list_threshold == 0 ? kLongListDefault : (uint32_t)f->long_list_threshold; }
// Whether a list of the frame can be longer than the threshold (a Gaussian is in a tile's list once): otherwise the kernels
// for such lists, which would find nothing to do, are not launched.
inline bool may_have_long_lists(const htgs_frame *f)
{
    return f->long_tiles != nullptr && (uint32_t)f->n_primitives > (chooses_threshold(f) ? kLeastThreshold : most_threshold(f));
}

// Several waves walk a tile's list (blend_waves.h); false: the launch is left to the kernels with one
bool blend_waves(const htgs_frame *f, int selector, uint32_t grid_w, uint32_t n_tiles);                 // blend_waves.hip
bool blend_forward_waves(const htgs_frame *f, int selector, uint32_t grid_w, uint32_t n_tiles);         // blend_forward_waves.hip

// The corner of a Gaussian's rectangle in its training record: row << column_bits | column.  A grid has at most 2^20 tiles
// (launch_scan), so that its rows and columns, each rounded up to a power of two, take 21 bits; unlike the corner's tile
// number it comes apart without a division.
__host__ __device__ __forceinline__ uint32_t column_bits(uint32_t grid_w) { return grid_w > 1u ? 32u - (uint32_t)__builtin_clz(grid_w - 1u) : 0u; }

// Workgroups go round the eight XCDs of the device in launch order, and each XCD has an L2 of its own.  Blocks that are
// neighbours in the input write neighbouring runs of every digit, a run being shorter than a cache line or two; handing
// every XCD a contiguous eighth of the input lets those partial lines meet in one L2 before they are written back.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_contiguous_block(uint32_t launched, uint32_t n_blocks)
{
    // (the launch may be larger than n_blocks asks for: its blocks beyond an XCD's share have nothing to do)
    const uint32_t per_xcd = (n_blocks + kXcds - 1) / kXcds;
    return launched / kXcds < per_xcd ? (launched % kXcds) * per_xcd + launched / kXcds : n_blocks;           // >= n_blocks: nothing to do
}
__device__ __forceinline__ uint32_t blocks_of(uint32_t n, uint32_t per_block) { return n / per_block + (n % per_block != 0u ? 1u : 0u); }
inline uint32_t xcd_padded_grid(uint32_t n_blocks) { return (n_blocks + kXcds - 1) / kXcds * kXcds; }

// host side error reporting (api.hip)
int fail(int code, const char *fmt, ...);
int check_launch(const char *what);

__device__ __forceinline__ float bits_to_float(uint32_t u) { return __uint_as_float(u); }
__device__ __forceinline__ uint32_t float_to_bits(float f) { return __float_as_uint(f); }

// ln x: x = m 2^e, m in [sqrt(1/2), sqrt(2)), s = (m-1)/(m+1), ln m = 2 s (1 + s^2/3 + ... + s^10/11)
__device__ __forceinline__ float d_logf(float x)
{
    if (x != x || x < 0.0f) return __builtin_nanf("");
    if (x == 0.0f) return -__builtin_huge_valf();
    if (x == __builtin_huge_valf()) return x;
    int e = 0;
    if (x < 1.17549435e-38f) { x = x * 8388608.0f; e = -23; }
    uint32_t ix = float_to_bits(x);
    e += (int)(ix >> 23) - 127;
    ix = (ix & 0x007fffffu) | 0x3f800000u;
    float m = bits_to_float(ix);
    if (m > 1.41421356237f) { m = m * 0.5f; e += 1; }
    const float s = (m - 1.0f) / (m + 1.0f);
    const float z = s * s;
    float p = 0.0909090909f;
    p = p * z + 0.1111111111f;
    p = p * z + 0.1428571429f;
    p = p * z + 0.2f;
    p = p * z + 0.3333333333f;
    p = p * z;
    const float lnm = 2.0f * (s + s * p);
    const float fe = (float)e;
    return fe * 0.693359375f + (lnm + fe * -2.12194440e-4f);
}

// 2^t for t in [-126, 1): n = rint(t), r = t - n, degree-5 polynomial of 2^r on [-1/2, 1/2] (relative error 2.7e-7).
// rint is taken by adding and subtracting 1.5 * 2^23 (exact for |t| < 2^22, ties to even like rint), which also leaves
// n in the low bits of the sum for the exponent: two full-rate additions instead of v_rndne_f32 and v_cvt_i32_f32.
__device__ __forceinline__ float d_exp2(float t)
{
    const float shifted = t + 12582912.0f;
    const float n = shifted - 12582912.0f;
    const float r = t - n;
    float p = 1.3381302124e-3f;
    p = __builtin_fmaf(p, r, 9.6663683653e-3f);
    p = __builtin_fmaf(p, r, 5.5503811687e-2f);
    p = __builtin_fmaf(p, r, 2.4022349715e-1f);
    p = __builtin_fmaf(p, r, 6.9314718246e-1f);
    p = __builtin_fmaf(p, r, 1.0f);
    return bits_to_float(float_to_bits(p) + (float_to_bits(shifted) << 23));
}

// 1 / x.  v_rcp_f32 followed by one fused Newton step is the correctly rounded quotient for every x with
// 2^-120 <= x < 2^121 on gfx950 (htgs_check_reciprocal compares all of them with the division); a wave in
// which any active lane is outside that range takes the division.
__device__ __forceinline__ bool rcp_in_range(float x) { return float_to_bits(x) - 0x03800000u < 0x78800000u; }
__device__ __forceinline__ float rcp_refined(float x)
{
    const float x0 = __builtin_amdgcn_rcpf(x);
    const float e = __builtin_fmaf(-x, x0, 1.0f);
    return __builtin_fmaf(x0, e, x0);
}
__device__ __forceinline__ float rcp_exact(float x)
{
    // (the short form first and unconditionally, the division over it where a lane needs it: one branch around a side
    // block instead of two ways that meet again)
    float r = rcp_refined(x);
    if (__builtin_expect(__any(!rcp_in_range(x)), 0)) r = 1.0f / x;
    return r;
}

// orders one wave's LDS writes before its later LDS reads (the LDS serves a wave's instructions in order; this only keeps
// the compiler from moving them)
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float clamp_pos(float v) { return v > 0.0f ? v : 0.0f; }
__device__ __forceinline__ float saturate(float v) { return v > 0.0f ? (v < 1.0f ? v : 1.0f) : 0.0f; }

}  // namespace htgs
