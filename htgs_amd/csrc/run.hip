// Whole passes in one call: the scratch carved out of two workspaces, every stage queued before the host knows the number of
// instances, and a wait for that one word instead of for the stream.
// Restates the drivers <mode>::inference / forward / update_max_weights (R/src/hybrid_blend/inference.cu:57-183,
// forward.cu:57-189, update_max_weights.cu:30-165).
//
// The number of instances decides the size of the per-instance buffers, so the reference stops the host at it.  Stopped
// there, the device runs dry until the host has read the number and queued the second half: 30 us of a frame, 100 us of a
// training step whose buffers are allocated in between.  Here a caller that has rendered before says how many instances to
// expect; duplication, sort and ranges are queued behind the scan, these kernels take the number from the device
// (InstanceCount), and the scan's last block also writes it to host memory, where this thread picks it up while the device
// sorts and queues the blend.  The blend waits for the number: with too many instances it would go over all tiles for
// nothing, which in a training pass writes the pixel records twice (1 M Gaussians at 1920x1080, a view with half as many instances
// again as expected: 200 us), and by the time the lists are sorted its launch is there.  Only where a pass is that short that the
// device waits for the host (kBlendAheadTiles) the blend is queued ahead as well.
#include "common.h"
#include <mutex>

namespace htgs {

// ---------------------------------------------------------------------------------------------
// Words in coherent host memory that a frame's scan writes and the host waits for.  One per call that is under way: taken
// from a free list and given back, a page of them at a time; the pages stay until the process ends.
// ---------------------------------------------------------------------------------------------
struct HostWord {
    unsigned long long value;              // tag << 32 | number of instances
    HostWord *next;                        // on the free list
    uint32_t tag;                          // of the last frame it was used for
    uint32_t pad[11];                      // a cache line each
};
static_assert(sizeof(HostWord) == 64, "a cache line each");
static std::mutex g_words_mutex;
static HostWord *g_free_words;
constexpr size_t kWordsPerPage = 64;

static HostWord *take_word()
{
    std::lock_guard<std::mutex> lock(g_words_mutex);
    if (!g_free_words) {
        void *page = nullptr;
        const hipError_t e = hipHostMalloc(&page, kWordsPerPage * sizeof(HostWord), hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent);
        if (e != hipSuccess || !page) {
            fail(HTGS_ERR_HIP, "htgs_run: hipHostMalloc: %s", hipGetErrorString(e));
            return nullptr;
        }
        HostWord *w = static_cast<HostWord *>(page);
        for (size_t i = 0; i < kWordsPerPage; ++i) {
            w[i].value = 0;
            w[i].tag = 0;
            w[i].next = g_free_words;
            g_free_words = w + i;
        }
    }
    HostWord *w = g_free_words;
    g_free_words = w->next;
    w->tag = w->tag == 0xffffffffu ? 1u : w->tag + 1u;     // (never 0, which the fresh word holds)
    return w;
}
static void give_back_word(HostWord *w)
{
    std::lock_guard<std::mutex> lock(g_words_mutex);
    w->next = g_free_words;
    g_free_words = w;
}

// Waits for the word: a busy loop that ends when the scan has run, or when the stream has nothing left to run (a stream
// that failed, say) and the word is still not there.
static int wait_for_word(const HostWord *w, hipStream_t s, uint64_t *n)
{
    for (uint32_t spin = 0;; ++spin) {
        const unsigned long long v = __atomic_load_n(&w->value, __ATOMIC_ACQUIRE);
        if ((uint32_t)(v >> 32) == w->tag) { *n = (uint32_t)v; return HTGS_OK; }
        if ((spin & 0xfffu) == 0xfffu) {
            const hipError_t e = hipStreamQuery(s);
            if (e == hipErrorNotReady) { (void)hipGetLastError(); continue; }
            if (e != hipSuccess) return fail(HTGS_ERR_HIP, "htgs_run: %s", hipGetErrorString(e));
            const unsigned long long last = __atomic_load_n(&w->value, __ATOMIC_ACQUIRE);
            if ((uint32_t)(last >> 32) == w->tag) { *n = (uint32_t)last; return HTGS_OK; }
            return fail(HTGS_ERR_HIP, "htgs_run: the number of instances did not arrive");
        }
        __builtin_ia32_pause();
    }
}

// ---------------------------------------------------------------------------------------------
// workspaces
// ---------------------------------------------------------------------------------------------
struct Carver {
    unsigned char *base;                   // nullptr: sizes only
    uint64_t used;
    template <typename T> T *take(uint64_t count)
    {
        T *p = base != nullptr && count > 0 ? reinterpret_cast<T *>(base + used) : nullptr;
        used += (count * sizeof(T) + 255) & ~255ull;
        return p;
    }
};

// The waves that a tile gets.  Blend of clusters of 1 and 3 M Gaussians (four views each), time with two waves over that with one,
// mean and worst view, on both sides of the lines:
//   images, K <= 16   14400 tiles 0.86 1.11, 16416 0.90 1.18, 22600 1.11 1.25 (HYBRID_BLEND); 0.92 1.23, 1.02 1.24, 1.26 1.31 (FIRST_K)
//   K = 32            12288 tiles 0.73 1.11, 14400 1.00 1.26;   image alone (fast_math): 12288 0.75 1.16, 14400 1.02 1.28
//   OIT_BLEND         16416 tiles 0.91 1.07, 22600 1.06 1.09
//   training, K <= 16 7500 tiles 0.81 0.86, 12288 1.02 1.25 (HYBRID_BLEND); 0.76 0.86, 1.08 1.33 (FIRST_K)
//   training, K = 32  7500 tiles 0.84 1.09 and 100 k Gaussians 1.13, 12288 1.29 1.45
// Four waves over two: 0.88 at 7500 tiles and 1.02 at 12288 (HYBRID_BLEND, images), but 1.25 at 7000 where lists are short (100 k
// Gaussians), which the line at 6144 is for.  HYBRID_BLEND's training pass with K = 32 never has four: what its waves leave for one
// another fills the LDS that a second workgroup would need (640x480: 193 us with one, 143 with two, 283 with four).
static int waves_of(const htgs_frame *f, int what, uint64_t n_tiles)
{
    if (f->mode == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING || what == HTGS_RUN_MAX_WEIGHTS) return 1;
    const bool train = what == HTGS_RUN_FORWARD, wide = htgs_effective_k(f->K) > 16;
    if (f->mode == HTGS_MODE_OIT_BLEND) return n_tiles <= 6144 ? 4 : n_tiles <= 16384 ? 2 : 1;
    if (train && wide && f->mode == HTGS_MODE_HYBRID_BLEND) return n_tiles <= 8192 ? 2 : 1;
    const uint64_t two = train ? (wide ? 8192 : 10240) : wide || f->fast_math ? 13312 : 15360;
    return n_tiles <= 6144 ? 4 : n_tiles <= two ? 2 : 1;
}
// From how many Gaussians on the instances are made in bins of depth.  The bins cost 10 us (the sample for their limits, a scan that cannot be
// left to the duplication, shorter runs of its output) and spare most insertions into a core: the more, the larger the core and
// the longer the lists.  Four waves that share a list gain little: the near batches come first, and each wave still fills a core of its
// own.  Whole passes, without / with bins, over clusters (and the stress scene) on both sides of the lines:
//   grids of four waves (374x512 to 640x480)   images, K = 16  200 k 0.89 to 0.93, 800 k 0.98 to 1.03, 1.5 M 1.00, 2 M 1.02 (640x480) and 0.99 (374x512),
//     3 M 1.05, 6 M 1.07 (250 k 0.82 to 0.89, 500 k 0.86 to 0.89);  K = 32  800 k 0.98, 1.5 M 1.00, 2 M 1.04;  K = 8  1 M 0.97, 2 M 0.99;  image alone  2 M 1.01;
//     FIRST_K  1 M 0.98, 2 M 1.00;  training  150 k 0.86 to 0.95, 400 k 0.97 (250 k 0.84 to 0.86, 500 k 0.82 to 0.88), 2 M 1.04, FIRST_K 2 M 1.10
//   up to 16384 tiles (900x700 to 1280x720)    images, K = 16  400 k 0.96 to 0.97, 800 k 1.02 (250 k 1.05 to 1.08, 500 k 1.01 to 1.02);  image alone
//     500 k 0.97, 1 M 1.01;  K = 32  400 k 0.99, 800 k 1.04;  training  150 k 0.98, 400 k 1.01 to 1.03 (130 k 1.03, 250 k 1.04 to 1.06)
//     FIRST_K, which looks at no instance behind its cores with or without bins:  K = 16  200 k 0.91, 400 k 0.94, 600 k 0.98, 800 k 1.01;  training 250 k 0.97
//   beyond (1920x1080)                         images, K = 16  200 k 0.97 to 0.98, 400 k 1.02, 800 k 1.06;  K = 32  400 k 1.01, 800 k 1.05;  training
//     150 k 0.99, 400 k 1.01 to 1.03;  image alone  200 k 0.98, 500 k 1.03;  FIRST_K  K = 16  400 k 0.99, 600 k 1.04;  K = 32  300 k 0.97;  training  300 k 0.99, 500 k 1.02
//   K = 8  400 k 0.93 to 1.0, 1 M 1.02 to 1.04 (1920x1080), 3 M 1.03 to 1.05, 2 M 1.00 (800x600);  FIRST_K 400 k 1.00, 800 k 1.03 (1920x1080);   K <= 4
//     0.92 (320 k) to 1.01 (3 M): never
//   weights (one wave)  HYBRID 1280x720 120 k 1.00, 200 k 0.97, 400 k 1.04;  1920x1080 250 k 0.96, 400 k 1.02;  640x480 150 k 0.96;  K = 32 200 k 0.93, K = 8 0.97
//     (150 k 1.05, 400 k 1.05);  FIRST_K 1280x720 120 k 0.96, 250 k 0.99, 500 k 1.05, 1 M 1.11;  1920x1080 250 k 0.94, 500 k 1.06, 1 M 1.18;  640x480 300 k 1.12 (250 k 0.96)
//     on the smallest grids the lists are long and walked in shares, the first of which then has the near Gaussians: stress scene 600 k at 309x378
//     K = 16 0.87, K = 32 0.84, 250 k at 400x400 0.92; clusters 400 k at 400x400 1.01 to 1.03
static bool takes_depth_bins(const htgs_frame *f, int what, uint64_t n_tiles)
{
    if (f->mode != HTGS_MODE_HYBRID_BLEND && f->mode != HTGS_MODE_ALPHA_BLEND_FIRST_K) return false;
    const int K = htgs_effective_k(f->K), n = f->n_primitives;
    const bool wide = n_tiles > 16384, first_k = f->mode == HTGS_MODE_ALPHA_BLEND_FIRST_K;
    if (K <= 4) return false;
    if (what == HTGS_RUN_MAX_WEIGHTS) return n_tiles > 4096 && n >= (wide ? 320000 : 300000);
    if (n_tiles <= 6144) return n >= 2000000;
    if (what == HTGS_RUN_FORWARD) return n >= (first_k ? (wide ? 300000 : 400000) : 200000);
    if (K == 8) return n >= (n_tiles >= 8192 ? 800000 : 2000000);
    return n >= (K == 16 ? (wide ? 300000 : first_k ? 700000 : 500000) : wide ? 400000 : first_k ? 700000 : 600000);
}
constexpr uint64_t kUnorderedTiles = 1280;      // workgroups of four waves
static uint64_t carve_front(htgs_frame *f, int what, void *base)
{
    Carver c = { static_cast<unsigned char *>(base), 0 };
    const uint64_t n = (uint64_t)f->n_primitives;
    const int tile = tile_size(f->mode);
    const uint64_t n_tiles = (uint64_t)div_up(f->width, tile) * div_up(f->height, tile);
    const bool train = what == HTGS_RUN_FORWARD;
    f->prim_floats = train ? HTGS_PRIM_FLOATS_TRAIN : HTGS_PRIM_FLOATS;
    f->n_touched = c.take<uint32_t>(n);
    f->offsets = c.take<uint32_t>(n);
    f->bounds = nullptr;
    f->touch = c.take<uint32_t>(4 * n);
    f->touch_cutoff_only = 0;
    f->prim = c.take<float>((uint64_t)f->prim_floats * n);
    f->clamp_info = train ? c.take<uint8_t>(3 * n) : nullptr;
    f->scan_tmp = c.take<uint32_t>(htgs_scan_tmp_words((int)n));
    f->n_instances_dev = c.take<uint32_t>(1);
    f->ranges = c.take<uint32_t>(2 * n_tiles);
    // (the modes that walk all of a list)
    f->long_tiles = f->mode != HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING ? c.take<uint32_t>(8 + 3 * n_tiles) : nullptr;
    f->long_counters = f->mode != HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING ? c.take<uint32_t>(HTGS_LONG_COUNTERS) : nullptr;
    f->waves_per_tile = waves_of(f, what, n_tiles);
    f->long_list_threshold = -1;                           // (ListThreshold)
    // (a grid whose workgroups are all on the device at once is taken in any order)
    f->tile_order = n_tiles > kUnorderedTiles ? c.take<uint32_t>(htgs_tile_order_words(f->mode, f->width, f->height)) : nullptr;
    // GLOBAL_ORDERING without a backward pass
    const bool by_depth = !train && f->mode == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING;
    f->depth_order = by_depth ? c.take<uint32_t>(htgs_depth_order_words((int)n)) : nullptr;
    f->depth_bins = takes_depth_bins(f, what, n_tiles) ? c.take<uint32_t>(htgs_depth_bins_words((int)n)) : nullptr;
    const bool has_core = f->mode == HTGS_MODE_HYBRID_BLEND || f->mode == HTGS_MODE_ALPHA_BLEND_FIRST_K;
    const bool has_tail = f->mode == HTGS_MODE_HYBRID_BLEND || f->mode == HTGS_MODE_OIT_BLEND;
    f->pixel_scratch = what == HTGS_RUN_MAX_WEIGHTS && has_tail ? c.take<float>(64 * n_tiles) : nullptr;
    const uint64_t records = 64 * n_tiles, K = (uint64_t)htgs_effective_k(f->K);
    f->core_idx = train && has_core ? c.take<uint32_t>(K * records) : nullptr;
    f->core_info = train && has_core ? c.take<float>(4 * K * records) : nullptr;
    f->tail_info = train && has_tail ? c.take<float>(6 * records) : nullptr;
    return c.used;
}
// (after carve_front: whether the frame has depth_order decides the width of its keys)
static uint64_t carve_back(htgs_frame *f, uint64_t n_instances, void *base)
{
    Carver c = { static_cast<unsigned char *>(base), 0 };
    const uint64_t m = n_instances > 0 ? n_instances : 1, kb = (uint64_t)htgs_frame_key_bytes(f);
    for (int i = 0; i < 2; ++i) f->keys[i] = c.take<unsigned char>(kb * m);
    for (int i = 0; i < 2; ++i) f->vals[i] = c.take<uint32_t>(m);
    f->sort_tmp = c.take<uint32_t>(htgs_sort_tmp_words(m));
    return c.used;
}
constexpr uint64_t kMostInstances = 0xfffffffeull;
// the number of instances that launches and buffers are sized for when `expected` are expected
static uint64_t with_headroom(uint64_t expected)
{
    const uint64_t n = expected + expected / 8 + 4096;
    return n < kMostInstances ? n : kMostInstances;
}
// the most instances from `least` to with_headroom(least) whose scratch fits into `bytes`, 0 if not even `least` do
static uint64_t fitting(htgs_frame *f, uint64_t least, uint64_t bytes)
{
    uint64_t lo = least, hi = with_headroom(least);
    if (carve_back(f, hi, nullptr) <= bytes) return hi;
    if (carve_back(f, lo, nullptr) > bytes) return 0;
    for (int step = 0; step < 5; ++step) {                 // (lo fits, hi does not)
        const uint64_t mid = lo + (hi - lo) / 2;
        if (carve_back(f, mid, nullptr) <= bytes) lo = mid; else hi = mid;
    }
    return lo;
}

// Frames of at most kBlendAheadGaussians on grids of no more tiles have their blend queued before the number is
// there: 20 k Gaussians at 400x304 in training 201 us a step so, 207 otherwise, and the records of 6144 tiles are written twice in 25 us.
constexpr uint64_t kBlendAheadTiles = 6144;
constexpr int kBlendAheadGaussians = 65536;
static int check_run(const htgs_frame *f, const htgs_workspace *w, const char *who)
{
    if (!f || !w) return fail(HTGS_ERR_ARGUMENT, "%s: null argument", who);
    if (f->mode < 0 || f->mode > 3) return fail(HTGS_ERR_MODE, "unsupported rasterizer mode");
    if (w->what < HTGS_RUN_RENDER || w->what > HTGS_RUN_MAX_WEIGHTS) return fail(HTGS_ERR_ARGUMENT, "%s: unknown pass", who);
    if (f->n_primitives < 0 || f->width <= 0 || f->height <= 0 || f->total_sh_bases < 0) return fail(HTGS_ERR_ARGUMENT, "%s: bad sizes", who);
    if (((uintptr_t)w->front | (uintptr_t)w->back) & 255) return fail(HTGS_ERR_ARGUMENT, "%s: workspaces must be 256-byte aligned", who);
    return HTGS_OK;
}

// The first half.  starts: the lists follow at once (FrameStart); *fused as in scan_offsets_publish.
static int queue_front(const htgs_frame *f, const htgs_workspace *w, HostWord *word, bool starts, bool *fused)
{
    htgs_frame t = *f;
    if (w->what != HTGS_RUN_RENDER) t.scale_modifier = 1.0f;       // as htgs_forward_front, htgs_max_weights_front
    if (w->what == HTGS_RUN_MAX_WEIGHTS) {
        t.sh_0 = t.sh_rest = nullptr;
        t.active_sh_bases = 1;
        t.total_sh_bases = 0;
    }
    FrameStart start = {};
    if (starts) {
        const int tile = tile_size(f->mode);
        const uint32_t n_tiles = (uint32_t)div_up(f->width, tile) * (uint32_t)div_up(f->height, tile);
        start.block_sums = f->scan_tmp;
        start.clear[0] = f->ranges; start.clear_words[0] = 2 * n_tiles;
        if (f->tile_order) {
            start.clear[1] = f->tile_order + n_tiles;
            start.clear_words[1] = (uint32_t)htgs_tile_order_words(f->mode, f->width, f->height) - n_tiles;
        }
        if (f->long_tiles) {
            start.clear[2] = f->long_tiles; start.clear_words[2] = 8;
            start.clear[4] = f->long_counters; start.clear_words[4] = HTGS_LONG_COUNTERS;
            if (f->tile_order) { start.clear[3] = f->long_tiles + 8 + 2 * (size_t)n_tiles; start.clear_words[3] = n_tiles < 132 ? n_tiles : 132; }
        }
    }
    const int rc = preprocess_and_start(&t, start);
    return rc != HTGS_OK ? rc : scan_offsets_publish(&t, &word->value, word->tag, starts, fused);
}
// The lists: duplication, sort, ranges; cleared: with what FrameStart left, fused: with the scan.
static int queue_lists(htgs_frame *f, htgs_workspace *w, bool cleared, HostWord *fused)
{
    bool ranged = false;
    int rc = fused ? create_instances_fused(f, &fused->value, fused->tag) : htgs_create_instances(f);
    if (rc == HTGS_OK) rc = sort_instances_of(f, &w->selector, &ranged);
    if (rc == HTGS_OK) rc = extract_ranges_of(f, w->selector, cleared, ranged);
    return rc;
}
static int queue_blend(htgs_frame *f, htgs_workspace *w)
{
    switch (w->what) {
        case HTGS_RUN_RENDER: return htgs_blend(f, w->selector);
        case HTGS_RUN_FORWARD: return htgs_blend_forward(f, w->selector);
        default: return htgs_max_weights_blend(f, w->selector, w->max_weights, w->weight_threshold);
    }
}

}  // namespace htgs

using namespace htgs;

extern "C" int htgs_run_sizes(const htgs_frame *f, htgs_workspace *w)
{
    const int rc = check_run(f, w, "htgs_run_sizes");
    if (rc != HTGS_OK) return rc;
    htgs_frame t = *f;
    w->front_needed = carve_front(&t, w->what, nullptr);
    t.depth_order = t.mode == HTGS_MODE_ALPHA_BLEND_GLOBAL_ORDERING && w->what != HTGS_RUN_FORWARD ? (uint32_t *)256 : nullptr;
    w->back_needed = carve_back(&t, with_headroom(w->expected), nullptr);
    return HTGS_OK;
}

extern "C" int htgs_run(htgs_frame *f, htgs_workspace *w)
{
    int rc = check_run(f, w, "htgs_run");
    if (rc != HTGS_OK) return rc;
    w->selector = 0;
    w->n_instances = 0;
    w->front_needed = carve_front(f, w->what, w->front);
    if (w->front == nullptr || w->front_bytes < w->front_needed) return HTGS_WORKSPACE;
    // (the tail's second walk of the weights takes fragments below the alpha threshold of 1/255; a tail's weight is at most
    // one per unit of alpha, so a weight threshold above leaves none of those)
    f->touch_cutoff_only = w->what == HTGS_RUN_MAX_WEIGHTS && !(w->weight_threshold > 0.004f) ? 1 : 0;
    hipStream_t s = (hipStream_t)f->stream;
    f->n_instances_live = nullptr;
    f->n_instances = 0;
    if (f->n_primitives == 0) return htgs_run_rest(f, w);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capture) == hipSuccess && capture != hipStreamCaptureStatusNone)
        return fail(HTGS_ERR_ARGUMENT, "htgs_run: the host waits for the number of instances, which a stream under capture never gives");
    HostWord *word = take_word();
    if (!word) return HTGS_ERR_HIP;
    const uint64_t queued_for = w->expected > 0 && w->back != nullptr ? fitting(f, w->expected, w->back_bytes) : 0;
    bool fused = false, blended = false;
    // (after a failure a kernel that was queued may still write the word: it is not used again)
    rc = queue_front(f, w, word, queued_for > 0, &fused);
    if (rc != HTGS_OK) return rc;
    if (queued_for > 0) {
        carve_back(f, queued_for, w->back);
        f->n_instances = queued_for;
        f->n_instances_live = f->n_instances_dev;
        rc = queue_lists(f, w, true, fused ? word : nullptr);
        const int tile = tile_size(f->mode);
        blended = fused && f->n_primitives <= kBlendAheadGaussians && (uint64_t)div_up(f->width, tile) * div_up(f->height, tile) <= kBlendAheadTiles;
        if (rc == HTGS_OK && blended) rc = queue_blend(f, w);
        f->n_instances_live = nullptr;
        if (rc != HTGS_OK) return rc;
    }
    uint64_t n = 0;
    rc = wait_for_word(word, s, &n);
    if (rc != HTGS_OK) return rc;
    give_back_word(word);
    w->n_instances = n;
    f->n_instances = n;
    if (n > kMostInstances) return HTGS_OK;                  // (the caller refuses the frame)
    if (queued_for == 0 || n > queued_for) return htgs_run_rest(f, w);
    return blended ? HTGS_OK : queue_blend(f, w);
}

extern "C" int htgs_run_rest(htgs_frame *f, htgs_workspace *w)
{
    int rc = check_run(f, w, "htgs_run_rest");
    if (rc != HTGS_OK) return rc;
    const uint64_t n = w->n_instances;
    if (n > kMostInstances) return fail(HTGS_ERR_ARGUMENT, "htgs_run_rest: more than 2^32-2 instances");
    f->n_instances = n;
    f->n_instances_live = nullptr;
    const uint64_t needed = carve_back(f, n, n > 0 ? w->back : nullptr);
    if (n > 0 && (w->back == nullptr || w->back_bytes < needed)) {
        w->back_needed = carve_back(f, with_headroom(n), nullptr);
        return HTGS_WORKSPACE;
    }
    rc = queue_lists(f, w, false, nullptr);
    return rc == HTGS_OK ? queue_blend(f, w) : rc;
}
