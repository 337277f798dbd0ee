// The plain forward frame (GaussianEngine::rasterFrame, GaussianEngine.cpp:621-712).
//
// The reference sorts its (tile, Gaussian) pairs by (tile, depth).  Here the Gaussians are sorted by
// depth first (stable, so equal depths keep Gaussian order), their pairs are emitted in that order and
// sorted by tile alone (stable): the same order, (tile, depth, Gaussian), with the depth's digits
// sorted once per visible Gaussian instead of once per pair, and 8-byte pairs instead of 12-byte ones.
//
// The whole frame is issued at once: its launches cover the pair capacity and read the pair count on
// the device.  The count reaches the host while the frame's sorts still run; a frame that turns out to
// have more pairs than the capacity, or a depth outside the window it is to be sorted on, stops there (every
// later kernel returns).  The first is issued again from its emission on, the second from the start.
#include "tpd_ctx.hpp"

#include <algorithm>
#include <chrono>
#include <thread>

namespace tpd {

// A frame sorted on the depth window although one of its depths lies outside is issued again on the wide
// key (1M Gaussians at 1920x1080: 125 us beside the frame's 405), where that key costs 10 us (one more pass
// of the item sort).  So it is kept for some frames after the last such depth: a camera whose farthest depth
// moves in and out by turns, 957 -> 780 us for two frames.
constexpr uint32_t kDepthHold = 64;

constexpr size_t kMinPairRoom = 1u << 20;

// Frames for which the room of the one with the most pairs is kept before it shrinks: a scene seen from many
// sides comes back to its widest view within some dozens.  40 views in random order where the room shrank at
// once: of 11M to 25M pairs 24 frames in 240 without room, of 0.6M to 1.3M 12 (227 us a frame, 224 with none).
constexpr uint32_t kRoomHold = 32;

// The arguments shared by the frame's item kernel, its emission and the item offsets.
static BatchArgs item_args(tpd_ctx* c) {
    BatchArgs a{};
    a.nitems = c->n;
    a.scan_desc = c->d_scan_desc;
    a.scan_desc2 = c->d_scan_desc2;
    a.counters = c->d_counters;
    a.splats = c->d_splats;
    a.tiles = c->d_tiles;
    a.offsets = c->d_offsets;
    a.rects = c->d_rects;
    a.item_keys = c->d_ikeys;
    a.keys = c->d_keys;
    a.vals = c->d_vals;
    a.totals_known = 1u;
    return a;
}

// Where each Gaussian's pairs lie in emission order: the exclusive scan of the tile counts, for a backward
// on the stream it runs on.  The frame's item kernel, complete when tpd_render returns, clears the scan's
// ticket and descriptors, and nothing else does: a second scan of one frame finds no partition left and
// keeps the first one's offsets, so every backward launches it, recorded into a caller's graph or not.
int launch_offsets(tpd_ctx* c, hipStream_t s) {
    if (c->n == 0) return TPD_OK;
    launch_batch_item_offsets(item_args(c), s);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TPD_OK : hip_fail(e, "item offsets");
}

// Waits until the frame's totals have reached h_counters (k_frame_offsets stores seq last).  An ordinary
// frame's are there within half a millisecond, looked for all the time; a frame behind long work on its
// stream looks every 50 us after the first 10 ms and leaves its core to others meanwhile (a look is up to
// 110 us late with the kernel's timer slack: one part in a hundred of such a wait).
static int wait_totals(tpd_ctx* c, hipStream_t s, uint32_t seq) {
    using clock = std::chrono::steady_clock;
    constexpr auto kSpin = std::chrono::milliseconds(10);
    constexpr auto kNap = std::chrono::microseconds(50);
    volatile uint32_t* const at = &c->h_counters[kHostSeq];
    clock::time_point begin{};
    bool naps = false;
    for (uint32_t spins = 1; __atomic_load_n(at, __ATOMIC_ACQUIRE) != seq; ++spins) {
        if (naps)
            std::this_thread::sleep_for(kNap);
        else if (spins % 4096u)
            continue;
        const hipError_t e = hipStreamQuery(s);
        if (e == hipErrorNotReady) {
            (void)hipGetLastError();  // not an error to be found by a later check
            const clock::time_point now = clock::now();
            if (begin == clock::time_point{}) begin = now;
            naps = now - begin >= kSpin;
            continue;
        }
        if (e != hipSuccess) return hip_fail(e, "frame");
        if (__atomic_load_n(at, __ATOMIC_ACQUIRE) != seq) return fail(TPD_ERR_STATE, "tpd_render: the frame ended without its totals");
    }
    return TPD_OK;
}

// What one frame is issued with.
struct FrameIssue {
    FrameArgs f{};
    uint32_t gx, gy, ntiles, lo_bits, key_bits, ishape, pshape;
};

// The room for pairs that a frame is issued with: what recent frames of the context needed and a quarter
// more, four pairs a Gaussian at least.  The grids of all that follows the item sort cover it and the
// emission's partitions are chosen by it, so that a small frame does not pay for a large one long ago
// (4k Gaussians at 256x144 after a frame of 17M pairs: 120 us with the buffers' whole room, 97 as without
// that frame).  The buffers keep the room of the largest frame: where a frame needs more than it was given,
// its pairs are issued once more (18 us).
static uint32_t pair_room(const tpd_ctx* c) {
    const size_t recent = (size_t)c->recent_pairs + c->recent_pairs / 4u;
    const size_t room = std::max(std::max<size_t>(4 * (size_t)c->n, kMinPairRoom), recent);
    return (uint32_t)std::min(std::min(room, c->cap_keys), (size_t)kMaxSortKeys);
}

// `room` pairs of the pair buffers as they are, for all that follows the item sort.  The pair sort's shape
// stays the one the pairs' digits were counted for.
static void set_pair_room(tpd_ctx* c, FrameIssue& q, uint32_t room) {
    BatchArgs& a = q.f.b;
    a.cap = room;
    a.keys = c->d_keys;
    a.vals = c->d_vals;
    a.hist_desc0 = c->ws.desc;
    a.pair_part_keys = sort_shape_keys(q.pshape);
}

static FrameIssue plan_frame(tpd_ctx* c, uint32_t gx, uint32_t gy) {
    FrameIssue q;
    q.gx = gx;
    q.gy = gy;
    q.ntiles = gx * gy;
    q.lo_bits = c->wide_frames ? kDepthWideBits : kDepthWindowBits;
    q.key_bits = bit_length(q.ntiles > 1 ? q.ntiles - 1 : 1);
    q.ishape = sort_shape_for(c->item_shape, c->n, q.lo_bits, 8);
    const uint32_t room = pair_room(c);
    q.pshape = sort_shape_for(c->pair_shape, expected_pairs(c->n, room), q.key_bits, 4);
    FrameArgs& f = q.f;
    f.b = item_args(c);
    BatchArgs& a = f.b;
    a.lo_bits = q.lo_bits;
    a.lo_base = c->wide_frames ? 0u : kDepthBase;
    a.hist_counts = c->ws.partials;
    a.hist_tickets = c->ws.tickets;
    a.hist_bits = sort_shape_bits(q.ishape);
    a.hist_plan = sort_digit_plan(q.ishape, q.lo_bits);
    a.hist_desc0_words = ((c->n + sort_shape_keys(q.ishape) - 1) / sort_shape_keys(q.ishape)) << a.hist_bits;
    a.pair_counts = c->ws.partials + kPairCountRow;
    a.pair_bits = sort_shape_bits(q.pshape);
    a.pair_plan = sort_digit_plan(q.pshape, q.key_bits);
    a.ranges = c->d_ranges;
    a.ntiles = q.ntiles;
    f.gauss = c->d_gauss;
    f.ent_idx = c->d_ent_idx;
    f.ent = c->d_ent_mats;
    f.cam = c->cam;
    f.n = c->n;
    f.sh_degree = c->sh_degree;
    f.gx = gx;
    f.gy = gy;
    f.offset_parts = item_offset_parts(c->n);
    set_pair_room(c, q, room);
    return q;
}

// The frame up to its Gaussians in depth order, and its totals on their way to the host.
static void issue_items(tpd_ctx* c, FrameIssue& q, hipStream_t s) {
    ++c->issues;
    BatchArgs& a = q.f.b;
    if (c->profile) hipEventRecord(c->ev[0], s);
    if (c->d_ent_idx)
        launch_entity_mats(c->d_models, c->n_ent, c->cam, c->d_ent_mats, s);
    else
        entity_mats(c->h_models.data(), c->cam, q.f.mats0);
    launch_frame_items(q.f, s);
    if (c->profile) hipEventRecord(c->ev[1], s);
    const FrameTotals totals{a.cap, q.lo_bits, c->n, ++c->frame_seq, c->d_host_counters};
    launch_sort_offsets(c->ws, q.ishape, a.hist_plan.passes, q.pshape, a.pair_plan.passes, c->d_counters, &totals, s);
    if (c->profile) hipEventRecord(c->ev[2], s);
    const bool items_alt = launch_sort_items(c->ws, q.ishape, c->d_ikeys, c->d_ivals, c->d_ikeys_alt, c->d_ivals_alt, c->n,
                                             q.lo_bits, &c->d_counters[kCtrItemsKept], s, &c->d_counters[kCtrSortItems]);
    a.kept_items = &c->d_counters[kCtrItemsKept];
    a.sorted_items = items_alt ? c->d_ivals_alt : c->d_ivals;
    a.sorted_keys64 = items_alt ? c->d_ikeys_alt : c->d_ikeys;
    if (c->profile) hipEventRecord(c->ev[3], s);
    c->emit_event = 3;
}

// The rest: the pairs, their sort and ranges, and the blend.
static int issue_pairs(tpd_ctx* c, const FrameIssue& q, hipStream_t s) {
    const BatchArgs& a = q.f.b;
    launch_batch_emit(a, s);
    if (c->profile) hipEventRecord(c->ev[4], s);
    const bool in_alt = launch_sort_pairs32(c->ws, q.pshape, c->d_keys, c->d_vals, c->d_keys_alt, c->d_vals_alt,
                                            &c->d_counters[kCtrSortPairs], a.cap, q.key_bits, s, true);
    if (c->profile) hipEventRecord(c->ev[5], s);
    c->sorted_keys = in_alt ? c->d_keys_alt : c->d_keys;
    c->sorted_vals = in_alt ? c->d_vals_alt : c->d_vals;
    c->last_passes = a.hist_plan.passes + a.pair_plan.passes;
    launch_ranges(c->sorted_keys, c->d_counters, a.cap, c->d_ranges, c->d_scan_desc,
                  emit_parts(c->n, a.cap), &c->d_counters[kCtrScanTicket], kDepthWideBits, s);
    launch_tile_order(c->d_ranges, q.ntiles, c->d_counters, c->d_tile_hist, c->d_jobs, q.gx, nullptr, nullptr, s);
    if (c->profile) hipEventRecord(c->ev[6], s);
    BlendArgs b{};
    b.counters = c->d_counters;
    b.jobs = c->d_jobs;
    b.vals = c->sorted_vals;
    b.splats = c->d_splats;
    b.width = c->cam.width;
    b.height = c->cam.height;
    b.gx = q.gx;
    b.ntiles = q.ntiles;
    b.image = c->d_image;
    b.rgba8 = c->d_rgba8;
    b.eval_count = nullptr;  // counted on request, by blending the frame once more
    b.final_T = c->d_final_T;  // kept for a backward of this frame
    b.final_last = c->d_final_last;
    b.tile_last = c->d_tile_last;
    launch_blend(b, s);
    c->last_blend = b;
    if (c->profile) hipEventRecord(c->ev[7], s);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TPD_OK : hip_fail(e, "forward launch");
}

int render_forward(tpd_ctx* c, hipStream_t s) {
    const uint32_t W = c->cam.width, H = c->cam.height;
    const uint32_t gx = (W + kTile - 1) / kTile, gy = (H + kTile - 1) / kTile;
    const uint32_t ntiles = gx * gy;
    hipError_t e;
    int rc;
    if ((rc = ensure_scene_buffers(c)) != TPD_OK) return rc;
    if ((rc = ensure_image_buffers(c)) != TPD_OK) return rc;

    if (c->n == 0) {
        // Empty scene: black image, empty ranges (GaussianEngine.cpp:362-365 renders nothing).
        e = hipMemsetAsync(c->d_image, 0, sizeof(float) * 3 * (size_t)W * H, s);
        if (e == hipSuccess) e = hipMemsetAsync(c->d_rgba8, 0, 4 * (size_t)W * H, s);
        if (e == hipSuccess) e = hipMemsetAsync(c->d_ranges, 0, sizeof(uint2) * ntiles, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) return hip_fail(e, "render empty scene");
        // RGBA8 alpha is 1 for every pixel (blend.slang:104 stores float4(C, 1)).
        std::vector<uint8_t> black(4 * (size_t)W * H, 0);
        for (size_t i = 3; i < black.size(); i += 4) black[i] = 255;
        e = hipMemcpy(c->d_rgba8, black.data(), black.size(), hipMemcpyHostToDevice);
        if (e != hipSuccess) return hip_fail(e, "render empty scene");
        c->last_pairs = 0;
        c->sorted_keys = c->d_keys;
        c->sorted_vals = c->d_vals;
        return TPD_OK;
    }

    if (c->cap_keys == 0 && (rc = ensure_pair_buffers(c, std::max<size_t>(4 * (size_t)c->n, kMinPairRoom), s)) != TPD_OK)
        return rc;
    if ((rc = ensure_sort_workspace(c, std::max<size_t>(c->n, c->cap_keys), s)) != TPD_OK) return rc;

    uint32_t P = 0;
    for (;;) {
        FrameIssue q = plan_frame(c, gx, gy);
        issue_items(c, q, s);
        if ((rc = issue_pairs(c, q, s)) != TPD_OK || (rc = wait_totals(c, s, c->frame_seq)) != TPD_OK) return rc;
        P = c->h_counters[kHostPairs];
        const bool depth_out = c->h_counters[kHostDepthOut] != 0, was_wide = c->wide_frames != 0;
        if (P > kMaxSortKeys) return fail(TPD_ERR_CAPACITY, "tpd_render: more than 2^30 - 1 tile/Gaussian pairs");
        if (P >= c->recent_pairs) {
            c->recent_pairs = P;
            c->recent_hold = kRoomHold;
        } else if (c->recent_hold) {
            --c->recent_hold;
        } else {
            c->recent_pairs = std::max(P, c->recent_pairs - c->recent_pairs / 8u);
        }
        if (P > c->cap_keys && (rc = ensure_pair_buffers(c, P, s)) != TPD_OK) return rc;
        if (depth_out) {
            c->wide_frames = kDepthHold;
            if (!was_wide) continue;  // issued again on the wide key
        } else if (was_wide) {
            --c->wide_frames;
        }
        if (c->h_counters[kHostOverflow]) {  // the Gaussians are in order: their pairs once more, with room
            ++c->resumes;
            set_pair_room(c, q, pair_room(c));
            launch_frame_resume(c->d_counters, s);
            if (c->profile) hipEventRecord(c->ev[8], s);
            c->emit_event = 8;
            if ((rc = issue_pairs(c, q, s)) != TPD_OK) return rc;
        }
        break;
    }
    c->last_pairs = P;
    c->has_blend = true;
    if (c->keep_unsorted && P) {
        if ((rc = launch_offsets(c, s)) != TPD_OK) return rc;
        if ((e = grow(c->d_keys_dbg, c->cap_keys_dbg, P, 1.25)) != hipSuccess ||
            (e = grow(c->d_vals_dbg, c->cap_vals_dbg, P, 1.25)) != hipSuccess)
            return hip_fail(e, "alloc unsorted pairs");
        launch_unsorted_pairs(c->d_splats, c->d_tiles, c->d_offsets, c->n, gx, gy, c->d_keys_dbg, c->d_vals_dbg, s);
        if ((e = hipGetLastError()) != hipSuccess) return hip_fail(e, "unsorted pairs");
    }
    return TPD_OK;
}

}  // namespace tpd
