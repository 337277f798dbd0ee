// Kernel argument blocks and launchers shared by the kernels and the C-ABI layer.
#pragma once

#include "tpd_device.hpp"

namespace tpd {

// Indices into the per-context device counter block.
enum : uint32_t {
    kCtrScanTicket = 0,   // partition ticket of the emission
    kCtrPairs = 1,        // pair count P: of the last emission partition, or in a plain frame of its totals
    kCtrOverflow = 2,     // 1 when P exceeded the frame's room or a depth lay outside the window sorted on:
                          // nothing that follows does anything
    kCtrDepthOut = 3,     // non-zero when an emitted depth lies outside the sort's depth window
    kCtrScanTicket2 = 4,  // partition ticket of a second scan in the frame (the item offsets), cleared by
                          // the item kernel
    kCtrSortPairs = 5,    // pair count for the pair sort and the ranges: P, or 0 when the frame overflowed
                          // (it is rendered again)
    kCtrTotal64 = 6,      // (two words) the plain frame's pair count, summed by its item kernel; zero between
                          // frames
    kCtrSortItems = 8,    // the plain frame's items to be sorted: all, or 0 when a depth lies outside the window
                          // that they would be sorted on
    kCtrItemsKept = 32,   // the visible items: those the item sort keeps (its later passes and
                          // the emission run on them).  128 bytes past the tickets: every emission
                          // block reads it right after its ticket atomic, and on the tickets' L2
                          // line that read would queue behind the other blocks' atomics
    kCtrCount = 64,
};

// The sort's depth window.  Culling keeps view depths inside [near, far], and depths in
// [2^-8, 2^8) have float bit patterns in [kDepthBase, kDepthBase + 2^27): such frames sort their items
// by the 27 bits (depth bits - kDepthBase), in the same order as the depth bits and with 4 bits less
// than a positive float.  A frame with any depth outside the window (flagged by its item kernel in
// kCtrDepthOut) sorts the 31-bit form.
constexpr uint32_t kDepthBase = 0x3B800000u;  // floatbits(2^-8)
constexpr uint32_t kDepthWindowBits = 27;
constexpr uint32_t kDepthWideBits = 31;
__device__ __forceinline__ bool depth_outside_window(float vz) {
    return __float_as_uint(vz) - kDepthBase >= (1u << kDepthWindowBits);
}

// The digits of an LSD radix sort's passes: pass p orders the bits [shift[p], shift[p + 1]) of the key.
// The key's bits are shared out evenly (13 bits in two passes: 6 and 7, not 8 and 5): fewer digits in
// a pass mean longer runs of equal digits, and the length of the runs it writes bounds a pass.
constexpr uint32_t kMaxPasses = 8;
struct DigitPlan {
    uint32_t passes;
    uint32_t shift[kMaxPasses + 1];
};

// A block of the blend: one tile, its sorted pairs and (in a batch) its view, in the launch order of
// launch_tile_order.  One 16-byte load by block index tells the block all it needs.
struct alignas(16) TileJob {
    uint32_t txy;         // tile column | tile row << 16, inside the view
    uint32_t start, end;  // the tile's range of the sorted pairs
    uint32_t view;        // batch: the tile's view (0 in a plain frame)
};

struct BlendArgs {
    const uint32_t* counters;    // the frame's kCtr* block: nothing is done after an overflow
    const TileJob* jobs;         // per block (heaviest tiles first)
    const uint32_t* vals;
    const Splat* splats;
    uint32_t width, height, gx, ntiles;
    float* image;            // H x W x 3 or null
    uint8_t* rgba8;          // H x W x 4 or null
    uint64_t* eval_count;    // when non-null, incremented by the number of evaluated pixel-splat pairs
    float* final_T;          // H x W final transmittance, for the backward (or null)
    int32_t* final_last;     // H x W sorted index of the last blended splat, -1 for none (or null)
    int32_t* tile_last;      // with final_T: per block and wave, the largest final_last
};

struct BackwardArgs {
    const TileJob* jobs;         // the forward frame's
    const uint32_t* vals;
    const Splat* splats;
    uint32_t width, height, gx, gy, ntiles;
    const float* dL_dimg;    // H x W x 3
    const uint32_t* offsets; // per-Gaussian exclusive scan of tile counts (pre-sort pair position)
    float* partials;         // P x 9 per (tile, splat) pair at its pre-sort position: dL/d(image x, y,
                             // conic a, b, c, r, g, b, opacity); every pair is written
    const float* final_T;    // the forward frame's per-pixel final transmittance
    const int32_t* final_last;  // and last blended splat
    const int32_t* tile_last;   // and its last blended splat per block and wave
};

struct PreBackwardArgs {
    const float* gauss;
    const uint32_t* ent_idx;     // N entity indices, or null: every Gaussian uses the first
    const EntityMats* ent;       // per entity
    CameraParams cam;
    uint32_t n, sh_degree;
    const uint32_t* tiles;
    const uint32_t* offsets;
    const float* partials;       // P x 9, summed per Gaussian over its tiles in tile order
    float* g2d;                  // N x 9 per-Gaussian sums (written, for inspection)
    float* grad_means;           // N x 3
    float* grad_log_scales;      // N x 3
    float* grad_quats;           // N x 4
    float* grad_opacity_logits;  // N
    float* grad_sh;              // N x 48
    uint32_t accumulate;         // add to the outputs instead of overwriting them
};

void launch_blend_bwd(const BackwardArgs& a, hipStream_t s);
void launch_preprocess_bwd(const PreBackwardArgs& a, hipStream_t s);

void launch_entity_mats(const float* models, uint32_t n_ent, const CameraParams& cam, EntityMats* out, hipStream_t s);
// Tile ranges of the P = min(counters[kCtrSortPairs], cap) sorted keys (tiles).  Also re-zeroes the scan
// descriptors and the emission's ticket for the next frame, and sets kCtrOverflow when a frame whose items
// were sorted on the depth-window key (lo_bits = kDepthWindowBits) has kCtrDepthOut set, which it clears
// otherwise.
void launch_ranges(const uint32_t* keys, uint32_t* counters, uint32_t cap, uint2* ranges, uint64_t* scan_desc,
                   uint32_t n_scan_desc, uint32_t* ticket, uint32_t lo_bits, hipStream_t s);
// The 64-bit keys (tile << 32) | floatbits(view depth) of n sorted tile keys, the depth from the splat
// of each value (for readers of the sorted pairs).
void launch_full_keys(const uint32_t* keys, const uint32_t* vals, const Splat* splats, uint32_t n, uint64_t* out,
                      hipStream_t s);
// The plain frame's pairs in the reference's emission order (Gaussian by Gaussian, row-major over each
// one's rectangle), 64-bit keys, at the scan of the tile counts (for readers of the unsorted pairs).
void launch_unsorted_pairs(const Splat* splats, const uint32_t* tiles, const uint32_t* offsets, uint32_t n, uint32_t gx,
                           uint32_t gy, uint64_t* keys, uint32_t* vals, hipStream_t s);
void launch_blend(const BlendArgs& a, hipStream_t s);
// The tiles in launch order for the blend: classes of pair count (bit length) from the heaviest
// down, empty tiles last, so that the longest tiles start first and the short ones fill the tail.
// counters (optional): nothing is done after a pair overflow.  `jobs` receives a job per tile in
// that order; `hist` is scratch for the per-chunk class counts.  grid_width > 0: the tile columns of
// the one view; 0: tile t belongs to view tile_view[t] of views.
constexpr uint32_t kOrderChunk = 1024;  // tiles per block
constexpr uint32_t kTileClasses = 33;   // pair-count bit lengths 0 .. 32
inline size_t tile_hist_words(size_t ntiles) { return kTileClasses * ((ntiles + kOrderChunk - 1) / kOrderChunk); }
struct BatchViewDev;
void launch_tile_order(const uint2* ranges, uint32_t ntiles, const uint32_t* counters, uint32_t* hist, TileJob* jobs,
                       uint32_t grid_width, const uint32_t* tile_view, const BatchViewDev* views, hipStream_t s);

// ------------------------------------------------------------------ batched rendering
//
// Many views of many scenes in one launch per stage.  Layout:
//   items   view-major: Gaussian g of view v is item views[v].item_base + g; per-item splats,
//           tile counts and pair offsets are indexed by item, pair values are items;
//   tiles   global tile t of view v is views[v].tile_base + (local tile); keys carry global
//           tiles, so one sort orders every view's pairs and the views' ranges are disjoint;
//   pixels  view v's image starts at pixel views[v].pix_base of the concatenated images;
//   blocks  preprocess block b covers Gaussians [256 (b - first_block), +256) of scene
//           block_scene[b] and projects them into every view of that scene, reading each
//           Gaussian record once;
//   order   items are sorted by depth key (stable: equal depths keep item order, which within a
//           view is Gaussian order), their pairs are emitted in that order, and the pairs are
//           then sorted by global tile alone (stable): within each tile they stay in (depth,
//           Gaussian) order, the order of the reference's (tile << 32 | depth) sort.

struct BatchSceneDev {
    const float* gauss;          // N x 60 records
    const uint32_t* ent_idx;     // N entity indices, or null
    const float* models;         // n_ent x 16 model matrices, or null (identity)
    uint32_t n, sh_degree, n_ent;
    uint32_t first_block;        // first preprocess block of the scene
    uint32_t view_begin, nviews; // the scene's views: scene_views[view_begin, view_begin + nviews)
    uint32_t pad;
};

struct BatchViewDev {
    CameraParams cam;
    uint32_t scene, gx, gy, tile_base;
    uint32_t item_base;          // item of Gaussian g = item_base + g
    uint32_t mat_base;           // entity matrices of this view at mats[mat_base + e]
    uint64_t pix_base;           // first pixel of this view in the concatenated images
};

struct BatchArgs {
    const BatchSceneDev* scenes;
    const BatchViewDev* views;
    const uint32_t* scene_views;  // view indices grouped by scene
    const uint32_t* block_scene;  // scene of each preprocess block
    uint32_t nblocks, nviews, nitems;
    const EntityMats* mats;
    uint64_t* scan_desc;          // look-back descriptors, zero on entry: one per emission partition ...
    uint64_t* scan_desc2;         // ... and one per partition of the item offsets
    uint32_t* counters;           // kCtr* block
    uint32_t cap;                 // pair capacity
    Splat* splats;                // per item (written for visible items only)
    uint32_t* tiles;              // per item tile counts, or null (kept for the backward)
    uint32_t* offsets;            // per item exclusive scan of the tile counts in item order, or null:
                                  // where the backward keeps the item's per-pair partial sums
    uint64_t* rects;              // per item emission record (pack_emit_rect), written only where the key
                                  // carries kRectLookup
    uint64_t* item_keys;          // per item: low word the depth key ((depth bits - lo_base) in lo_bits
                                  // bits, all ones within lo_bits when culled), high word the emission
                                  // record as inline_rect encodes it
    uint32_t lo_bits, lo_base;
    // the item sort's digit histograms, counted by the item kernel (the sort then skips its own):
    // counts as k_sort_hist leaves them (copy blockIdx mod kCountCopies), digit width and passes of
    // the item sort's shape; the first pass's look-back descriptors (desc0_words) and the tickets
    // are cleared here too
    uint32_t* hist_counts;
    uint32_t* hist_desc0;
    uint32_t* hist_tickets;
    uint32_t hist_bits, hist_desc0_words;
    DigitPlan hist_plan;
    // the pair sort's digit histograms, counted by the item kernel from each visible item's tile
    // rectangle (needs hist_counts): counts from row kPairCountRow of the sort's digit counts, digit
    // width and passes of the pair sort's shape; the emission clears the pair sort's first-pass
    // descriptors (a partition has pair_part_keys pairs, 0: none to clear) and the tickets
    uint32_t* pair_counts;
    uint32_t pair_bits, pair_part_keys;
    DigitPlan pair_plan;
    uint32_t totals_known;          // the emission finds P and the overflow flag in the counters (plain frame)
    const uint32_t* kept_items;     // emission input: the number of sorted items (the visible ones) ...
    const uint64_t* sorted_keys64;  // ... the item keys in depth order ...
    const uint32_t* sorted_items;   // ... and their items
    uint32_t* keys;               // pairs: global tile
    uint32_t* vals;               //        item
    uint2* ranges;                // all views' tiles, cleared by the item kernel
    uint32_t ntiles;
};

// The plain frame's items: one view of one scene, its tables in the kernel's arguments.
struct FrameArgs {
    BatchArgs b;
    const float* gauss;           // N x 60 records (any alignment)
    const uint32_t* ent_idx;      // N entity indices, or null: every Gaussian uses mats0
    EntityMats* ent;              // per entity; without ent_idx the kernel stores mats0 there, for the backward
    EntityMats mats0;
    CameraParams cam;
    uint32_t n, sh_degree, gx, gy;
    uint32_t offset_parts;        // partitions of the item offsets, whose descriptors are cleared
};

struct BatchBlendArgs {
    const BatchViewDev* views;
    const TileJob* jobs;          // per block (heaviest tiles first)
    const uint32_t* vals;
    const Splat* splats;
    uint32_t ntiles;
    const uint32_t* counters;     // the frame's kCtr* block: nothing is done after an overflow
    float* image;                 // concatenated H x W x 3 images, or null
    uint8_t* rgba8;               // concatenated H x W x 4 images, or null
    const float* dL_dimg;         // backward: concatenated H x W x 3 upstream gradients
    const uint32_t* offsets;      // backward: per item pre-sort pair offsets
    float* partials;              // backward: P x 9 per pair
    float* final_T;               // per pixel final transmittance: written by a forward kept for the
    int32_t* final_last;          // backward, read by it (with the last blended splat); or null
    int32_t* tile_last;           // the largest final_last per block and wave, likewise
    uint64_t* eval_count;         // forward: evaluated pixel-splat pairs are added here, or null
};

struct BatchGradsDev {            // one scene's parameter-gradient buffers
    float* means;                 // N x 3
    float* log_scales;            // N x 3
    float* quats;                 // N x 4
    float* opacity_logits;        // N
    float* sh;                    // N x 48
};

struct BatchPreBwdArgs {
    const BatchSceneDev* scenes;
    const BatchViewDev* views;
    const uint32_t* scene_views;
    const uint32_t* block_scene;
    uint32_t nblocks;
    const EntityMats* mats;
    const uint32_t* tiles;
    const uint32_t* offsets;
    const float* partials;
    const BatchGradsDev* grads;   // per scene
    const uint32_t* counters;     // nothing is written after an overflow
    uint32_t accumulate;
};

void launch_batch_mats(const BatchSceneDev* scenes, const BatchViewDev* views, uint32_t nviews, uint32_t max_ent,
                       EntityMats* mats, uint32_t* counters, hipStream_t s);
void launch_batch_items(const BatchArgs& a, hipStream_t s);
void launch_frame_items(const FrameArgs& a, hipStream_t s);
void launch_batch_emit(const BatchArgs& a, hipStream_t s);
void launch_batch_item_offsets(const BatchArgs& a, hipStream_t s);
// Partitions of the emission (of a frame with room for `cap` pairs, and the most of any) and of the item
// offsets.
uint32_t emit_parts(uint32_t nitems, uint32_t cap);
uint32_t emit_max_parts(uint32_t nitems);
uint32_t item_offset_parts(uint32_t nitems);
void launch_batch_blend(const BatchBlendArgs& a, hipStream_t s);
void launch_batch_blend_bwd(const BatchBlendArgs& a, hipStream_t s);
void launch_batch_preprocess_bwd(const BatchPreBwdArgs& a, hipStream_t s);

// ------------------------------------------------------------------ radix sort

constexpr uint32_t kMaxRadixBits = 9;                      // digit widths 8 and 9 bits
constexpr uint32_t kMaxRadix = 1u << kMaxRadixBits;
constexpr uint32_t kSortMinTile = 2048;                    // smallest partition of any block shape
constexpr uint32_t kCountCopies = 8;  // copies of the digit counts, block b adds into copy b mod 8
constexpr uint32_t kHistBlocks = 1024;                      // blocks of the digit-histogram kernel
constexpr uint32_t kMaxSortKeys = (1u << 30) - 1;          // 30-bit look-back values

constexpr uint32_t kShapeAuto = 0xFFFFFFFFu;  // the shape the key count and width ask for (sort_shape_for)

struct SortWorkspace {
    uint32_t* desc = nullptr;      // 2 regions x parts_cap x kMaxRadix look-back descriptors
    uint32_t parts_cap = 0;
    uint32_t* partials = nullptr;  // kCountCopies x kMaxPasses x kMaxRadix digit counts (zero between sorts)
    uint32_t* offsets = nullptr;   // kMaxPasses x kMaxRadix global exclusive digit offsets
    uint32_t* tickets = nullptr;   // kMaxPasses partition tickets
    uint32_t shape = kShapeAuto;   // onesweep block shape (index into the tuner's table), or kShapeAuto
};

// Partitions for n keys at the smallest partition size (descriptor capacity for every shape).
__host__ __device__ inline uint32_t sort_parts(uint32_t n) { return (n + kSortMinTile - 1) / kSortMinTile; }
uint32_t sort_num_shapes();
// The shape itself, or for kShapeAuto the one for n keys of key_bytes with key_bits sorted.
uint32_t sort_shape_for(uint32_t shape, uint32_t n, uint32_t key_bits, uint32_t key_bytes);
// The pair count a shape is chosen for before the pairs are counted: most frames have 1.5 to 4 pairs a
// Gaussian, and buffers keep the room of larger frames.
inline uint32_t expected_pairs(uint32_t nitems, uint32_t cap) { return nitems < cap / 4u ? 4u * nitems : cap; }
uint32_t sort_shape_keys(uint32_t shape);
uint32_t sort_shape_bits(uint32_t shape);                       // digit width of a shape
uint32_t sort_shape_passes(uint32_t shape, uint32_t key_bits);  // passes for key_bits bits
DigitPlan sort_digit_plan(uint32_t shape, uint32_t key_bits);

// Stable LSD sort of n (64-bit key, value) pairs by the low key_bits bits of the keys.  Returns true
// when the sorted data ended in the alternate buffers.
bool launch_sort_pairs(SortWorkspace& ws, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt,
                       uint32_t n, uint32_t key_bits, hipStream_t s);

// The frame's sorts, whose digit counts the item kernel has made (it also cleared the first pass's
// descriptors and the tickets): items in ws.partials from word 0 of each copy, pairs from word
// kPairCountRow.  launch_sort_offsets turns both into digit offsets (items from word 0 of ws.offsets,
// pairs from kPairCountRow) and re-zeroes the counts.  pair_shape with ppasses = 0: no counted pairs.
// With a frame (totals non-null) it also settles the frame's totals from the item kernel's: kCtrPairs,
// kCtrOverflow (more pairs than cap, or a depth outside the window of an item sort on it), kCtrSortPairs,
// kCtrSortItems, and tells the host.
constexpr uint32_t kMaxCountedPasses = 4;      // item passes whose counts the item kernel can make
constexpr uint32_t kMaxCountedPairPasses = 3;
constexpr uint32_t kPairCountRow = kMaxCountedPasses * kMaxRadix;
static_assert(kPairCountRow + kMaxCountedPairPasses * kMaxRadix <= kMaxPasses * kMaxRadix, "pair count rows");
enum : uint32_t { kHostPairs = 0, kHostOverflow = 1, kHostDepthOut = 2, kHostSeq = 3 };  // words of FrameTotals::host
struct FrameTotals {
    uint32_t cap, lo_bits, items;
    uint32_t seq;      // stored last, when the other words are there
    uint32_t* host;    // pinned host memory
};
void launch_sort_offsets(SortWorkspace& ws, uint32_t item_shape, uint32_t ipasses, uint32_t pair_shape, uint32_t ppasses,
                         uint32_t* counters, const FrameTotals* totals, hipStream_t s);
// Lets a frame that had no room for its pairs go on from its emission (the host has made room).
void launch_frame_resume(uint32_t* counters, hipStream_t s);
// Sorts the n items by the low lo_bits bits of their keys.  The first pass drops the keys whose high
// word is zero (the counts leave them out) and takes each key's index as its value; the later ones
// sort the *kept others.  count_ptr (optional): nothing is sorted when *count_ptr is 0.
bool launch_sort_items(SortWorkspace& ws, uint32_t shape, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt,
                       uint32_t* vals_alt, uint32_t n, uint32_t lo_bits, const uint32_t* kept, hipStream_t s,
                       const uint32_t* count_ptr = nullptr);
// Sorts the min(*count_ptr, n_max) pairs by the low key_bits bits of their 32-bit keys; without
// counted, their digits are counted first (after_count: recorded then).
bool launch_sort_pairs32(SortWorkspace& ws, uint32_t shape, uint32_t* keys, uint32_t* vals, uint32_t* keys_alt,
                         uint32_t* vals_alt, const uint32_t* count_ptr, uint32_t n_max, uint32_t key_bits, hipStream_t s,
                         bool counted, hipEvent_t after_count = nullptr);

}  // namespace tpd
