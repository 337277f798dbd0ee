// Batched rendering: many views of many scenes, one launch per stage.  The reference renders one
// camera per GaussianEngine::rasterFrame (GaussianEngine.h:26) and has no batched form; each view
// of a batch is rendered exactly as the plain frame renders it (same per-Gaussian projection,
// same per-view key order, same per-tile blend), only the index spaces are concatenated (the
// layout is described with BatchArgs).
//
//   k_batch_mats            entity matrices of every (view, entity)
//   k_batch_items           each block reads its 256 Gaussian records once and, for every view of
//                           its scene, projects them and writes per item the splat, the tile
//                           rectangle and a depth key; clears the tile ranges
//   k_frame_items           the same for the plain frame's one view
//   (item sort)             the items by depth key
//   k_batch_emit            the pairs in depth order: key = global tile, value = item, positions
//                           by a decoupled look-back scan over the sorted items; total P and the
//                           overflow flag
//   (pair sort, ranges)     the pairs by global tile alone, then the ranges
//   k_batch_item_offsets    for a backward, the items' first pairs in item order
//   k_batch_blend           one 16x16 tile of some view per block (blend_tile)
//   k_batch_blend_bwd       blend_bwd_tile per tile
//   k_batch_preprocess_bwd  per Gaussian, the chain rule summed over the views of its scene, into
//                           the scene's gradient buffers
#include "tpd_blend.hpp"
#include "tpd_grad.hpp"
#include "tpd_kernels.hpp"

#include <type_traits>

namespace tpd {

// Also clears the frame's depth-window flag, which the count pass that follows may set.
__global__ void k_batch_mats(const BatchSceneDev* __restrict__ scenes, const BatchViewDev* __restrict__ views,
                             EntityMats* __restrict__ mats, uint32_t* __restrict__ counters) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) counters[kCtrDepthOut] = 0u;
    const BatchViewDev& vw = views[blockIdx.y];
    const BatchSceneDev& sc = scenes[vw.scene];
    const uint32_t ne = sc.n_ent ? sc.n_ent : 1u;
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne) return;
    entity_mats(sc.models ? sc.models + 16 * (size_t)e : nullptr, vw.cam, mats[vw.mat_base + e]);
}

void launch_batch_mats(const BatchSceneDev* scenes, const BatchViewDev* views, uint32_t nviews, uint32_t max_ent,
                       EntityMats* mats, uint32_t* counters, hipStream_t s) {
    if (nviews == 0) return;
    const uint32_t ne = max_ent ? max_ent : 1u;
    hipLaunchKernelGGL(k_batch_mats, dim3((ne + 63) / 64, nviews), dim3(64), 0, s, scenes, views, mats, counters);
}

__device__ __forceinline__ bool project_in_view(const float* rec, const Cov3& cov, const EntityMats& m,
                                                const BatchViewDev& vw, uint32_t sh_degree, Projected& p) {
    return project_gaussian_cov(rec, [&cov] { return cov; }, m.vm, m.pvm, vw.cam.view,
                                (0.5f * (float)vw.cam.width) * vw.cam.focal_ndc[0],
                                (0.5f * (float)vw.cam.height) * vw.cam.focal_ndc[1], vw.cam.width, vw.cam.height,
                                vw.gx, vw.gy, sh_degree, p);
}

// ------------------------------------------------------------------ items

// The item kernel's digit histograms of the two sorts that follow it.
struct ItemCountLds {
    uint32_t item[kMaxCountedPasses][kMaxRadix];      // item key (depth key) digits, per pass
    uint32_t pair[kMaxCountedPairPasses][kMaxRadix];  // pair key (global tile) digits, per pass
    uint32_t pair_diff[kMaxRadix];  // pass 0: difference array (modulo 2^32) of the digit counts
    uint32_t pair_all;              // pass 0: added to every digit
    uint32_t wave_sum[kPreBlock / kWave];
};

// Counts the pair keys of a tile rectangle: tiles tile0 + r * gx + c, r < h, c < w (w, h >= 1).
// Row r's w tiles are consecutive, so their pass-0 digits are the circular run of w digits from
// d0 = first tile mod R: +1 at d0 and -1 at (d0 + w) mod R in the difference array, whose prefix
// sums then fall one short on every digit for each time the run passes digit R - 1, i.e.
// (d0 + w) / R times; that number goes into all0 (the thread's share of pair_all).  A higher
// pass adds the whole rectangle to one digit when its first and last tile share that digit's
// prefix, else each row's segments.
__device__ __forceinline__ void count_pair_digits(ItemCountLds& L, uint32_t& all0, uint32_t tile0, uint32_t gx,
                                                  uint32_t w, uint32_t h, const DigitPlan& plan) {
    const uint32_t last = tile0 + (h - 1u) * gx + (w - 1u);
    for (uint32_t q = 1; q < plan.passes; ++q) {
        const uint32_t sh = plan.shift[q], dmask = (1u << (plan.shift[q + 1] - sh)) - 1u;
        if ((tile0 >> sh) == (last >> sh)) {
            atomicAdd(&L.pair[q][(tile0 >> sh) & dmask], w * h);
            continue;
        }
        for (uint32_t r = 0; r < h; ++r) {
            uint32_t lo = tile0 + r * gx;
            const uint32_t hi = lo + (w - 1u);
            for (uint32_t seg = lo >> sh; seg <= (hi >> sh); ++seg) {
                const uint32_t end = min(hi, ((seg + 1u) << sh) - 1u);
                atomicAdd(&L.pair[q][seg & dmask], end - lo + 1u);
                lo = end + 1u;
            }
        }
    }
    const uint32_t bits = plan.shift[1], dmask = (1u << bits) - 1u;
    uint32_t t0 = tile0;
    for (uint32_t r = 0; r < h; ++r, t0 += gx) {
        const uint32_t d0 = t0 & dmask;
        atomicAdd(&L.pair_diff[d0], 1u);
        atomicSub(&L.pair_diff[(d0 + w) & dmask], 1u);
        all0 += (d0 + w) >> bits;
    }
}

// Clears the block's counters and its share of what the frame's sorts need cleared: the item sort's
// first descriptors, the tickets, and all tile ranges.
__device__ __forceinline__ void begin_items(const BatchArgs& a, ItemCountLds& L) {
    const uint32_t tid = threadIdx.x, gid = blockIdx.x * kPreBlock + tid, nthreads = gridDim.x * kPreBlock;
    for (uint32_t t = gid; t < a.ntiles; t += nthreads) a.ranges[t] = make_uint2(0u, 0u);
    for (uint32_t x = gid; x < a.hist_desc0_words; x += nthreads) a.hist_desc0[x] = 0u;
    if (blockIdx.x == 0 && tid < kMaxPasses && a.hist_tickets) a.hist_tickets[tid] = 0u;
    for (uint32_t x = tid; x < kMaxCountedPasses * kMaxRadix; x += kPreBlock) (&L.item[0][0])[x] = 0u;
    if (a.pair_counts) {
        for (uint32_t x = tid; x < kMaxCountedPairPasses * kMaxRadix; x += kPreBlock) (&L.pair[0][0])[x] = 0u;
        for (uint32_t x = tid; x < kMaxRadix; x += kPreBlock) L.pair_diff[x] = 0u;
        if (tid == 0) L.pair_all = 0u;
    }
    __syncthreads();
}

// One item in one view: its key (and rectangle record, and tile count for the backward), and the
// digits of its key and of its pairs' keys in the block's counts.  The splat is written already.
__device__ __forceinline__ void put_item(const BatchArgs& a, ItemCountLds& L, uint32_t& all0, uint32_t item, bool vis,
                                         const Projected& p, uint32_t tile_base, uint32_t gx) {
    const uint32_t culled_key = (1u << a.lo_bits) - 1u;  // lo_bits is 27 or 31
    uint64_t key = culled_key;
    if (vis) {
        const uint32_t tile0 = tile_base + (uint32_t)p.y0 * gx + (uint32_t)p.x0;
        const uint32_t w = (uint32_t)(p.x1 - p.x0), h = (uint32_t)(p.y1 - p.y0);
        const uint32_t r32 = inline_rect(tile0, gx, w, h);
        if (r32 == kRectLookup) a.rects[item] = pack_emit_rect(tile0, gx, w, h);
        const uint32_t k32 = (as_uint(p.vz) - a.lo_base) & culled_key;
        key = ((uint64_t)r32 << 32) | k32;
        if (a.pair_counts) count_pair_digits(L, all0, tile0, gx, w, h, a.pair_plan);
        for (uint32_t q = 0; q < a.hist_plan.passes; ++q)  // the item sort drops the culled items
            atomicAdd(&L.item[q][(k32 >> a.hist_plan.shift[q]) &
                                 ((1u << (a.hist_plan.shift[q + 1] - a.hist_plan.shift[q])) - 1u)], 1u);
    }
    a.item_keys[item] = key;
    if (a.tiles) a.tiles[item] = p.tiles;
}

// Adds the block's digit counts to the sorts' (copy blockIdx mod kCountCopies).
__device__ __forceinline__ void flush_item_counts(const BatchArgs& a, ItemCountLds& L, uint32_t all0) {
    const uint32_t tid = threadIdx.x, lane = __lane_id(), wave = tid / kWave;
    const bool pairs = a.pair_counts != nullptr;
    if (pairs) {
        const uint32_t s_all = wave_incl_scan(all0);
        if (lane == kWave - 1 && s_all) atomicAdd(&L.pair_all, s_all);
    }
    __syncthreads();
    const uint32_t R = 1u << a.hist_bits;
    const size_t copy = (blockIdx.x % kCountCopies) * (kMaxPasses * kMaxRadix);
    uint32_t* counts = a.hist_counts + copy;
    for (uint32_t x = tid; x < a.hist_plan.passes * R; x += kPreBlock) {
        const uint32_t v = L.item[x / R][x % R];
        if (v) atomicAdd(&counts[x], v);  // x = pass * R + digit, the layout of the sort's counts
    }
    if (!pairs) return;
    // pass 0 of the pair keys: pair_all plus the inclusive prefix sum of the difference array
    // (modulo 2^32, where its negative entries live); each thread takes PR / 256 consecutive
    // digits (PR = 256 or 512), of which the plan may use fewer
    const uint32_t PR = 1u << a.pair_bits, per = PR / kPreBlock, used = 1u << a.pair_plan.shift[1];
    uint32_t dv[2] = {0u, 0u}, local = 0;
    for (uint32_t i = 0; i < per; ++i) {
        dv[i] = L.pair_diff[tid * per + i];
        local += dv[i];
    }
    const uint32_t incl = wave_incl_scan(local);
    if (lane == kWave - 1) L.wave_sum[wave] = incl;
    __syncthreads();
    uint32_t run = incl - local + L.pair_all;
    for (uint32_t w = 0; w < wave; ++w) run += L.wave_sum[w];
    for (uint32_t i = 0; i < per; ++i) {
        run += dv[i];
        L.pair[0][tid * per + i] = tid * per + i < used ? run : 0u;
    }
    __syncthreads();
    uint32_t* pcounts = a.pair_counts + copy;
    for (uint32_t x = tid; x < a.pair_plan.passes * PR; x += kPreBlock) {
        const uint32_t v = L.pair[x / PR][x % PR];
        if (v) atomicAdd(&pcounts[x], v);
    }
}

// One Gaussian's items, for every view of its scene.  The record's 3D covariance is computed once for
// all views.  ENT: the scene has entities (a per-Gaussian entity index); without, every Gaussian of the
// block uses the view's first entity matrices, a block-uniform address (scalar loads).
template <bool ENT>
__device__ __forceinline__ void items_of_gaussian(const BatchArgs& a, const BatchSceneDev& sc,
                                                  const BatchViewDev* __restrict__ views,
                                                  const uint32_t* __restrict__ scene_views,
                                                  const EntityMats* __restrict__ mats, uint32_t g,
                                                  ItemCountLds& L, uint32_t& all0) {
    const uint32_t e = ENT ? sc.ent_idx[g] : 0u;

    // The record is read once and kept in registers for every view.
    float rec[60];
    const float4* r4 = reinterpret_cast<const float4*>(sc.gauss + (size_t)g * 60);
#pragma unroll
    for (int q = 0; q < 15; ++q) {
        const float4 t = r4[q];
        rec[4 * q + 0] = t.x; rec[4 * q + 1] = t.y; rec[4 * q + 2] = t.z; rec[4 * q + 3] = t.w;
    }
    bool depth_out = false;  // a visible depth outside the sort's depth window
    const OpacityTerms ot = opacity_terms(rec[3]);  // the same for every view
    const Cov3 cov = covariance3d(rec);
    for (uint32_t k = 0; k < sc.nviews; ++k) {
        const BatchViewDev& vw = views[scene_views[sc.view_begin + k]];
        const uint32_t item = vw.item_base + g;
        Projected p;
        const bool vis = project_in_view(rec, cov, mats[vw.mat_base + (ENT ? e : 0u)], vw, sc.sh_degree, p);
        if (vis) {
            store_splat(a.splats + item, p, ot);
            depth_out |= depth_outside_window(p.vz);
        }
        put_item(a, L, all0, item, vis, p, vw.tile_base, vw.gx);
    }
    if (depth_out) atomicOr(&a.counters[kCtrDepthOut], 1u);
}

// Per (Gaussian, view) item: project, write the splat record of a visible item, its emission
// record (and tile count for the backward) and its depth key for the item sort.
// Each block reads its 256 Gaussian records once, for all views of their scene.  It also counts in
// LDS the digits of the item keys (of the visible items) and, with a.pair_counts, of the pair keys
// the emission will write (every tile of each visible item's rectangle), and adds its counts into the
// sorts' digit counts: neither sort reads its keys for them.
__global__ __launch_bounds__(kPreBlock) void k_batch_items(const BatchArgs a, const BatchSceneDev* __restrict__ scenes,
                                                           const BatchViewDev* __restrict__ views,
                                                           const uint32_t* __restrict__ scene_views,
                                                           const uint32_t* __restrict__ block_scene,
                                                           const EntityMats* __restrict__ mats) {
    __shared__ ItemCountLds L;
    begin_items(a, L);
    const uint32_t b = blockIdx.x;
    if (b == 0 && threadIdx.x == 0) {
        a.counters[kCtrSortPairs] = 0u;    // set by the emission
        a.counters[kCtrScanTicket2] = 0u;  // of the item offsets
    }
    if (b >= a.nblocks) return;  // the one block of a batch without Gaussians only clears
    const BatchSceneDev& sc = scenes[block_scene[b]];
    const uint32_t g = (b - sc.first_block) * kPreBlock + threadIdx.x;
    uint32_t all0 = 0;
    if (g < sc.n) {
        if (sc.ent_idx)
            items_of_gaussian<true>(a, sc, views, scene_views, mats, g, L, all0);
        else
            items_of_gaussian<false>(a, sc, views, scene_views, mats, g, L, all0);
    }
    flush_item_counts(a, L, all0);
}

// The plain frame's items: Gaussian i is item i.  A grid of at most kFrameBlocks blocks (three stand on a
// CU at 143 registers; four at 128 took as long) strides over the Gaussians, 256 at a time, so that a block
// adds its counts to the sorts' once.  Also sums the frame's pair count.  Bound by HBM: 3M Gaussians 210 us
// for 0.94 GB.
constexpr uint32_t kFrameBlocks = 1024;
__global__ __launch_bounds__(kPreBlock) void k_frame_items(const FrameArgs f) {
    __shared__ ItemCountLds L;
    __shared__ uint64_t s_total[kPreBlock / kWave];
    const BatchArgs& a = f.b;
    begin_items(a, L);
    const uint32_t tid = threadIdx.x;
    // for a backward that may follow (a fill of its own costs it two launches): the offsets' ticket and
    // descriptors, and the matrices of a scene without entity indices
    if (blockIdx.x == 0) {
        if (tid == 0) a.counters[kCtrScanTicket2] = 0u;
        if (!f.ent_idx && tid < sizeof(EntityMats) / sizeof(float))
            reinterpret_cast<float*>(f.ent)[tid] = reinterpret_cast<const float*>(&f.mats0)[tid];
    }
    for (uint32_t x = blockIdx.x * kPreBlock + tid; x < f.offset_parts; x += gridDim.x * kPreBlock) a.scan_desc2[x] = 0;
    uint32_t all0 = 0;
    uint64_t total = 0;
    bool depth_out = false;
    for (uint32_t i = blockIdx.x * kPreBlock + tid; i < f.n; i += gridDim.x * kPreBlock) {
        // The record into registers at once, 16-byte loads when the records are 16-byte aligned.
        const float* g = f.gauss + (size_t)i * 60;
        float rec[60];
        if ((reinterpret_cast<uintptr_t>(f.gauss) & 15u) == 0u) {  // uniform
            const float4* r4 = reinterpret_cast<const float4*>(g);
#pragma unroll
            for (int q = 0; q < 15; ++q) {
                const float4 t = r4[q];
                rec[4 * q + 0] = t.x; rec[4 * q + 1] = t.y; rec[4 * q + 2] = t.z; rec[4 * q + 3] = t.w;
            }
        } else {
#pragma unroll
            for (int q = 0; q < 60; ++q) rec[q] = g[q];
        }
        Projected p;
        const float fx = (0.5f * (float)f.cam.width) * f.cam.focal_ndc[0];
        const float fy = (0.5f * (float)f.cam.height) * f.cam.focal_ndc[1];
        bool vis;
        if (f.ent_idx) {
            const EntityMats& m = f.ent[f.ent_idx[i]];
            vis = project_gaussian(rec, m.vm, m.pvm, f.cam.view, fx, fy, f.cam.width, f.cam.height, f.gx, f.gy,
                                   f.sh_degree, p);
        } else {
            vis = project_gaussian(rec, f.mats0.vm, f.mats0.pvm, f.cam.view, fx, fy, f.cam.width, f.cam.height, f.gx,
                                   f.gy, f.sh_degree, p);
        }
        if (vis) {
            store_splat(a.splats + i, p, opacity_terms(p.opacity));
            depth_out |= depth_outside_window(p.vz);
            total += p.tiles;
        }
        put_item(a, L, all0, i, vis, p, 0u, f.gx);
    }
    if (ballot(depth_out) != 0 && __lane_id() == 0) atomicOr(&a.counters[kCtrDepthOut], 1u);
    total = wave_sum_u64(total);
    if (__lane_id() == 0) s_total[tid / kWave] = total;
    flush_item_counts(a, L, all0);  // (its barriers order s_total too)
    if (tid == 0) {
        total = 0;
        for (uint32_t w = 0; w < kPreBlock / kWave; ++w) total += s_total[w];
        atomicAdd(reinterpret_cast<unsigned long long*>(a.counters + kCtrTotal64), (unsigned long long)total);
    }
}

void launch_frame_items(const FrameArgs& f, hipStream_t s) {
    const uint32_t chunks = (f.n + kPreBlock - 1) / kPreBlock;
    if (chunks == 0) return;
    hipLaunchKernelGGL(k_frame_items, dim3(chunks < kFrameBlocks ? chunks : kFrameBlocks), dim3(kPreBlock), 0, s, f);
}

void launch_batch_items(const BatchArgs& a, hipStream_t s) {
    const uint32_t nb = a.nblocks ? a.nblocks : 1u;  // one block clears the ranges of an empty batch
    hipLaunchKernelGGL(k_batch_items, dim3(nb), dim3(kPreBlock), 0, s, a, a.scenes, a.views, a.scene_views,
                       a.block_scene, a.mats);
}

// ------------------------------------------------------------------ pair emission in depth order

// Blocks take partitions of 512 x PT depth-sorted items (PT consecutive ones per thread) from an atomic
// ticket; item i's pairs go to base + the exclusive scan of the tile counts over the sorted items
// (decoupled look-back over the partitions), key = global tile, value = item.  The last partition
// stores the pair total and the overflow flag (unless a.totals_known).
//
// The pairs are made position by position: a thread takes 8 consecutive places of the output, aligned
// so that it stores them with 16-byte stores, and needs the item each belongs to.  Items mark the place
// of their first pair in LDS and a maximum scan (thread, wave, block) spreads the marks, so every place
// costs the same whatever the rectangles' sizes: bound by the stores.  (Small rectangles written by
// their own thread and the places of large ones found by a binary search over the block's items, 13
// dependent LDS reads each: 534 us for 22M pairs of 1M items, 500 us for 61M pairs of 32M items;
// this way 125 and 256 us.)
constexpr uint32_t kEmitThreads = 512;
constexpr uint32_t kEmitRun = 8;                              // places per thread
constexpr uint32_t kEmitChunk = kEmitThreads * kEmitRun;      // places per round of the block

template <uint32_t PT>
struct EmitLds {
    uint4 item[kEmitThreads * PT];  // first place, first tile, width | grid width << 16, item
    alignas(16) uint16_t own[kEmitChunk];  // 1 + the block's item whose pairs begin at the place, else 0
    uint32_t wave_sum[kEmitThreads / kWave], wave_max[kEmitThreads / kWave];
    uint64_t base;
    uint32_t part;
};

template <uint32_t PT>
__global__ __launch_bounds__(kEmitThreads) void k_batch_emit(const BatchArgs a) {
    constexpr uint32_t kItems = kEmitThreads * PT;
    __shared__ EmitLds<PT> L;
    const uint32_t tid = threadIdx.x, wave = tid / kWave, lane = __lane_id();
    if (a.totals_known && a.counters[kCtrOverflow]) return;  // the frame is rendered again
    // the pair sort's counts come from the item kernel: its first pass's descriptors (which the
    // item sort's last pass may have used) and the tickets are cleared here, for the pairs where their
    // number is known, else for the room
    if (a.pair_part_keys) {
        const uint32_t pairs = a.totals_known ? a.counters[kCtrSortPairs] : a.cap;
        const uint32_t words = ((pairs + a.pair_part_keys - 1) / a.pair_part_keys) << a.pair_bits;
        for (uint32_t x = blockIdx.x * kEmitThreads + tid; x < words; x += gridDim.x * kEmitThreads) a.hist_desc0[x] = 0u;
        if (blockIdx.x == 0 && tid < kMaxPasses) a.hist_tickets[tid] = 0u;
    }
    // The sorted items are the visible ones (the item sort dropped the culled).  The grid is sized
    // for all items; the blocks past the visible items' partitions leave before taking a ticket
    // (the tickets, one atomic each on one address, pace the blocks' starts), so that exactly the
    // first nparts blocks take tickets 0 .. nparts - 1.
    const uint32_t nitems =
        __builtin_amdgcn_readfirstlane(a.kept_items ? min(*a.kept_items, a.nitems) : a.nitems);
    const uint32_t nparts = (nitems + kItems - 1) / kItems;
    if (blockIdx.x >= nparts) {
        if (blockIdx.x == 0 && tid == 0 && !a.totals_known) {  // no visible item: the totals the last partition would store
            a.counters[kCtrPairs] = 0u;
            a.counters[kCtrOverflow] = 0u;
            a.counters[kCtrSortPairs] = 0u;
        }
        return;
    }
    if (tid == 0) L.part = atomicAdd(&a.counters[kCtrScanTicket], 1u);
    __syncthreads();
    const uint32_t part = __builtin_amdgcn_readfirstlane(L.part);
    if (part >= nparts) return;  // never: the first nparts blocks share nparts tickets
    const uint32_t i0 = part * kItems + tid * PT;

    uint32_t item[PT], rect[PT];  // rect: the key's high word (inline_rect)
    if (PT > 1 && i0 + PT <= nitems) {
#pragma unroll
        for (uint32_t j = 0; j + 1 < PT; j += 2) {  // i0 is a multiple of PT, which is even
            const ulonglong2 k = *reinterpret_cast<const ulonglong2*>(a.sorted_keys64 + i0 + j);
            rect[j] = (uint32_t)(k.x >> 32); rect[j + 1] = (uint32_t)(k.y >> 32);
        }
        if constexpr (PT % 4 == 0) {
#pragma unroll
            for (uint32_t j = 0; j < PT; j += 4) {
                const uint4 v = *reinterpret_cast<const uint4*>(a.sorted_items + i0 + j);
                item[j] = v.x; item[j + 1] = v.y; item[j + 2] = v.z; item[j + 3] = v.w;
            }
        } else if constexpr (PT == 2) {
            const uint2 v = *reinterpret_cast<const uint2*>(a.sorted_items + i0);
            item[0] = v.x; item[1] = v.y;
        }
    } else {
#pragma unroll
        for (uint32_t j = 0; j < PT; ++j) {
            item[j] = i0 + j < nitems ? a.sorted_items[i0 + j] : 0u;
            rect[j] = i0 + j < nitems ? (uint32_t)(a.sorted_keys64[i0 + j] >> 32) : 0u;
        }
    }
    // The items' tile counts, and the places of their first pairs in the block.
    uint32_t t[PT], mine = 0;
    uint4 rec[PT];
#pragma unroll
    for (uint32_t j = 0; j < PT; ++j) {
        const uint64_t r = rect_of(rect[j], a.rects, item[j]);
        t[j] = rect[j] ? emit_rect_w(r) * emit_rect_h(r) : 0u;  // 0: past the end
        rec[j] = make_uint4(mine, emit_rect_tile0(r), emit_rect_w(r) | emit_rect_gx(r) << 16, item[j]);
        mine += t[j];
    }
    const uint32_t incl_w = wave_incl_scan(mine);
    if (lane == kWave - 1) L.wave_sum[wave] = incl_w;
    *reinterpret_cast<uint4*>(&L.own[tid * kEmitRun]) = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    uint32_t wave_off = 0, block_total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kEmitThreads / kWave; ++w) {
        const uint32_t v = L.wave_sum[w];
        wave_off += (w < wave) ? v : 0u;
        block_total += v;
    }
    const uint32_t start = wave_off + incl_w - mine;
#pragma unroll
    for (uint32_t j = 0; j < PT; ++j) {
        rec[j].x += start;
        L.item[tid * PT + j] = rec[j];
    }
    if (wave == 0) {
        if (lane == 0) store_relaxed(&a.scan_desc[part], (part == 0 ? kDescP : kDescA) | (uint64_t)block_total);
        uint64_t excl = 0;
        if (part > 0) excl = scan_lookback(a.scan_desc, part);
        if (lane == 0) {
            if (part > 0) store_relaxed(&a.scan_desc[part], kDescP | (excl + block_total));
            L.base = excl;
            if (part == nparts - 1 && !a.totals_known) {
                const uint64_t total = excl + block_total;
                a.counters[kCtrPairs] = total > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)total;
                a.counters[kCtrOverflow] = total > a.cap ? 1u : 0u;
                a.counters[kCtrSortPairs] = total > a.cap ? 0u : (uint32_t)total;
            }
        }
    }
    __syncthreads();
    const uint64_t base = L.base;
    // Places are counted from the output position at or below base that is a multiple of 8: place p is
    // position base - lead + p, and the block's pairs are places [lead, lead + block_total).
    const uint32_t lead = (uint32_t)base & (kEmitRun - 1u), end = lead + block_total;
    const uint64_t pos0 = base - lead;
    uint32_t carry = 0;  // 1 + the last item whose pairs began before this round
    for (uint32_t c0 = 0; c0 < end; c0 += kEmitChunk) {
        if (pos0 + c0 >= a.cap) break;  // a batch without room: nothing that is left is stored
#pragma unroll
        for (uint32_t j = 0; j < PT; ++j) {
            const uint32_t p = lead + rec[j].x - c0;  // wraps below c0: then not < kEmitChunk
            if (t[j] != 0u && p < kEmitChunk) L.own[p] = (uint16_t)(tid * PT + j + 1u);
        }
        __syncthreads();
        uint4* const mark = reinterpret_cast<uint4*>(&L.own[tid * kEmitRun]);
        const uint4 m = *mark;
        *mark = make_uint4(0u, 0u, 0u, 0u);
        uint32_t o[kEmitRun] = {m.x & 0xFFFFu, m.x >> 16, m.y & 0xFFFFu, m.y >> 16,
                                m.z & 0xFFFFu, m.z >> 16, m.w & 0xFFFFu, m.w >> 16};
#pragma unroll
        for (uint32_t q = 1; q < kEmitRun; ++q) o[q] = max(o[q], o[q - 1]);
        const uint32_t scan = wave_incl_max(o[kEmitRun - 1]);
        if (lane == kWave - 1) L.wave_max[wave] = scan;
        __syncthreads();
        uint32_t before = max(carry, wave_below(scan));
#pragma unroll
        for (uint32_t w = 0; w < kEmitThreads / kWave; ++w) {
            const uint32_t v = L.wave_max[w];
            before = w < wave ? max(before, v) : before;
            carry = max(carry, v);
        }
        const uint32_t p0 = c0 + tid * kEmitRun;
        if (p0 >= end) continue;
        uint32_t key[kEmitRun], val[kEmitRun];
#pragma unroll
        for (uint32_t q = 0; q < kEmitRun; ++q) {
            const uint32_t owner = max(max(o[q], before), 1u) - 1u;  // (item 0 for the places before the first)
            const uint4 r = L.item[owner];
            // row and column of the pair in the rectangle: k / w through an approximate reciprocal,
            // corrected by one step either way (k < 2^22: grids are at most 2048 x 2048 tiles)
            const uint32_t k = p0 + q - lead - r.x, w = r.z & 0xFFFFu;
            int32_t ry = (int32_t)((float)k * __builtin_amdgcn_rcpf((float)w));
            int32_t rx = (int32_t)k - ry * (int32_t)w;
            if (rx < 0) { --ry; rx += (int32_t)w; }
            if (rx >= (int32_t)w) { ++ry; rx -= (int32_t)w; }
            key[q] = r.y + (uint32_t)ry * (r.z >> 16) + (uint32_t)rx;
            val[q] = r.w;
        }
        const uint64_t pos = pos0 + p0;
        if (p0 >= lead && p0 + kEmitRun <= end && pos + kEmitRun <= a.cap) {
            uint4* const dk = reinterpret_cast<uint4*>(a.keys + pos);
            uint4* const dv = reinterpret_cast<uint4*>(a.vals + pos);
            dk[0] = make_uint4(key[0], key[1], key[2], key[3]);
            dk[1] = make_uint4(key[4], key[5], key[6], key[7]);
            dv[0] = make_uint4(val[0], val[1], val[2], val[3]);
            dv[1] = make_uint4(val[4], val[5], val[6], val[7]);
        } else {
#pragma unroll
            for (uint32_t q = 0; q < kEmitRun; ++q)
                if (p0 + q >= lead && p0 + q < end && pos + q < a.cap) {
                    a.keys[pos + q] = key[q];
                    a.vals[pos + q] = val[q];
                }
        }
    }
}

// For frames kept for a backward: the exclusive scan of the items' tile counts in item order,
// where the backward keeps each item's per-pair partial sums (consecutive Gaussians of a view then
// have adjacent partials, which the parameter-gradient pass reads item by item).  Partitions of
// 512 x PT items, decoupled look-back over a.scan_desc2.
template <uint32_t PT>
__global__ __launch_bounds__(kEmitThreads) void k_batch_item_offsets(const BatchArgs a) {
    constexpr uint32_t kItems = kEmitThreads * PT;
    __shared__ uint32_t s_part;
    __shared__ uint32_t s_wave_sum[kEmitThreads / kWave];
    __shared__ uint64_t s_base;
    const uint32_t tid = threadIdx.x, wave = tid / kWave, lane = __lane_id();
    if (tid == 0) s_part = atomicAdd(&a.counters[kCtrScanTicket2], 1u);
    __syncthreads();
    const uint32_t part = __builtin_amdgcn_readfirstlane(s_part);
    const uint32_t nparts = (a.nitems + kItems - 1) / kItems;
    if (part >= nparts) return;
    uint64_t* desc = a.scan_desc2;
    // A wave takes PT / 4 rows of 256 consecutive items, a lane 4 of each row.
    constexpr uint32_t kRows = PT / 4u;
    const uint32_t i0 = part * kItems + wave * (kWave * PT) + 4u * lane;
    const bool full = (part + 1u) * kItems <= a.nitems;
    uint4 t[kRows];
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r) {
        const uint32_t i = i0 + r * 4u * kWave;
        if (full) {
            t[r] = *reinterpret_cast<const uint4*>(a.tiles + i);
        } else {
            t[r].x = i < a.nitems ? a.tiles[i] : 0u;
            t[r].y = i + 1u < a.nitems ? a.tiles[i + 1u] : 0u;
            t[r].z = i + 2u < a.nitems ? a.tiles[i + 2u] : 0u;
            t[r].w = i + 3u < a.nitems ? a.tiles[i + 3u] : 0u;
        }
    }
    uint32_t before[kRows], incl_w = 0;  // the wave's tiles before the lane's items of a row; in all its rows
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r) {
        const uint32_t own = (t[r].x + t[r].y) + (t[r].z + t[r].w), incl = wave_incl_scan(own);
        before[r] = incl_w + incl - own;
        incl_w += (uint32_t)__builtin_amdgcn_readlane(incl, kWave - 1);
    }
    if (lane == kWave - 1) s_wave_sum[wave] = incl_w;
    __syncthreads();
    uint32_t wave_off = 0, block_total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kEmitThreads / kWave; ++w) {
        const uint32_t v = s_wave_sum[w];
        wave_off += (w < wave) ? v : 0u;
        block_total += v;
    }
    if (wave == 0) {
        if (lane == 0) store_relaxed(&desc[part], (part == 0 ? kDescP : kDescA) | (uint64_t)block_total);
        uint64_t excl = 0;
        if (part > 0) excl = scan_lookback(desc, part);
        if (lane == 0) {
            if (part > 0) store_relaxed(&desc[part], kDescP | (excl + block_total));
            s_base = excl;
        }
    }
    __syncthreads();
    const uint32_t base = (uint32_t)s_base + wave_off;
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r) {
        const uint32_t i = i0 + r * 4u * kWave, o = base + before[r];
        const uint4 off = make_uint4(o, o + t[r].x, o + t[r].x + t[r].y, o + t[r].x + t[r].y + t[r].z);
        if (full) {
            *reinterpret_cast<uint4*>(a.offsets + i) = off;
        } else {
            if (i < a.nitems) a.offsets[i] = off.x;
            if (i + 1u < a.nitems) a.offsets[i + 1u] = off.y;
            if (i + 2u < a.nitems) a.offsets[i + 2u] = off.z;
            if (i + 3u < a.nitems) a.offsets[i + 3u] = off.w;
        }
    }
}

// Items per thread of the offsets' scan.  Its partitions finish at the rate of the look-back (about 16 ns
// each), so many items want large ones: at 8 / 16 / 32 per thread 33.8M items take 125 / 95 / 85 us, 3M 19 / 13 / 11.
static uint32_t offsets_per_thread(uint32_t nitems) { return nitems >= (1u << 21) ? 32u : 8u; }

uint32_t item_offset_parts(uint32_t nitems) {
    const uint32_t n = offsets_per_thread(nitems) * kEmitThreads;
    return (nitems + n - 1) / n;
}

void launch_batch_item_offsets(const BatchArgs& a, hipStream_t s) {
    const uint32_t nparts = item_offset_parts(a.nitems);
    if (nparts == 0 || !a.offsets || !a.tiles) return;
    const auto kernel = offsets_per_thread(a.nitems) == 32u ? k_batch_item_offsets<32> : k_batch_item_offsets<8>;
    hipLaunchKernelGGL(kernel, dim3(nparts), dim3(kEmitThreads), 0, s, a);
}

// Items per thread of the emission, by the items and the room for their pairs.  The partitions finish at
// the rate of the look-back, so many items want large ones; few items want enough blocks; and items of
// many pairs each (the nearest partition of 1,024 then holds six times the mean) want the smallest, as
// the block with the most pairs ends last.  Measured, us at 1 / 2 / 4 / 8 items per thread:
//     100k items, 2.4 pairs each    10 /  12 /  15 /  25
//     0.8M items, 1.5 pairs         37 /  27 /  21 /  24
//     1M items, 2.8 pairs           38 /  29 /  29 /  41
//     1M items, 22 pairs            80 / 117 / 176 / 312
//     3M items, 2 pairs             82 /  56 /  46 /  58
//     32M items, 2 pairs           619 / 411 / 300 / 254
static uint32_t emit_per_thread(uint32_t nitems, uint32_t cap) {
    if (nitems < (1u << 18) || cap / 8u >= nitems) return 1u;
    return nitems < (1u << 19) ? 2u : nitems < (1u << 23) ? 4u : 8u;
}

uint32_t emit_max_parts(uint32_t nitems) { return (nitems + kEmitThreads - 1) / kEmitThreads; }

uint32_t emit_parts(uint32_t nitems, uint32_t cap) {
    const uint32_t n = emit_per_thread(nitems, cap) * kEmitThreads;
    return (nitems + n - 1) / n;
}

void launch_batch_emit(const BatchArgs& a, hipStream_t s) {
    const uint32_t nparts = emit_parts(a.nitems, a.cap), per = emit_per_thread(a.nitems, a.cap);
    if (nparts == 0) return;
    const auto kernel = per == 8u ? k_batch_emit<8> : per == 4u ? k_batch_emit<4> : per == 2u ? k_batch_emit<2> : k_batch_emit<1>;
    hipLaunchKernelGGL(kernel, dim3(nparts), dim3(kEmitThreads), 0, s, a);
}

// ------------------------------------------------------------------ blend, forward and backward

__device__ __forceinline__ TileView batch_tile_view(const BatchViewDev* __restrict__ views, const TileJob& j) {
    const BatchViewDev& vw = views[j.view];
    return TileView{j.txy & 0xFFFFu, j.txy >> 16, vw.cam.width, vw.cam.height, vw.gx, vw.gy, vw.pix_base};
}

// COUNT: also adds the evaluated pixel-splat pairs to a.eval_count (a separate launch for the
// FLOP count, so that the frame's own blend is timed without the counting).
template <bool COUNT>
__global__ __launch_bounds__(kTilePixels, 8) void k_batch_blend(const BatchBlendArgs a,
                                                             const BatchViewDev* __restrict__ views) {
    __shared__ BlendFwdLds lds;
    const TileJob j = a.jobs[blockIdx.x];  // loaded beside the flag (meaningless after an overflow)
    if (a.counters[kCtrOverflow]) return;  // the frame is rendered again with larger buffers
    const TileView tv = batch_tile_view(views, j);
    blend_tile<COUNT>(lds, tv, make_uint2(j.start, j.end), a.vals, a.splats, a.image, a.rgba8, a.eval_count, a.final_T,
                      a.final_last, a.tile_last + 4 * (size_t)blockIdx.x);
}

void launch_batch_blend(const BatchBlendArgs& a, hipStream_t s) {
    if (a.ntiles == 0) return;
    if (a.eval_count)
        hipLaunchKernelGGL(k_batch_blend<true>, dim3(a.ntiles), dim3(kTilePixels), 0, s, a, a.views);
    else
        hipLaunchKernelGGL(k_batch_blend<false>, dim3(a.ntiles), dim3(kTilePixels), 0, s, a, a.views);
}

__global__ __launch_bounds__(kTilePixels, 6) void k_batch_blend_bwd(const BatchBlendArgs a,
                                                                 const BatchViewDev* __restrict__ views) {
    __shared__ BlendBwdLds lds;
    const TileJob j = a.jobs[blockIdx.x];
    const int4 last = reinterpret_cast<const int4*>(a.tile_last)[blockIdx.x];
    if (a.counters[kCtrOverflow]) return;
    const TileView tv = batch_tile_view(views, j);
    blend_bwd_tile(lds, tv, make_uint2(j.start, j.end), a.vals, a.splats, a.dL_dimg, a.offsets, a.partials, a.final_T,
                   a.final_last, last);
}

void launch_batch_blend_bwd(const BatchBlendArgs& a, hipStream_t s) {
    if (a.ntiles == 0) return;
    hipLaunchKernelGGL(k_batch_blend_bwd, dim3(a.ntiles), dim3(kTilePixels), 0, s, a, a.views);
}

// ------------------------------------------------------------------ preprocess backward

// Three waves per SIMD: 168 registers and 12 bytes of scratch for 175 registers and two waves.
__global__ __launch_bounds__(kGradBlock, 3) void k_batch_preprocess_bwd(const BatchPreBwdArgs a,
                                                                        const BatchSceneDev* __restrict__ scenes,
                                                                        const BatchViewDev* __restrict__ views,
                                                                        const uint32_t* __restrict__ scene_views,
                                                                        const uint32_t* __restrict__ block_scene,
                                                                        const EntityMats* __restrict__ mats,
                                                                        const BatchGradsDev* __restrict__ grads) {
    // The block's records (consecutive Gaussians, 240 B each) are read from HBM once and kept in LDS for
    // the views of their scene: read again per view, the records of the resident blocks (about 6 MB per
    // XCD) outgrow the XCD's L2.  The same LDS later holds the block's SH gradients (48 floats per
    // Gaussian), stored to HBM the same way.
    __shared__ alignas(16) float s_rec[kGradBlock * kRecStride];
    if (a.counters[kCtrOverflow]) return;  // gradients are left untouched; the step is run again
    constexpr uint32_t kParts = kPreBlock / kGradBlock;  // blocks per item block of block_scene
    const uint32_t b = blockIdx.x / kParts;
    const uint32_t si = block_scene[b];
    const BatchSceneDev& sc = scenes[si];
    const uint32_t g0 = (b - sc.first_block) * kPreBlock + (blockIdx.x % kParts) * kGradBlock;
    if (g0 >= sc.n) return;
    const uint32_t g = g0 + threadIdx.x;
    const uint32_t nvalid = min(kGradBlock, sc.n - g0);
    const bool valid = threadIdx.x < nvalid;           // every thread stays for the barriers
    load_records_block(reinterpret_cast<const float4*>(sc.gauss + (size_t)g0 * 60), nvalid, s_rec);
    __syncthreads();
    const float* rec = s_rec + threadIdx.x * kRecStride;
    const uint32_t e = (valid && sc.ent_idx) ? sc.ent_idx[g] : 0u;
    // The same FP32 operations as a plain backward per view accumulated into the gradient buffers:
    // every log-scale, quaternion, opacity and SH entry receives one term per view, added to the
    // running sum directly; a mean receives three terms per view, so they are summed on their own
    // first and then added.
    float gm[3] = {0.f, 0.f, 0.f}, gls[3] = {0.f, 0.f, 0.f}, gq[4] = {0.f, 0.f, 0.f, 0.f}, gop = 0.f;
    float gsh[48];
#pragma unroll
    for (int k = 0; k < 48; ++k) gsh[k] = 0.f;
    // ent: the scene has entities; without, every Gaussian uses the view's first entity matrices,
    // a block-uniform address (scalar loads)
    // The next view's tile count and offset are loaded ahead of this view's work: each view is a chain of
    // count, partials and arithmetic, with few waves to hide it (64 views of 16 scenes, us: 2179, with three
    // waves per SIMD 2069, with both 1887; the 4.2 GB it moves take 790).
    const auto views_of = [&](auto ent) {
        if (sc.nviews == 0) return;
        uint32_t next_view = scene_views[sc.view_begin];
        uint32_t next_item = views[next_view].item_base + g;
        uint32_t next_tiles = a.tiles[next_item], next_off = a.offsets[next_item];
        for (uint32_t k = 0; k < sc.nviews; ++k) {
            const BatchViewDev& vw = views[next_view];
            const uint32_t tiles = next_tiles, off = next_off;
            next_view = scene_views[sc.view_begin + min(k + 1u, sc.nviews - 1u)];
            next_item = views[next_view].item_base + g;
            next_tiles = a.tiles[next_item];
            next_off = a.offsets[next_item];
            if (tiles == 0) continue;
            float gr[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) gr[q] = 0.0f;
            sum_pair_partials(a.partials + (size_t)off * 9, tiles, gr);
            const EntityMats& m = mats[vw.mat_base + (decltype(ent)::value ? e : 0u)];
            float vm[3] = {0.f, 0.f, 0.f};
            accumulate_param_grads(rec, m.vm, m.pvm, vw.cam, sc.sh_degree, gr, vm, gls, gq, gop, gsh);
#pragma unroll
            for (int c = 0; c < 3; ++c) gm[c] += vm[c];
        }
    };
    if (valid) {
        if (sc.ent_idx)
            views_of(std::true_type{});
        else
            views_of(std::false_type{});
    }
    const BatchGradsDev& gd = grads[si];
    if (valid) store_param_grads_but_sh(g, a.accumulate != 0, gm, gls, gq, gop, gd.means, gd.log_scales, gd.quats,
                                        gd.opacity_logits);
    __syncthreads();  // the records are done with: the LDS takes the SH gradients
    if (valid) {
        float4* d = reinterpret_cast<float4*>(s_rec + threadIdx.x * 48u);
#pragma unroll
        for (int k = 0; k < 12; ++k) d[k] = make_float4(gsh[4 * k], gsh[4 * k + 1], gsh[4 * k + 2], gsh[4 * k + 3]);
    }
    __syncthreads();
    store_sh_grads_block(reinterpret_cast<const float4*>(s_rec), nvalid, a.accumulate != 0,
                         reinterpret_cast<float4*>(gd.sh + (size_t)g0 * 48));
}

void launch_batch_preprocess_bwd(const BatchPreBwdArgs& a, hipStream_t s) {
    if (a.nblocks == 0) return;
    hipLaunchKernelGGL(k_batch_preprocess_bwd, dim3(a.nblocks * (kPreBlock / kGradBlock)), dim3(kGradBlock), 0, s, a, a.scenes, a.views,
                       a.scene_views, a.block_scene, a.mats, a.grads);
}

}  // namespace tpd
