// Per-tile blend bodies shared by the plain and the batched kernels: the forward front-to-back
// composite (blend.slang:22-105) and its backward.  A kernel maps its block to a tile (TileView)
// and calls blend_tile / blend_bwd_tile with its block's LDS.
#pragma once

#include "tpd_device.hpp"

namespace tpd {

// Where a tile's pixels lie: tile coordinates inside its view, the view's size and tile grid,
// and the view's first pixel in the (concatenated) image buffers.
struct TileView {
    uint32_t tx, ty;
    uint32_t width, height;
    uint32_t gx, gy;
    uint64_t pix_base;
};

constexpr uint32_t kSub = 4;                              // 4x4-pixel sub-blocks ...
constexpr uint32_t kSubBlocks = kTilePixels / (kSub * kSub);  // ... 16 per tile, one per 16-lane row
constexpr uint32_t kSplatGrads = 9;  // dL/d(image x, y, conic a, b, c, r, g, b, opacity)

// A staging round holds up to N splats of the tile's sorted list in slots 0..N-1; slot N is a
// sentinel that no pixel can take (skip threshold +inf).  Sub-block lists hold the byte offsets
// of the slots of the splats that can reach the sub-block, in sorted order, padded with the
// sentinel up to the longest list of the wave.
//
// Both kernels wait for LDS and for their own arithmetic, so the blocks a CU holds decide their speed: N,
// the slots' layout and the launch bounds are chosen for eight blocks of the forward (64 registers, 18.7 KB
// of LDS; 5 / 6 / 7 / 8 blocks: 3.70 / 3.39 / 3.16 / 3.00 ms for 64 views of 46.5M pixels and 62.9M pairs)
// and six of the backward (80 registers, 26.3 KB; 3 / 4 / 5 / 6 blocks: 9.86 / 8.42 / 7.77 / 7.69 ms).
struct BlendSlot {
    float2 xy, ab;  // centre; conic a, b
    float2 cs, po;  // conic c, skip threshold; opacity, red
    float2 gb;      // green, blue
};
// The backward's slot also holds the tile's gradient sums of its splat, so that a list entry is the
// address of both.
struct alignas(16) BlendBwdSlot {
    double acc[kSplatGrads];
    float2 gb;
    float2 xy, ab;
    float2 cs, po;
};

template <typename SLOT, uint32_t N>
struct BlendLds {
    static constexpr uint32_t kSlots = N;
    static constexpr uint32_t kSentinel = N * sizeof(SLOT);  // byte offset of the slot no pixel takes
    static_assert(kSentinel < 65536u && (N & 7u) == 0u && N <= kTilePixels, "list entries");
    SLOT slot[N + 1];
    alignas(16) uint16_t list[kSubBlocks][N];
    alignas(16) uint32_t cnt[kBlendWaves][kSubBlocks];  // [staging wave][sub-block]
    alignas(16) uint32_t done[kBlendWaves];             // per wave: all of its pixels have terminated
    __device__ __forceinline__ SLOT& at(uint32_t off) {
        return *reinterpret_cast<SLOT*>(reinterpret_cast<char*>(slot) + off);
    }
};
using BlendFwdLds = BlendLds<BlendSlot, kTilePixels>;
using BlendBwdLds = BlendLds<BlendBwdSlot, 184>;

// Sub-blocks are numbered row-major inside the tile: q = 4 * row + column (4x4 pixels each).
__device__ __forceinline__ void sub_block_origin(const TileView& tv, uint32_t q, uint32_t& x0, uint32_t& y0) {
    x0 = tv.tx * kTile + (q & 3u) * kSub;
    y0 = tv.ty * kTile + (q >> 2) * kSub;
}

// Sub-block walked by row g (0..3) of wave w: wave w owns the 8x8 quadrant (w & 1, w >> 1) of the
// tile, row g the 4x4 block (g & 1, g >> 1) inside it.
__device__ __forceinline__ uint32_t sub_block_of(uint32_t w, uint32_t g) {
    return (((w >> 1) * 2u + (g >> 1)) * 4u) + (w & 1u) * 2u + (g & 1u);
}

// Pixel of this thread: the sub-block of its wave and 16-lane row, lanes row-major inside it.
__device__ __forceinline__ void tile_pixel(const TileView& tv, uint32_t& px, uint32_t& py) {
    const uint32_t wave = threadIdx.x / kWave, lane = __lane_id();
    uint32_t x0, y0;
    sub_block_origin(tv, sub_block_of(wave, lane >> 4), x0, y0);
    px = x0 + (lane & 3u);
    py = y0 + ((lane >> 2) & 3u);
}

// Stages a round of the tile's sorted list in LDS and builds one
// compacted list per 4x4 sub-block (sorted order kept) of the splats that may reach
// alpha >= 1/255 at some pixel centre of the sub-block (sub_block_mask, with the per-splat part
// the preprocess stored in the record).  Returns the number
// of list entries this wave walks: the longest of its four lists (the shorter ones are padded
// with the sentinel).  Ends with a barrier.
// This thread's splat of a staging round: whether the slot holds one, its index and its record.
struct StagedSplat {
    bool valid;
    uint32_t g;
    Splat sp;
};

// Both loads are unconditional (slot past the end: value 0 and record 0, which every non-empty
// buffer has), so that a load issued a round ahead stays in flight in its own registers.
__device__ __forceinline__ uint32_t load_value(const uint32_t* __restrict__ vals, uint32_t k, uint32_t end) {
    return vals[k < end ? k : 0u];
}

__device__ __forceinline__ StagedSplat load_staged(const Splat* __restrict__ splats, uint32_t g, uint32_t k,
                                                   uint32_t end) {
    StagedSplat t;
    t.valid = k < end;
    t.g = g;
    t.sp = splats[t.valid ? g : 0u];
    return t;
}

template <typename LDS>
__device__ __forceinline__ uint32_t blend_stage_loaded(LDS& s, const TileView& tv, const StagedSplat& in) {
    const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = __lane_id();
    {
        constexpr uint32_t words = sizeof(s.list) / sizeof(uint4);
        uint32_t s2 = LDS::kSentinel | (LDS::kSentinel << 16);
        asm volatile("" : "+s"(s2));  // made anew each round: four registers held through the walk spill
        uint4* lw = reinterpret_cast<uint4*>(&s.list[0][0]);
        static_assert(words > kTilePixels && words <= 2 * kTilePixels, "list fill");
        lw[tid] = make_uint4(s2, s2, s2, s2);
        if (tid < words - kTilePixels) lw[tid + kTilePixels] = make_uint4(s2, s2, s2, s2);
        if (tid == 0) {
            auto& e = s.at(LDS::kSentinel);
            e.xy = e.ab = e.po = e.gb = make_float2(0.0f, 0.0f);
            e.cs = make_float2(0.0f, __builtin_inff());
        }
    }
    uint32_t mask = 0;
    // the tile's bands, in scalar registers
    float band_y[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        band_y[k] = as_float(__builtin_amdgcn_readfirstlane(as_uint((float)(tv.ty * kTile + kSub * k))));
    if (in.valid) {
        const Splat& sp = in.sp;
        const float4 p = sp.xyzr;
        const float4 c = sp.conop;
        auto& e = s.slot[tid];
        e.xy = make_float2(p.x, p.y);
        e.ab = make_float2(c.x, c.y);
        e.cs = make_float2(c.z, sp.aux.x);
        e.po = make_float2(c.w, sp.rgb.x);
        e.gb = make_float2(sp.rgb.y, sp.rgb.z);
        const uint32_t reach = sub_block_mask_bands(p.x, p.y, c.x, c.y, c.z,
                                                    SubBlockReach{sp.aux.y, sp.aux.z, sp.aux.w, sp.rgb.w},
                                                    (float)(tv.tx * kTile), band_y);
        // sub-blocks with at least one pixel inside the view
        const uint32_t vx = min((tv.width - tv.tx * kTile + kSub - 1) / kSub, 4u);
        const uint32_t vy = min((tv.height - tv.ty * kTile + kSub - 1) / kSub, 4u);
        const uint32_t vcols = (1u << vx) - 1u;
        const uint32_t vrows = (1u << vy) - 1u;
        const uint32_t vspread = (vrows & 1u) | ((vrows & 2u) << 3) | ((vrows & 4u) << 6) | ((vrows & 8u) << 9);
        mask = reach & (vcols * vspread);
    }
    uint64_t bal[kSubBlocks];
#pragma unroll
    for (uint32_t q = 0; q < kSubBlocks; ++q) bal[q] = ballot((mask >> q) & 1u);
    if (lane == 0) {
#pragma unroll
        for (uint32_t q = 0; q < kSubBlocks; ++q) s.cnt[wave][q] = (uint32_t)__popcll(bal[q]);
    }
    __syncthreads();
    // lane q < 16: this wave's start in sub-block q's list, and the list's length
    uint32_t start = 0, total = 0;
    if (lane < kSubBlocks) {
#pragma unroll
        for (uint32_t w = 0; w < kBlendWaves; ++w) {
            const uint32_t n = s.cnt[w][lane];
            start += w < wave ? n : 0u;
            total += n;
        }
    }
    // The lanes with bit q set are exactly bal[q]: it serves as the execution mask, and the
    // lane's rank among them is a masked bit count.
#pragma unroll
    for (uint32_t q = 0; q < kSubBlocks; ++q) {
        if (lane_on(bal[q])) {
            const uint32_t off = (uint32_t)__builtin_amdgcn_readlane(start, q) + lanes_below(bal[q]);
            s.list[q][off] = (uint16_t)(tid * sizeof(s.slot[0]));
        }
    }
    uint32_t walk = 0;
#pragma unroll
    for (uint32_t g = 0; g < 4; ++g) walk = max(walk, (uint32_t)__builtin_amdgcn_readlane(total, sub_block_of(wave, g)));
    __syncthreads();
    return walk;
}

// Forward composite of one tile.  Per pixel the operations and their order are the reference's;
// the shortcuts around them change no pixel:
//   - the sub-block lists of blend_stage drop only splats no pixel of the sub-block can take;
//   - skip = log(1/(255 o)) - 0.01: a power below it gives o * exp(power) < 0.99/255, so the
//     alpha < 1/255 test would discard the splat anyway; exp() runs only if some lane needs it;
//   - a wave leaves the round as soon as all its pixels have terminated.
// Each 16-lane row of a wave walks its own sub-block's list, so one wave step evaluates up to four
// different splats.  COUNT adds up the pixel-splat pairs whose power is evaluated (for the FLOP
// roofline; sentinel entries are not counted).  With final_T / final_last, each pixel's final
// transmittance and the sorted index of the last splat it blended (-1: none) are stored for the
// backward, which then need not run the composite again, and the largest index of each wave in
// tile_last[0 .. 3], from which the backward knows where to start before it has a pixel's.
template <bool COUNT>
__device__ __forceinline__ void blend_tile(BlendFwdLds& s, const TileView& tv, uint2 range,
                                           const uint32_t* __restrict__ vals, const Splat* __restrict__ splats,
                                           float* __restrict__ image, uint8_t* __restrict__ rgba8,
                                           uint64_t* eval_count, float* __restrict__ final_T,
                                           int32_t* __restrict__ final_last, int32_t* __restrict__ tile_last) {
    const uint32_t tid = threadIdx.x, wave = tid / kWave, lane = __lane_id();
    uint32_t pxl, pyl;
    tile_pixel(tv, pxl, pyl);
    const bool inside = pxl < tv.width && pyl < tv.height;
    const float fx = (float)pxl, fy = (float)pyl;

    // The per-pixel state machine runs on wave-uniform lane masks (scalar instructions) rather
    // than per-lane booleans: live = pixels not yet terminated.
    float T = 1.0f, cr = 0.0f, cg = 0.0f, cb = 0.0f;
    int32_t last = -1;
    uint64_t live = ballot(inside);
    uint32_t evals = 0;
    const uint16_t* list = s.list[sub_block_of(wave, lane >> 4)];
    // The global loads of staging are issued a round ahead: the record of round r + 1 and the
    // value of round r + 2 are in flight while round r blends.
    StagedSplat next = load_staged(splats, load_value(vals, range.x + tid, range.y), range.x + tid, range.y);
    uint32_t g_after = load_value(vals, range.x + kTilePixels + tid, range.y);
    for (uint32_t base = range.x; base < range.y; base += kTilePixels) {
        // The block leaves once every pixel has terminated: one flag per wave and one barrier
        // (a wave rewrites its flag only after this round's staging barriers, so no wave can
        // overwrite a flag another is still reading).
        if (lane == 0) s.done[wave] = live == 0 ? 1u : 0u;
        __syncthreads();
        const uint4 done = *reinterpret_cast<const uint4*>(s.done);
        if ((done.x & done.y & done.z & done.w) != 0u) break;
        const uint32_t walk = blend_stage_loaded(s, tv, next);
        next = load_staged(splats, g_after, base + kTilePixels + tid, range.y);
        g_after = load_value(vals, base + 2 * kTilePixels + tid, range.y);
        if (live == 0) continue;
        uint32_t taken = BlendFwdLds::kSentinel;  // the last slot blended in this round
        // Two list entries per step: both splats' powers are formed before the first one updates
        // the pixel (power does not depend on T), then the two updates run in list order.  An odd
        // walk reads one sentinel entry (every list is padded with it), which no lane takes.
        const auto power_of = [&](const float2& xy, const float2& ab, const float2& cs) {
            const float dx = xy.x - fx, dy = xy.y - fy;
            return -0.5f * ((ab.x * dx) * dx + (cs.x * dy) * dy) - (ab.y * dx) * dy;
        };
        // power <= 0 equals !(power > 0) except for NaN, whose exp is 0 and whose alpha therefore
        // fails the 1/255 test: either way the splat is skipped.  Active lanes have power in
        // [skip, 0] with skip >= log(1/255) - 0.01, inside soft_expf_inrange's range.
        const auto blend_one = [&](uint32_t off, float power, uint64_t act) {
            const float2 po = s.at(off).po;
            float alpha = po.x * soft_expf_inrange(power);
            alpha = alpha < 0.99f ? alpha : 0.99f;
            const float tn = T * (1.0f - alpha);
            const uint64_t ok = act & ballot(!(alpha < 1.0f / 255.0f));
            const uint64_t low = ballot(tn < 0.0001f);
            if (lane_on(ok & ~low)) {
                const float2 gb = s.at(off).gb;
                cr = cr + (po.y * alpha) * T;
                cg = cg + (gb.x * alpha) * T;
                cb = cb + (gb.y * alpha) * T;
                T = tn;
                taken = off;
            }
            live &= ~(ok & low);
        };
        for (uint32_t i = 0; i < walk; i += 2) {
            const uint32_t o1 = list[i], o2 = list[i + 1];
            const BlendSlot &S1 = s.at(o1), &S2 = s.at(o2);
            const float2 xy1 = S1.xy, ab1 = S1.ab, cs1 = S1.cs, xy2 = S2.xy, ab2 = S2.ab, cs2 = S2.cs;
            const float p1 = power_of(xy1, ab1, cs1), p2 = power_of(xy2, ab2, cs2);
            const uint64_t act1 = ballot(p1 <= 0.0f) & ballot(!(p1 < cs1.y)) & live;
            const uint64_t can2 = ballot(p2 <= 0.0f) & ballot(!(p2 < cs2.y));
            if (COUNT) evals += (lane_on(live) && o1 != BlendFwdLds::kSentinel) ? 1u : 0u;
            if (act1 != 0) blend_one(o1, p1, act1);
            if (COUNT) evals += (lane_on(live) && o2 != BlendFwdLds::kSentinel) ? 1u : 0u;
            const uint64_t act2 = can2 & live;
            if (act2 != 0) blend_one(o2, p2, act2);
            if (live == 0) break;
        }
        if (taken != BlendFwdLds::kSentinel) last = (int32_t)(base + taken / (uint32_t)sizeof(BlendSlot));
    }
    if (final_T) {
        const int32_t m = wave_max(last);
        if (lane == 0) tile_last[wave] = m;
    }
    if (COUNT) {
        const uint64_t sum = wave_sum_u64(evals);
        if (lane == 0) atomicAdd(reinterpret_cast<unsigned long long*>(eval_count), (unsigned long long)sum);
    }
    if (inside) {
        const size_t o = tv.pix_base + (size_t)pyl * tv.width + pxl;
        if (image) {
            image[o * 3 + 0] = cr;
            image[o * 3 + 1] = cg;
            image[o * 3 + 2] = cb;
        }
        if (rgba8) {
            uchar4 q;
            q.x = unorm8(cr); q.y = unorm8(cg); q.z = unorm8(cb); q.w = 255;
            reinterpret_cast<uchar4*>(rgba8)[o] = q;
        }
        if (final_T) {
            final_T[o] = T;
            final_last[o] = last;
        }
    }
}

// Pre-sort position of the pair (this tile, splat g): g's first pair (offset) + the row-major rank of
// the tile in g's rectangle (from its record's position and radius).
__device__ __forceinline__ size_t pair_position(const TileView& tv, const float4& xyzr, uint32_t offset) {
    int32_t x0, y0, x1, y1;
    bounding_rect(xyzr.x, xyzr.y, xyzr.w, tv.gx, tv.gy, x0, y0, x1, y1);
    return (size_t)offset + (size_t)((int32_t)tv.ty - y0) * (size_t)(x1 - x0) + (size_t)((int32_t)tv.tx - x0);
}

// Stores the gradient sums of a pair at its pre-sort position; zeros when out is null.
__device__ __forceinline__ void store_partial_at(size_t pos, float* __restrict__ partials, const float* out) {
    float* dst = partials + pos * kSplatGrads;
#pragma unroll
    for (uint32_t q = 0; q < kSplatGrads; ++q) dst[q] = out ? out[q] : 0.0f;
}

// The same for the pair (this tile, splat g), its record and offset read here.
__device__ __forceinline__ void store_pair_partial(const TileView& tv, uint32_t g, const Splat* __restrict__ splats,
                                                   const uint32_t* __restrict__ offsets, float* __restrict__ partials,
                                                   const float* out) {
    store_partial_at(pair_position(tv, splats[g].xyzr, offsets[g]), partials, out);
}

// Backward of one tile.  The forward frame stored each pixel's final transmittance and last
// contributor (blend_tile's final_T / final_last) and each wave's last contributor (tile_last); the
// tile's splats are walked back to front
// recovering T_i = T_{i+1} / (1 - a_i) and the colour accumulated behind each splat, producing per splat dL/d(image x, y), dL/d(conic a, b, c), dL/d(rgb), dL/d(opacity).
// Each 16-lane row (one 4x4 sub-block) sums its lanes with DPP row operations in a fixed order;
// the rows' sums for a splat (at most one per sub-block, 16 in all) are added in LDS with float64
// atomics.  Those FP32 row sums add exactly in float64 unless their magnitudes span more than
// 2^25, so the tile's total, rounded once to FP32, does not depend on the order in which the rows
// arrive, and a frame's gradients repeat bit for bit from run to run (the exception would need
// row sums 2^25 apart whose float64 rounding then also moves the FP32 result).  Each (tile,
// splat) pair's sums are stored once, at the pair's pre-sort position offsets[g] + row-major rank
// of the tile in g's rectangle, so no global atomics are needed, and the per-Gaussian sum over
// its tiles runs in tile order.  Every pair of the tile's range is written (zeros behind the last
// contributor), so the partials need no clearing beforehand.
//
// Bound: VALU issue, once six blocks stand on a CU (BlendLds).  An entry's update is about 100
// instructions: only what changes the pixel's state or reads the upstream gradient runs under the
// lanes' mask, the colour behind is advanced where alpha and 1 - alpha are at hand, products shared
// with the power are kept, and the nine row sums end in two masked LDS additions (130 instructions
// with every value zeroed and formed under the mask, three additions, and the splat's colour carried
// to the next update).  A tile has few rounds, so its first loads are kept to a chain of three: the
// tile's job and tile_last by block index, then the values, then the records and offsets.  Together,
// in a step of 64 views, k_batch_blend_bwd 9.81 -> 8.39 ms, k_blend_bwd at 3M Gaussians / 1920x1080
// 0.96 -> 0.87 ms; with the sums in the splats' slots and six blocks to a CU 7.69 and 0.83 ms.
__device__ __forceinline__ void blend_bwd_tile(BlendBwdLds& L, const TileView& tv, uint2 range,
                                               const uint32_t* __restrict__ vals, const Splat* __restrict__ splats,
                                               const float* __restrict__ dL_dimg, const uint32_t* __restrict__ offsets,
                                               float* __restrict__ partials, const float* __restrict__ final_T,
                                               const int32_t* __restrict__ final_last, const int4 tile_last) {
    constexpr uint32_t kG = kSplatGrads, kN = BlendBwdLds::kSlots;
    const uint32_t tid = threadIdx.x, wave = tid / kWave, lane = __lane_id();
    uint32_t pxl, pyl;
    tile_pixel(tv, pxl, pyl);
    const bool inside = pxl < tv.width && pyl < tv.height;
    const float fx = (float)pxl, fy = (float)pyl;
    if (tid < kN)
#pragma unroll
        for (uint32_t q = 0; q < kG; ++q) L.slot[tid].acc[q] = 0.0;
    const uint32_t stage_end = tid < kN ? range.y : 0u;  // threads past the slots stage nothing
    const uint16_t* list = L.list[sub_block_of(wave, lane >> 4)];
    // what the lane keeps and adds of a row's nine sums (entry_update)
    const bool b0 = (lane & 1u) != 0u, b1 = (lane & 2u) != 0u;
    const bool first_quad = (lane & 12u) == 0u, last_lane = (lane & 15u) == 15u, adds = first_quad || last_lane;
    const uint32_t acc_lane = last_lane ? 64u : (b0 ? 32u : 0u) + (b1 ? 16u : 0u);

    // The forward frame stored each pixel's final transmittance and last blended splat.
    float T = 1.0f;
    int32_t last = -1;
    const size_t o = tv.pix_base + (size_t)pyl * tv.width + pxl;
    if (inside) {
        T = final_T[o];
        last = final_last[o];
    }
    const int32_t block_last = max(max(tile_last.x, tile_last.y), max(tile_last.z, tile_last.w));

    // ---- back to front
    float g_r = 0.0f, g_g = 0.0f, g_b = 0.0f;
    if (inside) {
        g_r = dL_dimg[o * 3 + 0];
        g_g = dL_dimg[o * 3 + 1];
        g_b = dL_dimg[o * 3 + 2];
    }
    float acc_r = 0.0f, acc_g = 0.0f, acc_b = 0.0f;  // colour accumulated behind the current splat
    const int32_t first_chunk = block_last < 0 ? -1 : (int32_t)(((uint32_t)block_last - range.x) / kN);
    // Loads a chunk ahead, as the forward does: while chunk c is walked, the record and the offset of
    // this thread's splat of chunk c - 1 and the value of chunk c - 2 are in flight.  The offset gives
    // the pair's pre-sort position once the record is there, so the partial sums of the thread's slot
    // are stored after the walk without reading anything more.
    const auto value_of = [&](int32_t c) -> uint32_t {
        return c >= 0 ? load_value(vals, range.x + (uint32_t)c * kN + tid, stage_end) : 0u;
    };
    const auto offset_of = [&](int32_t c, uint32_t g) -> uint32_t {
        return c >= 0 && range.x + (uint32_t)c * kN + tid < stage_end ? offsets[g] : 0u;
    };
    uint32_t g_next = value_of(first_chunk);
    StagedSplat next = load_staged(splats, g_next, range.x + (uint32_t)first_chunk * kN + tid,
                                   first_chunk < 0 ? 0u : stage_end);
    uint32_t off_next = offset_of(first_chunk, g_next);
    uint32_t g_after = value_of(first_chunk - 1);
    for (int32_t chunk = first_chunk; chunk >= 0; --chunk) {
        const uint32_t base = range.x + (uint32_t)chunk * kN;
        const StagedSplat cur = next;
        const size_t pos = cur.valid ? pair_position(tv, cur.sp.xyzr, off_next) : 0;
        __syncthreads();
        const uint32_t walk = blend_stage_loaded(L, tv, cur);
        if (chunk > 0) {
            next = load_staged(splats, g_after, base - kN + tid, stage_end);
            off_next = offset_of(chunk - 1, g_after);
            g_after = value_of(chunk - 2);
        }
        // Two list entries per step, back to front: both splats' powers, exponentials and alphas
        // are formed first (none depends on the transmittance), then the two updates run in order.
        // A step past the list's start reads the sentinel entry, which no lane takes.
        // of the last blended splat (or past the slots, or before the first)
        const int32_t last_off = min(max(last - (int32_t)base, -1), (int32_t)kN) * (int32_t)sizeof(BlendBwdSlot);
        const auto entry_update = [&](uint32_t off, float con_b, float red, float cdy, float adx, float bdx, float dx, float dy,
                                      float G, float raw, float alpha, uint64_t updm) {
            float p = 0.0f, v5 = 0.0f, v6 = 0.0f, v7 = 0.0f, v8 = 0.0f;
            if (lane_on(updm)) {
                const float2 gb = L.at(off).gb;
                // transmittance in front of this splat: 1 - alpha >= 0.01, so the hardware reciprocal
                // (about 1 ulp) stands in for the correctly rounded division (the gradients are
                // checked against float64, not bit for bit; plain and batched frames run this same code)
                const float om = 1.0f - alpha;
                T = T * __builtin_amdgcn_rcpf(om);
                const float w = alpha * T;
                v5 = w * g_r;
                v6 = w * g_g;
                v7 = w * g_b;
                const float dL_dalpha = T * ((red - acc_r) * g_r + (gb.x - acc_g) * g_g + (gb.y - acc_b) * g_b);
                const bool unclamped = raw < 0.99f;  // alpha = o * G
                v8 = unclamped ? dL_dalpha * G : 0.0f;
                p = unclamped ? dL_dalpha * alpha : 0.0f;  // dL/dpower
                acc_r = alpha * red + om * acc_r;
                acc_g = alpha * gb.x + om * acc_g;
                acc_b = alpha * gb.y + om * acc_b;
            }
            // Position and conic gradients, in every lane (p is 0 where the splat is not taken).
            // Multiplying by a power of two does not round, so -0.5 moves freely.
            const float hp = -0.5f * p;
            const float v0 = p * (-adx - con_b * dy), v1 = p * (-cdy - bdx);
            const float v2 = hp * (dx * dx), v3 = -p * (dx * dy), v4 = hp * (dy * dy);
            // Row sums.  v0 .. v7 by a reduce-scatter: lanes exchange half of their values with the
            // lane across bit 0, then across bit 1 (quad_perm), keeping the halves whose index bits
            // match their own, and the four quads of the row add up by rotations; lane (b0, b1) of
            // every quad then holds the row sums of values 4 b0 + 2 b1 + {0, 1}.  v8 by a plain row
            // reduction.  The order of every addition is fixed.
            const float x0 = (b0 ? v4 : v0) + dpp_mov<0xB1>(b0 ? v0 : v4);  // quad_perm [1, 0, 3, 2]
            const float x1 = (b0 ? v5 : v1) + dpp_mov<0xB1>(b0 ? v1 : v5);
            const float x2 = (b0 ? v6 : v2) + dpp_mov<0xB1>(b0 ? v2 : v6);
            const float x3 = (b0 ? v7 : v3) + dpp_mov<0xB1>(b0 ? v3 : v7);
            float y0 = (b1 ? x2 : x0) + dpp_mov<0x4E>(b1 ? x0 : x2);        // quad_perm [2, 3, 0, 1]
            float y1 = (b1 ? x3 : x1) + dpp_mov<0x4E>(b1 ? x1 : x3);
            y0 += dpp_mov<0x124>(y0);  // row_ror:4
            y1 += dpp_mov<0x124>(y1);
            y0 += dpp_mov<0x128>(y0);  // row_ror:8
            y1 += dpp_mov<0x128>(y1);
            const float s8 = row_sum16(v8);
            // Into the tile's float64 sums: the row's first quad adds y0 and y1, its last lane v8's
            // sum beside y0 (acc_lane: the byte offset of the lane's first value).
            const float z = last_lane ? s8 : y0;
            char* const acc = reinterpret_cast<char*>(L.slot) + (off + acc_lane);
            if (adds && z != 0.0f) atomicAdd(reinterpret_cast<double*>(acc), (double)z);
            if (first_quad && y1 != 0.0f) atomicAdd(reinterpret_cast<double*>(acc) + 1, (double)y1);
        };
        for (int32_t i = (int32_t)walk - 1; i >= 0; i -= 2) {
            const uint32_t o1 = list[i], o2 = i >= 1 ? list[i - 1] : BlendBwdLds::kSentinel;
            // lanes whose last blended splat lies at or behind the entry
            const uint64_t mine1 = ballot((int32_t)o1 <= last_off);
            const uint64_t mine2 = ballot((int32_t)o2 <= last_off);
            if ((mine1 | mine2) == 0) continue;
            const BlendBwdSlot &S1 = L.at(o1), &S2 = L.at(o2);
            const float2 xy1 = S1.xy, ab1 = S1.ab, cs1 = S1.cs, po1 = S1.po;
            const float2 xy2 = S2.xy, ab2 = S2.ab, cs2 = S2.cs, po2 = S2.po;
            const float dx1 = xy1.x - fx, dy1 = xy1.y - fy, dx2 = xy2.x - fx, dy2 = xy2.y - fy;
            const float adx1 = ab1.x * dx1, bdx1 = ab1.y * dx1, cdy1 = cs1.x * dy1;
            const float adx2 = ab2.x * dx2, bdx2 = ab2.y * dx2, cdy2 = cs2.x * dy2;
            const float p1 = -0.5f * (adx1 * dx1 + cdy1 * dy1) - bdx1 * dy1;
            const float p2 = -0.5f * (adx2 * dx2 + cdy2 * dy2) - bdx2 * dy2;
            const uint64_t act1 = ballot(p1 <= 0.0f) & ballot(!(p1 < cs1.y)) & mine1;
            const uint64_t act2 = ballot(p2 <= 0.0f) & ballot(!(p2 < cs2.y)) & mine2;
            if ((act1 | act2) == 0) continue;
            const float G1 = soft_expf_inrange(p1), G2 = soft_expf_inrange(p2);
            const float raw1 = po1.x * G1, raw2 = po2.x * G2;
            const float alpha1 = raw1 < 0.99f ? raw1 : 0.99f, alpha2 = raw2 < 0.99f ? raw2 : 0.99f;
            const uint64_t updm1 = act1 & ballot(!(alpha1 < 1.0f / 255.0f));
            const uint64_t updm2 = act2 & ballot(!(alpha2 < 1.0f / 255.0f));
            if (updm1 != 0) entry_update(o1, ab1.y, po1.y, cdy1, adx1, bdx1, dx1, dy1, G1, raw1, alpha1, updm1);
            if (updm2 != 0) entry_update(o2, ab2.y, po2.y, cdy2, adx2, bdx2, dx2, dy2, G2, raw2, alpha2, updm2);
        }
        __syncthreads();
        if (cur.valid) {
            float out[kG];
#pragma unroll
            for (uint32_t q = 0; q < kG; ++q) {
                out[q] = (float)L.slot[tid].acc[q];
                L.slot[tid].acc[q] = 0.0;
            }
            store_partial_at(pos, partials, out);
        }
    }
    // Pairs behind the tile's last contributor (all of them when no pixel blended anything) get
    // zero gradients.
    for (uint32_t k = range.x + (uint32_t)(first_chunk + 1) * kN + tid; k < range.y; k += kTilePixels)
        store_pair_partial(tv, vals[k], splats, offsets, partials, nullptr);
}

}  // namespace tpd
