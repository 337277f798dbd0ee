// Forward path kernels of a frame besides its items and their pairs (k_batch.hip): entity matrices,
// tile ranges, tile order, and the front-to-back blend.
//
// Reference: torpedo/volumetric/assets/gaussian/{project,range,blend}.slang and the dispatch sequence
// of GaussianEngine::recordSplat/recordBlend (GaussianEngine.cpp:777-863).
#include "tpd_blend.hpp"
#include "tpd_kernels.hpp"

namespace tpd {

// ------------------------------------------------------------------ entity matrices

__global__ void k_entity_mats(const float* __restrict__ models, uint32_t n_ent, CameraParams cam,
                              EntityMats* __restrict__ out) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n_ent) return;
    entity_mats(models ? models + 16 * (size_t)e : nullptr, cam, out[e]);
}

void launch_entity_mats(const float* models, uint32_t n_ent, const CameraParams& cam, EntityMats* out,
                        hipStream_t s) {
    const uint32_t ne = n_ent ? n_ent : 1u;
    hipLaunchKernelGGL(k_entity_mats, dim3((ne + 63) / 64), dim3(64), 0, s, models, ne, cam, out);
}

// ------------------------------------------------------------------ ranges

// Each thread takes runs of kRangeRun consecutive sorted keys, read with 16-byte loads, and
// compares each key (a tile) with the one before it (the key before the run is one more load).
constexpr uint32_t kRangeRun = 8;

// range.slang:16-35.  Empty tiles keep the (0, 0) written by the item kernel (the reference clears
// with fillBuffer, GaussianEngine.cpp:843-848).  The kernel also re-zeroes the scan descriptors and
// the scan ticket for the next frame.  A batch frame whose items were sorted on the depth-window key
// although one of its depths lies outside the window (kCtrDepthOut) has some pairs out of depth order
// inside their tiles (never in the wrong tile); it is marked overflowed, so that every later kernel
// skips it and the host renders it again on the wider key.
__global__ void k_ranges(const uint32_t* __restrict__ keys, uint32_t* __restrict__ counters, uint32_t cap,
                         uint2* __restrict__ ranges, uint64_t* scan_desc, uint32_t n_scan_desc, uint32_t* ticket,
                         uint32_t lo_bits) {
    const uint32_t P = min(counters[kCtrSortPairs], cap);
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t nthreads = gridDim.x * blockDim.x;
    for (uint32_t d = gid; d < n_scan_desc; d += nthreads) scan_desc[d] = 0;
    if (gid == 0) {
        *ticket = 0;
        if (lo_bits != kDepthWindowBits)
            counters[kCtrDepthOut] = 0;  // (always, in a plain frame: the host has it)
        else if (counters[kCtrDepthOut])
            counters[kCtrOverflow] = 1u;
    }
    uint32_t* r = reinterpret_cast<uint32_t*>(ranges);
    const uint32_t runs = (P + kRangeRun - 1) / kRangeRun;
    for (uint32_t run = gid; run < runs; run += nthreads) {
        const uint32_t i0 = run * kRangeRun, n = min(kRangeRun, P - i0);
        uint32_t t[kRangeRun];
        if (n == kRangeRun) {
            const uint4* v = reinterpret_cast<const uint4*>(keys + i0);
            const uint4 x = v[0], y = v[1];
            t[0] = x.x; t[1] = x.y; t[2] = x.z; t[3] = x.w;
            t[4] = y.x; t[5] = y.y; t[6] = y.z; t[7] = y.w;
        } else {
#pragma unroll
            for (uint32_t j = 0; j < kRangeRun; ++j) t[j] = j < n ? keys[i0 + j] : 0u;
        }
        uint32_t prev = i0 > 0 ? keys[i0 - 1] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < kRangeRun; ++j) {
            if (j >= n) break;
            const uint32_t idx = i0 + j, cur = t[j];
            if (idx == 0) {
                r[2 * cur] = 0;
            } else if (cur != prev) {
                r[2 * prev + 1] = idx;
                r[2 * cur] = idx;
            }
            if (idx == P - 1) r[2 * cur + 1] = P;
            prev = cur;
        }
    }
}

void launch_ranges(const uint32_t* keys, uint32_t* counters, uint32_t cap, uint2* ranges, uint64_t* scan_desc,
                   uint32_t n_scan_desc, uint32_t* ticket, uint32_t lo_bits, hipStream_t s) {
    uint32_t work = (cap + kRangeRun - 1) / kRangeRun;
    work = work > n_scan_desc ? work : n_scan_desc;
    uint32_t nb = (work + 255) / 256;
    nb = nb < 1 ? 1 : (nb > 8192 ? 8192 : nb);
    hipLaunchKernelGGL(k_ranges, dim3(nb), dim3(256), 0, s, keys, counters, cap, ranges, scan_desc, n_scan_desc, ticket,
                       lo_bits);
}

// ------------------------------------------------------------------ the reference's keys, for readers

__global__ void k_full_keys(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                            const Splat* __restrict__ splats, uint32_t n, uint64_t* __restrict__ out) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        out[i] = ((uint64_t)keys[i] << 32) | as_uint(splats[vals[i]].xyzr.z);
}

void launch_full_keys(const uint32_t* keys, const uint32_t* vals, const Splat* splats, uint32_t n, uint64_t* out,
                      hipStream_t s) {
    if (n == 0) return;
    uint32_t nb = (n + 255) / 256;
    nb = nb > 8192 ? 8192 : nb;
    hipLaunchKernelGGL(k_full_keys, dim3(nb), dim3(256), 0, s, keys, vals, splats, n, out);
}

// keygen.slang:21-54.
__global__ void k_unsorted_pairs(const Splat* __restrict__ splats, const uint32_t* __restrict__ tiles,
                                 const uint32_t* __restrict__ offsets, uint32_t n, uint32_t gx, uint32_t gy,
                                 uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || tiles[i] == 0) return;
    const float4 c = splats[i].xyzr;
    int32_t x0, y0, x1, y1;
    bounding_rect(c.x, c.y, c.w, gx, gy, x0, y0, x1, y1);
    uint32_t pos = offsets[i];
    for (int32_t y = y0; y < y1; ++y)
        for (int32_t x = x0; x < x1; ++x, ++pos) {
            keys[pos] = ((uint64_t)((uint32_t)y * gx + (uint32_t)x) << 32) | as_uint(c.z);
            vals[pos] = i;
        }
}

void launch_unsorted_pairs(const Splat* splats, const uint32_t* tiles, const uint32_t* offsets, uint32_t n, uint32_t gx,
                           uint32_t gy, uint64_t* keys, uint32_t* vals, hipStream_t s) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_unsorted_pairs, dim3((n + 255) / 256), dim3(256), 0, s, splats, tiles, offsets, n, gx, gy, keys,
                       vals);
}

// ------------------------------------------------------------------ tile order

// Tiles are ordered by class (bit length of the pair count, 0 for an empty tile), heaviest class
// first.  One 1024-thread block per chunk of 1024 tiles needs its start in each class (the tiles of all
// heavier classes, then those of the class in earlier chunks) and scatters its tiles.  Up to
// kOrderOwnChunks chunks every block counts all tiles itself, one launch; beyond, a launch before
// counts each chunk's tiles per class into hist[class * chunks + chunk], as a block's own count
// takes longer (both launches and the one, us: 144 tiles 8.5 and 5.1, 3,600 9.6 and 7.9, 8,160 11.3 and
// 10.9).  Within a chunk and class the order is the order in which waves claim slots.  Every wave combines its lanes of one class into one LDS atomic.  Inside each
// class's range of launch positions the tiles are placed by xcd_unmap, so that each XCD (blocks
// go to the 8 XCDs round-robin) takes one contiguous run of the class's tiles, in index order by
// chunks: neighbouring tiles, which share splats, then mostly meet in one L2.

constexpr uint32_t kOrderOwnChunks = 4;

__device__ __forceinline__ uint32_t tile_class(const uint2* __restrict__ ranges, uint32_t t) {
    const uint2 r = ranges[t];
    const uint32_t n = r.y > r.x ? r.y - r.x : 0u;
    return n ? 32u - (uint32_t)__builtin_clz(n) : 0u;  // 0 .. 32
}

// Adds, for each lane with `valid`, one to slot[cls] and returns the lane's slot value before
// the addition (lanes of one class in lane order).
__device__ __forceinline__ uint32_t claim_class_slot(uint32_t* slot, uint32_t cls, bool valid) {
    const uint32_t lane = __lane_id();
    const uint64_t lt = lanemask_lt();
    uint64_t todo = ballot(valid);
    uint32_t mine = 0;
    while (todo) {
        const uint32_t leader = (uint32_t)__builtin_ctzll(todo);
        const uint32_t c = __builtin_amdgcn_readlane(cls, leader);
        const uint64_t peers = ballot(valid && cls == c) & todo;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(&slot[c], (uint32_t)__popcll(peers));
        base = __builtin_amdgcn_readlane(base, leader);
        if ((peers >> lane) & 1ull) mine = base + (uint32_t)__popcll(peers & lt);
        todo &= ~peers;
    }
    return mine;
}

__global__ __launch_bounds__(kOrderChunk) void k_tile_class_count(const uint2* __restrict__ ranges, uint32_t ntiles,
                                                                  const uint32_t* counters,
                                                                  uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[kTileClasses];
    const uint32_t tid = threadIdx.x, chunks = gridDim.x;
    if (counters && counters[kCtrOverflow]) return;
    if (tid < kTileClasses) cnt[tid] = 0;
    __syncthreads();
    const uint32_t t = blockIdx.x * kOrderChunk + tid;
    (void)claim_class_slot(cnt, t < ntiles ? tile_class(ranges, t) : 0u, t < ntiles);
    __syncthreads();
    if (tid < kTileClasses) hist[tid * chunks + blockIdx.x] = cnt[tid];
}

// Adds the wave's tiles per class to count[class]: lanes of one class found with a ballot per bit of the
// class, one LDS addition each; kTileClasses: no tile.
__device__ __forceinline__ void count_classes(uint32_t* count, uint32_t cls) {
    uint64_t peers = ~0ull;
#pragma unroll
    for (uint32_t b = 0; b < 6; ++b) {
        const uint64_t bal = ballot((cls >> b) & 1u);
        peers &= ((cls >> b) & 1u) ? bal : ~bal;
    }
    if (cls < kTileClasses && (peers & lanemask_lt()) == 0) atomicAdd(&count[cls], (uint32_t)__popcll(peers));
}

// hist: the chunks' counts, or null: every block counts them.
__global__ __launch_bounds__(kOrderChunk) void k_tile_order(const uint2* __restrict__ ranges, uint32_t ntiles,
                                                            const uint32_t* counters, const uint32_t* __restrict__ hist,
                                                            TileJob* __restrict__ jobs, uint32_t grid_width,
                                                            const uint32_t* __restrict__ tile_view,
                                                            const BatchViewDev* __restrict__ views) {
    __shared__ uint32_t slot[kTileClasses], total[kTileClasses], cstart[kTileClasses];
    const uint32_t tid = threadIdx.x, lane = __lane_id(), wave = tid / kWave, chunks = gridDim.x;
    if (counters && counters[kCtrOverflow]) return;
    if (!hist) {
        if (tid < kTileClasses) slot[tid] = total[tid] = 0;
        __syncthreads();
        uint32_t cls[kOrderOwnChunks];  // all loads in flight together
#pragma unroll
        for (uint32_t k = 0; k < kOrderOwnChunks; ++k)
            cls[k] = k * kOrderChunk + tid < ntiles ? tile_class(ranges, k * kOrderChunk + tid) : kTileClasses;
#pragma unroll
        for (uint32_t k = 0; k < kOrderOwnChunks; ++k)  // total: of this chunk and the later ones, until below
            if (k < chunks) count_classes(k < blockIdx.x ? slot : total, cls[k]);
        __syncthreads();
        if (tid < kTileClasses) total[tid] += slot[tid];
    } else {
        for (uint32_t c = wave; c < kTileClasses; c += kOrderChunk / kWave) {
            uint64_t all = 0, before = 0;
            for (uint32_t k = lane; k < chunks; k += kWave) {
                const uint32_t v = hist[c * chunks + k];
                all += v;
                before += k < blockIdx.x ? v : 0u;
            }
            all = wave_sum_u64(all);
            before = wave_sum_u64(before);
            if (lane == 0) {
                total[c] = (uint32_t)all;
                slot[c] = (uint32_t)before;
            }
        }
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t pos = 0;
        for (int c = (int)kTileClasses - 1; c >= 0; --c) {
            cstart[c] = pos;
            slot[c] += pos;
            pos += total[c];
        }
    }
    __syncthreads();
    const uint32_t t = blockIdx.x * kOrderChunk + tid;
    const uint32_t cls = t < ntiles ? tile_class(ranges, t) : 0u;
    const uint32_t pos = claim_class_slot(slot, cls, t < ntiles);
    if (t >= ntiles) return;
    const uint2 r = ranges[t];
    uint32_t v = 0, local = t, gx = grid_width;
    if (grid_width == 0) {
        v = tile_view[t];
        local = t - views[v].tile_base;
        gx = views[v].gx;
    }
    const uint32_t ty = local / gx;
    jobs[cstart[cls] + xcd_unmap(pos - cstart[cls], total[cls])] = TileJob{(local - ty * gx) | ty << 16, r.x, r.y, v};
}

void launch_tile_order(const uint2* ranges, uint32_t ntiles, const uint32_t* counters, uint32_t* hist, TileJob* jobs,
                       uint32_t grid_width, const uint32_t* tile_view, const BatchViewDev* views, hipStream_t s) {
    if (ntiles == 0) return;
    const uint32_t chunks = (ntiles + kOrderChunk - 1) / kOrderChunk;
    const bool own = chunks <= kOrderOwnChunks;
    if (!own)
        hipLaunchKernelGGL(k_tile_class_count, dim3(chunks), dim3(kOrderChunk), 0, s, ranges, ntiles, counters, hist);
    hipLaunchKernelGGL(k_tile_order, dim3(chunks), dim3(kOrderChunk), 0, s, ranges, ntiles, counters,
                       own ? nullptr : (const uint32_t*)hist, jobs, grid_width, tile_view, views);
}

// ------------------------------------------------------------------ blend

// blend.slang:22-105.  One 16x16 tile per 256-thread block (blend_tile).
template <bool COUNT>
__global__ __launch_bounds__(kTilePixels, 8) void k_blend(const BlendArgs a) {
    __shared__ BlendFwdLds lds;
    const TileJob j = a.jobs[blockIdx.x];  // loaded beside the flag (meaningless after an overflow)
    if (a.counters[kCtrOverflow]) return;  // the frame is rendered again
    const TileView tv{j.txy & 0xFFFFu, j.txy >> 16, a.width, a.height, a.gx, 0, 0};
    blend_tile<COUNT>(lds, tv, make_uint2(j.start, j.end), a.vals, a.splats, a.image, a.rgba8, a.eval_count, a.final_T,
                      a.final_last, a.tile_last + 4 * (size_t)blockIdx.x);
}

void launch_blend(const BlendArgs& a, hipStream_t s) {
    if (a.ntiles == 0) return;
    if (a.eval_count)
        hipLaunchKernelGGL(k_blend<true>, dim3(a.ntiles), dim3(kTilePixels), 0, s, a);
    else
        hipLaunchKernelGGL(k_blend<false>, dim3(a.ntiles), dim3(kTilePixels), 0, s, a);
}

}  // namespace tpd
