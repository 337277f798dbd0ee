// Stable LSD radix sort of (32- or 64-bit key, 32-bit value) pairs, one pass per digit of BITS bits
// (8 or 9; sort_shape_for or an autotuner picks the shape, digit width included).  A frame sorts its
// items by depth with 64-bit keys, then their pairs by tile with 32-bit ones.
//
// Replaces the reference's 2-bit "4-way" sorter (radix-shuffle/-prefixA/-prefixB/-mapping.slang,
// 4 dispatches per 2 bits, GaussianEngine.cpp:819-841) with:
//   k_sort_hist + k_sort_offsets  one read of the keys computes the digit histograms of every pass
//                                 and their global exclusive offsets (a frame's counts come from
//                                 its item kernel, k_frame_offsets scans those of both sorts);
//   k_onesweep (once per pass)    each block takes the next partition of BLOCK x ITEMS keys from an
//                                 atomic ticket, ranks its keys by digit with wave64 ballot
//                                 matching (stable: element order inside a wave, then waves in
//                                 order), publishes its per-digit counts with a decoupled
//                                 look-back, reorders the partition in LDS and writes every digit
//                                 run out contiguously.
// The result equals a stable sort by key, i.e. the reference's order (tile, depth, index).
#include "tpd_kernels.hpp"

#include <type_traits>

namespace tpd {

constexpr uint32_t kFlagA = 1u << 30;
constexpr uint32_t kFlagP = 2u << 30;
constexpr uint32_t kValMask = (1u << 30) - 1u;
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;  // kKeys64Drop: the rank of a dropped key

template <typename KT>
__device__ __forceinline__ uint32_t digit_of(KT k, uint32_t shift, uint32_t mask) {
    return (uint32_t)(k >> shift) & mask;
}

// ------------------------------------------------------------------ histograms

// Digit histograms of every pass in one read of the keys.  Consecutive keys often share a digit
// (all pairs of one Gaussian share its depth bits; neighbouring tiles share the high tile bits),
// so each wave first collapses runs of equal digits (run heads found with one shuffle and one
// ballot) and only run heads add their run length to the block's LDS histogram.  Each thread
// keeps kHistUnroll loads in flight; blocks add their non-zero bins to the global counts, block b
// into copy b mod kCountCopies (kCountCopies x kMaxPasses x kMaxRadix, zero on entry), so that
// each counter takes 1/kCountCopies of the blocks' atomics; k_sort_offsets sums the copies and
// re-zeroes them.
constexpr uint32_t kHistUnroll = 8;

// The key of the lane below (lane 0 keeps its own) by a wave-wide DPP shift: register moves, no
// LDS traffic (a shuffle per digit and pass goes through the LDS crossbar).
constexpr int kWaveShr1 = 0x138;  // DPP control wave_shr:1
__device__ __forceinline__ uint64_t key_of_lane_below(uint64_t k) {
    const int lo = (int)(uint32_t)k, hi = (int)(uint32_t)(k >> 32);
    const uint32_t plo = (uint32_t)__builtin_amdgcn_update_dpp(lo, lo, kWaveShr1, 0xF, 0xF, false);
    const uint32_t phi = (uint32_t)__builtin_amdgcn_update_dpp(hi, hi, kWaveShr1, 0xF, 0xF, false);
    return ((uint64_t)phi << 32) | plo;
}
__device__ __forceinline__ uint32_t key_of_lane_below(uint32_t k) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)k, (int)k, kWaveShr1, 0xF, 0xF, false);
}

template <uint32_t BITS, typename KT>
__global__ __launch_bounds__(256) void k_sort_hist(const KT* __restrict__ keys, const uint32_t* count_ptr,
                                                   uint32_t n_imm, const DigitPlan plan, uint32_t tile_keys,
                                                   uint32_t* __restrict__ counts, uint32_t* __restrict__ desc0,
                                                   uint32_t* __restrict__ tickets) {
    constexpr uint32_t R = 1u << BITS;
    __shared__ uint32_t h[kMaxPasses][R];
    const uint32_t n = count_ptr ? min(*count_ptr, n_imm) : n_imm;  // device count, capped by the capacity
    const uint32_t tid = threadIdx.x, lane = __lane_id();
    const uint32_t passes = plan.passes;
    for (uint32_t x = tid; x < kMaxPasses * R; x += 256) (&h[0][0])[x] = 0;
    // The first onesweep pass needs region 0 of the look-back descriptors and all tickets at zero.
    const uint32_t nparts = (n + tile_keys - 1) / tile_keys;
    for (uint32_t x = blockIdx.x * 256 + tid; x < nparts * R; x += gridDim.x * 256) desc0[x] = 0;
    if (blockIdx.x == 0 && tid < kMaxPasses) tickets[tid] = 0;
    __syncthreads();

    constexpr uint32_t kChunk = 256 * kHistUnroll;
    const uint64_t above = lane == 63 ? 0ull : (~0ull << (lane + 1));
    for (uint32_t c0 = blockIdx.x * kChunk; c0 < n; c0 += gridDim.x * kChunk) {
        KT k[kHistUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kHistUnroll; ++u) {
            const uint32_t i = c0 + u * 256 + tid;
            k[u] = i < n ? keys[i] : KT(0);
        }
#pragma unroll
        for (uint32_t u = 0; u < kHistUnroll; ++u) {
            const uint32_t i = c0 + u * 256 + tid;
            const bool valid = i < n;
            const uint64_t vmask = ballot(valid);
            const KT below = key_of_lane_below(k[u]);
#pragma unroll
            for (uint32_t p = 0; p < kMaxPasses; ++p) {
                if (p >= passes) break;
                const uint32_t mask = (1u << (plan.shift[p + 1] - plan.shift[p])) - 1u;
                const uint32_t d = digit_of(k[u], plan.shift[p], mask);
                const uint32_t prev = digit_of(below, plan.shift[p], mask);
                const bool head = valid && (lane == 0 || prev != d);
                const uint64_t heads = ballot(head) | ~vmask;  // invalid lanes end runs
                if (head) {
                    const uint64_t nxt = heads & above;
                    const uint32_t end = nxt ? (uint32_t)__builtin_ctzll(nxt) : 64u;
                    atomicAdd(&h[p][d], end - lane);
                }
            }
        }
    }
    __syncthreads();
    for (uint32_t p = 0; p < passes; ++p)
        for (uint32_t d = tid; d < R; d += 256) {
            const uint32_t v = h[p][d];
            if (v) atomicAdd(&counts[(blockIdx.x % kCountCopies) * (kMaxPasses * kMaxRadix) + p * R + d], v);
        }
}

// Exclusive scan of one pass's 2^bits digit counts (bits 8 or 9) summed over their kCountCopies copies,
// by a block of 256 threads (each takes a contiguous run of digits); every copy is then re-zeroed.
// Returns, in thread 255, the number of keys counted.
__device__ __forceinline__ uint32_t scan_digit_counts(uint32_t* __restrict__ counts, uint32_t* __restrict__ offsets,
                                                      uint32_t bits, uint32_t* s_w) {
    const uint32_t t = threadIdx.x, dpt = bits == 9 ? 2u : 1u;
    uint32_t c[2] = {0u, 0u};
    for (uint32_t i = 0; i < dpt; ++i) {
#pragma unroll
        for (uint32_t k = 0; k < kCountCopies; ++k) {
            uint32_t* q = counts + k * (kMaxPasses * kMaxRadix) + t * dpt + i;
            c[i] += *q;
            *q = 0;
        }
    }
    const uint32_t local = c[0] + c[1];
    const uint32_t incl = wave_incl_scan(local);
    const uint32_t w = t / kWave;
    if (__lane_id() == kWave - 1) s_w[w] = incl;
    __syncthreads();
    uint32_t off = incl - local;
    for (uint32_t q = 0; q < w; ++q) off += s_w[q];
    for (uint32_t i = 0; i < dpt; ++i) {
        offsets[t * dpt + i] = off;
        off += c[i];
    }
    return off;
}

__global__ __launch_bounds__(256) void k_sort_offsets(uint32_t* __restrict__ counts, uint32_t* __restrict__ offsets,
                                                      uint32_t bits) {
    __shared__ uint32_t s_w[4];
    const uint32_t row = blockIdx.x << bits;
    (void)scan_digit_counts(counts + row, offsets + row, bits, s_w);
}

// The frame's two sorts at once, one block per pass of either (launch_sort_offsets).
__global__ __launch_bounds__(256) void k_frame_offsets(uint32_t* __restrict__ counts, uint32_t* __restrict__ offsets,
                                                       uint32_t ibits, uint32_t ipasses, uint32_t pbits,
                                                       uint32_t* __restrict__ counters, const FrameTotals totals) {
    __shared__ uint32_t s_w[4];
    const uint32_t b = blockIdx.x;
    const bool items = b < ipasses;
    const uint32_t row = items ? b << ibits : kPairCountRow + ((b - ipasses) << pbits);
    const uint32_t depth_out = counters[kCtrDepthOut];  // (loaded beside the counts)
    const uint32_t n = scan_digit_counts(counts + row, offsets + row, items ? ibits : pbits, s_w);
    // no item is sorted on a window that does not hold its depth: the frame is issued again
    const bool depth_over = totals.host && totals.lo_bits == kDepthWindowBits && depth_out != 0;
    if (b == 0 && items && threadIdx.x == 255) {
        counters[kCtrItemsKept] = depth_over ? 0u : n;
        counters[kCtrSortItems] = depth_over ? 0u : totals.items;
    }
    if (totals.host && b == gridDim.x - 1 && threadIdx.x == 0) {
        // the 64-bit total, as the digit counts may have wrapped
        uint64_t* const t64 = reinterpret_cast<uint64_t*>(counters + kCtrTotal64);
        const uint64_t total = *t64;
        const uint32_t P = total > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)total;
        const bool over = total > totals.cap || depth_over;
        *t64 = 0;
        counters[kCtrPairs] = P;
        counters[kCtrOverflow] = over ? 1u : 0u;
        counters[kCtrSortPairs] = over ? 0u : P;
        totals.host[kHostPairs] = P;
        totals.host[kHostOverflow] = over ? 1u : 0u;
        totals.host[kHostDepthOut] = depth_out;
        __hip_atomic_store(&totals.host[kHostSeq], totals.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// A frame whose pairs had no room, found room for meanwhile: its totals stand, its emission may run.
__global__ void k_frame_resume(uint32_t* counters) {
    counters[kCtrOverflow] = 0u;
    counters[kCtrSortPairs] = counters[kCtrPairs];
}

void launch_frame_resume(uint32_t* counters, hipStream_t s) {
    hipLaunchKernelGGL(k_frame_resume, dim3(1), dim3(1), 0, s, counters);
}

// ------------------------------------------------------------------ one pass

// Key widths of a pass: kKeys64 and kKeys32 read and write 64- and 32-bit keys.  kKeys64Drop is kKeys64
// that also drops the keys whose high word is zero (the culled items, which the digit counts leave
// out): they take no part in the ranking, get no LDS slot and are never written.  Its values are the
// keys' indices (the items), generated rather than read.
enum : uint32_t { kKeys64 = 0, kKeys32 = 1, kKeys64Drop = 2 };

struct OnesweepArgs {
    const void* keys_in;
    const uint32_t* vals_in;
    void* keys_out;
    uint32_t* vals_out;
    const uint32_t* count_ptr;  // the key count, capped by n_imm (kKeys64Drop: n_imm keys, none when it is 0)
    uint32_t n_imm;
    uint32_t shift, digit_mask;  // this pass's digit
    const uint32_t* offsets;   // 2^BITS global exclusive offsets of this pass's digits
    uint32_t* desc;            // this pass's look-back region (parts x 2^BITS), zero on entry
    uint32_t* desc_next;       // the other region, cleared here for the next pass
    uint32_t* ticket;
};

// LDS of one partition of BLOCK x ITEMS keys (of type KT) with 2^BITS digits.
template <uint32_t BITS, uint32_t BLOCK, uint32_t ITEMS, typename KT>
struct OnesweepLds {
    static constexpr uint32_t R = 1u << BITS;
    static constexpr uint32_t kWaves = BLOCK / kWave;
    static constexpr uint32_t kTileKeys = BLOCK * ITEMS;
    uint16_t whist[kWaves][R];  // per wave digit counters (then wave offsets), zero on entry
    uint32_t bstart[R];
    uint32_t adj[R];
    uint32_t wtot[8];
    uint32_t nkeep;             // kKeys64Drop: the partition's kept keys
    uint32_t part;
    KT keys[kTileKeys];         // the partition reordered by digit (then its values)
};

// Decoupled look-back of one digit: kLookback predecessor descriptors are loaded at once (before
// partition 0 a virtual inclusive prefix of 0), consumed in order up to the first inclusive
// prefix; an unpublished one is re-read after a short sleep.  Returns the exclusive prefix.
template <uint32_t R>
__device__ __forceinline__ uint32_t onesweep_lookback(const uint32_t* desc, uint32_t part, uint32_t d) {
    constexpr int32_t kLookback = 8;
    uint32_t excl = 0;
    int32_t jj = (int32_t)part - 1;
    while (true) {
        uint32_t dsc[kLookback];
#pragma unroll
        for (int32_t u = 0; u < kLookback; ++u)
            dsc[u] = jj - u >= 0 ? load_relaxed(&desc[(uint32_t)(jj - u) * R + d]) : kFlagP;
        uint32_t add = 0;
        int32_t used = 0;
        bool found = false, blocked = false;
#pragma unroll
        for (int32_t u = 0; u < kLookback; ++u) {
            if (!found && !blocked) {
                const uint32_t f = dsc[u] & ~kValMask;
                if (f == 0) {
                    blocked = true;
                } else {
                    add += dsc[u] & kValMask;
                    used = u + 1;
                    found = f == kFlagP;
                }
            }
        }
        excl += add;
        jj -= used;
        if (found) return excl;
        if (blocked) __builtin_amdgcn_s_sleep(1);
    }
}

// The digits are owned by DTH threads, each taking DPT consecutive digits for the per-digit
// bookkeeping and the look-back.
template <uint32_t BITS, uint32_t BLOCK, uint32_t ITEMS, uint32_t MODE>
__global__ __launch_bounds__(BLOCK) void k_onesweep(const OnesweepArgs a) {
    constexpr bool DROP = MODE == kKeys64Drop;
    constexpr bool WIDE = MODE != kKeys32;
    using KT = typename std::conditional<WIDE, uint64_t, uint32_t>::type;  // key type after the load
    using Lds = OnesweepLds<BITS, BLOCK, ITEMS, KT>;
    constexpr uint32_t R = Lds::R;
    constexpr uint32_t kWaves = Lds::kWaves;
    constexpr uint32_t kTileKeys = Lds::kTileKeys;
    constexpr uint32_t DTH = R < BLOCK ? R : BLOCK;  // threads owning digits
    constexpr uint32_t DPT = R / DTH;                // digits per owning thread
    static_assert(R >= 256 && (R % BLOCK == 0 || BLOCK % R == 0), "digits and threads must tile");
    static_assert(DTH / kWave <= 8, "at most 8 digit-owning waves");
    __shared__ Lds L;

    const uint32_t n = a.count_ptr && !DROP ? min(*a.count_ptr, a.n_imm) : a.n_imm;
    const uint32_t nparts = (n + kTileKeys - 1) / kTileKeys;
    const uint32_t tid = threadIdx.x, wave = tid / kWave, lane = __lane_id();
    // The grid covers the most keys there may be: the blocks past the partitions leave before they
    // take a ticket, so that exactly nparts blocks share nparts tickets.
    if (blockIdx.x >= nparts) return;
    if (tid == 0) L.part = atomicAdd(a.ticket, 1u);
    const uint32_t any = DROP && a.count_ptr ? *a.count_ptr : 1u;  // (on its way while the ticket is)
    for (uint32_t x = tid; x < kWaves * R / 2; x += BLOCK) reinterpret_cast<uint32_t*>(&L.whist[0][0])[x] = 0;
    __syncthreads();
    const uint32_t part = __builtin_amdgcn_readfirstlane(L.part);  // block-uniform: keep it scalar
    if (part >= nparts || any == 0u) return;
    if (a.desc_next)
        for (uint32_t d = tid; d < R; d += BLOCK) a.desc_next[part * R + d] = 0;

    // Load ITEMS keys and values per thread, wave-striped: element e = wave*(ITEMS*64) + j*64 +
    // lane; past the end keys are all ones (kKeys64Drop: zero, i.e. dropped).  Every partition but the
    // last is full: its loads (and, without dropped keys, its stores) need no bounds checks.
    const uint32_t base = part * kTileKeys;
    const uint32_t wbase = base + wave * (ITEMS * kWave) + lane;
    const bool full = base + kTileKeys <= n;
    const auto load_key = [&](uint32_t idx) -> KT {
        return static_cast<const KT*>(a.keys_in)[idx];
    };
    KT k[ITEMS];
    if (full) {
#pragma unroll
        for (uint32_t j = 0; j < ITEMS; ++j) k[j] = load_key(wbase + j * kWave);
    } else {
#pragma unroll
        for (uint32_t j = 0; j < ITEMS; ++j) {
            const uint32_t idx = wbase + j * kWave;
            k[j] = idx < n ? load_key(idx) : (DROP ? KT(0) : ~KT(0));
        }
    }

    // Rank within the wave: peers with the same digit found with BITS ballots; the lowest lane of
    // each group advances the wave's running digit counter.  This matching is most of the pass's
    // arithmetic, and arithmetic and LDS are most of its time: a bit costs four instructions (nine
    // as peers &= bit ? bal : ~bal; a pass over 62.9M 32-bit keys 326 -> 285 us, 20M 64-bit 150 -> 126).  Digits are recomputed from the keys
    // wherever they are needed (a few instructions) rather than kept in registers or LDS.
    const auto digit = [&](KT key) -> uint32_t {
        return digit_of(key, a.shift, a.digit_mask);
    };
    const auto dropped = [&](KT key) { return DROP && (uint32_t)((uint64_t)key >> 32) == 0u; };
    uint32_t rank[ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const uint32_t d = digit(k[j]);
        uint32_t plo = ~0u, phi = ~0u;
        constexpr uint32_t kAndXnor = 0x90;  // a & ~(b ^ c)
#pragma unroll
        for (uint32_t b = 0; b < BITS; ++b) {
            uint32_t m = (uint32_t)((int32_t)(d << (31u - b)) >> 31);  // all ones where the bit is set
            asm("" : "+v"(m));  // one value for the ballot and the masks
            const uint64_t bal = ballot(m != 0u);
            plo = __builtin_amdgcn_bitop3_b32(plo, (uint32_t)bal, m, kAndXnor);
            phi = __builtin_amdgcn_bitop3_b32(phi, (uint32_t)(bal >> 32), m, kAndXnor);
        }
        if constexpr (DROP) {
            // a dropped key is nobody's peer and gets no rank (kNoSlot)
            const bool cull = dropped(k[j]);
            const uint64_t gone = ballot(cull);
            plo &= ~(uint32_t)gone;
            phi &= ~(uint32_t)(gone >> 32);
            const uint32_t below = __builtin_amdgcn_mbcnt_hi(phi, __builtin_amdgcn_mbcnt_lo(plo, 0u));
            const uint32_t pre = L.whist[wave][d];
            if (!cull && below == 0) L.whist[wave][d] = (uint16_t)(pre + __popc(plo) + __popc(phi));
            rank[j] = cull ? kNoSlot : pre + below;
        } else {
            const uint32_t below = __builtin_amdgcn_mbcnt_hi(phi, __builtin_amdgcn_mbcnt_lo(plo, 0u));
            const uint32_t pre = L.whist[wave][d];
            if (below == 0) L.whist[wave][d] = (uint16_t)(pre + __popc(plo) + __popc(phi));
            rank[j] = pre + below;
        }
    }
    __syncthreads();

    // Per digit: wave exclusive offsets and the partition's digit counts (published); then the
    // digits' block-local starts by an exclusive scan over the digit-owning threads.
    uint32_t tot[DPT];
    uint32_t tstart = 0;
    if (tid < DTH) {
        uint32_t local = 0;
#pragma unroll
        for (uint32_t i = 0; i < DPT; ++i) {
            const uint32_t d = tid * DPT + i;
            uint32_t acc = 0;
#pragma unroll
            for (uint32_t w = 0; w < kWaves; ++w) {
                const uint32_t c = L.whist[w][d];
                L.whist[w][d] = (uint16_t)acc;
                acc += c;
            }
            tot[i] = acc;
            local += acc;
            store_relaxed(&a.desc[part * R + d], (part == 0 ? kFlagP : kFlagA) | acc);
        }
        const uint32_t incl = wave_incl_scan(local);
        if (lane == kWave - 1) L.wtot[wave] = incl;
        tstart = incl - local;
    }
    __syncthreads();
    if (tid < DTH) {
        for (uint32_t w = 0; w < wave; ++w) tstart += L.wtot[w];
#pragma unroll
        for (uint32_t i = 0; i < DPT; ++i) {
            L.bstart[tid * DPT + i] = tstart;
            tstart += tot[i];
        }
        if (DROP && tid == DTH - 1) L.nkeep = tstart;  // the kept keys of all digits
    }
    __syncthreads();

    // Reorder the partition by digit in LDS (local position = digit start + wave offset + rank).
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const uint32_t d = digit(k[j]);
        if (DROP && rank[j] == kNoSlot) continue;
        const uint32_t lp = L.bstart[d] + L.whist[wave][d] + rank[j];
        rank[j] = lp;
        L.keys[lp] = k[j];
    }

    // The values, wanted last: their registers are free only now that the keys are in LDS.
    uint32_t v[ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const uint32_t idx = wbase + j * kWave;
        v[j] = DROP ? idx : a.vals_in[full || idx < n ? idx : 0u];
    }

    // Look-back per digit, then the global position adjustment of each digit run.
    if (tid < DTH) {
#pragma unroll
        for (uint32_t i = 0; i < DPT; ++i) {
            const uint32_t d = tid * DPT + i;
            uint32_t excl = 0;
            if (part > 0) {
                excl = onesweep_lookback<R>(a.desc, part, d);
                store_relaxed(&a.desc[part * R + d], kFlagP | (excl + tot[i]));
            }
            L.adj[d] = a.offsets[d] + excl - L.bstart[d];
        }
    }
    __syncthreads();

    // Keys out, each to its digit's global start + its place in the partition; the global position
    // of each output slot is kept for the values (the keys' LDS is reused for them).
    // (the past-the-end keys are in the last digit, after the others; dropped keys have no slot)
    const uint32_t nvalid = DROP ? L.nkeep : min(kTileKeys, n - base);
    const bool all_valid = full && !DROP;
    uint32_t gpos[ITEMS];
#pragma unroll
    for (uint32_t t = 0; t < ITEMS; ++t) {
        const uint32_t i = t * BLOCK + tid;
        const KT key = L.keys[i];
        gpos[t] = L.adj[digit(key)] + i;
        if (all_valid || i < nvalid) static_cast<KT*>(a.keys_out)[gpos[t]] = key;
    }
    __syncthreads();
    uint32_t* s_vals = reinterpret_cast<uint32_t*>(L.keys);
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j)
        if (!DROP || rank[j] != kNoSlot) s_vals[rank[j]] = v[j];
    __syncthreads();
#pragma unroll
    for (uint32_t t = 0; t < ITEMS; ++t) {
        const uint32_t i = t * BLOCK + tid;
        if (all_valid || i < nvalid) a.vals_out[gpos[t]] = s_vals[i];
    }
}

// Shapes the tuner chooses from: {digit bits, threads, keys per thread}; kernel[mode].
struct SortShape {
    uint32_t bits, block, items;
    void (*kernel[3])(const OnesweepArgs);
};
#define TPD_SHAPE(B, T, I)                                                                                \
    {                                                                                                     \
        B, T, I, { k_onesweep<B, T, I, kKeys64>, k_onesweep<B, T, I, kKeys32>, k_onesweep<B, T, I, kKeys64Drop> } \
    }
static const SortShape kShapes[] = {
    TPD_SHAPE(8, 256, 16), TPD_SHAPE(8, 256, 8),  TPD_SHAPE(8, 256, 12), TPD_SHAPE(8, 512, 8),
    TPD_SHAPE(8, 512, 12), TPD_SHAPE(8, 256, 20), TPD_SHAPE(9, 512, 12), TPD_SHAPE(9, 512, 8),
    TPD_SHAPE(9, 512, 16), TPD_SHAPE(9, 1024, 16), TPD_SHAPE(9, 1024, 12), TPD_SHAPE(8, 1024, 12),
};
#undef TPD_SHAPE
constexpr uint32_t kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);

uint32_t sort_num_shapes() { return kNumShapes; }
uint32_t sort_shape_keys(uint32_t shape) { return kShapes[shape % kNumShapes].block * kShapes[shape % kNumShapes].items; }
uint32_t sort_shape_bits(uint32_t shape) { return kShapes[shape % kNumShapes].bits; }
uint32_t sort_shape_passes(uint32_t shape, uint32_t key_bits) {
    const uint32_t b = sort_shape_bits(shape);
    return (key_bits + b - 1) / b;
}
DigitPlan sort_digit_plan(uint32_t shape, uint32_t key_bits) {
    DigitPlan p{};
    p.passes = sort_shape_passes(shape, key_bits);
    for (uint32_t i = 0; i <= p.passes && i <= kMaxPasses; ++i) p.shift[i] = key_bits * i / (p.passes ? p.passes : 1u);
    return p;
}

// Wide digits where they save a pass (27-bit depths 3 passes for 4, 45-bit keys 5 for 6, 17-bit tiles 2
// for 3), and blocks as large as still fill the chip: few keys want many small partitions, many keys
// few look-back steps and long digit runs; 3 * 2^20 keys are the most whose partitions of 12,288 stand on
// 256 CUs at once.  us a pass:
//   64-bit keys       8-bit 256x8  512x8  512x12  1024x12    9-bit 512x8  512x12  1024x12  1024x16
//     3k                      6.2    6.1     7.1      9.7          6.8     7.7      9.7     12.1
//     100k                    8.6    8.6    10.0     11.8          9.9    11.1     13.2     15.8
//     1M                       21     16      16       16           17      17       18       20
//     3M                       40     28      24       21           32      27       23       25
//     4M                       54     37      33       31           43      37       35       27
//     20M                     212    152     130      122          193     158      136      126
//   32-bit keys
//     0.24M                    16     12      13       13           14      14       14       16
//     0.7M                     31     21      19       18           23      21       19       20
//     2.8M                     45     29      24       20           32      26       21       23
//     22M                     187    128     106      101          149     119      110      110
//     62M                     490    347     271      270          461     364      313      286
uint32_t sort_shape_for(uint32_t shape, uint32_t n, uint32_t key_bits, uint32_t key_bytes) {
    if (shape != kShapeAuto) return shape % kNumShapes;
    constexpr uint32_t k8_256x8 = 1, k8_512x8 = 3, k9_512x8 = 7, k9_1024x16 = 9, k9_1024x12 = 10, k8_1024x12 = 11;
    const uint32_t large = key_bytes == 4 ? 1u << 19 : 1500000u;
    if ((key_bits + 8) / 9 < (key_bits + 7) / 8)
        return n < large ? k9_512x8 : n <= (key_bytes == 4 ? 1u << 23 : 3u << 20) ? k9_1024x12 : k9_1024x16;
    return n < (1u << 16) ? k8_256x8 : n < large ? k8_512x8 : k8_1024x12;
}

// A block per 2,048 keys, what its threads load at once: a block that takes four such chunks one after
// the other is alone on its CU below 2M keys (200k keys 18.6 -> 8.2 us, 1M 19.1 -> 12.8, 4M 23.2 and 23.0).
static uint32_t hist_blocks(uint32_t n_max) {
    uint32_t hb = (n_max + 256 * kHistUnroll - 1) / (256 * kHistUnroll);
    return hb < 1 ? 1 : (hb > kHistBlocks ? kHistBlocks : hb);
}

// Counts the digits of every pass and scans them (offsets from word 0 of ws.offsets).
template <typename KT>
static void launch_count(SortWorkspace& ws, uint32_t shape, const DigitPlan& plan, const KT* keys,
                         const uint32_t* count_ptr, uint32_t n_max, hipStream_t s) {
    const uint32_t hb = hist_blocks(n_max), bits = sort_shape_bits(shape), tile = sort_shape_keys(shape);
    if (bits == 8)
        hipLaunchKernelGGL((k_sort_hist<8, KT>), dim3(hb), dim3(256), 0, s, keys, count_ptr, n_max, plan, tile,
                           ws.partials, ws.desc, ws.tickets);
    else
        hipLaunchKernelGGL((k_sort_hist<9, KT>), dim3(hb), dim3(256), 0, s, keys, count_ptr, n_max, plan, tile,
                           ws.partials, ws.desc, ws.tickets);
    hipLaunchKernelGGL(k_sort_offsets, dim3(plan.passes), dim3(256), 0, s, ws.partials, ws.offsets, bits);
}

// The passes of one sort, its digit offsets in `offsets`.  kept (optional): the first pass drops the
// keys whose high word is zero, the later ones run on the *kept others.
template <typename KT>
static bool launch_passes(SortWorkspace& ws, uint32_t shape, const DigitPlan& plan, const uint32_t* offsets, KT* keys,
                          uint32_t* vals, KT* keys_alt, uint32_t* vals_alt, const uint32_t* count_ptr, uint32_t n_max,
                          const uint32_t* kept, hipStream_t s) {
    const SortShape& sh = kShapes[shape];
    const uint32_t R = 1u << sh.bits, tile = sh.block * sh.items, parts = (n_max + tile - 1) / tile;
    const KT* kin = keys;
    const uint32_t* vin = vals;
    KT* kout = keys_alt;
    uint32_t* vout = vals_alt;
    for (uint32_t p = 0; p < plan.passes; ++p) {
        OnesweepArgs o;
        o.keys_in = kin; o.vals_in = vin; o.keys_out = kout; o.vals_out = vout;
        o.count_ptr = (kept && p > 0) ? kept : count_ptr;
        o.n_imm = n_max;
        o.shift = plan.shift[p];
        o.digit_mask = (1u << (plan.shift[p + 1] - plan.shift[p])) - 1u;
        o.offsets = offsets + p * R;
        o.desc = ws.desc + (size_t)(p & 1u) * ws.parts_cap * R;
        o.desc_next = ws.desc + (size_t)((p + 1) & 1u) * ws.parts_cap * R;
        o.ticket = ws.tickets + p;
        const uint32_t mode = sizeof(KT) == 4 ? kKeys32 : (kept && p == 0) ? kKeys64Drop : kKeys64;
        hipLaunchKernelGGL(sh.kernel[mode], dim3(parts), dim3(sh.block), 0, s, o);
        KT* const tk = kout; kout = const_cast<KT*>(kin); kin = tk;
        uint32_t* const tv = vout; vout = const_cast<uint32_t*>(vin); vin = tv;
    }
    return (plan.passes & 1u) != 0;
}

bool launch_sort_pairs(SortWorkspace& ws, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt,
                       uint32_t n, uint32_t key_bits, hipStream_t s) {
    const uint32_t shape = sort_shape_for(ws.shape, n, key_bits, 8);
    const DigitPlan plan = sort_digit_plan(shape, key_bits);
    if (n == 0 || plan.passes == 0 || plan.passes > kMaxPasses) return false;
    launch_count(ws, shape, plan, (const uint64_t*)keys, nullptr, n, s);
    return launch_passes(ws, shape, plan, ws.offsets, keys, vals, keys_alt, vals_alt, nullptr, n, nullptr, s);
}

void launch_sort_offsets(SortWorkspace& ws, uint32_t item_shape, uint32_t ipasses, uint32_t pair_shape, uint32_t ppasses,
                         uint32_t* counters, const FrameTotals* totals, hipStream_t s) {
    hipLaunchKernelGGL(k_frame_offsets, dim3(ipasses + ppasses), dim3(256), 0, s, ws.partials, ws.offsets,
                       sort_shape_bits(item_shape), ipasses, sort_shape_bits(pair_shape), counters,
                       totals ? *totals : FrameTotals{});
}

bool launch_sort_items(SortWorkspace& ws, uint32_t shape, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt,
                       uint32_t* vals_alt, uint32_t n, uint32_t lo_bits, const uint32_t* kept, hipStream_t s,
                       const uint32_t* count_ptr) {
    return launch_passes(ws, shape, sort_digit_plan(shape, lo_bits), ws.offsets, keys, vals, keys_alt, vals_alt, count_ptr,
                         n, kept, s);
}

bool launch_sort_pairs32(SortWorkspace& ws, uint32_t shape, uint32_t* keys, uint32_t* vals, uint32_t* keys_alt,
                         uint32_t* vals_alt, const uint32_t* count_ptr, uint32_t n_max, uint32_t key_bits, hipStream_t s,
                         bool counted, hipEvent_t after_count) {
    const DigitPlan plan = sort_digit_plan(shape, key_bits);
    const bool run = n_max != 0 && plan.passes != 0 && plan.passes <= kMaxPasses;
    if (run && !counted) launch_count(ws, shape, plan, (const uint32_t*)keys, count_ptr, n_max, s);
    if (after_count) hipEventRecord(after_count, s);
    if (!run) return false;
    return launch_passes(ws, shape, plan, ws.offsets + (counted ? kPairCountRow : 0u), keys, vals, keys_alt, vals_alt,
                         count_ptr, n_max, nullptr, s);
}

}  // namespace tpd
