// The context behind the opaque tpd_ctx handle, and the host-side helpers shared by the C-ABI
// translation units.
#pragma once

#include "tpd_kernels.hpp"
#include "../../include/tpd_hip.h"

#include <string>
#include <vector>

namespace tpd {
struct BackwardState;
struct BatchState;
}  // namespace tpd

struct tpd_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    bool keep_unsorted = false;

    // scene (GaussianEngine::compile)
    float* d_gauss = nullptr;  // N x 60
    bool own_gauss = true;
    uint32_t n = 0, sh_degree = 3;
    uint32_t* d_ent_idx = nullptr;
    float* d_models = nullptr;
    uint32_t n_ent = 1;
    std::vector<float> h_models;
    bool have_scene = false;

    // camera
    tpd::CameraParams cam{};
    bool have_camera = false;

    // per-Gaussian frame buffers
    tpd::EntityMats* d_ent_mats = nullptr; size_t cap_ent_mats = 0;
    tpd::Splat* d_splats = nullptr; size_t cap_splats = 0;
    uint32_t* d_tiles = nullptr; size_t cap_tiles = 0;
    uint32_t* d_offsets = nullptr; size_t cap_offsets = 0;
    uint64_t* d_scan_desc = nullptr; size_t cap_scan_desc = 0;    // the emission's, zero between frames
    uint64_t* d_scan_desc2 = nullptr; size_t cap_scan_desc2 = 0;  // the item offsets', cleared by the frame
    uint32_t* d_counters = nullptr;
    uint32_t* h_counters = nullptr;  // pinned: the frame's totals (kHost*), written by the device
    uint32_t* d_host_counters = nullptr;  // the same memory as the device addresses it

    uint64_t* d_ikeys = nullptr; size_t cap_ikeys = 0;   // item sort: depth keys (+ tile rectangles) and
    uint64_t* d_ikeys_alt = nullptr; size_t cap_ikeys_alt = 0;  // Gaussian indices, ping-pong
    uint32_t* d_ivals = nullptr; size_t cap_ivals = 0;
    uint32_t* d_ivals_alt = nullptr; size_t cap_ivals_alt = 0;
    uint64_t* d_rects = nullptr; size_t cap_rects = 0;   // rectangles that do not fit their item's key
    uint32_t frame_seq = 0;                              // of the totals in h_counters

    // pairs (tiles and Gaussian indices) + sort
    uint32_t* d_keys = nullptr; size_t cap_keys = 0;
    uint32_t* d_vals = nullptr; size_t cap_vals = 0;
    uint32_t* d_keys_alt = nullptr; size_t cap_keys_alt = 0;
    uint32_t* d_vals_alt = nullptr; size_t cap_vals_alt = 0;
    uint64_t* d_keys_dbg = nullptr; size_t cap_keys_dbg = 0;
    uint32_t* d_vals_dbg = nullptr; size_t cap_vals_dbg = 0;
    uint64_t* d_full_keys = nullptr; size_t cap_full_keys = 0;  // 64-bit keys rebuilt for readers
    tpd::SortWorkspace ws;  // shared by the frame's sorts and the stand-alone one; ws.shape: the latter's
    uint32_t item_shape = tpd::kShapeAuto, pair_shape = tpd::kShapeAuto;  // of the frame's sorts
    const uint32_t* sorted_keys = nullptr;
    const uint32_t* sorted_vals = nullptr;
    uint32_t wide_frames = 0;   // frames still to be sorted on the wide depth key (kDepthHold, render.cpp)
    uint64_t issues = 0;        // item launches of all frames: one a frame, two where a depth left the window
    uint64_t resumes = 0;       // frames whose pairs were issued again with more room

    // image
    uint2* d_ranges = nullptr; size_t cap_ranges = 0;
    uint32_t* d_tile_hist = nullptr; size_t cap_tile_hist = 0;
    tpd::TileJob* d_jobs = nullptr; size_t cap_jobs = 0;         // the blend's blocks, heaviest tiles first
    int32_t* d_tile_last = nullptr; size_t cap_tile_last = 0;    // per block and wave, for the backward
    float* d_image = nullptr; size_t cap_image = 0;
    uint8_t* d_rgba8 = nullptr; size_t cap_rgba8 = 0;
    // per pixel final transmittance and last blended splat of the frame, for the backward
    float* d_final_T = nullptr; size_t cap_final_T = 0;
    int32_t* d_final_last = nullptr; size_t cap_final_last = 0;

    uint32_t last_pairs = 0;
    uint32_t recent_pairs = 0;  // the most pairs of recent frames, after recent_hold frames of fewer an eighth less
    uint32_t recent_hold = 0;   // with each
    uint32_t last_passes = 0;
    bool rendered = false;

    // stage timing with HIP events on the render stream (tpd_set_profiling)
    bool profile = false;
    hipEvent_t ev[9] = {};
    uint32_t emit_event = 3;  // where the emission that made the frame's pairs began: 3, or 8 for a resumed frame
    uint64_t* d_eval_count = nullptr;  // blend evaluations, counted on request (tpd_get_blend_evaluations)
    tpd::BlendArgs last_blend{};       // the last rendered frame's blend, for that count
    bool has_blend = false;

    // backward and batched state (backward.cpp, batch.cpp)
    tpd::BackwardState* bwd = nullptr;
    tpd::BatchState* batch = nullptr;
};

namespace tpd {
extern thread_local std::string g_last_error;
int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);
uint32_t bit_length(uint32_t v);
int ensure_scene_buffers(tpd_ctx* c);
int ensure_image_buffers(tpd_ctx* c);
// s: the stream that uses them first
int ensure_pair_buffers(tpd_ctx* c, size_t pairs, hipStream_t s);
int ensure_sort_workspace(tpd_ctx* c, size_t pairs, hipStream_t s);
int render_forward(tpd_ctx* c, hipStream_t s);
int launch_offsets(tpd_ctx* c, hipStream_t s);
void backward_release(tpd_ctx* c);
void batch_release(tpd_ctx* c);
void batch_set_sort_shape(tpd_ctx* c, uint32_t shape);
int batch_view_rgba8(tpd_ctx* c, uint32_t view, const uint8_t** d_rgba, uint32_t* width, uint32_t* height);
int noalloc_setup(int device);  // device address of the allocation-free sort's scratch (noalloc.hip)

// Grows a device allocation to hold at least `count` elements (contents are not preserved).
template <typename T>
inline hipError_t grow(T*& p, size_t& cap, size_t count, double headroom = 1.0) {
    if (p && cap >= count) return hipSuccess;
    if (p) {
        hipError_t e = hipFree(p);
        if (e != hipSuccess) return e;
        p = nullptr;
    }
    size_t want = (size_t)((double)count * headroom);
    if (want < count) want = count;
    if (want < 1) want = 1;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&p), want * sizeof(T));
    if (e != hipSuccess) {
        cap = 0;
        p = nullptr;
        return e;
    }
    cap = want;
    return hipSuccess;
}

// Zeroes device memory before anything uses it.  hipMemset goes to the null stream and may return before it
// has run (8 GiB: 3 us, then 1.4 ms of work), and the streams frames run on do not wait for the null stream.
inline hipError_t clear_now(void* p, size_t bytes) {
    const hipError_t e = hipMemset(p, 0, bytes);
    return e == hipSuccess ? hipStreamSynchronize(nullptr) : e;
}

template <typename T>
inline void release(T*& p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}
}  // namespace tpd
