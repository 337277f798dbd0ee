// Autotuner: picks launch shapes by timing them on the context's own last frame.  Only choices
// that leave every output bit-identical are tuned (radix-pass block shape here); the reference
// has no counterpart (its shapes are compile-time constants, GaussianEngine.h:121-124).
#include "tpd_ctx.hpp"

#include <algorithm>
#include <vector>

using namespace tpd;

extern "C" {

static void set_shapes(tpd_ctx* c, uint32_t shape) {
    c->ws.shape = c->item_shape = c->pair_shape = shape;
    batch_set_sort_shape(c, shape);
}

int tpd_set_sort_shape(tpd_ctx* c, uint32_t shape) {
    if (!c) return fail(TPD_ERR_INVALID, "null context");
    if (shape >= sort_num_shapes()) return fail(TPD_ERR_INVALID, "tpd_set_sort_shape: no such shape");
    set_shapes(c, shape);
    return TPD_OK;
}

int tpd_reset_sort_shape(tpd_ctx* c) {
    if (!c) return fail(TPD_ERR_INVALID, "null context");
    set_shapes(c, kShapeAuto);
    return TPD_OK;
}

// Times both sorts (items by depth, pairs by tile) of whole frames per shape and keeps the fastest
// shape for each; sort_ms[shape] = both sorts' time, *best = the pair sort's shape.  The stand-alone sorts,
// of other keys and key counts, keep their own (200k 43-bit keys 84 us; with a frame's best 106).
int tpd_autotune(tpd_ctx* c, float* sort_ms, uint32_t capacity, uint32_t* n_shapes, uint32_t* best) {
    if (!c) return fail(TPD_ERR_INVALID, "null context");
    hipSetDevice(c->device);
    const uint32_t ns = sort_num_shapes();
    if (n_shapes) *n_shapes = ns;
    if (!c->rendered || c->n == 0 || c->last_pairs == 0)
        return fail(TPD_ERR_STATE, "tpd_autotune: render a non-empty frame first");
    hipStream_t s = c->stream;
    const uint32_t keep_items = c->item_shape, keep_pairs = c->pair_shape;
    const bool keep_profile = c->profile;
    int rc = tpd_set_profiling(c, 1);
    std::vector<float> med(ns, 0.0f), items(ns, 0.0f), pairs(ns, 0.0f);
    for (uint32_t sh = 0; sh < ns && rc == TPD_OK; ++sh) {
        c->item_shape = c->pair_shape = sh;
        std::vector<float> ti, tp, t;
        for (int rep = 0; rep < 4 && rc == TPD_OK; ++rep) {
            if ((rc = render_forward(c, s)) != TPD_OK) break;
            float mi = 0.0f, mp = 0.0f;
            if (hipEventSynchronize(c->ev[5]) != hipSuccess ||
                hipEventElapsedTime(&mi, c->ev[2], c->ev[3]) != hipSuccess ||
                hipEventElapsedTime(&mp, c->ev[4], c->ev[5]) != hipSuccess) {
                rc = fail(TPD_ERR_HIP, "tpd_autotune: timing");
                break;
            }
            if (rep > 0) {  // first run warms up
                ti.push_back(mi);
                tp.push_back(mp);
                t.push_back(mi + mp);
            }
        }
        const auto median = [](std::vector<float>& v) {
            std::sort(v.begin(), v.end());
            return v.empty() ? 0.0f : v[v.size() / 2];
        };
        items[sh] = median(ti);
        pairs[sh] = median(tp);
        med[sh] = median(t);
    }
    c->profile = keep_profile;
    if (rc != TPD_OK) {
        c->item_shape = keep_items;
        c->pair_shape = keep_pairs;
        return rc;
    }
    uint32_t bi = 0, bp = 0;
    for (uint32_t sh = 1; sh < ns; ++sh) {
        if (items[sh] < items[bi]) bi = sh;
        if (pairs[sh] < pairs[bp]) bp = sh;
    }
    c->item_shape = bi;
    c->pair_shape = bp;
    if (best) *best = bp;
    if (sort_ms)
        for (uint32_t sh = 0; sh < ns && sh < capacity; ++sh) sort_ms[sh] = med[sh];
    // Leave a consistent frame behind (keys/ranges/image of the current camera).
    return render_forward(c, s);
}

}  // extern "C"
