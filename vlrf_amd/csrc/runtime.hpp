// runtime.hpp - the context object behind vlrf_hip_ctx_t.
#pragma once

#include "internal.hpp"

#include <vector>

struct vlrf_hip_ctx {
    int device = 0;
    int num_cus = 0;
    char name[256] = {0};
    hipStream_t stream = nullptr;   // default priority, non-blocking
    hipEvent_t ev0 = nullptr, ev1 = nullptr;

    struct RopeTab {
        int max_seq = 0, d_head = 0;
        float theta = 0.f;
        float* cos_t = nullptr;
        float* sin_t = nullptr;
    };
    std::vector<RopeTab> ropes;      // RoPE tables per (max_seq, d_head, theta)
    void* scratch_buf = nullptr;     // split-K partials of the standalone ops
    size_t scratch_bytes = 0;
    // Outgrown buffers that a captured launch addresses, kept for the graph's
    // replays until the context ends.  A buffer at least doubles when one is put
    // here, so together they stay below the current one.
    static constexpr int kMaxKept = 64;
    bool scratch_captured = false;   // the current buffer was handed out under capture
    int n_kept = 0;
    void* kept[kMaxKept] = {};
    size_t kept_bytes = 0;
    float* noalloc_scratch = nullptr;   // this device's fixed array for vlrf_hip_attn_decode_noalloc
    int* small_tile_ctr = nullptr;      // small-M linear: row-tile counters (zero between calls)

    // Device cos/sin tables built on the host as RopeCache::init does.
    int rope_tables(int max_seq, int d_head, float theta, const float** c, const float** s);
    // Grows the shared scratch buffer (waits for queued work before freeing the old one).
    int scratch(size_t bytes, float** out);
    // The same for a caller that can do without: null where it cannot be had
    // (bytes 0, the stream under capture, no memory).
    float* try_scratch(size_t bytes);
    ~vlrf_hip_ctx();
};

namespace vlrf_hip {
using Ctx = ::vlrf_hip_ctx;
}
