// lif_rows.h -- which currents each thread of the LIF scan over runs of rows
// (k_lif_rows, spiking.hip) loads.  Plain C++, so that the bounds can be checked
// on the host over every block of a plane.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define HSES_LIF_HD __host__ __device__ __forceinline__
#else
#define HSES_LIF_HD inline
#endif

namespace hses {

constexpr int32_t kLifRowsThreads = 512, kLifRowsMaxT = 64;

// Rows of a block: the first multiple of 4 whose threads fill 7/8 of their waves,
// or the fullest; 0 where four rows are too wide.
inline int32_t lif_rows_block(int32_t h) {
    int32_t best = 0, best_fill = 0;
    for (int32_t rb = 4; (int64_t)rb * h / 4 <= kLifRowsThreads; rb += 4) {
        const int32_t lanes = rb * h / 4, fill = lanes * 256 / ((lanes + 63) & ~63);
        if (fill > best_fill) best = rb, best_fill = fill;
        if (fill >= 224) break;
    }
    return best;
}

// Threads of a block of rb rows: four columns each, whole waves.
inline int32_t lif_rows_threads(int32_t rb, int32_t h) { return (rb * h / 4 + 63) & ~63; }

// A thread's four columns of a plane: e, the first one it loads; own, the columns
// from its first to the block's end (<= 0: an idle thread); over, how many of the
// four are its neighbour's and are dropped.
struct LifCols {
    int64_t e;
    int32_t own, over;
};

// Thread tid of the block whose rb rows start at row0, in a plane of at least four
// columns.  A block's rows are a multiple of 4 (the last block aside), so only the
// plane's last columns can be fewer than four: their thread loads the plane's last
// four.  Idle threads load the block's first four, or the plane's last where the block
// holds fewer (rows of one to three columns), and nothing of them is kept.
HSES_LIF_HD LifCols lif_rows_cols(int64_t row0, int32_t rb, int32_t h, int32_t tid, int64_t plane) {
    LifCols c;
    c.own = rb * h - 4 * tid;
    c.over = c.own > 0 && c.own < 4 ? 4 - c.own : 0;
    const int64_t first = row0 * h;
    if (c.own > 0) c.e = first + 4 * tid - c.over;
    else c.e = first < plane - 4 ? first : plane - 4;
    return c;
}

}  // namespace hses
