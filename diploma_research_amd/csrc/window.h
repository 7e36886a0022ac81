// Products of matrices whose elements lie within a band (window.hip).
#pragma once

#include "dim_internal.h"
#include "kernels.h"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace dimgpu {

constexpr uint32_t kWindowGroup = 16; // tiles whose column span is kept; wavefronts of a workgroup
constexpr uint32_t kWindowMaxPer = 4;
constexpr uint32_t kWindowMaxSigma = 16;
// 64 workgroups: smaller matrices leave most CUs without one. Not the crossing
// but a little above it: FP32 products at 1074 tiles of sigma 16 take 9.5 us by
// the tile kernel and 9.2 by windows, transposed ones 19.5 sorted at 940 tiles
// and 15.2 by windows at 1031 (band of 2000).
constexpr uint32_t kWindowMinTiles = 1024;

// What else a plain product by windows needs to be the faster one; uneven rows,
// microseconds, tile kernel and windows:
// - Row sums that a wavefront keeps in LDS (256 of a tile): rows so short that
//   tiles hold more are written one by one. 206 starts a tile on average (sigma
//   16, 8200 tiles, FP64, band 200): 35.3 and 33.8; 256: 36.0 and 45.7; 342: 38.2
//   and 64.3.
constexpr uint32_t kWindowMaxStarts = 208;
// - Elements: sigma 4, 2100 tiles, rows of 2, FP64 7.0 and 7.9, FP32 5.6 and 5.9;
//   3900 tiles, rows of 3, band 6000: FP64 10.9 and 9.1, FP32 7.6 and 6.9.
constexpr uint64_t kWindowElements = 750000;
// - In FP64, with twice the bytes to move before a workgroup's first sum, more
//   workgroups: sigma 16, rows of 12, 1074 tiles, band 200: 10.8 and 15.0; 1097,
//   band 8000: 13.4 and 16.3; 2004, band 8000: 18.9 and 17.7; 2435, band 200: 19.0
//   and 17.1.
constexpr uint32_t kWindowMinTiles64 = 2048;
// - In FP64 and within a narrow band, where the tile kernel finds x in L1 anyway,
//   more elements: sigma 4, 2054 tiles, band 200: 5.7 and 6.9; sigma 8, 2924 tiles,
//   band 200: 9.0 and 9.2; but sigma 4, 3017 tiles, band 2000: 9.1 and 7.2. Narrow:
//   a window that reaches less far past the rows' own share of the columns than
//   2/5 of the workgroup's elements.
constexpr uint64_t kWindowNarrowElements = 1500000;

// How a product is cut: workgroups of 16 wavefronts with `per` tiles each, and
// the largest window, in entries of x; blocks == 0: the tile kernel's.
struct WindowShape {
    uint32_t per = 0, blocks = 0, width = 0;
};

struct WindowPlan {
    uint32_t* span = nullptr; // lowest and highest column of every 16 tiles
    WindowShape f64, f32;
    WindowShape sums; // of the transposed product (transpose.hip)
};

// The shape for values of vb bytes, from the spans and the tile flags (tiles + 1
// entries).
WindowShape window_shape(const DevFormat& A, const std::vector<uint32_t>& span,
                         const std::vector<uint8_t>& tile_flags, size_t vb);

WindowShape window_sums_shape(uint32_t tiles, uint32_t sigma, const std::vector<uint32_t>& span);

namespace detail {

// The columns [lo, lo + w) of workgroup b's tiles.
__device__ __forceinline__ void window_of(const uint32_t* span, uint32_t tiles, const WindowShape& S, uint32_t b,
                                          uint32_t* lo, uint32_t* w) {
    const uint32_t groups = (tiles + kWindowGroup - 1) / kWindowGroup;
    const uint32_t g0 = b * S.per, g1 = min(g0 + S.per, groups);
    uint32_t l = 0xffffffffu, h = 0;
    for (uint32_t g = g0; g < g1; ++g) {
        l = min(l, span[2 * g]);
        h = max(h, span[2 * g + 1]);
    }
    *lo = l;
    *w = min(h - l + 1u, S.width);
}

} // namespace detail

hipError_t launch_spans(const DevFormat& A, uint32_t* span, hipStream_t stream);

// y = A x.
hipError_t launch_window_spmv(const DevFormat& A, const WindowPlan& P, bool f32, const void* x, void* y,
                              hipStream_t stream);

} // namespace dimgpu
