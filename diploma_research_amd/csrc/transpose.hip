// y = A^T x.
//
// Adding every product into y where it belongs costs one memory-side atomic
// per element, and those are slow (FP64, 4.2M elements within a band of 18000
// columns: 235 us, where the bytes take 10). Large products are sorted instead:
// the columns are cut into bins, the first kernel writes each product to its
// column's bin, and the second sums each bin in LDS and writes its part of y
// once. Where a workgroup's products of a bin go follows from the pattern
// alone; it is counted with a matrix's first product (3 small kernels) and kept.
//
// Where the elements lie within a band, a workgroup's columns fit LDS and
// nothing is sorted: it adds its products up there, writes the sums of its
// window, and a second kernel adds the windows up (4.1M elements within a band
// of 18000 columns, FP64: 27.6 us against 68.5 sorted).
#include "handle.h"
#include "spmv_impl.h"

#include <algorithm>

namespace dimgpu {

namespace {

using detail::DescWord;
using detail::element_row;
using detail::sload;
using detail::wave_incl_scan;
using detail::xcd_remap;

constexpr int kSortThreads = 512;
constexpr uint32_t kSortWaves = kSortThreads / 64;
constexpr uint32_t kMaxBins = 2048;   // counters of a workgroup, in LDS
constexpr uint32_t kMaxShift = 13;    // columns of a bin: at most 8192 (64 KB of FP64 sums)
constexpr uint32_t kSortBlocks = 512;
// Below this many elements the atomics are faster than two kernels and the
// round trip through the bins.
constexpr uint64_t kSortElements = 1u << 15;

template<typename V>
__global__ void k_fill(V* y, size_t n, V value, const int* done) {
    if (done && *done)
        return;
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        y[i] = value;
}

// Calls f(row, column, value's place) for every element of tile t that this
// lane holds.
template<int SIGMA, typename F>
__device__ __forceinline__ void over_tile(const DevFormat& A, uint32_t t, F&& f) {
    const int lane = threadIdx.x & 63;
    using W = typename DescWord<SIGMA>::type;
    const size_t base = static_cast<size_t>(t) * (64 * SIGMA);
    const uint32_t bits = static_cast<uint32_t>(static_cast<const W*>(A.bit_flag)[static_cast<size_t>(t) * 64 + lane]) |
                          (lane == 0 ? 1u : 0u);
    const uint32_t tpw = A.tile_ptr[t];
    const bool dirty = (tpw & kDirty) != 0;
    const uint32_t row0 = tpw & ~kDirty;
    const uint32_t* tdo = dirty ? A.tile_desc_offset + A.tile_desc_offset_ptr[t] : nullptr;
    const int nb = __popc(bits);
    const int y_off = wave_incl_scan(nb, lane) - nb;
    const uint64_t first = base + static_cast<size_t>(lane) * SIGMA; // the lane's first element
    const int have = first >= A.nnz ? 0 : A.nnz - first < SIGMA ? static_cast<int>(A.nnz - first) : SIGMA;
#pragma unroll
    for (int r = 0; r < SIGMA; ++r)
        if (r < have) {
            const size_t pos = base + static_cast<size_t>(r) * 64 + lane;
            f(element_row(bits, r, y_off, row0, dirty, tdo), A.col_idx[pos], pos);
        }
}

// y[col] += a_ij * x[row] by floating-point atomics.
template<typename V, int SIGMA>
__global__ __launch_bounds__(256) void k_transpose_atomic(DevFormat A, const V* __restrict__ vals,
                                                          const V* __restrict__ x, V* y, const int* done) {
    if (done && *done)
        return;
    const uint32_t t = xcd_remap(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6);
    if (t >= A.tiles)
        return;
    over_tile<SIGMA>(A, t, [&](uint32_t row, uint32_t col, size_t pos) { unsafeAtomicAdd(y + col, vals[pos] * x[row]); });
}

// ---- the pattern's part: where each workgroup's products of a bin go ------

// counts[b * bins + bin]: elements of workgroup b's tiles in each bin
__global__ __launch_bounds__(kSortThreads) void k_count_bins(uint64_t nnz, uint64_t per, uint32_t shift, uint32_t bins,
                                                             uint64_t tile, const uint32_t* __restrict__ col_idx,
                                                             uint32_t* __restrict__ counts) {
    __shared__ uint32_t n[kMaxBins];
    for (uint32_t i = threadIdx.x; i < bins; i += kSortThreads)
        n[i] = 0;
    __syncthreads();
    const uint64_t e0 = blockIdx.x * per * tile;
    const uint64_t total = (nnz + tile - 1) / tile * tile, e1 = e0 + per * tile < total ? e0 + per * tile : total;
    const uint32_t sigma = static_cast<uint32_t>(tile / 64);
    for (uint64_t e = e0 + threadIdx.x; e < e1; e += kSortThreads) {
        // (the padding of the last tile is no element)
        const uint64_t t0 = e / tile * tile, in = e - t0;
        if (t0 + (in & 63u) * sigma + (in >> 6) < nnz)
            atomicAdd(&n[col_idx[e] >> shift], 1u);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < bins; i += kSortThreads)
        counts[static_cast<size_t>(blockIdx.x) * bins + i] = n[i];
}

// counts to each workgroup's offset within the bin (in place), and the bins'
// totals: 64 bins per workgroup, the workgroups' counts in 16 pieces
__global__ __launch_bounds__(1024) void k_bin_offsets(uint32_t blocks, uint32_t bins, uint32_t* counts,
                                                      uint32_t* totals) {
    __shared__ uint32_t sum[16][64];
    const uint32_t c = threadIdx.x & 63, piece = threadIdx.x >> 6;
    const uint32_t bin = blockIdx.x * 64 + c;
    const uint32_t per = (blocks + 15) / 16, b0 = min(piece * per, blocks), b1 = min(b0 + per, blocks);
    uint32_t s = 0;
    if (bin < bins)
        for (uint32_t b = b0; b < b1; ++b)
            s += counts[static_cast<size_t>(b) * bins + bin];
    sum[piece][c] = s;
    __syncthreads();
    uint32_t at = 0, all = 0;
    for (uint32_t q = 0; q < 16; ++q) {
        at += q < piece ? sum[q][c] : 0u;
        all += sum[q][c];
    }
    if (bin < bins) {
        for (uint32_t b = b0; b < b1; ++b) {
            const uint32_t n = counts[static_cast<size_t>(b) * bins + bin];
            counts[static_cast<size_t>(b) * bins + bin] = at;
            at += n;
        }
        if (piece == 0)
            totals[bin] = all;
    }
}

// start[bin] = the bin's first place, start[bins] = the element count
__global__ __launch_bounds__(1024) void k_bin_starts(uint32_t bins, const uint32_t* totals, uint32_t* start) {
    __shared__ uint32_t sum[1024];
    const uint32_t per = (bins + 1023) / 1024, i0 = min(threadIdx.x * per, bins), i1 = min(i0 + per, bins);
    uint32_t s = 0;
    for (uint32_t i = i0; i < i1; ++i)
        s += totals[i];
    sum[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t d = 1; d < 1024; d <<= 1) {
        const uint32_t u = threadIdx.x >= d ? sum[threadIdx.x - d] : 0u;
        __syncthreads();
        sum[threadIdx.x] += u;
        __syncthreads();
    }
    uint32_t at = sum[threadIdx.x] - s;
    for (uint32_t i = i0; i < i1; ++i) {
        start[i] = at;
        at += totals[i];
    }
    if (threadIdx.x == 1023)
        start[bins] = sum[1023];
}

// ---- the product -----------------------------------------------------------

// Every product to its bin. The workgroups of one XCD take neighbouring tiles,
// whose runs in a bin are neighbours too and meet in its L2.
template<typename V, int SIGMA>
__global__ __launch_bounds__(kSortThreads) void k_sort_products(DevFormat A, TransposePlan T,
                                                                const V* __restrict__ vals, const V* __restrict__ x,
                                                                const int* done) {
    if (done && *done)
        return;
    __shared__ uint32_t next[kMaxBins];
    const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t* off = T.off + static_cast<size_t>(b) * T.bins;
    for (uint32_t i = threadIdx.x; i < T.bins; i += kSortThreads)
        next[i] = T.start[i] + off[i];
    __syncthreads();
    V* prod = static_cast<V*>(T.prod);
    const uint32_t t1 = min((b + 1) * T.per, A.tiles);
    const uint32_t mask = (1u << T.shift) - 1u;
    for (uint32_t t = b * T.per + (threadIdx.x >> 6); t < t1; t += kSortWaves)
        over_tile<SIGMA>(A, t, [&](uint32_t row, uint32_t col, size_t pos) {
            const V v = vals[pos] * x[row];
            const uint32_t at = atomicAdd(&next[col >> T.shift], 1u);
            prod[at] = v;
            T.col[at] = static_cast<uint16_t>(col & mask);
        });
}

// Sums one bin (a share of it) in LDS, in FP64 (FP32 products too: the FP64
// adds are also the faster ones there). With one share per bin y is
// written, so it needs no clearing; with more, every share adds its sums to a
// cleared y.
template<typename V>
__global__ __launch_bounds__(kSortThreads) void k_sum_bins(TransposePlan T, uint32_t cols, uint32_t shares, V* y,
                                                           const int* done) {
    if (done && *done)
        return;
    extern __shared__ double sum[];
    const uint32_t bin = blockIdx.x / shares, share = blockIdx.x - bin * shares;
    const uint32_t c0 = bin << T.shift, n = min(1u << T.shift, cols - c0);
    for (uint32_t i = threadIdx.x; i < n; i += kSortThreads)
        sum[i] = 0.0;
    __syncthreads();
    const uint32_t a = T.start[bin], e = T.start[bin + 1];
    const uint32_t per = (e - a + shares - 1) / shares;
    const uint32_t i0 = min(a + share * per, e), i1 = min(i0 + per, e);
    const V* __restrict__ prod = static_cast<const V*>(T.prod);
    const uint16_t* __restrict__ col = T.col;
    constexpr uint32_t U = 4;
    uint32_t i = i0 + threadIdx.x;
    for (; i + (U - 1) * kSortThreads < i1; i += U * kSortThreads) {
        V v[U];
        uint32_t c[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            v[u] = prod[i + u * kSortThreads];
            c[u] = col[i + u * kSortThreads];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            unsafeAtomicAdd(sum + c[u], static_cast<double>(v[u]));
    }
    for (; i < i1; i += kSortThreads)
        unsafeAtomicAdd(sum + col[i], static_cast<double>(prod[i]));
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < n; q += kSortThreads) {
        if (shares == 1)
            y[c0 + q] = static_cast<V>(sum[q]);
        else
            unsafeAtomicAdd(y + c0 + q, static_cast<V>(sum[q]));
    }
}

// ---- matrices within a band ------------------------------------------------

constexpr int kBandThreads = 64 * static_cast<int>(kWindowGroup);
static_assert(kBandThreads == 1024, "one workgroup per CU: its window may take all of the LDS");

// Workgroup b's sums of its window, to sums[b * width]. One workgroup of 16
// wavefronts per CU; the products of one column meet in LDS in no fixed order
// (FP64 sums, for FP32 products too).
template<typename V, int SIGMA>
__global__ __launch_bounds__(kBandThreads) void k_band_products(DevFormat A, const uint32_t* __restrict__ span,
                                                                WindowShape S, const V* __restrict__ vals,
                                                                const V* __restrict__ x, double* __restrict__ sums,
                                                                const int* done) {
    if (done && *done)
        return;
    extern __shared__ double sum[];
    const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
    uint32_t lo, w;
    detail::window_of(span, A.tiles, S, b, &lo, &w);
    for (uint32_t i = threadIdx.x; i < w; i += kBandThreads)
        sum[i] = 0.0;
    __syncthreads();
    const uint32_t tb = b * kWindowGroup * S.per, te = min(tb + kWindowGroup * S.per, A.tiles);
    const int lane = threadIdx.x & 63;
    const uint32_t ulane = static_cast<uint32_t>(lane);
    for (uint32_t t = tb + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); t < te; t += kWindowGroup) {
        // (all of a tile's loads in flight together)
        using W = typename DescWord<SIGMA>::type;
        const size_t base = static_cast<size_t>(t) * (64 * SIGMA);
        const uint32_t bits =
          static_cast<uint32_t>(static_cast<const W*>(A.bit_flag)[static_cast<size_t>(t) * 64 + ulane]) |
          (lane == 0 ? 1u : 0u);
        uint32_t col[SIGMA], row[SIGMA];
        V v[SIGMA], xv[SIGMA];
#pragma unroll
        for (int r = 0; r < SIGMA; ++r) {
            v[r] = __builtin_nontemporal_load(vals + base + r * 64 + ulane);
            col[r] = __builtin_nontemporal_load(A.col_idx + base + r * 64 + ulane);
        }
        const uint32_t tpw = sload(A.tile_ptr + t), row0 = tpw & ~kDirty;
        const int nb = __popc(bits);
        const uint32_t y_off = static_cast<uint32_t>(wave_incl_scan(nb, lane) - nb);
#pragma unroll
        for (int r = 0; r < SIGMA; ++r)
            row[r] = y_off - 1u + static_cast<uint32_t>(__popc(bits & ((2u << r) - 1u)));
        if (tpw & kDirty) {
            const uint32_t* tdo = A.tile_desc_offset + sload(A.tile_desc_offset_ptr + t);
#pragma unroll
            for (int r = 0; r < SIGMA; ++r)
                row[r] = tdo[row[r]];
        }
#pragma unroll
        for (int r = 0; r < SIGMA; ++r)
            xv[r] = x[row0 + row[r]];
        const uint64_t left = A.nnz - base; // (the last tile has padding)
#pragma unroll
        for (int r = 0; r < SIGMA; ++r)
            if (ulane * SIGMA + r < left)
                unsafeAtomicAdd(sum + (col[r] - lo), static_cast<double>(v[r] * xv[r]));
    }
    __syncthreads();
    double* out = sums + static_cast<size_t>(b) * S.width;
    for (uint32_t i = threadIdx.x; i < w; i += kBandThreads)
        out[i] = sum[i];
}

// y: every column's sums over the windows that hold it, in the workgroups'
// order. The windows are looked through 256 at a time; those that meet the
// workgroup's 256 columns are listed in LDS.
template<typename V>
__global__ __launch_bounds__(256) void k_band_sum(const uint32_t* __restrict__ span, uint32_t tiles, WindowShape S,
                                                  uint32_t cols, const double* __restrict__ sums, V* __restrict__ y,
                                                  const int* done) {
    if (done && *done)
        return;
    __shared__ uint32_t at_s[256], lo_s[256], w_s[256], n_s[4];
    const uint32_t c0 = blockIdx.x * 256, c = c0 + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double s = 0.0;
    for (uint32_t b0 = 0; b0 < S.blocks; b0 += 256) {
        const uint32_t b = b0 + threadIdx.x;
        uint32_t lo = 0, w = 0;
        if (b < S.blocks)
            detail::window_of(span, tiles, S, b, &lo, &w);
        const bool meets = lo < c0 + 256 && c0 < lo + w;
        const uint64_t m = __ballot(meets);
        if (lane == 0)
            n_s[wave] = __popcll(m);
        __syncthreads();
        uint32_t k = __popcll(m & ((1ull << lane) - 1ull)), n = 0;
        for (uint32_t q = 0; q < 4; ++q) {
            k += q < wave ? n_s[q] : 0u;
            n += n_s[q];
        }
        if (meets) {
            at_s[k] = b;
            lo_s[k] = lo;
            w_s[k] = w;
        }
        __syncthreads();
        constexpr uint32_t U = 8;
        for (uint32_t i = 0; i < n; i += U) {
            double v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                const uint32_t q = min(i + u, n - 1u);
                const uint32_t o = c - lo_s[q];
                v[u] = i + u < n && o < w_s[q] ? sums[static_cast<size_t>(at_s[q]) * S.width + o] : 0.0;
            }
#pragma unroll
            for (uint32_t u = 0; u < U; ++u)
                s += v[u];
        }
        __syncthreads();
    }
    if (c < cols)
        y[c] = static_cast<V>(s);
}

template<typename V, int SIGMA>
hipError_t launch_band(const dim_csr5* h, const V* vals, const V* x, V* y, hipStream_t stream, const int* done) {
    const WindowShape& S = h->win.sums;
    const uint32_t bytes = S.width * static_cast<uint32_t>(sizeof(double));
    const void* f = reinterpret_cast<const void*>(&k_band_products<V, SIGMA>);
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    if (e != hipSuccess)
        return e;
    double* sums = static_cast<double*>(h->tplan.prod);
    hipLaunchKernelGGL((k_band_products<V, SIGMA>), dim3(S.blocks), dim3(kBandThreads), bytes, stream, h->f,
                       static_cast<const uint32_t*>(h->win.span), S, vals, x, sums, done);
    hipLaunchKernelGGL(k_band_sum<V>, dim3((h->f.cols + 255) / 256), dim3(256), 0, stream,
                       static_cast<const uint32_t*>(h->win.span), h->f.tiles, S, h->f.cols,
                       static_cast<const double*>(sums), y, done);
    return hipGetLastError();
}

// ---- which of them ---------------------------------------------------------

// The matrix's plan, made with its first product; sorted == false when it
// keeps the atomics (few elements, very many columns, no room, or a stream
// that is being captured before the plan exists).
dim_status transpose_plan(dim_csr5* h, hipStream_t stream, bool* sorted) {
    const DevFormat& A = h->f;
    TransposePlan& T = h->tplan;
    *sorted = T.bins != 0 || T.band;
    if (*sorted || T.refused || A.nnz < kSortElements)
        return DIM_SUCCESS;
    const bool band = h->win.sums.blocks != 0;
    // about 512 bins, of 64 to 8192 columns
    uint32_t shift = 6;
    while (shift < kMaxShift && (A.cols >> shift) >= 512)
        ++shift;
    const uint32_t bins = (A.cols + (1u << shift) - 1) >> shift;
    if (bins > kMaxBins && !band) {
        T.refused = true;
        return DIM_SUCCESS;
    }
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return DIM_SUCCESS;
    }
    if (band) {
        double* sums = nullptr;
        const hipError_t e = dev_alloc(h, sums, size_t{h->win.sums.blocks} * h->win.sums.width);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            T.refused = true;
            return DIM_SUCCESS;
        }
        DIM_HIP_TRY(e);
        T.prod = sums;
        T.band = *sorted = true;
        return DIM_SUCCESS;
    }
    TransposePlan p;
    p.shift = shift;
    p.bins = bins;
    p.per = std::max<uint32_t>((A.tiles + kSortBlocks - 1) / kSortBlocks, kSortWaves / 4);
    p.blocks = (A.tiles + p.per - 1) / p.per;
    const size_t kept = h->allocations.size();
    const uint64_t kept_bytes = h->device_bytes;
    uint32_t* totals = nullptr;
    double* prod = nullptr;
    hipError_t e = dev_alloc(h, p.off, size_t{p.blocks} * bins);
    if (e == hipSuccess)
        e = dev_alloc(h, p.start, bins + 1);
    if (e == hipSuccess)
        e = dev_alloc(h, totals, bins);
    if (e == hipSuccess)
        e = dev_alloc(h, p.col, A.nnz);
    if (e == hipSuccess)
        e = dev_alloc(h, prod, A.nnz);
    p.prod = prod;
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        for (; h->allocations.size() > kept; h->allocations.pop_back())
            (void)hipFree(h->allocations.back());
        h->device_bytes = kept_bytes;
        T.refused = true;
        return DIM_SUCCESS;
    }
    DIM_HIP_TRY(e);
    hipLaunchKernelGGL(k_count_bins, dim3(p.blocks), dim3(kSortThreads), 0, stream, A.nnz, uint64_t{p.per}, shift, bins,
                       uint64_t{64} * A.sigma, static_cast<const uint32_t*>(A.col_idx), p.off);
    hipLaunchKernelGGL(k_bin_offsets, dim3((bins + 63) / 64), dim3(1024), 0, stream, p.blocks, bins, p.off, totals);
    hipLaunchKernelGGL(k_bin_starts, dim3(1), dim3(1024), 0, stream, bins, static_cast<const uint32_t*>(totals),
                       p.start);
    DIM_HIP_TRY(hipGetLastError());
    T = p;
    *sorted = true;
    return DIM_SUCCESS;
}

template<typename V>
hipError_t product(const dim_csr5* h, bool sorted, const V* vals, const V* x, V* y, hipStream_t stream,
                   const int* done) {
    const DevFormat& A = h->f;
    const TransposePlan& T = h->tplan;
    // enough workgroups for the chip where the bins are few
    if (T.band) {
        switch (A.sigma) {
#define DIM_B(S)                                                                                                      \
    case S:                                                                                                           \
        return launch_band<V, S>(h, vals, x, y, stream, done);
            DIM_B(4) DIM_B(5) DIM_B(6) DIM_B(7) DIM_B(8) DIM_B(10) DIM_B(12) DIM_B(14) DIM_B(16)
#undef DIM_B
            default: return hipErrorInvalidValue;
        }
    }
    const uint32_t shares = sorted ? std::max(1u, 256u / T.bins) : 0u;
    if (shares != 1)
        hipLaunchKernelGGL(k_fill<V>, dim3(1024), dim3(256), 0, stream, y, static_cast<size_t>(A.cols), V(0), done);
    if (!A.tiles)
        return hipGetLastError();
    const uint32_t grid = (A.tiles + 3) / 4;
    switch (A.sigma) {
#define DIM_T(S)                                                                                                      \
    case S:                                                                                                           \
        if (sorted)                                                                                                   \
            hipLaunchKernelGGL((k_sort_products<V, S>), dim3(T.blocks), dim3(kSortThreads), 0, stream, A, T, vals, x, \
                               done);                                                                                 \
        else                                                                                                          \
            hipLaunchKernelGGL((k_transpose_atomic<V, S>), dim3(grid), dim3(256), 0, stream, A, vals, x, y, done);    \
        break;
        DIM_FOR_EACH_SIGMA(DIM_T)
#undef DIM_T
        default: return hipErrorInvalidValue;
    }
    if (sorted)
        hipLaunchKernelGGL(k_sum_bins<V>, dim3(T.bins * shares), dim3(kSortThreads), sizeof(double) << T.shift, stream, T,
                           A.cols, shares, y, done);
    return hipGetLastError();
}

} // namespace

dim_status launch_spmv_transpose(dim_csr5* h, bool f32, const void* x, void* y, hipStream_t stream, const int* done) {
    bool sorted = false;
    if (dim_status st = transpose_plan(h, stream, &sorted))
        return st;
    if (f32)
        DIM_HIP_TRY(product<float>(h, sorted, h->f.vals32, static_cast<const float*>(x), static_cast<float*>(y), stream,
                                   done));
    else
        DIM_HIP_TRY(product<double>(h, sorted, h->f.vals64, static_cast<const double*>(x), static_cast<double*>(y),
                                    stream, done));
    return DIM_SUCCESS;
}

} // namespace dimgpu
