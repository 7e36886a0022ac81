// CSR -> CSR5 (omega = 64) conversion on the GPU, from device CSR arrays.
//
// Produces exactly the format of the host builder (format.cpp), following
// the reference conversion (include/dim/mat/storage_formats/csr5.h:
// generate_tile_pointer 411-431, set_bit_flag 323-340, generate_tile_offset
// 363-397, transpose 463-493), one wavefront per tile:
//   1. the CSR arrays are checked and the empty rows counted;
//   2. a tile's first row by a 64-way search in row_ptr, then its row starts by
//      a walk over row_ptr, 64 rows at a time: bit flags, tile flags, dirty mark;
//   3. the per-tile transpose of values and column indices, through LDS, and
//      the column spans of every 16 tiles;
//   4. only if there are empty rows: the segment -> row maps of dirty tiles (a
//      scan of their segment counts, then the walk again) and the list of
//      empty rows.
// Everything the handle keeps is one allocation and the temporaries another:
// an allocation or free takes longer than most of the kernels.
#include "handle.h"
#include "spmv_impl.h"

#include <hip/hip_runtime.h>

#include <memory>

namespace dimgpu {

namespace {

using detail::wave_incl_scan;

constexpr int kT = 256;

struct Counts {
    int bad;           // 1: row_ptr decreases, 2: column out of range, 4: row_ptr's ends
    uint32_t n_empty;  // rows without elements
    uint32_t n_dirty;  // tiles that hold one
    uint32_t ntdo;     // segments of dirty tiles
};

__global__ void k_zero_counts(Counts* c) {
    *c = Counts{};
}

// row_ptr[0] == 0, monotone, row_ptr[rows] == nnz, col_idx < cols; the empty rows
__global__ __launch_bounds__(kT) void k_check(uint32_t rows, uint32_t cols, uint64_t nnz,
                                              const uint32_t* __restrict__ rp, const uint32_t* __restrict__ ci,
                                              Counts* out) {
    const size_t tid = blockIdx.x * static_cast<size_t>(kT) + threadIdx.x;
    const size_t stride = static_cast<size_t>(gridDim.x) * kT;
    int bad = 0;
    uint32_t empty = 0;
    for (size_t r = tid; r < rows; r += stride) {
        const uint32_t a = rp[r], b = rp[r + 1];
        bad |= b < a ? 1 : 0;
        empty += a == b ? 1u : 0u;
    }
    size_t k = tid;
    for (; k + 3 * stride < nnz; k += 4 * stride) {
        const uint32_t a = ci[k], b = ci[k + stride], c = ci[k + 2 * stride], d = ci[k + 3 * stride];
        bad |= max(max(a, b), max(c, d)) >= cols ? 2 : 0;
    }
    for (; k < nnz; k += stride)
        bad |= ci[k] >= cols ? 2 : 0;
    if (tid == 0 && (rp[0] != 0 || rp[rows] != nnz))
        bad |= 4;
    if (bad)
        atomicOr(&out->bad, bad);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        empty += __shfl_xor(empty, d, 64);
    if ((threadIdx.x & 63) == 0 && empty)
        atomicAdd(&out->n_empty, empty);
}

// What no tile writes: the ends of the arrays, the flag words' padding (they
// are read 4 bytes at a time), the product's counters; with no empty rows, the
// segment offsets too.
__global__ __launch_bounds__(kT) void k_ends(uint32_t T, uint32_t rows, uint32_t flag_bytes, bool clean,
                                             uint32_t* tile_ptr, uint8_t* tile_flags, uint32_t* tdo_ptr, uint32_t* tdo,
                                             uint32_t* queue, uint32_t* span) {
    const uint32_t tid = blockIdx.x * kT + threadIdx.x, stride = gridDim.x * kT;
    if (tid == 0) {
        tile_ptr[T] = rows;
        tile_flags[T] = kStartsRow;
        tdo[0] = 0;
    }
    for (uint32_t i = T + 1 + tid; i < flag_bytes; i += stride)
        tile_flags[i] = 0;
    for (uint32_t i = tid; i < kQueueWords; i += stride)
        queue[i] = 0;
    if (clean)
        for (uint32_t i = tid; i <= T; i += stride)
            tdo_ptr[i] = 0;
    if (span) // (the lowest and the highest column of no tiles)
        for (uint32_t i = tid; i < 2 * ((T + kWindowGroup - 1) / kWindowGroup); i += stride)
            span[i] = i & 1u ? 0u : 0xffffffffu;
}

// The last row r with rp[r] <= b (b < rp[rows]), found by the whole wavefront.
__device__ __forceinline__ uint32_t first_row(const uint32_t* __restrict__ rp, uint32_t rows, uint32_t b, int lane) {
    uint32_t lo = 0, hi = rows; // rp[lo] <= b < rp[hi]
    while (hi - lo > 1) {
        const uint32_t step = (hi - lo + 63) / 64;
        const uint64_t at = static_cast<uint64_t>(lo) + static_cast<uint64_t>(lane + 1) * step;
        const uint32_t n = __popcll(__ballot(at < hi && rp[at < hi ? at : lo] <= b));
        lo += n * step;
        hi = hi - lo > step ? lo + step : hi;
    }
    return lo;
}

// One wavefront per tile: first row, row starts, flags, dirty mark (an empty
// row among the rows from the tile's first up to the next tile's first).
template<typename W>
__global__ __launch_bounds__(kT) void k_tiles(uint32_t T, uint32_t rows, uint32_t nnz, uint32_t sigma,
                                              const uint32_t* __restrict__ rp, uint32_t* __restrict__ tile_ptr,
                                              W* __restrict__ bits, uint8_t* __restrict__ tile_flags,
                                              uint32_t* __restrict__ nseg_dirty) {
    __shared__ uint32_t words[kT / 64][64];
    const uint32_t t = blockIdx.x * (kT / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (t >= T)
        return; // wave-uniform
    uint32_t* w = words[threadIdx.x >> 6];
    w[lane] = 0;
    __builtin_amdgcn_wave_barrier(); // a wavefront's LDS accesses run in order
    const uint32_t tile = kOmega * sigma;
    const uint32_t b = t * tile;
    const uint32_t e = nnz - b > tile ? b + tile : nnz;
    const uint32_t start = __builtin_amdgcn_readfirstlane(first_row(rp, rows, b, lane));
    if (lane == 0 && rp[start] == b)
        w[0] = 1u;
    __builtin_amdgcn_wave_barrier();
    bool dirty = false;
    for (uint64_t r0 = uint64_t{start} + 1; r0 < rows; r0 += 64) { // wave-uniform
        const uint64_t r = r0 + lane;
        const bool in = r < rows;
        const uint32_t s = in ? rp[r] : 0xffffffffu;
        const uint32_t n = in ? rp[r + 1] : 0xffffffffu;
        if (in && s < e && n > s) {
            const uint32_t at = s - b;
            atomicOr(&w[at / sigma], 1u << (at % sigma));
        }
        dirty = dirty || __ballot(in && n == s && s <= e) != 0ull;
        // done past the tile's end; the rows at its end can only be empty
        // (or the next tile's first)
        if (__ballot(!in || s > e) || (dirty && __ballot(lane == 0 && s >= e)))
            break;
    }
    __builtin_amdgcn_wave_barrier();
    const uint32_t word = w[lane];
    bits[static_cast<size_t>(t) * kOmega + lane] = static_cast<W>(word);
    int n = __popc(word | (lane == 0 ? 1u : 0u));
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        n += __shfl_xor(n, d, 64);
    if (lane == 0) {
        tile_ptr[t] = start | (dirty ? kDirty : 0u);
        tile_flags[t] = static_cast<uint8_t>(((word & 1u) ? kStartsRow : 0) | (n > 1 ? kMultiSeg : 0));
        nseg_dirty[t] = dirty ? static_cast<uint32_t>(n) : 0u;
    }
}

// Exclusive scan of in[0..n) to out[0..n], out[n] the total (also to *total; the
// number of entries that are not 0 is added to *nonzero), by one workgroup.
// (Dirty tiles are counted here: an atomic add of each, 586k of them in 150M
// elements at sigma 4, made a conversion of 3.2 ms take 8.7.)
__global__ __launch_bounds__(1024) void k_scan(uint32_t n, const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                               uint32_t* total, uint32_t* nonzero) {
    __shared__ uint32_t wave_sum[16], carry_s;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t carry = 0, filled = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += 1024) {
        const uint32_t i = i0 + threadIdx.x;
        const uint32_t v = i < n ? in[i] : 0u;
        filled += v ? 1u : 0u;
        const uint32_t incl = static_cast<uint32_t>(wave_incl_scan(static_cast<int>(v), lane));
        if (lane == 63)
            wave_sum[w] = incl;
        __syncthreads();
        uint32_t before = carry;
        for (int q = 0; q < w; ++q)
            before += wave_sum[q];
        if (i < n)
            out[i] = before + incl - v;
        if (threadIdx.x == 1023)
            carry_s = before + incl;
        __syncthreads();
        carry = carry_s;
    }
    if (threadIdx.x == 0) {
        out[n] = carry;
        if (total)
            *total = carry;
    }
    if (nonzero && filled)
        atomicAdd(nonzero, filled);
}

// Segment -> row offsets of dirty tiles: segment 0 lies in the tile's first row,
// the others in its non-empty rows in order.
__global__ __launch_bounds__(kT) void k_tile_offsets(uint32_t T, uint32_t rows, uint32_t nnz, uint32_t tile,
                                                     const uint32_t* __restrict__ rp,
                                                     const uint32_t* __restrict__ tile_ptr,
                                                     const uint32_t* __restrict__ tdo_ptr, uint32_t* __restrict__ tdo) {
    const uint32_t t = blockIdx.x * (kT / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (t >= T || !(tile_ptr[t] & kDirty))
        return; // wave-uniform
    const uint32_t start = tile_ptr[t] & ~kDirty;
    const uint32_t b = t * tile, e = nnz - b > tile ? b + tile : nnz;
    uint32_t* out = tdo + tdo_ptr[t];
    if (lane == 0)
        out[0] = 0;
    uint32_t seg = 1;
    for (uint64_t r0 = uint64_t{start} + 1; r0 < rows; r0 += 64) {
        const uint64_t r = r0 + lane;
        const bool in = r < rows;
        const uint32_t s = in ? rp[r] : 0xffffffffu;
        const bool starts = in && s < e && rp[r + 1] > s;
        const uint64_t m = __ballot(starts);
        if (starts)
            out[seg + __popcll(m & ((1ull << lane) - 1ull))] = static_cast<uint32_t>(r) - start;
        seg += __popcll(m);
        if (__ballot(!in || s >= e))
            break;
    }
}

constexpr uint32_t kRowBlock = 4096;

// empty rows of each kRowBlock rows
__global__ __launch_bounds__(kT) void k_count_empty(uint32_t rows, const uint32_t* __restrict__ rp, uint32_t* counts) {
    __shared__ uint32_t n;
    if (threadIdx.x == 0)
        n = 0;
    __syncthreads();
    const uint64_t r0 = static_cast<uint64_t>(blockIdx.x) * kRowBlock;
    uint32_t mine = 0;
    for (uint32_t i = threadIdx.x; i < kRowBlock; i += kT)
        if (r0 + i < rows)
            mine += rp[r0 + i] == rp[r0 + i + 1] ? 1u : 0u;
    if (mine)
        atomicAdd(&n, mine);
    __syncthreads();
    if (threadIdx.x == 0)
        counts[blockIdx.x] = n;
}

// the empty rows in ascending order, each block's from first[block] on
__global__ __launch_bounds__(64) void k_list_empty(uint32_t rows, const uint32_t* __restrict__ rp,
                                                   const uint32_t* __restrict__ first, uint32_t* __restrict__ list) {
    const int lane = threadIdx.x;
    const uint64_t r0 = static_cast<uint64_t>(blockIdx.x) * kRowBlock;
    uint32_t at = first[blockIdx.x];
    if (at == first[blockIdx.x + 1])
        return;
    for (uint32_t i = 0; i < kRowBlock; i += 64) {
        const uint64_t r = r0 + i + lane;
        const bool empty = r < rows && rp[r] == rp[r + 1];
        const uint64_t m = __ballot(empty);
        if (empty)
            list[at + __popcll(m & ((1ull << lane) - 1ull))] = static_cast<uint32_t>(r);
        at += __popcll(m);
    }
}

// Values and columns in tile order, through LDS (each lane's elements an odd
// number of entries apart, as in values.hip): consecutive reads and writes on
// both sides.
template<int SIGMA>
__global__ __launch_bounds__(kT) void k_transpose(uint32_t T, uint64_t nnz, const uint32_t* __restrict__ ci,
                                                  const double* __restrict__ v, uint32_t* __restrict__ ci_out,
                                                  double* __restrict__ v_out, float* __restrict__ v32_out,
                                                  uint32_t* span) {
    __shared__ double stage[kT / 64][64 * (SIGMA | 1)];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t t = blockIdx.x * (kT / 64) + (threadIdx.x >> 6);
    if (t >= T)
        return; // wave-uniform
    double* s = stage[threadIdx.x >> 6];
    uint32_t* sc = reinterpret_cast<uint32_t*>(s);
    const uint64_t base = static_cast<uint64_t>(t) * (64 * SIGMA);
    const uint32_t left = static_cast<uint32_t>(nnz - base < 64 * SIGMA ? nnz - base : 64 * SIGMA);
    double a[SIGMA];
    uint32_t c[SIGMA];
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const uint32_t e = r * 64 + lane;
        a[r] = e < left ? v[base + e] : 0.0;
        c[r] = e < left ? ci[base + e] : 0u;
    }
    if (span) {
        uint32_t l = 0xffffffffu, h = 0;
#pragma unroll
        for (int r = 0; r < SIGMA; ++r) {
            l = min(l, r * 64 + lane < left ? c[r] : 0xffffffffu);
            h = max(h, c[r]);
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            l = min(l, static_cast<uint32_t>(__shfl_xor(static_cast<int>(l), d, 64)));
            h = max(h, static_cast<uint32_t>(__shfl_xor(static_cast<int>(h), d, 64)));
        }
        if (lane == 0) {
            atomicMin(span + 2 * (t / kWindowGroup), l);
            atomicMax(span + 2 * (t / kWindowGroup) + 1, h);
        }
    }
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const uint32_t e = r * 64 + lane;
        s[(e / SIGMA) * (SIGMA | 1) + e % SIGMA] = a[r];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const double x = s[lane * (SIGMA | 1) + r];
        v_out[base + r * 64 + lane] = x;
        if (v32_out)
            v32_out[base + r * 64 + lane] = static_cast<float>(x);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const uint32_t e = r * 64 + lane;
        sc[(e / SIGMA) * (SIGMA | 1) + e % SIGMA] = c[r];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < SIGMA; ++r)
        ci_out[base + r * 64 + lane] = sc[lane * (SIGMA | 1) + r];
}

template<typename W>
dim_status convert(uint32_t rows, uint32_t cols, uint64_t nnz, const uint32_t* rp, const uint32_t* ci,
                   const double* v, uint32_t sigma, bool keep_f32, hipStream_t s, dim_csr5** out) {
    std::unique_ptr<dim_csr5, void (*)(dim_csr5*)> h(new dim_csr5, free_handle);
    DIM_HIP_TRY(hipGetDevice(&h->device));
    const uint64_t tile = uint64_t{kOmega} * sigma;
    const uint64_t T64 = (nnz + tile - 1) / tile;
    if (T64 >= kDirty)
        return fail(DIM_INVALID_ARGUMENT, "too many tiles");
    const uint32_t T = static_cast<uint32_t>(T64);
    const uint32_t n32 = static_cast<uint32_t>(nnz);
    DevFormat& d = h->f;
    d.rows = rows;
    d.cols = cols;
    d.sigma = sigma;
    d.tiles = T;
    d.nnz = nnz;
    d.padded = T64 * tile;

    // temporaries
    const uint32_t row_blocks = (rows + kRowBlock - 1) / kRowBlock;
    Arena tmp;
    Counts* counts = nullptr;
    uint32_t *nseg_dirty = nullptr, *empty_counts = nullptr, *empty_first = nullptr;
    tmp.add(counts, 1);
    tmp.add(nseg_dirty, size_t{T} + 1);
    tmp.add(empty_counts, row_blocks);
    tmp.add(empty_first, size_t{row_blocks} + 1);
    void* tmp_base = nullptr;
    DIM_HIP_TRY(tmp.commit(&tmp_base));
    std::unique_ptr<void, void (*)(void*)> tmp_guard(tmp_base, [](void* p) { (void)hipFree(p); });

    Counts got{};
    hipLaunchKernelGGL(k_zero_counts, dim3(1), dim3(1), 0, s, counts);
    hipLaunchKernelGGL(k_check, dim3(1024), dim3(kT), 0, s, rows, cols, nnz, rp, ci, counts);
    DIM_HIP_TRY(hipMemcpyAsync(&got, counts, sizeof(Counts), hipMemcpyDeviceToHost, s));
    DIM_HIP_TRY(hipStreamSynchronize(s));
    if (got.bad & 1)
        return fail(DIM_INVALID_ARGUMENT, "row_ptr must be non-decreasing");
    if (got.bad & 2)
        return fail(DIM_INVALID_ARGUMENT, "column index out of range");
    if (got.bad & 4)
        return fail(DIM_INVALID_ARGUMENT, "row_ptr must start at 0 and end at nnz");
    const uint32_t n_empty = got.n_empty;
    d.n_empty = n_empty;

    Arena keep;
    W* bits = nullptr;
    // flag words are read 4 bytes at a time: pad to a multiple of 4 plus 4
    const size_t flag_bytes = (size_t{T} + 1 + 3) / 4 * 4 + 4;
    keep.add(d.col_idx, d.padded);
    keep.add(d.vals64, d.padded);
    if (keep_f32)
        keep.add(d.vals32, d.padded);
    keep.add(bits, size_t{T} * kOmega);
    keep.add(d.tile_ptr, size_t{T} + 1);
    keep.add(d.tile_flags, flag_bytes);
    keep.add(d.tile_desc_offset_ptr, size_t{T} + 1);
    // (a dirty tile has a segment for each of its non-empty rows, and one)
    keep.add(d.tile_desc_offset, n_empty ? size_t{rows} - n_empty + T : 1);
    keep.add(d.empty_rows, n_empty);
    const bool spans = T >= kWindowMinTiles && sigma <= kWindowMaxSigma;
    const size_t groups = (size_t{T} + kWindowGroup - 1) / kWindowGroup;
    if (spans)
        keep.add(h->win.span, 2 * groups);
    add_scratch(keep, h->s, T);
    DIM_HIP_TRY(keep.commit_block(h.get()));
    d.bit_flag = bits;

    const dim3 tile_grid((T + kT / 64 - 1) / (kT / 64)), block(kT);
    hipLaunchKernelGGL(k_ends, dim3(n_empty ? 1 : 32), block, 0, s, T, rows, static_cast<uint32_t>(flag_bytes),
                       n_empty == 0, d.tile_ptr, d.tile_flags, d.tile_desc_offset_ptr, d.tile_desc_offset, h->s.queue, h->win.span);
    if (T) {
        hipLaunchKernelGGL((k_tiles<W>), tile_grid, block, 0, s, T, rows, n32, sigma, rp, d.tile_ptr, bits,
                           d.tile_flags, nseg_dirty);
        switch (sigma) {
#define DIM_TRANSPOSE(S)                                                                                              \
    case S:                                                                                                           \
        hipLaunchKernelGGL((k_transpose<S>), tile_grid, block, 0, s, T, nnz, ci, v, d.col_idx, d.vals64, d.vals32,    \
                           h->win.span);                                                                              \
        break;
            DIM_FOR_EACH_SIGMA(DIM_TRANSPOSE)
#undef DIM_TRANSPOSE
            default: break;
        }
    }
    if (n_empty) {
        hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, T, static_cast<const uint32_t*>(nseg_dirty),
                           d.tile_desc_offset_ptr, &counts->ntdo, &counts->n_dirty);
        if (T)
            hipLaunchKernelGGL(k_tile_offsets, tile_grid, block, 0, s, T, rows, n32, static_cast<uint32_t>(tile), rp,
                               static_cast<const uint32_t*>(d.tile_ptr),
                               static_cast<const uint32_t*>(d.tile_desc_offset_ptr), d.tile_desc_offset);
        hipLaunchKernelGGL(k_count_empty, dim3(row_blocks), block, 0, s, rows, rp, empty_counts);
        hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, row_blocks, static_cast<const uint32_t*>(empty_counts),
                           empty_first, static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr));
        hipLaunchKernelGGL(k_list_empty, dim3(row_blocks), dim3(64), 0, s, rows, rp,
                           static_cast<const uint32_t*>(empty_first), d.empty_rows);
        DIM_HIP_TRY(hipMemcpyAsync(&got, counts, sizeof(Counts), hipMemcpyDeviceToHost, s));
    }
    DIM_HIP_TRY(hipGetLastError());
    // host copy of the tile flags for the launch planner
    std::vector<uint8_t> hflags(size_t{T} + 1);
    std::vector<uint32_t> hspan(spans ? 2 * groups : 0);
    DIM_HIP_TRY(hipMemcpyAsync(hflags.data(), d.tile_flags, size_t{T} + 1, hipMemcpyDeviceToHost, s));
    if (spans)
        DIM_HIP_TRY(hipMemcpyAsync(hspan.data(), h->win.span, hspan.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    DIM_HIP_TRY(hipStreamSynchronize(s));
    if (spans)
        shape_windows(h.get(), hspan, hflags);
    h->binfo.assign(std::move(hflags));
    d.binfo = &h->binfo;
    d.any_dirty = got.ntdo != 0;
    h->n_dirty = got.n_dirty;
    h->sys_row = {0, rows};
    h->sys_tile = {0, T};
    h->sys_nnz_csr = {0, nnz};
    h->nnz_logical = nnz;
    *out = h.release();
    return DIM_SUCCESS;
}

} // namespace
} // namespace dimgpu

using namespace dimgpu;

extern "C" dim_status dim_csr5_from_csr_device(uint32_t rows, uint32_t cols, uint64_t nnz, const uint32_t* row_ptr,
                                               const uint32_t* col_idx, const double* vals, const dim_csr5_opts* opts,
                                               void* stream, dim_csr5** out) {
    if (!out)
        return fail(DIM_INVALID_ARGUMENT, "out is null");
    *out = nullptr;
    if (!row_ptr || (nnz && (!col_idx || !vals)))
        return fail(DIM_INVALID_ARGUMENT, "null CSR array");
    if (rows >= kDirty)
        return fail(DIM_INVALID_ARGUMENT, "row count must be below 2^31");
    if (nnz >= (uint64_t{1} << 32))
        return fail(DIM_INVALID_ARGUMENT, "non-zero count must fit in 32 bits");
    const uint32_t sigma = opts && opts->sigma ? opts->sigma : 16;
    if (!sigma_supported(sigma))
        return fail(DIM_INVALID_ARGUMENT, "unsupported sigma");
    const bool keep_f32 = opts && (opts->flags & DIM_CSR5_KEEP_F32);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (sigma <= 16)
        return convert<uint16_t>(rows, cols, nnz, row_ptr, col_idx, vals, sigma, keep_f32, s, out);
    return convert<uint32_t>(rows, cols, nnz, row_ptr, col_idx, vals, sigma, keep_f32, s, out);
}
