// Kernels between the CSR order of the stored elements and the tile layout:
// new values, their diagonal form, and the sampled outer product.
//
// A lane's elements are consecutive in CSR order, so read or written where a
// lane needs them, a wavefront's accesses are sigma elements apart. They go
// through LDS instead (one region per wavefront, each lane's elements an odd
// number of words apart, so that both sides are free of bank conflicts), and
// memory sees consecutive elements only.
#include "handle.h"
#include "spmv_impl.h"

#include <algorithm>

namespace dimgpu {

namespace {

using detail::DescWord;
using detail::element_row;
using detail::wave_incl_scan;

// The tiles of a matrix, or of one system of a batch (blockIdx.y).
struct Tiles {
    uint32_t begin, end; // tiles
    uint64_t nnz0, nnz;  // its elements in CSR order
};

__device__ __forceinline__ Tiles tiles_of(const DevFormat& A, const SystemTiles* sys) {
    if (!sys)
        return {0, A.tiles, 0, A.nnz};
    const SystemTiles s = sys[blockIdx.y];
    return {s.tile0, s.tile1, s.nnz0, s.nnz};
}

// place of element e of a tile (CSR order within the tile) in its LDS region
template<int SIGMA>
__device__ __forceinline__ uint32_t staged(uint32_t e) {
    return (e / SIGMA) * (SIGMA | 1) + e % SIGMA;
}

// out[csr(e)] = scale * u[row(e)] * v[col(e)]
template<int SIGMA>
__global__ __launch_bounds__(256) void k_sampled_outer(DevFormat A, const SystemTiles* sys, double scale,
                                                       const double* __restrict__ u, const double* __restrict__ v,
                                                       double* __restrict__ out) {
    __shared__ double stage[4][64 * (SIGMA | 1)];
    const uint32_t lane = threadIdx.x & 63;
    const Tiles T = tiles_of(A, sys);
    const uint32_t t = T.begin + blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T.end)
        return; // wave-uniform
    double* s = stage[threadIdx.x >> 6];
    using W = typename DescWord<SIGMA>::type;
    const size_t base = static_cast<size_t>(t) * (64 * SIGMA);
    const uint64_t first = static_cast<uint64_t>(t - T.begin) * (64 * SIGMA); // the tile's first element
    const uint32_t left = static_cast<uint32_t>(T.nnz - first < 64 * SIGMA ? T.nnz - first : 64 * SIGMA);
    const uint32_t bits = static_cast<uint32_t>(static_cast<const W*>(A.bit_flag)[static_cast<size_t>(t) * 64 + lane]) |
                          (lane == 0 ? 1u : 0u);
    const uint32_t tpw = A.tile_ptr[t];
    const bool dirty = (tpw & kDirty) != 0;
    const uint32_t row0 = tpw & ~kDirty;
    const uint32_t* tdo = dirty ? A.tile_desc_offset + A.tile_desc_offset_ptr[t] : nullptr;
    const int nb = __popc(bits);
    const int y_off = wave_incl_scan(nb, static_cast<int>(lane)) - nb;
#pragma unroll
    for (int r = 0; r < SIGMA; ++r)
        if (lane * SIGMA + r < left) {
            const uint32_t row = element_row(bits, r, y_off, row0, dirty, tdo);
            s[lane * (SIGMA | 1) + r] = scale * u[row] * v[A.col_idx[base + r * 64 + lane]];
        }
    __builtin_amdgcn_wave_barrier(); // a wavefront's LDS accesses run in order
    double* o = out + T.nnz0 + first;
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const uint32_t e = r * 64 + lane;
        if (e < left)
            o[e] = s[staged<SIGMA>(e)];
    }
}

// Tile-layout values from CSR-order values (the same permutation as the
// conversion's transpose), in FP64 and, if kept, FP32; DIA: the diagonal form
// too. There a lane takes a row: its elements from LDS in CSR order, their
// diagonals from the row's word, so that a wavefront writes 64 neighbouring
// places of a diagonal at a time (7 diagonals, 10^6 rows, FP64 and FP32, sigma
// 16: 63 us; element by element from the tile layout, with the diagonal
// looked up by its column, 257; without the diagonal form 50).
template<int SIGMA, bool DIA>
__global__ __launch_bounds__(256) void k_set_values(DevFormat A, DiaForm D, const SystemTiles* sys,
                                                    const double* __restrict__ src) {
    __shared__ double stage[4][64 * (SIGMA | 1)];
    const uint32_t lane = threadIdx.x & 63;
    const Tiles T = tiles_of(A, sys);
    const uint32_t t = T.begin + blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T.end)
        return; // wave-uniform
    double* s = stage[threadIdx.x >> 6];
    const size_t base = static_cast<size_t>(t) * (64 * SIGMA);
    const uint64_t first = static_cast<uint64_t>(t - T.begin) * (64 * SIGMA);
    const uint32_t left = static_cast<uint32_t>(T.nnz - first < 64 * SIGMA ? T.nnz - first : 64 * SIGMA);
    const double* in = src + T.nnz0 + first;
    uint32_t flags = 0, row0 = 0;
    if constexpr (DIA) { // (in flight with the values)
        using W = typename DescWord<SIGMA>::type;
        flags = static_cast<const W*>(A.bit_flag)[static_cast<size_t>(t) * 64 + lane];
        row0 = A.tile_ptr[t] & ~kDirty; // a matrix kept by diagonals has no dirty tiles
    }
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const uint32_t e = r * 64 + lane;
        s[staged<SIGMA>(e)] = e < left ? in[e] : 0.0;
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const size_t pos = base + r * 64 + lane;
        const double a = s[lane * (SIGMA | 1) + r];
        A.vals64[pos] = a;
        if (A.vals32)
            A.vals32[pos] = static_cast<float>(a);
    }
    if constexpr (DIA) {
        __shared__ uint16_t starts[4][64 * SIGMA];
        uint16_t* start = starts[threadIdx.x >> 6];
        const uint32_t bits = flags | (lane == 0 ? 1u : 0u);
        const bool continues = (__ballot(flags & 1u) & 1ull) == 0ull; // the first element's row began in an earlier tile
        const int nb = __popc(bits);
        const int incl = wave_incl_scan(nb, static_cast<int>(lane));
        const uint32_t rows = static_cast<uint32_t>(detail::lane_value(incl, 63));
        uint32_t k = static_cast<uint32_t>(incl - nb);
#pragma unroll
        for (int r = 0; r < SIGMA; ++r)
            if ((bits >> r) & 1u)
                start[k++] = static_cast<uint16_t>(lane * SIGMA + r);
        __builtin_amdgcn_wave_barrier();
        for (uint32_t i = lane; i < rows; i += 64) {
            const uint32_t row = row0 + i;
            uint32_t at = start[i];
            const uint32_t end = i + 1 < rows ? start[i + 1] : left;
            const uint32_t held = D.meta[row] & ((1u << kDiaSplitShift) - 1u);
            // (of a row that began earlier, the last elements)
            uint32_t skip = i == 0 && continues ? static_cast<uint32_t>(__popc(held)) - (end - at) : 0u;
#pragma unroll
            for (uint32_t d = 0; d < kDiaMax; ++d)
                if ((held >> d) & 1u) {
                    if (skip) {
                        --skip;
                    } else if (at < end) { // (of a row that ends in the next tile, the first)
                        const double a = s[staged<SIGMA>(at++)];
                        D.v64[d * D.ld + row] = a;
                        if (D.v32)
                            D.v32[d * D.ld + row] = static_cast<float>(a);
                    }
                }
        }
    }
}

// Values of the diagonal form from the tile layout: one wavefront per tile,
// every element's diagonal found among the nd offsets.
template<int SIGMA>
__global__ __launch_bounds__(256) void k_dia_fill(DevFormat A, DiaForm D, const SystemTiles* sys) {
    const uint32_t lane = threadIdx.x & 63;
    const Tiles T = tiles_of(A, sys);
    const uint32_t t = T.begin + blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T.end)
        return;
    using W = typename DescWord<SIGMA>::type;
    const size_t base = static_cast<size_t>(t) * (64 * SIGMA);
    const uint64_t first = static_cast<uint64_t>(t - T.begin) * (64 * SIGMA);
    const uint32_t bits = static_cast<uint32_t>(static_cast<const W*>(A.bit_flag)[static_cast<size_t>(t) * 64 + lane]) |
                          (lane == 0 ? 1u : 0u);
    const uint32_t row0 = A.tile_ptr[t] & ~kDirty;
    const int nb = __popc(bits);
    const int y_off = wave_incl_scan(nb, static_cast<int>(lane)) - nb;
    int32_t off[kDiaMax];
    const int32_t* o = D.sys_off ? D.sys_off + blockIdx.y * kDiaMax : nullptr;
#pragma unroll
    for (uint32_t q = 0; q < kDiaMax; ++q)
        off[q] = o ? o[q] : D.off[q];
#pragma unroll
    for (int r = 0; r < SIGMA; ++r) {
        const size_t pos = base + r * 64 + lane;
        if (first + lane * SIGMA + r >= T.nnz)
            continue;
        const uint32_t row = element_row(bits, r, y_off, row0, false, nullptr);
        const int32_t diff = static_cast<int32_t>(A.col_idx[pos]) - static_cast<int32_t>(row);
        uint32_t d = D.nd;
#pragma unroll
        for (int q = kDiaMax - 1; q >= 0; --q)
            d = (static_cast<uint32_t>(q) < D.nd && off[q] == diff) ? static_cast<uint32_t>(q) : d;
        if (d < D.nd && row < D.rows) {
            D.v64[d * D.ld + row] = A.vals64[pos];
            if (D.v32)
                D.v32[d * D.ld + row] = A.vals32[pos];
        }
    }
}

// Calls f(grid, sys, dia) for the whole matrix: four tiles per block; a
// batch's systems along y (at most 65535 of them in one launch), each with as
// many blocks as the one with the most tiles needs.
template<typename F>
hipError_t over_tiles(const dim_csr5* h, F&& f) {
    if (!h->f.tiles)
        return hipSuccess;
    if (!h->sys_tab) {
        f(dim3((h->f.tiles + 3) / 4), static_cast<const SystemTiles*>(nullptr), h->dia);
        return hipGetLastError();
    }
    constexpr uint32_t kMaxY = 65535;
    for (uint32_t s0 = 0; s0 < h->n_systems; s0 += kMaxY) {
        const uint32_t s1 = std::min(h->n_systems, s0 + kMaxY);
        uint32_t most = 0;
        for (uint32_t s = s0; s < s1; ++s)
            most = std::max(most, h->sys_tile[s + 1] - h->sys_tile[s]);
        DiaForm D = h->dia;
        if (D.sys_off)
            D.sys_off += size_t{s0} * kDiaMax;
        if (most)
            f(dim3((most + 3) / 4, s1 - s0), static_cast<const SystemTiles*>(h->sys_tab + s0), D);
    }
    return hipGetLastError();
}

} // namespace

hipError_t launch_set_values(const dim_csr5* h, const double* vals_csr, hipStream_t stream) {
    return over_tiles(h, [&](dim3 grid, const SystemTiles* sys, const DiaForm& D) {
        switch (h->f.sigma) {
#define DIM_SV(S)                                                                                                     \
    case S:                                                                                                           \
        if (D.nd)                                                                                                     \
            hipLaunchKernelGGL((k_set_values<S, true>), grid, dim3(256), 0, stream, h->f, D, sys, vals_csr);          \
        else                                                                                                          \
            hipLaunchKernelGGL((k_set_values<S, false>), grid, dim3(256), 0, stream, h->f, D, sys, vals_csr);         \
        break;
            DIM_FOR_EACH_SIGMA(DIM_SV)
#undef DIM_SV
            default: break;
        }
    });
}

hipError_t launch_sampled_outer(const dim_csr5* h, double scale, const double* u, const double* v, double* out,
                                hipStream_t stream) {
    return over_tiles(h, [&](dim3 grid, const SystemTiles* sys, const DiaForm&) {
        switch (h->f.sigma) {
#define DIM_O(S)                                                                                                      \
    case S: hipLaunchKernelGGL((k_sampled_outer<S>), grid, dim3(256), 0, stream, h->f, sys, scale, u, v, out); break;
            DIM_FOR_EACH_SIGMA(DIM_O)
#undef DIM_O
            default: break;
        }
    });
}

hipError_t launch_dia_fill(const dim_csr5* h, hipStream_t stream) {
    return over_tiles(h, [&](dim3 grid, const SystemTiles* sys, const DiaForm& D) {
        switch (h->f.sigma) {
#define DIM_DIA_FILL(S)                                                                                               \
    case S: hipLaunchKernelGGL((k_dia_fill<S>), grid, dim3(256), 0, stream, h->f, D, sys); break;
            DIM_FOR_EACH_SIGMA(DIM_DIA_FILL)
#undef DIM_DIA_FILL
            default: break;
        }
    });
}

} // namespace dimgpu
