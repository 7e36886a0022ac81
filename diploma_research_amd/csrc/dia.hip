// Products of matrices kept by diagonals (stencil operators).
//
// The tile kernels (spmv_impl.h) decode every element's row and column and
// gather x element by element; they are bound by the L2 latency of those
// gathers. A matrix whose elements fill a few diagonals needs neither: with
// one row per lane, step d reads 64 consecutive values of diagonal d and 64
// consecutive x entries, every load of a row is independent of every other,
// and the kernel is bound by the stream of values.
#include "dia.h"
#include "spmv_impl.h"

namespace dimgpu {

namespace {

using detail::xcd_remap;

struct DiaArgs {
    const uint16_t* meta;
    uint64_t ld;
    uint32_t rows, cols;
    int32_t off[kDiaMax];
};

// Sum of one row's products, diagonal by diagonal: the part of the row in its
// first lane of the tile layout, then the part in the next lane, then their
// sum, each part a chain of fused multiply-adds from 0 (the tile kernels'
// order). Places without an element are skipped, so that x there, finite or
// not, has no effect.
template<typename V, int ND>
__device__ __forceinline__ V row_sum(const V (&v)[ND], const V (&xv)[ND], uint32_t meta) {
    const uint32_t split = meta >> kDiaSplitShift;
    V first = V(0), acc = V(0);
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const bool cut = split == static_cast<uint32_t>(d);
        first = cut ? acc : first;
        acc = cut ? V(0) : acc;
        const V t = fma(v[d], xv[d], acc);
        acc = ((meta >> d) & 1u) ? t : acc;
    }
    return first + acc;
}

// Row + offset, held to the column range: a missing element's place reads a
// valid x entry that is not used.
__device__ __forceinline__ uint32_t dia_col(uint32_t row, int32_t off, uint32_t cols) {
    const int c = static_cast<int>(row) + off;
    return static_cast<uint32_t>(max(0, min(c, static_cast<int>(cols) - 1)));
}

// Load of a value that a product reads once (NT: see stream_values).
template<bool NT, typename V>
__device__ __forceinline__ V load_value(const V* p) {
    if constexpr (NT)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

// One row per thread: two or four rows of a thread in flight, or two
// neighbouring rows with 16-byte loads, are slower (7 diagonals, FP64, 128^3
// rows: 26.5 us, against 29.4, 31.8 and 27.6 us; the tile kernel with column
// codes 35.4 us). Bound by the stream of values: 155 MB at 5.9 TB/s. The
// blocks of one XCD take one contiguous eighth of the rows, so that the x
// entries of neighbouring rows meet in its L2 (without: 31.0 us).
template<typename V, int ND, bool NT>
__global__ __launch_bounds__(256) void k_dia_spmv(DiaArgs a, const V* __restrict__ vals, const V* __restrict__ x,
                                                  V* __restrict__ y) {
    const uint32_t b0 = xcd_remap(blockIdx.x, gridDim.x) * 256u;
    const uint32_t left = a.rows - b0; // rows from b0 on (at least 1)
    const uint32_t i = min(threadIdx.x, left - 1u);
    const uint32_t meta = (a.meta + b0)[i];
    V v[ND], xv[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        v[d] = load_value<NT>(vals + d * a.ld + b0 + i);
        xv[d] = *reinterpret_cast<const V*>(reinterpret_cast<const char*>(x) +
                                            dia_col(b0 + i, a.off[d], a.cols) * static_cast<uint32_t>(sizeof(V)));
    }
    const V s = row_sum<V, ND>(v, xv, meta);
    if (threadIdx.x < left)
        (y + b0)[i] = s;
}

// Column-major blocks: one row per lane, its values kept in registers while
// the columns go by. One column at a time: the wavefronts of an XCD then work
// on the same columns of neighbouring rows, and the x entries they share stay
// in its L2.
template<typename V, int ND>
__global__ __launch_bounds__(256) void k_dia_spmm_cols(DiaArgs a, int k, uint64_t ldx, uint64_t ldy,
                                                       const V* __restrict__ vals, const V* __restrict__ X,
                                                       V* __restrict__ Y) {
    const uint32_t b0 = xcd_remap(blockIdx.x, gridDim.x) * 256u;
    const uint32_t left = a.rows - b0;
    const uint32_t i = min(threadIdx.x, left - 1u);
    const uint32_t meta = (a.meta + b0)[i];
    V v[ND];
    uint32_t at[ND]; // byte offset of x in its column
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        v[d] = (vals + d * a.ld + b0)[i];
        at[d] = dia_col(b0 + i, a.off[d], a.cols) * static_cast<uint32_t>(sizeof(V));
    }
    for (int j = 0; j < k; ++j) {
        const char* xj = reinterpret_cast<const char*>(X + static_cast<uint64_t>(j) * ldx);
        V xv[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d)
            xv[d] = *reinterpret_cast<const V*>(xj + at[d]);
        const V s = row_sum<V, ND>(v, xv, meta);
        if (threadIdx.x < left)
            (Y + static_cast<uint64_t>(j) * ldy + b0)[i] = s;
    }
}

// Row-major blocks: L lanes per row, each with W neighbouring columns in one
// load (the last lane's columns end at the row's end, so where W does not
// divide k two lanes compute the same columns and write the same bits). A
// wavefront so reads and writes consecutive memory, and a row's x entries for
// all columns come with one line. The loads need no more than an element's
// alignment. No transposes around it: 8 FP64 columns of 112^3 rows, three
// matrices and blocks in turn, take 71 us (61 where one stays in the Infinity
// Cache), where the tile kernel between two transposes took 196.
// One column per lane: 90 us, twice the loads.
template<typename V, int ND, int W>
__global__ __launch_bounds__(256) void k_dia_spmm_rows(DiaArgs a, uint32_t k, uint32_t L, uint32_t inv_L,
                                                       uint32_t rows_per, const V* __restrict__ vals,
                                                       const V* __restrict__ X, V* __restrict__ Y) {
    typedef V VW __attribute__((ext_vector_type(W), aligned(sizeof(V))));
    const uint64_t b0 = static_cast<uint64_t>(xcd_remap(blockIdx.x, gridDim.x)) * rows_per;
    const uint32_t work = min(rows_per, a.rows - static_cast<uint32_t>(b0)) * L;
    const uint32_t e = min(threadIdx.x, work - 1u);
    const uint32_t i = (e * inv_L) >> 16; // e / L
    const uint32_t c = min((e - i * L) * W, k - W);
    const uint32_t meta = (a.meta + b0)[i];
    V v[ND];
    VW xv[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        v[d] = (vals + d * a.ld + b0)[i];
        const uint64_t at = static_cast<uint64_t>(dia_col(static_cast<uint32_t>(b0) + i, a.off[d], a.cols)) * k + c;
        xv[d] = *reinterpret_cast<const VW*>(X + at);
    }
    VW s;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        V xw[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d)
            xw[d] = xv[d][w];
        s[w] = row_sum<V, ND>(v, xw, meta);
    }
    if (threadIdx.x < work)
        *reinterpret_cast<VW*>(Y + b0 * k + i * k + c) = s;
}

DiaArgs make_args(const DiaForm& D) {
    DiaArgs a;
    a.meta = D.meta;
    a.ld = D.ld;
    a.rows = D.rows;
    a.cols = D.cols;
    for (uint32_t d = 0; d < kDiaMax; ++d)
        a.off[d] = D.off[d];
    return a;
}

// F<ND>::run for the compiled diagonal counts
template<typename F>
hipError_t by_diagonals(uint32_t nd, F&& f) {
    switch (nd) {
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 7: f(std::integral_constant<int, 7>{}); break;
        case 9: f(std::integral_constant<int, 9>{}); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template<typename V>
const V* values_of(const DiaForm& D) {
    if constexpr (std::is_same<V, float>::value)
        return D.v32;
    else
        return D.v64;
}

// The values of a single-vector product are read non-temporally when its
// streams (values, row words, x and y) take more than half of the 256 MB
// Infinity Cache, so that they do not push x out of L2 and two such matrices
// in turn do not evict each other. 7 diagonals, FP64, 128^3 rows (155 MB): 26.5
// us non-temporal, and with ordinary loads 20.1 us where one matrix is
// multiplied over and over but 32.2 us for three in turn: the line is drawn for
// programs that touch other data between two products, and costs those that do
// nothing else 6 us. FP32, 114^3 (56 MB): 9.0-9.9 against 8.6 us, so smaller
// products use ordinary loads. Products of several columns always do: their
// values are the smaller part. 8 FP64 columns, ordinary and non-temporal values:
// 112^3 rows, three matrices in turn 73.4 and 72.1 us, one over and over 61.5 and
// 66.5; 64^3 in turn 12.0 and 14.7; 160^3 in turn 207.6 and 205.1.
template<typename V>
bool stream_values(const DiaForm& D) {
    const uint64_t row = (uint64_t{D.nd} + 2) * sizeof(V) + sizeof(uint16_t);
    return row * D.rows > (uint64_t{128} << 20);
}

template<typename V>
hipError_t spmv(const DiaForm& D, const void* x, void* y, hipStream_t st) {
    const DiaArgs a = make_args(D);
    const dim3 grid((D.rows + 255) / 256), block(256);
    return by_diagonals(D.nd, [&](auto nd) {
        constexpr int ND = decltype(nd)::value;
        if (stream_values<V>(D))
            hipLaunchKernelGGL((k_dia_spmv<V, ND, true>), grid, block, 0, st, a, values_of<V>(D),
                               static_cast<const V*>(x), static_cast<V*>(y));
        else
            hipLaunchKernelGGL((k_dia_spmv<V, ND, false>), grid, block, 0, st, a, values_of<V>(D),
                               static_cast<const V*>(x), static_cast<V*>(y));
    });
}

template<typename V, int W>
hipError_t spmm_rows(const DiaForm& D, int k, const void* X, void* Y, hipStream_t st) {
    const DiaArgs a = make_args(D);
    const uint32_t uk = static_cast<uint32_t>(k), L = (uk + W - 1) / W, rows_per = 256 / L;
    const uint32_t inv_L = (65536 + L - 1) / L; // (e * inv_L) >> 16 == e / L for e < 256, L <= 16
    const dim3 grid((D.rows + rows_per - 1) / rows_per), block(256);
    return by_diagonals(D.nd, [&](auto nd) {
        constexpr int ND = decltype(nd)::value;
        hipLaunchKernelGGL((k_dia_spmm_rows<V, ND, W>), grid, block, 0, st, a, uk, L, inv_L, rows_per,
                           values_of<V>(D), static_cast<const V*>(X), static_cast<V*>(Y));
    });
}

template<typename V>
hipError_t spmm(const DiaForm& D, int k, const void* X, void* Y, uint64_t ldx, uint64_t ldy, hipStream_t st) {
    if (ldx) {
        const DiaArgs a = make_args(D);
        const dim3 grid((D.rows + 255) / 256), block(256);
            return by_diagonals(D.nd, [&](auto nd) {
            constexpr int ND = decltype(nd)::value;
            hipLaunchKernelGGL((k_dia_spmm_cols<V, ND>), grid, block, 0, st, a, k, ldx, ldy, values_of<V>(D),
                               static_cast<const V*>(X), static_cast<V*>(Y));
        });
    }
    if (k == 1) // a row is one element either way
        return spmv<V>(D, X, Y, st);
    constexpr int kWide = 16 / static_cast<int>(sizeof(V));
    return k >= kWide ? spmm_rows<V, kWide>(D, k, X, Y, st) : spmm_rows<V, 2>(D, k, X, Y, st);
}

} // namespace

hipError_t launch_dia_spmv(const DiaForm& D, bool f32, const void* x, void* y, hipStream_t stream) {
    return f32 ? spmv<float>(D, x, y, stream) : spmv<double>(D, x, y, stream);
}

hipError_t launch_dia_spmm(const DiaForm& D, bool f32, int k, const void* X, void* Y, uint64_t ldx, uint64_t ldy,
                           hipStream_t stream) {
    if (k < 1 || k > kMaxK)
        return hipErrorInvalidValue;
    return f32 ? spmm<float>(D, k, X, Y, ldx, ldy, stream) : spmm<double>(D, k, X, Y, ldx, ldy, stream);
}

} // namespace dimgpu
