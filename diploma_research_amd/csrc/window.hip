// Single-vector products of matrices whose elements lie within a band.
//
// The tile kernel (spmv_impl.h) gathers x element by element from L1 and L2:
// every lane of a gather takes a cycle of the CU's address unit and most of
// them a line of L2 (8.2M elements of uneven rows within a band of 8000
// columns, FP64: 0.6 GB from L2 for 66 MB of values). Here a workgroup of 16
// wavefronts takes 16 or more neighbouring tiles and first copies the part of x
// that their columns span, its window, into LDS; the gathers are then LDS
// reads, and what is left is the stream of the matrix, read one tile ahead.
// That product: 54.4 us by the tile kernel, 32.6 us here (112 MB, 3.4 TB/s).
//
// A row belongs to the workgroup in which it starts. Inside the workgroup its
// parts meet in LDS; what lies in the next workgroup's first tile is added by
// the row's owner, and matrices with rows that reach further keep the tile
// kernel, as do those whose windows do not fit.
#include "window.h"
#include "spmv_impl.h"

#include <algorithm>

namespace dimgpu {

namespace {

using detail::DescWord;
using detail::dpp_val;
using detail::kDppWaveShr1;
using detail::lane_value;
using detail::sload;
using detail::sload_flag;
using detail::wave_incl_scan;
using detail::wave_seg_scan;
using detail::xcd_remap;

constexpr int kWaves = static_cast<int>(kWindowGroup);
constexpr int kThreads = 64 * kWaves;
constexpr int kStageRows = 256; // row sums of a tile that a wavefront keeps in LDS
constexpr uint32_t kLdsBytes = 160 * 1024;
constexpr uint32_t kStaticLds = 1024; // what the kernels keep besides

struct Args {
    const uint32_t* tile_ptr;
    const void* bit_flag;
    const uint8_t* tile_flags;
    const uint32_t* tdo_ptr;
    const uint32_t* tdo;
    const uint32_t* col_idx;
    const uint32_t* empty_rows;
    const uint32_t* span;
    uint64_t nnz;
    uint32_t tiles, n_empty;
    WindowShape S;
};

// Bound by the stream of the matrix and, with few tiles per wavefront, by the
// first tile's way through. One workgroup per CU, 16 wavefronts of at most 128
// VGPRs: a tile's values and columns are 48 of them at sigma 16 in FP64, so each
// is loaded for the next tile as soon as it has been used. (The loads are there
// whether or not a tile follows: one step loop for both, as two loops, one of
// them without loads, kept the arrays in scratch memory: 51.4 us.)
template<typename V, int SIGMA>
__global__ __launch_bounds__(kThreads) void k_window_spmv(Args a, const V* __restrict__ vals,
                                                          const V* __restrict__ x, V* __restrict__ y) {
    using W = typename DescWord<SIGMA>::type;
    extern __shared__ double lds[];
    __shared__ V head_s[kWaves], tail_s[kWaves], look_s;
    __shared__ uint32_t row_s[kWaves];
    __shared__ int start_s[kWaves];
    const int lane = threadIdx.x & 63;
    const uint32_t ulane = static_cast<uint32_t>(lane);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t tb = b * (kWindowGroup * a.S.per), te = min(tb + kWindowGroup * a.S.per, a.tiles);
    const uint32_t t0 = min(tb + wave * a.S.per, te), t1 = min(t0 + a.S.per, te);
    uint32_t lo, w;
    detail::window_of(a.span, a.tiles, a.S, b, &lo, &w);
    V* win = reinterpret_cast<V*>(lds);
    V* stage = win + ((a.S.width + 2u) & ~1u) + wave * kStageRows;
    const W* __restrict__ flags = static_cast<const W*>(a.bit_flag);

    // ---- the window, the first tile, the next workgroup's part of the last row
    constexpr int U = 8;
    V part[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
        part[u] = (x + lo)[min(u * kThreads + threadIdx.x, w - 1u)];
    V v[SIGMA];
    uint32_t col[SIGMA], bits = 0, tpw = 0, tdo_at = 0;
    if (t0 < t1) {
        const size_t base = static_cast<size_t>(t0) * 64;
        bits = (flags + base)[ulane];
        tpw = sload(a.tile_ptr + t0);
        tdo_at = sload(a.tdo_ptr + t0);
#pragma unroll
        for (int r = 0; r < SIGMA; ++r)
            col[r] = __builtin_nontemporal_load(a.col_idx + base * SIGMA + r * 64 + ulane);
#pragma unroll
        for (int r = 0; r < SIGMA; ++r)
            v[r] = __builtin_nontemporal_load(vals + base * SIGMA + r * 64 + ulane);
    }
    const bool looks = wave == kWaves - 1 && te < a.tiles && !(sload_flag(a.tile_flags + te) & kStartsRow);
    uint32_t ahead = 0;
    if (looks)
        ahead = (flags + static_cast<size_t>(te) * 64)[ulane];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t i = u * kThreads + threadIdx.x;
        if (i < w)
            win[i] = part[u];
    }
    for (uint32_t i0 = U * kThreads; i0 < w; i0 += U * kThreads) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            part[u] = (x + lo)[min(i0 + u * kThreads + threadIdx.x, w - 1u)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + u * kThreads + threadIdx.x;
            if (i < w)
                win[i] = part[u];
        }
    }
    if (threadIdx.x == 0)
        win[w] = V(0); // (what the padding of the last tile reads)
    if (wave == kWaves - 1) {
        V s = V(0);
        if (looks) {
            // the elements before the tile's first row start, in CSR order
            const int ls = __ffsll(static_cast<long long>(__ballot(ahead != 0))) - 1;
            const int rs = __ffs(__builtin_amdgcn_readlane(static_cast<int>(ahead), ls)) - 1;
            const uint32_t n = static_cast<uint32_t>(ls * SIGMA + rs);
            const size_t base = static_cast<size_t>(te) * (64 * SIGMA);
            for (uint32_t i = ulane; i < n; i += 64) {
                const size_t at = base + (i % SIGMA) * 64 + i / SIGMA;
                s = fma(vals[at], x[a.col_idx[at]], s);
            }
            s = detail::wave_sum(s);
        }
        if (lane == 0)
            look_s = s;
    }
    __syncthreads();

    // ---- the tiles
    V carry = V(0);       // the open row's sum so far
    uint32_t row = 0;     // and the row, once one has started in these tiles
    bool started = false;
    for (uint32_t t = t0; t < t1; ++t) {
        const uint32_t my_bits = bits;
        const uint32_t row0 = tpw & ~kDirty;
        const uint32_t* off = (tpw & kDirty) ? a.tdo + tdo_at : nullptr;
        const int nb = __popc(my_bits);
        const int incl = wave_incl_scan(nb, lane);
        const int first = incl - nb;             // row starts of the lanes below
        const int n = lane_value(incl, 63);      // and of the tile
        const uint64_t who = __ballot(nb > 0);
        // start k of the tile begins segment k + s_lo (segment 0 lies in row0)
        const int s_lo = lane_value(static_cast<int>(my_bits & 1u), 0) ? 0 : 1;
        // (clean tiles: segment k lies in row0 + k)
        const bool staged = n <= kStageRows;
        if (t + 1 == a.tiles) {
            const uint32_t left = static_cast<uint32_t>(a.nnz - static_cast<uint64_t>(t) * (64 * SIGMA));
#pragma unroll
            for (int r = 0; r < SIGMA; ++r)
                col[r] = ulane * SIGMA + r < left ? col[r] : 0xffffffffu;
        }
        V cur = V(0), red = V(0);
        bool has = false;
        int k = first - 1; // the start that the running sum belongs to
        // The next tile's loads follow each step's use; after the last tile
        // they re-read one line a step of this one.
        const bool more = t + 1 < t1;
        const uint32_t tn = more ? t + 1 : t;
        const uint32_t ln = more ? ulane : 0u;
        const W* nf = flags + static_cast<size_t>(tn) * 64;
        const uint32_t* nc = a.col_idx + static_cast<size_t>(tn) * (64 * SIGMA);
        const V* nv = vals + static_cast<size_t>(tn) * (64 * SIGMA);
        bits = nf[ln];
        tpw = sload(a.tile_ptr + tn);
        tdo_at = sload(a.tdo_ptr + tn);
#pragma unroll
        for (int r = 0; r < SIGMA; ++r) {
            const V xv = win[min(col[r] - lo, w)];
            col[r] = __builtin_nontemporal_load(nc + r * 64 + ln);
            const bool starts = (my_bits >> r) & 1u;
            if (starts && has && staged)
                stage[k] = cur;
            if (!staged) { // wave-uniform
                if (starts && has)
                    y[row0 + (off ? off[k + s_lo] : static_cast<uint32_t>(k + s_lo))] = cur;
            }
            red = starts && !has ? cur : red;
            k += starts ? 1 : 0;
            has = has || starts;
            cur = fma(v[r], xv, starts ? V(0) : cur);
            v[r] = __builtin_nontemporal_load(nv + r * 64 + ln);
        }

        // A lane in which a row starts closes the row left open below it: the
        // trailing sum of the last such lane and the leading sums in between.
        const V trail = has ? cur : V(0);
        V A[1] = {has ? red : cur};
        V below = V(0);
        if (who == ~0ull) {
            below = dpp_val<kDppWaveShr1, 0xf>(trail);
        } else {
            int f = lane == 0 ? 1 : static_cast<int>((who >> (lane - 1)) & 1ull);
            wave_seg_scan<V, 1>(A, f, 1);
            const uint64_t under = who & ((1ull << lane) - 1ull);
            const V got = __shfl(trail, under ? 63 - __clzll(under) : 0, 64);
            below = under ? got : V(0);
        }
        const V tot = below + A[0];
        if (nb > 0 && first > 0) {
            if (staged)
                stage[first - 1] = tot;
            else
                y[row0 + (off ? off[first - 1 + s_lo] : static_cast<uint32_t>(first - 1 + s_lo))] = tot;
        }
        if (n == 0) { // the whole tile continues the open row
            carry = carry + lane_value(A[0], 63);
        } else {
            const int f0 = __ffsll(static_cast<long long>(who)) - 1, l0 = 63 - __clzll(who);
            const V closed = carry + lane_value(tot, f0);
            if (lane == 0) {
                if (started)
                    y[row] = closed;
                else
                    head_s[wave] = closed;
            }
            started = true;
            const V last = lane_value(trail, l0);
            carry = l0 == 63 ? last : last + lane_value(A[0], 63);
            row = row0 + (off ? off[n - 1 + s_lo] : static_cast<uint32_t>(n - 1 + s_lo));
            if (staged) {
                // the wave barriers keep the compiler from moving these LDS
                // accesses across one another's; a wavefront's run in order
                __builtin_amdgcn_wave_barrier();
                for (int i = lane; i < n - 1; i += 64)
                    y[row0 + (off ? off[i + s_lo] : static_cast<uint32_t>(i + s_lo))] = stage[i];
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    for (uint32_t i = b * kThreads + threadIdx.x; i < a.n_empty; i += gridDim.x * kThreads)
        y[a.empty_rows[i]] = V(0);

    // ---- the rows that cross wavefronts
    if (lane == 0) {
        start_s[wave] = started ? 1 : 0;
        tail_s[wave] = carry;
        row_s[wave] = row;
        if (!started)
            head_s[wave] = carry;
    }
    __syncthreads();
    if (threadIdx.x < kWaves && start_s[threadIdx.x]) {
        V s = tail_s[threadIdx.x];
        int u = static_cast<int>(threadIdx.x) + 1;
        for (; u < kWaves; ++u) {
            s = s + head_s[u];
            if (start_s[u])
                break;
        }
        if (u == kWaves)
            s = s + look_s;
        y[row_s[threadIdx.x]] = s;
    }
}

// Column span of every 16 tiles, one workgroup for each.
__global__ __launch_bounds__(256) void k_spans(uint32_t sigma, uint32_t tiles, uint64_t nnz,
                                               const uint32_t* __restrict__ col_idx, uint32_t* __restrict__ span) {
    __shared__ uint32_t l_s[4], h_s[4];
    const uint32_t lane = threadIdx.x & 63, tile = 64 * sigma;
    uint32_t l = 0xffffffffu, h = 0;
    for (uint32_t q = threadIdx.x >> 6; q < kWindowGroup; q += 4) {
        const uint32_t t = blockIdx.x * kWindowGroup + q;
        if (t >= tiles)
            break;
        const uint64_t base = static_cast<uint64_t>(t) * tile, left = nnz - base;
        for (uint32_t r = 0; r < sigma; ++r)
            if (lane * sigma + r < left) { // (the padding is no element)
                const uint32_t c = col_idx[base + r * 64 + lane];
                l = min(l, c);
                h = max(h, c);
            }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        l = min(l, static_cast<uint32_t>(__shfl_xor(static_cast<int>(l), d, 64)));
        h = max(h, static_cast<uint32_t>(__shfl_xor(static_cast<int>(h), d, 64)));
    }
    if ((threadIdx.x & 63) == 0) {
        l_s[threadIdx.x >> 6] = l;
        h_s[threadIdx.x >> 6] = h;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        span[2 * blockIdx.x] = min(min(l_s[0], l_s[1]), min(l_s[2], l_s[3]));
        span[2 * blockIdx.x + 1] = max(max(h_s[0], h_s[1]), max(h_s[2], h_s[3]));
    }
}

template<typename V>
uint32_t spmv_lds(uint32_t width) {
    return (((width + 2u) & ~1u) + kWaves * kStageRows) * static_cast<uint32_t>(sizeof(V));
}

template<typename V, int SIGMA>
hipError_t launch(const Args& a, uint32_t blocks, const V* vals, const V* x, V* y, hipStream_t s) {
    const uint32_t bytes = spmv_lds<V>(a.S.width);
    const void* f = reinterpret_cast<const void*>(&k_window_spmv<V, SIGMA>);
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL((k_window_spmv<V, SIGMA>), dim3(blocks), dim3(kThreads), bytes, s, a, vals, x, y);
    return hipGetLastError();
}

template<typename V>
hipError_t spmv(const DevFormat& A, const WindowShape& S, const uint32_t* span, const V* vals, const void* x, void* y,
                hipStream_t s) {
    Args a;
    a.tile_ptr = A.tile_ptr;
    a.bit_flag = A.bit_flag;
    a.tile_flags = A.tile_flags;
    a.tdo_ptr = A.tile_desc_offset_ptr;
    a.tdo = A.tile_desc_offset;
    a.col_idx = A.col_idx;
    a.empty_rows = A.empty_rows;
    a.span = span;
    a.nnz = A.nnz;
    a.tiles = A.tiles;
    a.n_empty = A.n_empty;
    a.S = S;
    const V* xv = static_cast<const V*>(x);
    V* yv = static_cast<V*>(y);
    switch (A.sigma) {
#define DIM_W(S_)                                                                                                     \
    case S_:                                                                                                          \
        return launch<V, S_>(a, S.blocks, vals, xv, yv, s);
        DIM_W(4) DIM_W(5) DIM_W(6) DIM_W(7) DIM_W(8) DIM_W(10) DIM_W(12) DIM_W(14) DIM_W(16)
#undef DIM_W
        default: return hipErrorInvalidValue;
    }
}

} // namespace

// The largest window where a wavefront has `per` tiles.
static uint32_t widest(const std::vector<uint32_t>& span, uint32_t groups, uint32_t per) {
    uint32_t width = 0;
    for (uint32_t g = 0; g < groups; g += per) {
        uint32_t l = 0xffffffffu, h = 0;
        for (uint32_t i = g; i < std::min(g + per, groups); ++i) {
            l = std::min(l, span[2 * i]);
            h = std::max(h, span[2 * i + 1]);
        }
        width = std::max(width, h - l + 1);
    }
    return width;
}

// As many tiles per wavefront as give every CU one workgroup, or fewer: those
// whose window is at most `most` entries and `times` the workgroup's elements
// (copying a wider one moves more than gathering would).
static WindowShape cut(uint32_t tiles, uint32_t sigma, const std::vector<uint32_t>& span, uint64_t most,
                       uint32_t times) {
    WindowShape s;
    if (sigma > kWindowMaxSigma || tiles < kWindowMinTiles)
        return s;
    const uint32_t groups = (tiles + kWindowGroup - 1) / kWindowGroup;
    for (uint32_t per = std::min((groups + 255) / 256, kWindowMaxPer); per; --per) {
        const uint32_t width = widest(span, groups, per);
        if (width <= most && width <= times * kWindowGroup * 64 * sigma * per) {
            s.per = per;
            s.width = width;
            s.blocks = (groups + per - 1) / per;
            break;
        }
    }
    return s;
}

WindowShape window_shape(const DevFormat& A, const std::vector<uint32_t>& span,
                         const std::vector<uint8_t>& tile_flags, size_t vb) {
    const uint32_t tiles = A.tiles, sigma = A.sigma;
    const bool f64 = vb == sizeof(double);
    if (A.rows - A.n_empty > uint64_t{kWindowMaxStarts} * tiles || A.nnz < kWindowElements ||
        (f64 && tiles < kWindowMinTiles64))
        return {};
    const WindowShape s = cut(tiles, sigma, span, (kLdsBytes - kStaticLds) / vb - kWaves * kStageRows - 2, 2);
    const double each = double{kWindowGroup} * 64 * sigma * s.per; // elements of a workgroup
    const double past = s.width - each * A.cols / A.nnz;
    if (f64 && past < 0.4 * each && A.nnz < kWindowNarrowElements)
        return {};
    // every workgroup's first tile has a row start
    for (uint64_t t = 0; s.blocks && t < tiles; t += uint64_t{kWindowGroup} * s.per)
        if (!(tile_flags[t] & (kStartsRow | kMultiSeg)))
            return {};
    return s;
}

WindowShape window_sums_shape(uint32_t tiles, uint32_t sigma, const std::vector<uint32_t>& span) {
    return cut(tiles, sigma, span, (kLdsBytes - kStaticLds) / sizeof(double), 2);
}

hipError_t launch_spans(const DevFormat& A, uint32_t* span, hipStream_t stream) {
    if (A.tiles)
        hipLaunchKernelGGL(k_spans, dim3((A.tiles + kWindowGroup - 1) / kWindowGroup), dim3(256), 0, stream, A.sigma,
                           A.tiles, A.nnz, static_cast<const uint32_t*>(A.col_idx), span);
    return hipGetLastError();
}

hipError_t launch_window_spmv(const DevFormat& A, const WindowPlan& P, bool f32, const void* x, void* y,
                              hipStream_t stream) {
    return f32 ? spmv<float>(A, P.f32, P.span, A.vals32, x, y, stream)
               : spmv<double>(A, P.f64, P.span, A.vals64, x, y, stream);
}

} // namespace dimgpu
