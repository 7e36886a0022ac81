// The dim_csr5 handle behind the C ABI, and error plumbing shared by the
// C ABI translation units.
#pragma once

#include "dia.h"
#include "dim_internal.h"
#include "kernels.h"
#include "resident.h"
#include "window.h"
#include "../../include/dim_gpu.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <string>
#include <vector>

namespace dimgpu {
struct CgCache;
void free_cg_cache(CgCache* c);
struct BatchCache;
void free_batch_cache(BatchCache* c);
// A system of a batch: tiles [tile0, tile1) and nnz elements from element nnz0
// of the CSR order on.
struct SystemTiles {
    uint32_t tile0, tile1;
    uint64_t nnz0, nnz;
};
// Where the products of y = A^T x go before they are summed (transpose.hip):
// workgroup b (tiles [b * per, (b + 1) * per)) writes its products of columns
// [bin << shift, (bin + 1) << shift) from place start[bin] + off[b * bins + bin] on.
struct TransposePlan {
    uint32_t shift = 0, bins = 0, per = 0, blocks = 0; // bins == 0: no plan
    uint32_t* off = nullptr;
    uint32_t* start = nullptr; // bins + 1
    void* prod = nullptr;      // a product per element, FP64-sized
    uint16_t* col = nullptr;   // and its column within the bin
    bool refused = false;      // the matrix keeps the atomics
    bool band = false;         // by windows (window.h) instead: prod holds their sums
};
} // namespace dimgpu

struct dim_csr5 {
    dimgpu::DevFormat f;
    dimgpu::Scratch s;
    int device = 0;
    uint32_t n_dirty = 0;
    uint64_t device_bytes = 0;
    std::vector<void*> allocations;
    void* block = nullptr; // the arrays of the format and the scratch (take_block)
    size_t block_bytes = 0;
    // block-diagonal batches: system i owns rows [sys_row[i], sys_row[i+1]) and
    // tiles [sys_tile[i], sys_tile[i+1])
    uint32_t n_systems = 1;
    std::vector<uint32_t> sys_row, sys_tile;
    std::vector<uint64_t> sys_nnz_csr;
    // chunks of system s in the chunk table: [sys_chunk[s], sys_chunk[s + 1])
    std::vector<uint32_t> sys_chunk;
    uint32_t* d_sys_chunk = nullptr;
    // batches: tiles and elements of each system, on the device (values.hip)
    dimgpu::SystemTiles* sys_tab = nullptr;
    std::vector<int32_t> sys_off; // batches kept by diagonals: dia.sys_off's entries
    uint64_t nnz_logical = 0; // stored elements (the format's nnz counts padding inside a batch)
    dimgpu::BoundaryInfo binfo; // host copy of the tile flags (f.binfo points here)
    dimgpu::DiaForm dia;        // stencil matrices: the values by diagonal (dia.h)
    dimgpu::WindowPlan win;     // matrices within a band (window.h)
    dimgpu::TransposePlan tplan; // made with the first transposed product
    dimgpu::ResidentTrial resident;
    // Column slices for plain products (capi.cpp): xs is the matrix whose
    // rows are the (column slice s, row i) pairs that hold elements, in the
    // order of s*rows + i. That stacked handle also owns the partial products
    // (ystack, one FP64-sized entry per stacked row), the bit map of the
    // pairs (present, bit s*rows + i) and the set bits before each word of
    // it (present_rank).
    dim_csr5* xs = nullptr;
    uint32_t xs_slices = 0;
    void* ystack = nullptr;
    uint32_t* present = nullptr;
    uint32_t* present_rank = nullptr;
    // column-major staging of row-major multi-RHS blocks (dim_csr5_spmm),
    // grown on demand
    void* mm_scratch = nullptr;
    size_t mm_bytes = 0;
    // device copies of host vectors for the host-pointer entry points
    // (dim_csr5_spmv_host, dim_cg_host): cols + rows FP64-sized entries,
    // allocated on first use
    void* host_stage = nullptr;
    // work buffers, pinned state and captured iteration graph of the last
    // dim_cg / dim_cg_multi solve, kept for the next solve of the same shape
    // (cg.hip); freed with the handle
    dimgpu::CgCache* cg_cache = nullptr;
    // the same for dim_cg_batched (batched.hip): block tables and buffers
    // sized by the batch, kept from the first batched solve
    dimgpu::BatchCache* batch_cache = nullptr;
};

namespace dimgpu {

void set_error(const std::string& msg);
dim_status fail(dim_status st, const std::string& msg);
dim_status hip_fail(hipError_t e, const char* what);

// The staging area of the host-pointer entry points: cols + rows entries of
// 8 bytes on the matrix's device (*x at the start, *y after it), allocated
// with the handle's arrays on first use.
dim_status stage_host_vectors(dim_csr5* A, char** x, char** y);

#define DIM_HIP_TRY(expr)                                                                                          \
    do {                                                                                                           \
        hipError_t e_ = (expr);                                                                                    \
        if (e_ != hipSuccess)                                                                                      \
            return ::dimgpu::hip_fail(e_, #expr);                                                                  \
    } while (0)

// The block of a handle's arrays. Allocating and freeing one of more than 64 MB
// costs 0.35 ms (a program that converts matrix after matrix spends more on it
// than on the conversion, and after a thousand of them 2 ms each), so the last
// one freed, if it is between 16 and 256 MiB, is kept for the next conversion:
// one block per device, freed when the next request does not fit it, when
// another takes its place, or when an allocation of the library finds no room.
// give_block() expects that no work on the block is in flight.
hipError_t take_block(size_t bytes, void** p, size_t* got);
void give_block(int device, void* p, size_t bytes);
// Frees the current device's kept block; false if there is none.
bool drop_block();

// hipMalloc that gives up the kept block before it fails.
inline hipError_t malloc_or_drop(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && drop_block()) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    return e;
}

// device allocation owned by the handle
template<typename T>
hipError_t dev_alloc(dim_csr5* h, T*& p, size_t count) {
    p = nullptr;
    const size_t bytes = count ? count * sizeof(T) : sizeof(T);
    void* q = nullptr;
    hipError_t e = malloc_or_drop(&q, bytes);
    if (e != hipSuccess)
        return e;
    h->allocations.push_back(q);
    h->device_bytes += bytes;
    p = static_cast<T*>(q);
    return hipSuccess;
}

// Several device arrays in one allocation, each on a 256-byte boundary: add()
// them, then commit() once.
class Arena {
  public:
    template<typename T>
    void add(T*& p, size_t count) {
        p = nullptr;
        parts_.push_back({[&p](char* at) { p = reinterpret_cast<T*>(at); }, bytes_});
        bytes_ += (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
    }
    void add_bytes(void*& p, size_t bytes) {
        p = nullptr;
        parts_.push_back({[&p](char* at) { p = at; }, bytes_});
        bytes_ += (std::max<size_t>(bytes, 1) + 255) / 256 * 256;
    }
    // the caller frees *base
    hipError_t commit(void** base) {
        *base = nullptr;
        const hipError_t e = malloc_or_drop(base, std::max<size_t>(bytes_, 1));
        if (e == hipSuccess)
            place(*base);
        return e;
    }
    // the handle frees it
    hipError_t commit(dim_csr5* h) {
        void* base = nullptr;
        const hipError_t e = commit(&base);
        if (e == hipSuccess) {
            h->allocations.push_back(base);
            h->device_bytes += bytes_;
        }
        return e;
    }
    // as the handle's block
    hipError_t commit_block(dim_csr5* h) {
        const hipError_t e = take_block(std::max<size_t>(bytes_, 1), &h->block, &h->block_bytes);
        if (e == hipSuccess) {
            place(h->block);
            h->device_bytes += bytes_;
        }
        return e;
    }

  private:
    void place(void* base) {
        for (const Part& p : parts_)
            p.set(static_cast<char*>(base) + p.at);
    }
    struct Part {
        std::function<void(char*)> set;
        size_t at;
    };
    std::vector<Part> parts_;
    size_t bytes_ = 0;
};

// The products' scratch for a matrix of T tiles (the queue must be cleared).
inline void add_scratch(Arena& a, Scratch& s, uint32_t T) {
    const size_t n = std::max<size_t>(T, 1);
    a.add_bytes(s.head, n * kMaxK * sizeof(double));
    a.add_bytes(s.tail, n * kMaxK * sizeof(double));
    a.add(s.chunk_flags, n);
    a.add(s.dot_chunk, n * kMaxK);
    a.add(s.dot_blk, ((n + 255) / 256) * kMaxK);
    a.add(s.queue, kQueueWords);
}

template<typename T>
hipError_t upload(dim_csr5* h, T*& p, const std::vector<T>& v) {
    hipError_t e = dev_alloc(h, p, v.size());
    if (e != hipSuccess)
        return e;
    if (!v.empty())
        e = hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
    return e;
}

// Uploads a host format into a fresh handle (allocates scratch too).
// plain_columns: leave out the column codes (products stream col_idx).
dim_status upload_format(const HostFormat& f, bool keep_f32, dim_csr5** out, bool plain_columns = false);

void free_handle(dim_csr5* h);

// The windows of a matrix on the device, from its spans on the host (window.h).
inline void shape_windows(dim_csr5* h, const std::vector<uint32_t>& span, const std::vector<uint8_t>& tile_flags) {
    h->win.f64 = window_shape(h->f, span, tile_flags, sizeof(double));
    h->win.sums = window_sums_shape(h->f.tiles, h->f.sigma, span);
    if (h->f.vals32)
        h->win.f32 = window_shape(h->f, span, tile_flags, sizeof(float));
}

// New values (CSR order) into the tile layout, FP64 and, if kept, FP32, and into
// the diagonal form.
hipError_t launch_set_values(const dim_csr5* h, const double* vals_csr, hipStream_t stream);

// out[e] = scale * u[row(e)] * v[col(e)] for every stored element e, in CSR order.
hipError_t launch_sampled_outer(const dim_csr5* h, double scale, const double* u, const double* v, double* out,
                                hipStream_t stream);

// y = A^T x (x has rows entries, y has cols entries). done: as launch_spmv.
dim_status launch_spmv_transpose(dim_csr5* h, bool f32, const void* x, void* y, hipStream_t stream,
                                 const int* done = nullptr);

// Writes the values of the diagonal form from the tile layout. The places
// without an element are not written: they must hold 0.
hipError_t launch_dia_fill(const dim_csr5* h, hipStream_t stream);

// Device memory of a diagonal form with nd diagonals (values zeroed, FP32 ones
// if the handle keeps them) and `meta` row words; hipSuccess with D.nd == 0 when
// there is no room.
hipError_t alloc_diagonals(dim_csr5* h, uint32_t nd, size_t meta, DiaForm& D);

} // namespace dimgpu

// For the tests, and so in no public header: how many resident launches of the
// handle's solves iterated since the last call; from the next launch but `from`
// on they fail as `fault` (ResidentTrial::Fault) says. The kernels end by
// themselves in every case.
extern "C" uint32_t dim_test_resident(dim_csr5* A, uint32_t fault, uint32_t from);
