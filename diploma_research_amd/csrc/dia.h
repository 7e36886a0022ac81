// The diagonal form of a matrix on the device and its products (dia.hip).
#pragma once

#include "kernels.h"
#include "dim_internal.h"

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dimgpu {

// Values by diagonal: element (row, row + off[d]) at v64[d * ld + row], 0 where
// the row has no such element; meta as HostFormat::dia_meta. nd is 0 when the
// matrix has no diagonal form.
struct DiaForm {
    uint32_t nd = 0; // 3, 5, 7 or 9
    uint32_t rows = 0, cols = 0;
    uint64_t ld = 0;
    int32_t off[kDiaMax] = {};
    // batches: each system's offsets (kDiaMax of them), off unused; a system's
    // rows follow one another as in the batch's vectors
    const int32_t* sys_off = nullptr;
    double* v64 = nullptr;
    float* v32 = nullptr;
    uint16_t* meta = nullptr;
    // plain products use it: the matrix keeps column codes or could, and no
    // row spans three lanes (the summation order is then the tile kernels')
    bool products = false;
};

// y = A x.
hipError_t launch_dia_spmv(const DiaForm& D, bool f32, const void* x, void* y, hipStream_t stream);

// Y = A X for k columns. ldx = ldy = 0: row-major n x k blocks; otherwise
// column-major with those leading dimensions.
hipError_t launch_dia_spmm(const DiaForm& D, bool f32, int k, const void* X, void* Y, uint64_t ldx, uint64_t ldy,
                           hipStream_t stream);

} // namespace dimgpu
