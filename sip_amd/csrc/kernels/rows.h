// Contiguous C2C rows, single LDS plane (split_rows in stockham_device.h): the first pass reads and the
// last writes HBM, T threads per transform, F transforms per workgroup. W: waves per SIMD the register
// budget is held to (0 = the compiler's choice). Threads and radices per length: row_shapes.py.
#pragma once
#include "stockham_device.h"

namespace sip {

template <int W, int L, int T, int S, int... Rs>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(W))) void stockham_rows_kernel(const StockhamArgs a)
{
    extern __shared__ float lds[];
    split_rows<L, T, S, false, Rs...>(a, lds, tile_index(a));
}

}  // namespace sip
