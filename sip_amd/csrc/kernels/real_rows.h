// Real-transform rows, single LDS plane: MODE 1 = R2C (half-length C2C + pair post-process), MODE 2 =
// C2R (pair pre-process + half-length C2C). W: waves per SIMD the register budget is held to (0 = the
// compiler's choice). Threads and radices per half length: real_shapes.py.
#pragma once
#include "stockham_device.h"

namespace sip {

template <int W, int L, int T, int S, int MODE, int... Rs>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(W))) void stockham_real_rows_kernel(const StockhamArgs a)
{
    extern __shared__ float lds[];
    if constexpr (MODE == 1)
        split_rows<L, T, S, true, Rs...>(a, lds, tile_index(a));
    else
        split_rows_c2r<L, T, S, Rs...>(a, lds, tile_index(a));
}

}  // namespace sip
