// Rows in, columns out (split_rows_cols in stockham_device.h): the second stage of a four-step split.
// W: waves per SIMD the register budget is held to (0 = the compiler's choice): 1000 points as 50 threads of
// 10 x 10 x 10 within 64 registers, two 800-thread tiles per CU, 3.61 TB/s; as the leaf's 20 x 10 x 5 2.89.
#pragma once
#include "stockham_device.h"

namespace sip {

template <int W, int L, int T, int S, int... Rs>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(W))) void stockham_rc_kernel(const StockhamArgs a)
{
    extern __shared__ float lds[];
    split_rows_cols<L, T, S, Rs...>(a, lds, tile_index(a));
}

}  // namespace sip
