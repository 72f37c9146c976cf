// Column-tile kernels, single LDS plane (split_cols in stockham_device.h). TW4: the stage applies the
// four-step twiddle on store. W: waves per SIMD the register budget is held to (0 = the compiler's
// choice): with W = 8 (64 registers) two 1024-thread tiles share a CU, one loading while the other
// computes. 1024 points with the twiddle took 76 registers, one tile per CU: 1048576 x 8, stage A of 64 MiB
// 37.4 us, with W = 8 and 16 x 4 x 16 26 us.
#pragma once
#include "stockham_device.h"

namespace sip {

template <int W, int L, int T, int S, bool TW4, int... Rs>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(W))) void stockham_cols_kernel(const StockhamArgs a)
{
    extern __shared__ float lds[];
    split_cols<L, T, S, TW4, Rs...>(a, lds, tile_index(a));
}

}  // namespace sip
