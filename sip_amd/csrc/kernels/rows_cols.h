// Rows in, columns out (split_rows_cols in stockham_device.h): the second stage of a four-step split.
#pragma once
#include "stockham_device.h"

namespace sip {

template <int L, int T, int S, int... Rs>
__global__ __launch_bounds__(1024) void stockham_rc_kernel(const StockhamArgs a)
{
    extern __shared__ float lds[];
    split_rows_cols<L, T, S, Rs...>(a, lds, tile_index(a));
}

}  // namespace sip
