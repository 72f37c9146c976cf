// Registry entries of the kernels that run several stages of a plan in one launch.
#pragma once
#include "stockham_args.h"

namespace sip {

// One-launch Bluestein transform on convolutions of M points (bluestein.h). The forward FFT's radices
// are given; the inverse runs them in reverse. Launch arguments: in_len = N, rtw = chirp, tw / tw2 =
// pass twiddles of the forward / inverse FFT, tw4_lo = kernel spectrum, col_direct = lanes walk
// adjacent transforms.
struct BluesteinInstance {
    int32_t M, T, npass;
    int32_t radix[4];
    const void *fn;
};

}  // namespace sip
