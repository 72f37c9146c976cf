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
    int32_t rows, cols;  // rows / adjacent columns from which the one launch is faster than the stages
};

// One-launch inverse short-time transform (istft.h).
struct IstftArgs {
    const float2 *in;     // spectra (channel, n, frames)
    float2 *out;          // samples (channel, out_len)
    const float2 *tw;     // pass twiddles of the inverse n-point FFT
    const float *win;     // window, n values
    int64_t frames, hop, out_len;
    int64_t start;        // first sample of the overlap-add span that is written
    int64_t tiles;        // tiles per channel
    int64_t keep;         // frames a tile advances by
    int32_t halo;         // frames of a tile that the tile before ends: ceil(n / hop) - 1
    int32_t F, LP;        // frames per tile, LDS pitch of a frame
    FastDiv div_F, div_tiles, div_hop;
};

struct IstftInstance {
    int32_t L, T, npass;
    int32_t radix[8];
    const void *fn;
};

}  // namespace sip
