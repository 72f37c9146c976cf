// Real transforms of odd length n (no half-length transform exists), contiguous rows, single LDS plane:
// the n-point complex passes straight from and to HBM. MODE 1 = R2C: the first pass reads reals (the zero
// imaginary parts fold away at compile time) and the last writes bins 0 .. n/2. MODE 2 = C2R: the first
// pass reads bin j or the conjugate of bin n - j (the second reader of a line finds it in the cache), the
// last computes and writes real parts only.
#pragma once
#include "fused_args.h"
#include "stockham_device.h"

namespace sip {

struct HalfOut {
    static constexpr bool kPairTail = false;
    static constexpr bool kRegTail = false;
    float2 *__restrict__ out;
    int last;  // n / 2
    template <int R, int NS>
    __device__ __forceinline__ void store_bf(int d, const float2 (&v)[R]) const
    {
#pragma unroll
        for (int r = 0; r < R; r++)
            if (d + r * NS <= last) gstore(out + d + r * NS, v[r]);
    }
};

struct RealOut {
    static constexpr bool kPairTail = false;
    static constexpr bool kRegTail = false;
    float *__restrict__ out;
    template <int R, int NS>
    __device__ __forceinline__ void store_bf(int d, const float2 (&v)[R]) const
    {
#pragma unroll
        for (int r = 0; r < R; r++) out[d + r * NS] = v[r].x;
    }
};

template <int L, int T, int S, int MODE, int R0, int... Rest>
__global__ __launch_bounds__(1024) void real_odd_kernel(const StockhamArgs a)
{
    static_assert(L % 2 == 1, "even lengths run half-length transforms");
    extern __shared__ float pl[];
    constexpr int NBF0 = L / R0, NB0 = (NBF0 + T - 1) / T;
    constexpr bool EXACT0 = (NBF0 % T) == 0;
    const int tid = threadIdx.x, flp = tid / T, t = tid - flp * T;
    const int64_t f = tile_index(a) * a.F + flp;
    const bool active = f < a.nfft;
    int64_t ib = 0, ob = 0;
    if (active) {
        ib = tile_base((uint32_t)f, a.tin);
        ob = tile_base((uint32_t)f, a.tout);
    }
    float2 v[NB0][R0];
#pragma unroll
    for (int q = 0; q < NB0; q++) {
        const int b = t + q * T;
        if (active && (EXACT0 || b < NBF0)) {
#pragma unroll
            for (int r = 0; r < R0; r++) {
                const int j = b + r * NBF0;
                if constexpr (MODE == 1) {
                    v[q][r] = make_float2(static_cast<const float *>(a.in)[ib + j], 0.f);
                } else {
                    v[q][r] = gload(static_cast<const float2 *>(a.in) + ib + (j <= L / 2 ? j : L - j));
                }
            }
            if constexpr (MODE == 2) {
#pragma unroll
                for (int r = 0; r < R0; r++) {
                    const int j = b + r * NBF0;
                    if (j > L / 2) v[q][r].y = -v[q][r].y;
                }
                if (b == 0) v[q][0].y = 0.f;  // the imaginary part of bin 0 is dropped
            }
        }
    }
    if constexpr (MODE == 1)
        split_chain<L, T, S, 1, R0, Rest...>(pl, a.tw, flp * a.LP, t, active, v,
                                             HalfOut{static_cast<float2 *>(a.out) + ob, L / 2});
    else
        split_chain<L, T, S, 1, R0, Rest...>(pl, a.tw, flp * a.LP, t, active, v, RealOut{static_cast<float *>(a.out) + ob});
}

}  // namespace sip
