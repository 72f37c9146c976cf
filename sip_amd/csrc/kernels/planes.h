// Contiguous C2C rows whose real and imaginary parts are arrays of their own (split planes), single LDS
// plane per transform. Forward only: exchanging the two planes on both sides gives the inverse
// (i conj(z) swaps the parts, and conj(DFT(conj z)) is the inverse), so the host swaps pointers.
//
// What bounds the split form is the number of memory instructions in flight: staged through LDS element
// by element (a loop of 4-byte loads, each waited for) 256 x 32768 reached 3.0 TB/s. Here every thread
// issues all loads of its first pass at once, straight from both planes, and stores its last pass the same
// way (runs of T floats): 256 x 32768 45.3 -> 28.8 us, 1000 x 8388 57 -> 28, 100 x 83886 54 -> 30. Rows of at most 48 points, whose runs would be a few floats, go through LDS
// in line order instead (16 to 48 points: 4.8-5.9 TB/s, from their own threads 2.1-4.7), also with all
// loads in flight.
#pragma once
#include "stockham_device.h"

namespace sip {

struct PlanesIo {
    static constexpr bool kPairTail = false;
    static constexpr bool kRegTail = false;
    float *__restrict__ re;
    float *__restrict__ im;
    template <int R, int NS>
    __device__ __forceinline__ void store_bf(int d, const float2 (&v)[R]) const
    {
#pragma unroll
        for (int r = 0; r < R; r++) re[d + r * NS] = v[r].x;
#pragma unroll
        for (int r = 0; r < R; r++) im[d + r * NS] = v[r].y;
    }
};

template <int W, int L, int T, int R0, int... Rest>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(W))) void planes_rows_kernel(const StockhamArgs a)
{
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
    const float *gr = static_cast<const float *>(a.in) + ib, *gi = a.in_im + ib;
    float2 v[NB0][R0];
#pragma unroll
    for (int q = 0; q < NB0; q++) {
        const int b = t + q * T;
        if (active && (EXACT0 || b < NBF0)) {
#pragma unroll
            for (int r = 0; r < R0; r++) v[q][r].x = gr[b + r * NBF0];
#pragma unroll
            for (int r = 0; r < R0; r++) v[q][r].y = gi[b + r * NBF0];
        }
    }
    split_chain<L, T, -1, 1, R0, Rest...>(pl, a.tw, flp * a.LP, t, active, v,
                                          PlanesIo{static_cast<float *>(a.out) + ob, a.out_im + ob});
}

// Rows in line order: element i = tid + u (F T) of the workgroup's F L contiguous elements. The exchange
// between line order and the passes' order goes through the plane in two halves on both sides. Rows of a
// tile are contiguous (the host checks that a row starts where the one before ends).
template <int L, int T, int... Rs>
__global__ __launch_bounds__(1024) void planes_small_kernel(const StockhamArgs a)
{
    extern __shared__ float pl[];
    constexpr int R0 = first_of<Rs...>(), RL = last_of<Rs...>();
    constexpr int NBF0 = L / R0, NB0 = (NBF0 + T - 1) / T, NBFL = L / RL, NBL = (NBFL + T - 1) / T;
    constexpr int NG = (L + T - 1) / T;
    const int F = a.F, tid = threadIdx.x, nt = blockDim.x;
    const int flp = tid / T, t = tid - flp * T;
    const int64_t f0 = (int64_t)blockIdx.x * F;
    const int nf = (int)(a.nfft - f0 < F ? a.nfft - f0 : F);
    const bool active = flp < nf;
    const int total = nf * L;
    const float *gr = static_cast<const float *>(a.in) + f0 * L, *gi = a.in_im + f0 * L;
    float2 e[NG];
#pragma unroll
    for (int u = 0; u < NG; u++) {
        const int i = tid + u * nt;
        if (i < total) e[u] = make_float2(gr[i], gi[i]);
    }
    const int lbase = flp * a.LP;
    float2 v[NB0][R0];
#pragma unroll
    for (int plane = 0; plane < 2; plane++) {
        if (plane) __syncthreads();
#pragma unroll
        for (int u = 0; u < NG; u++) {
            const int i = tid + u * nt, f = i / L;
            if (i < total) pl[f * a.LP + lds_pad(i - f * L)] = plane ? e[u].y : e[u].x;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NB0; q++) {
            const int b = t + q * T;
            if (active && (NBF0 % T == 0 || b < NBF0)) {
#pragma unroll
                for (int r = 0; r < R0; r++) {
                    const float x = pl[lbase + lds_idx_read<NBF0>(b, r)];
                    if (plane)
                        v[q][r].y = x;
                    else
                        v[q][r].x = x;
                }
            }
        }
    }
    __syncthreads();
    float2 w[NBL][RL];
    split_chain<L, T, -1, 1, Rs...>(pl, a.tw, lbase, t, active, v, RegTail<RL>{w});
#pragma unroll
    for (int plane = 0; plane < 2; plane++) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NBL; q++) {
            const int b = t + q * T;
            if (active && (NBFL % T == 0 || b < NBFL)) {
#pragma unroll
                for (int r = 0; r < RL; r++)
                    pl[lbase + lds_idx_write<NBFL, RL>(0, b, r)] = plane ? w[q][r].y : w[q][r].x;
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NG; u++) {
            const int i = tid + u * nt, f = i / L;
            if (i < total) {
                const float x = pl[f * a.LP + lds_pad(i - f * L)];
                if (plane)
                    e[u].y = x;
                else
                    e[u].x = x;
            }
        }
    }
    float *dr = static_cast<float *>(a.out) + f0 * L, *di = a.out_im + f0 * L;
#pragma unroll
    for (int u = 0; u < NG; u++) {
        const int i = tid + u * nt;
        if (i < total) {
            dr[i] = e[u].x;
            di[i] = e[u].y;
        }
    }
}

}  // namespace sip
