// Bluestein's chirp-z transform of length N in one launch (gfx950).
//
// X[k] = c[k] sum_n (x[n] c[n]) conj c[k - n] with c[n] = e^{s i pi n^2 / N}: a circular convolution
// of M >= 2 N - 1 points. A workgroup owns F transforms: the first pass of the forward M-point FFT
// reads x from HBM and multiplies by the chirp, the kernel spectrum D (already divided by M) is
// applied to the forward FFT's outputs in registers, and the last pass of the inverse FFT applies
// the chirp again and writes the N outputs. Nothing of the M-point sequences leaves the CU.
//
// What bounds it: run as stages (chirp, FFT, multiply, FFT, chirp) the transform moves 56 M + 16 N
// bytes through HBM for 16 N bytes of input and output; here HBM carries the 16 N and the work is
// the two FFTs' LDS exchanges and butterflies. Measured on MI355X, staged / one launch: 1009 x 4096
// 138 / 26.5 us, 17 x 123361 122 / 22.5 us, 509 x 4120 73 / 20 us, 4099 x 511 133 / 38 us, 16381 x
// 128 104 / 56 us.
//   * M is even, so N <= M / 2 and the first pass's slots r >= R0 / 2 are zero, and the last
//     pass's outputs r >= R / 2 unused, at compile time: half of those butterflies folds away.
//   * The inverse runs the forward's radices in reverse. The forward's last pass of radix R leaves
//     elements b + r M / R in the thread's registers, which is what the inverse's first pass of the
//     same radix reads: no exchange between the two FFTs.
//   * One LDS plane per transform (the exchange of stockham_device.h), 4 (M + M / 16 + 1) bytes.
// Lanes walk the transform (rows) or F adjacent transforms (columns), chosen per launch.
#pragma once
#include "fused_args.h"
#include "stockham2d.h"

namespace sip {

// Output side of the inverse FFT: out[j] = v[j] chirp[j] for j < n, interleaved or in two planes.
struct BlueOut {
    static constexpr bool kPairTail = false;
    static constexpr bool kRegTail = false;
    float2 *__restrict__ out;
    float *out_re, *out_im;  // split planes (out_im != null)
    const float2 *__restrict__ chirp;
    int64_t es;
    int n;
    template <int R, int NS>
    __device__ __forceinline__ void store_bf(int d, const float2 (&v)[R]) const
    {
        // d + r NS >= NS R / 2 = M / 2 >= n for r >= R / 2
        constexpr int H = R / 2;
        float2 c[H];
#pragma unroll
        for (int r = 0; r < H; r++) {
            const int j = d + r * NS;
            c[r] = chirp[j < n ? j : n - 1];
        }
#pragma unroll
        for (int r = 0; r < H; r++) {
            const int j = d + r * NS;
            if (j >= n) continue;
            const float2 y = cmul(v[r], c[r]);
            if (out_im) {
                out_re[(int64_t)j * es] = y.x;
                out_im[(int64_t)j * es] = y.y;
            } else {
                out[(int64_t)j * es] = y;
            }
        }
    }
};

template <int M, int T, class RF, class RI>
struct Bluestein;

template <int M, int T, int... RF, int... RI>
struct Bluestein<M, T, Radices<RF...>, Radices<RI...>> {
    static constexpr int R0 = first_of<RF...>(), RL = last_of<RF...>();
    static_assert(M % 2 == 0 && R0 % 2 == 0, "zero folding needs even M and first radix");
    static_assert(RL == first_of<RI...>() && R0 == last_of<RI...>(), "the inverse reverses the radices");
    static constexpr int NBF0 = M / R0, NB0 = (NBF0 + T - 1) / T;
    static constexpr int NBFL = M / RL, NBL = (NBFL + T - 1) / T;

    __device__ __forceinline__ static void run(const StockhamArgs &a, float *pl)
    {
        const int F = a.F, tid = threadIdx.x, n = a.in_len;
        int t, flp;
        if (a.col_direct) {
            t = (int)fdiv((uint32_t)tid, a.div_F);
            flp = tid - t * F;
        } else {
            flp = tid / T;
            t = tid - flp * T;
        }
        const int64_t f = tile_index(a) * F + flp;
        const bool active = f < a.nfft;
        int64_t ib = 0, ob = 0;  // a lane without a transform reads transform 0's elements, stores none
        if (active) {
            ib = tile_base((uint32_t)f, a.tin);
            ob = tile_base((uint32_t)f, a.tout);
        }
        const float2 *chirp = a.rtw;
        float2 v[NB0][R0];
        {
            constexpr int H = R0 / 2;
            float2 c[NB0][H];
#pragma unroll
            for (int q = 0; q < NB0; q++)
#pragma unroll
                for (int r = 0; r < H; r++) {
                    const int j = t + q * T + r * NBF0;
                    const int jj = j < n ? j : n - 1;
                    const int64_t o = ib + (int64_t)jj * a.tin.es;
                    if (a.in_sep)
                        v[q][r] = make_float2(static_cast<const float *>(a.in)[o], a.in_im[o]);
                    else
                        v[q][r] = gload(static_cast<const float2 *>(a.in) + o);
                    c[q][r] = chirp[jj];
                }
#pragma unroll
            for (int q = 0; q < NB0; q++)
#pragma unroll
                for (int r = 0; r < R0; r++) {
                    const int j = t + q * T + r * NBF0;
                    if (r < H && j < n)
                        v[q][r] = cmul(v[q][r], c[q][r < H ? r : 0]);
                    else
                        v[q][r] = make_float2(0.f, 0.f);
                }
        }
        const int lbase = flp * a.LP;
        float2 w[NBL][RL];
        split_chain<M, T, -1, 1, RF...>(pl, a.tw, lbase, t, active, v, RegTail<RL>{w});
#pragma unroll
        for (int q = 0; q < NBL; q++)
#pragma unroll
            for (int r = 0; r < RL; r++) {
                const int b = t + q * T;
                if (NBFL % T == 0 || b < NBFL) w[q][r] = cmul(w[q][r], a.tw4_lo[b + r * NBFL]);
            }
        __syncthreads();  // the forward FFT's last readers of the plane are done
        const BlueOut io{static_cast<float2 *>(a.out) + ob, static_cast<float *>(a.out) + ob,
                         a.out_sep ? a.out_im + ob : nullptr, chirp, a.tout.es, n};
        split_chain<M, T, 1, 1, RI...>(pl, a.tw2, lbase, t, active, w, io);
    }
};

template <int M, int T, class RF, class RI>
__global__ __launch_bounds__(1024) void bluestein_kernel(const StockhamArgs a)
{
    extern __shared__ float lds[];
    Bluestein<M, T, RF, RI>::run(a, lds);
}

}  // namespace sip
