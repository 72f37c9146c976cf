// Inverse short-time transform in one launch (gfx950): the inverse DFTs of a run of adjacent frames
// and their windowed overlap-add.
//
// Spectra X[c][k][t] (bin k of frame (c, t) at (c n + k) frames + t). A workgroup transforms F frames
// t0 .. t0 + F - 1 of one channel (lanes walk adjacent frames, so the loads are runs of F values),
// puts the frames into LDS and sums the samples that no other frame covers: of the F frames the
// first halo = ceil(n / hop) - 1 only contribute to samples of the tile before, so a tile ends
// keep * hop samples, keep = F - halo.
//
// What bounds it: as stages (column DFTs to a frame array, then the overlap-add) the spectra's
// 8 n frames bytes are read, written and read again; here they are read F / keep times, the
// repeated frames mostly from the caches, and only the samples are written. Tiles of one channel
// go to one XCD in order, so that the halo frames are in its L2. Measured on MI355X, staged / one
// launch: 8 channels x 2049 frames of 1024, hop 256 126.5 / 67.7 us; 4 channels, 2^23 points in all:
// 256, hop 64 53 / 32 us, 400, hop 100 69 / 34, 1000, hop 250 83 / 47, 1200, hop 300 223 / 55.
//
// W: waves per SIMD the register budget is held to (8: 64 registers, two 1024-thread tiles per CU; 0: the
// compiler's choice, for the lengths that would spill, gen_instances.py).
//
// The sums run in the order, and with the operations, of the staged overlap-add (aux.hip). LDS: one
// plane, the real parts of all frames summed first, then the imaginary parts.
#pragma once
#include "fused_args.h"
#include "stockham_device.h"

namespace sip {

template <int W, int L, int T, int... Rs>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(W))) void istft_kernel(const IstftArgs a)
{
    extern __shared__ float pl[];
    constexpr int R0 = first_of<Rs...>(), NBF0 = L / R0, NB0 = (NBF0 + T - 1) / T;
    constexpr bool EXACT0 = (NBF0 % T) == 0;
    constexpr int RL = last_of<Rs...>(), NBFL = L / RL, NBL = (NBFL + T - 1) / T;
    constexpr bool EXACTL = (NBFL % T) == 0;
    const int F = a.F, tid = threadIdx.x, nthreads = blockDim.x;
    const int64_t tile = xcd_tile();
    const uint32_t c = fdiv((uint32_t)tile, a.div_tiles);
    const int64_t k = tile - (int64_t)c * a.tiles;
    const int64_t t0 = k * a.keep - a.halo;  // first frame of the tile
    const int t = (int)fdiv((uint32_t)tid, a.div_F);
    const int fl = tid - t * F;
    const int64_t fr = t0 + fl;
    const bool active = fr >= 0 && fr < a.frames;
    const float2 *src = a.in + (int64_t)c * L * a.frames + (active ? fr : 0);
    float2 v[NB0][R0];
#pragma unroll
    for (int q = 0; q < NB0; q++) {
        const int b = t + q * T;
        if (active && (EXACT0 || b < NBF0)) {
#pragma unroll
            for (int r = 0; r < R0; r++) v[q][r] = gload(src + (int64_t)(b + r * NBF0) * a.frames);
        }
    }
    float2 w[NBL][RL];
    split_chain<L, T, 1, 1, Rs...>(pl, a.tw, fl * a.LP, t, active, v, RegTail<RL>{w});

    // frames lo .. hi of the tile exist
    const int lo = t0 < 0 ? (int)-t0 : 0;
    const int hi = (int)((t0 + F < a.frames ? t0 + F : a.frames) - 1 - t0);
    const int hop = (int)a.hop;
    // samples s = 0 .. keep hop - 1 of the tile are m = base + s of the overlap-add span
    const int64_t base = k * a.keep * a.hop;
    const int ns = (int)(a.keep * a.hop);
    float *dst = reinterpret_cast<float *>(a.out + (int64_t)c * a.out_len);
#pragma unroll
    for (int plane = 0; plane < 2; plane++) {
        __syncthreads();  // earlier readers of the plane are done
#pragma unroll
        for (int q = 0; q < NBL; q++) {
            const int b = t + q * T;
            if (active && (EXACTL || b < NBFL)) {
#pragma unroll
                for (int r = 0; r < RL; r++)
                    pl[fl * a.LP + lds_idx_write<NBFL, RL>(0, b, r)] = plane ? w[q][r].y : w[q][r].x;
            }
        }
        __syncthreads();
        // The two halves of a sample are stored apart (the L2 merges them): keeping the real parts in
        // registers until the imaginary ones are summed costs 16 of them, and with 64 or fewer two
        // 1024-thread workgroups fit on a CU.
        for (int s = tid; s < ns; s += nthreads) {
            const int64_t m = base + s;
            if (m < a.start || m >= a.start + a.out_len) continue;
            // frames f0 .. f1 (relative to t0) cover sample m; frame f holds it at j, which falls by hop
            const int rel = (int)fdiv((uint32_t)s, a.div_hop);  // m / hop = k keep + rel = t0 + halo + rel
            int j = s - rel * hop;                              // m - (m / hop) hop
            const int back = (int)fdiv((uint32_t)(L - 1 - j), a.div_hop);  // frames before m / hop that cover m
            int f0 = rel + a.halo - back, f1 = rel + a.halo;
            j += back * hop;
            if (f0 < lo) {
                j -= (lo - f0) * hop;
                f0 = lo;
            }
            if (f1 > hi) f1 = hi;
            float acc = 0.f, e = 0.f;
            for (int f = f0; f <= f1; f++, j -= hop) {
                const float wj = a.win[j];
                acc = fmaf(pl[f * a.LP + lds_pad(j)], wj, acc);
                e = fmaf(wj, wj, e);
            }
            dst[2 * (m - a.start) + plane] = acc / ((float)L * e);
        }
    }
}

}  // namespace sip
