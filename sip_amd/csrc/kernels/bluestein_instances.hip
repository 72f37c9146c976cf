// One-launch Bluestein instances: convolution lengths M with at most 32 values per thread in any
// pass and even first radix, closely enough spaced that the zero padding of 2 N - 1 to M stays
// below a third. Above 16384 points a transform is one 1024-thread workgroup's chain of eight passes
// (20480 points 32 us, 24576 38, 32768 47, whatever their number up to 256), which the stages, spread over the
// chip, undercut while there are few transforms: rows of 9973 8 / 12 staged 28 / 35 us, 12277 12 / 16 35 /
// 39, 16381 20 / 24 45 / 48; columns, whose runs are narrow, staged / one launch 9973 x 24 49 / 49, 12277 x 48
// 67 / 65, 16381 x 64 75 / 75.
#include "bluestein.h"

namespace sip {

#define SIP_ARG(...) __VA_ARGS__
#define SIP_BLUE_FROM(M, T, NP, RF, RI, ROWS, COLS) \
    {M, T, NP, {RF}, (const void *)&bluestein_kernel<M, T, Radices<RF>, Radices<RI>>, ROWS, COLS}
#define SIP_BLUE(M, T, NP, RF, RI) SIP_BLUE_FROM(M, T, NP, SIP_ARG(RF), SIP_ARG(RI), 1, 1)

extern const BluesteinInstance g_bluestein[] = {
    SIP_BLUE(48, 6, 2, SIP_ARG(8, 6), SIP_ARG(6, 8)),
    SIP_BLUE(64, 8, 2, SIP_ARG(8, 8), SIP_ARG(8, 8)),
    SIP_BLUE(80, 8, 2, SIP_ARG(10, 8), SIP_ARG(8, 10)),
    SIP_BLUE(96, 8, 2, SIP_ARG(12, 8), SIP_ARG(8, 12)),
    SIP_BLUE(128, 8, 2, SIP_ARG(16, 8), SIP_ARG(8, 16)),
    SIP_BLUE(160, 10, 2, SIP_ARG(16, 10), SIP_ARG(10, 16)),
    SIP_BLUE(192, 12, 2, SIP_ARG(16, 12), SIP_ARG(12, 16)),
    SIP_BLUE(256, 16, 2, SIP_ARG(16, 16), SIP_ARG(16, 16)),
    SIP_BLUE(320, 16, 2, SIP_ARG(20, 16), SIP_ARG(16, 20)),
    SIP_BLUE(384, 48, 3, SIP_ARG(8, 8, 6), SIP_ARG(6, 8, 8)),
    SIP_BLUE(512, 64, 3, SIP_ARG(8, 8, 8), SIP_ARG(8, 8, 8)),
    SIP_BLUE(640, 64, 3, SIP_ARG(10, 8, 8), SIP_ARG(8, 8, 10)),
    SIP_BLUE(768, 64, 3, SIP_ARG(12, 8, 8), SIP_ARG(8, 8, 12)),
    SIP_BLUE(1024, 64, 3, SIP_ARG(16, 8, 8), SIP_ARG(8, 8, 16)),
    SIP_BLUE(1280, 80, 3, SIP_ARG(16, 10, 8), SIP_ARG(8, 10, 16)),
    SIP_BLUE(1536, 96, 3, SIP_ARG(16, 12, 8), SIP_ARG(8, 12, 16)),
    SIP_BLUE(2048, 128, 3, SIP_ARG(16, 16, 8), SIP_ARG(8, 16, 16)),
    SIP_BLUE(2560, 160, 3, SIP_ARG(16, 16, 10), SIP_ARG(10, 16, 16)),
    SIP_BLUE(3072, 192, 3, SIP_ARG(16, 16, 12), SIP_ARG(12, 16, 16)),
    SIP_BLUE(4096, 256, 3, SIP_ARG(16, 16, 16), SIP_ARG(16, 16, 16)),
    SIP_BLUE(5120, 256, 3, SIP_ARG(20, 16, 16), SIP_ARG(16, 16, 20)),
    SIP_BLUE(6144, 512, 4, SIP_ARG(12, 8, 8, 8), SIP_ARG(8, 8, 8, 12)),
    SIP_BLUE(8192, 512, 4, SIP_ARG(16, 8, 8, 8), SIP_ARG(8, 8, 8, 16)),
    SIP_BLUE(10240, 640, 4, SIP_ARG(16, 10, 8, 8), SIP_ARG(8, 8, 10, 16)),
    SIP_BLUE(12288, 768, 4, SIP_ARG(16, 12, 8, 8), SIP_ARG(8, 8, 12, 16)),
    SIP_BLUE(16384, 1024, 4, SIP_ARG(16, 16, 8, 8), SIP_ARG(8, 8, 16, 16)),
    SIP_BLUE_FROM(20480, 1024, 4, SIP_ARG(20, 16, 8, 8), SIP_ARG(8, 8, 16, 20), 12, 24),
    SIP_BLUE_FROM(24576, 1024, 4, SIP_ARG(16, 16, 12, 8), SIP_ARG(8, 12, 16, 16), 16, 48),
    SIP_BLUE_FROM(32768, 1024, 4, SIP_ARG(16, 16, 16, 8), SIP_ARG(8, 16, 16, 16), 24, 64),
};
extern const int g_bluestein_count = (int)(sizeof(g_bluestein) / sizeof(g_bluestein[0]));

}  // namespace sip
