"""Shapes of the column-tile kernels (columns.h): threads per column, radices, and the waves per SIMD the
kernel is held to (8: at most 64 registers, so that two 1024-thread workgroups share a CU; 0: the
compiler's choice). Lengths that are not listed take the leaf's threads and radices.

What bounds a column tile is how many workgroups a CU holds, one loading while another computes, so the
best shapes keep 16 x T <= 1024 threads and 16-20 values per thread: 1000 as 50 threads of 10 x 10 x 10
where the leaf's 20 x 10 x 5 takes 80 registers and one workgroup per CU. With the four-step twiddle the
store of one butterfly of radix R derives its R factors from 1 + log2 R table products, so the largest
radix comes last: 1024 as 16 x 4 x 16 5.10 TB/s, as 16 x 8 x 8 3.94.

Measured on MI355X over 64 MiB of columns, 16 wide: every listed shape was the fastest of the leaf's
shape and three to six others by cost (passes, idle rounds, values per thread), with and without the
register limit. The figures are GB/s of the leaf's shape / of this one.
"""

# without the four-step twiddle
COLUMN_SHAPES = {
    150: (15, [15, 10], 0),  # 6269 / 6502
    160: (16, [16, 10], 8),  # 6354 / 6995
    162: (27, [9, 6, 3], 8),  # 5258 / 5697
    216: (27, [9, 8, 3], 8),  # 5290 / 5615
    240: (16, [16, 15], 0),  # 6240 / 6770
    270: (30, [10, 9, 3], 0),  # 4996 / 5782
    300: (30, [12, 5, 5], 0),  # 5112 / 5551
    324: (36, [12, 9, 3], 0),  # 5105 / 5318
    384: (32, [16, 6, 4], 0),  # 5464 / 6033
    540: (60, [12, 9, 5], 0),  # 4141 / 5070
    600: (60, [12, 10, 5], 0),  # 4254 / 4860
    675: (45, [15, 9, 5], 0),  # 4312 / 4545
    720: (48, [16, 15, 3], 0),  # 5028 / 5250
    729: (41, [9, 9, 9], 0),  # 3881 / 4419
    750: (50, [15, 10, 5], 8),  # 3570 / 4382
    768: (64, [16, 12, 4], 0),  # 4993 / 5426
    810: (54, [15, 9, 6], 8),  # 3454 / 4484
    864: (54, [16, 9, 6], 8),  # 3727 / 4078
    900: (60, [15, 15, 4], 8),  # 3385 / 4380
    960: (64, [16, 15, 4], 8),  # 4178 / 4478
    972: (54, [12, 9, 9], 8),  # 3575 / 3796
    1000: (50, [10, 10, 10], 8),  # 2910 / 3704
}

# Columns tiles (16 wide) from which a shape is used. Up to one tile per CU a launch is bounded by one tile's chain
# of exchanges, which these shapes, of fewer threads or held to 64 registers, make longer; the two-plane leaf
# halves it. Start / shape / two planes: 729 x 64 6.39 / 7.68 / 5.78 us, x 2048 10.8 / 11.3 / 9.6; 864 x 4096
# 15.9 / 17.8 / 15.3; 972 x 64 7.6 / 8.3 / 6.9; from 385 tiles the shape wins (729 x 8192 28.4 / 24.2, 972 x 8192
# 43.3 / 35.9). Both run the same radices.
COLUMN_FROM = {729: 385, 864: 385, 972: 385}

# with the four-step twiddle applied on store
COLUMN_TW_SHAPES = {
    64: (4, [4, 16], 0),  # 5902 / 6189
    72: (9, [8, 9], 0),  # 5152 / 5880
    75: (5, [5, 15], 0),  # 3968 / 5197
    80: (10, [8, 10], 0),  # 5352 / 6001
    90: (8, [6, 15], 0),  # 4936 / 5687
    96: (8, [12, 8], 0),  # 4862 / 5973
    100: (10, [10, 10], 0),  # 4113 / 5710
    108: (12, [12, 9], 0),  # 5276 / 5880
    128: (8, [8, 16], 0),  # 5641 / 6163
    135: (9, [9, 15], 0),  # 5252 / 5523
    150: (15, [15, 10], 0),  # 5254 / 5791
    160: (10, [8, 20], 0),  # 5660 / 6312
    162: (27, [6, 3, 9], 0),  # 4021 / 4769
    180: (15, [12, 15], 0),  # 5701 / 6294
    192: (16, [12, 16], 0),  # 5741 / 6399
    200: (10, [10, 20], 0),  # 5189 / 5638
    216: (18, [6, 3, 12], 0),  # 4104 / 4528
    240: (16, [15, 16], 0),  # 5612 / 6185
    243: (27, [9, 3, 9], 0),  # 4097 / 4569
    250: (25, [5, 5, 10], 0),  # 3961 / 4309
    270: (30, [9, 3, 10], 0),  # 3805 / 4694
    288: (36, [8, 4, 9], 0),  # 4161 / 4660
    300: (24, [20, 15], 0),  # 3936 / 5517
    320: (24, [20, 16], 0),  # 4151 / 5466
    324: (36, [9, 3, 12], 0),  # 4031 / 4432
    360: (24, [8, 3, 15], 0),  # 3940 / 4756
    375: (25, [5, 5, 15], 0),  # 3745 / 3987
    384: (24, [8, 3, 16], 0),  # 3809 / 4545
    405: (45, [9, 5, 9], 0),  # 3848 / 4234
    432: (36, [12, 3, 12], 8),  # 3677 / 4445
    450: (30, [15, 2, 15], 0),  # 3857 / 4074
    480: (32, [8, 4, 15], 8),  # 4095 / 4541
    486: (54, [9, 6, 9], 0),  # 3337 / 3688
    500: (25, [5, 5, 20], 0),  # 3795 / 4204
    512: (32, [16, 2, 16], 8),  # 4394 / 5513
    576: (48, [12, 4, 12], 0),  # 3812 / 4193
    600: (30, [10, 3, 20], 0),  # 3307 / 3984
    625: (42, [5, 5, 5, 5], 8),  # - / 2696
    640: (32, [8, 4, 20], 0),  # 3975 / 5392
    648: (54, [9, 6, 12], 8),  # 3832 / 4043
    675: (45, [15, 3, 15], 0),  # 3666 / 4392
    720: (60, [12, 4, 15], 8),  # 3501 / 4260
    729: (41, [9, 9, 9], 8),  # - / 3679
    750: (50, [10, 5, 15], 8),  # 2695 / 3681
    768: (64, [8, 6, 16], 8),  # 3493 / 4340
    800: (40, [8, 5, 20], 0),  # 3345 / 4125
    864: (54, [9, 6, 16], 8),  # 2783 / 3497
    900: (60, [15, 4, 15], 8),  # 3416 / 3753
    960: (64, [8, 8, 15], 8),  # 4276 / 4490
    972: (54, [9, 9, 12], 8),  # - / 3463
    1000: (50, [10, 5, 20], 8),  # 2973 / 3578
    1024: (64, [16, 4, 16], 8),  # 3942 / 5099
}

# as COLUMN_FROM
COLUMN_TW_FROM = {625: 257, 729: 257, 972: 257}
# Points up to which a shape is used: with two tiles per CU the input and the intermediate share the last-level cache,
# which beyond 96 MiB of each costs more than the overlap gains (two-plane leaf / shape: 995328 x 16 as 972 x 1024 146 /
# 165 us, 1000000 x 16 167 / 185, x 32 330 / 351, 1024000 x 32 297 / 326; 1000000 x 8 87 / 79).
COLUMN_TW_POINTS = {972: 12 << 20, 1000: 12 << 20}

# Whole axes above 1024 points in one pass (no four-step twiddle), with the columns per tile: 16 columns
# take 32 values per thread (waves per SIMD 4: 128 registers, one workgroup per CU), 8 fewer but half
# lines; both were timed. GB/s of the one pass / of the two four-step passes, 64 MiB of columns, three buffer
# sets in turn. 2560, 3072 and 4096 points are left to the two passes: one 1024-thread tile per CU wins only where
# the tiles fill whole waves of 256 (us in two passes / one: 2560 x 2560 42.3 / 51.8, 3072 x 2051 42.1 / 51.4, 4096 x
# 2560 62.8 / 78.7; 4096 x 3584 86.4 / 84.3).
LONG_COLUMN_SHAPES = {
    1080: (60, [20, 9, 6], 8, 16),  # 3793 / 2624
    1125: (75, [15, 15, 5], 8, 8),  # 2865 / 2149
    1152: (72, [16, 9, 8], 8, 8),  # 3395 / 2403
    1200: (60, [12, 10, 10], 8, 16),  # 3352 / 2492
    1215: (45, [15, 9, 9], 4, 16),  # 2809 / 2222
    1250: (125, [10, 5, 5, 5], 8, 8),  # 2776 / 2124
    1280: (64, [20, 8, 8], 4, 16),  # 3022 / 2533
    1296: (48, [16, 9, 9], 4, 16),  # 3101 / 2062
    1350: (113, [15, 15, 6], 8, 8),  # 3163 / 2386
    1440: (120, [16, 15, 6], 8, 8),  # 3226 / 2620
    1458: (81, [9, 9, 6, 3], 8, 8),  # 2246 / 2197
    1500: (100, [20, 15, 5], 8, 8),  # 2884 / 2540
    1536: (64, [16, 12, 8], 4, 16),  # 2990 / 2616
    1600: (107, [20, 16, 5], 8, 8),  # 3140 / 2293
    1620: (90, [20, 9, 9], 8, 8),  # 2847 / 2086
    1728: (108, [16, 9, 4, 3], 8, 8),  # 2573 / 2381
    1800: (120, [15, 15, 8], 8, 8),  # 2965 / 2320
    1875: (125, [15, 5, 5, 5], 8, 8),  # 2509 / 2133
    1920: (128, [16, 15, 8], 8, 8),  # 2930 / 2353
    1944: (122, [9, 9, 8, 3], 8, 8),  # 2759 / 2184
    2000: (100, [20, 10, 10], 8, 8),  # 2517 / 2260
    2025: (113, [9, 9, 5, 5], 8, 8),  # 2455 / 2177
    2048: (64, [16, 16, 8], 4, 16),  # 3849 / 2532
    2160: (80, [16, 15, 9], 4, 8),  # 3131 / 2201
    2250: (75, [15, 15, 10], 4, 8),  # 2732 / 2176
    2304: (96, [16, 12, 12], 4, 8),  # 3108 / 2350
    2400: (80, [16, 15, 10], 4, 8),  # 2785 / 2455
    2880: (120, [16, 15, 12], 4, 8),  # 2703 / 2324
}

# Tiles from which the one pass is used, where not 128: us in two passes / one, 1458 x 1024 15.2 / 17.9, x 2112
# (264 tiles) 23.6 / 25.8, x 3072 32.0 / 29.1; 1944 x 2112 29.2 / 31.3, x 2560 39.9 / 32.9; 2025 x 2112 30.3 / 35.1, x
# 2560 42.6 / 40.1; 1728 x 2051 26.0 / 28.3.
LONG_COLUMN_FROM = {1458: 320, 1728: 288, 1944: 320, 2025: 320}
