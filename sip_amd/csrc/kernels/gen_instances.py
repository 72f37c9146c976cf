"""Generates the Stockham kernel instances compiled into libsip_fft.so.

Every leaf length L (a transform that fits one workgroup's LDS) gets one kernel per direction,
with its radix sequence and threads-per-transform fixed at compile time. The leaf set is every
2,3,5-smooth length up to 16384 (powers of two included), and lengths carrying one factor 7, 11
or 13 up to 4096; longer or other lengths are planned on the host as several leaf passes
(four-step) or Bluestein.

Usage: python gen_instances.py OUTDIR NPARTS   (writes OUTDIR/stockham_part_<k>.hip and
OUTDIR/stockham_parts.inc). The output is a pure function of this file.
"""
from __future__ import annotations

import hashlib
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))  # also when loaded from a path
from column_shapes import (COLUMN_FROM, COLUMN_SHAPES, COLUMN_TW_FROM, COLUMN_TW_POINTS, COLUMN_TW_SHAPES, LONG_COLUMN_FROM,
                           LONG_COLUMN_SHAPES)
from real_shapes import REAL_SHAPES, ROWS_COLS_FROM, ROWS_COLS_SHAPES
from row_shapes import ROW_FROM, ROW_SHAPES
from split_rates import SPLIT_RATES

MAX_SMOOTH = 16384
MAX_POW2 = 16384
MAX_PRIME_FACTOR_LEN = 4096


def smooth_lengths():
    out = set()
    for a in range(15):
        for b in range(10):
            for c in range(7):
                n = 2 ** a * 3 ** b * 5 ** c
                if n <= MAX_SMOOTH:
                    out.add(n)
    for a in range(15):
        if 2 ** a <= MAX_POW2:
            out.add(2 ** a)
    base = sorted(x for x in out if x <= MAX_PRIME_FACTOR_LEN)
    for p in (7, 11, 13):
        for m in base:
            if m * p <= MAX_PRIME_FACTOR_LEN:
                out.add(m * p)
    out.discard(1)
    return sorted(out)


def factor(n):
    f = {}
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            f[p] = f.get(p, 0) + 1
            n //= p
    assert n == 1, n
    return f


# Radix sequences chosen by measurement where the cost model's first choice measured slower: tuning
# builds took the second and third sequence by cost (same pass count) for every length above 1024
# where one exists (118 lengths), then the fourth and the best with one pass more (165 lengths),
# each timed as C2C rows of 128 MiB on MI355X, best of two runs per build; kept where the
# alternative was faster by more than 5 % (run-to-run spread: median 0.6 %, at most 3.4 % in the
# first round, 6.2 % in the second, whose kept gains are all above 10 %). Old / new microseconds in
# the comments.
LEAF_SEQ = {
    1120: [16, 10, 7],       # 51.6 / 46.6
    1200: [20, 12, 5],       # 49.6 / 46.6
    1280: [16, 10, 8],       # 46.0 / 40.9
    1320: [15, 11, 8],       # 54.6 / 50.9
    1760: [16, 11, 10],      # 52.3 / 46.5
    1920: [16, 12, 10],      # 51.0 / 47.7
    2100: [10, 10, 7, 3],    # 62.9 / 56.0
    2500: [10, 10, 5, 5],    # 54.3 / 50.4
    2520: [12, 7, 6, 5],     # 62.7 / 56.0
    2916: [12, 9, 9, 3],     # 56.6 / 53.2
    3000: [15, 8, 5, 5],     # 60.2 / 54.0
    3300: [15, 11, 5, 4],    # 58.7 / 55.2
    5760: [16, 10, 9, 4],    # 55.1 / 50.4
    5832: [12, 9, 9, 6],     # 63.6 / 53.1
    6000: [20, 12, 5, 5],    # 66.9 / 56.1
    6144: [16, 16, 6, 4],    # 47.6 / 43.2
    6480: [16, 9, 9, 5],     # 62.9 / 54.5
    6750: [15, 15, 6, 5],    # 63.0 / 57.3
    6912: [16, 9, 8, 6],     # 51.0 / 47.7
    9600: [20, 20, 6, 4],    # 50.7 / 46.9
    11520: [16, 16, 9, 5],   # 66.6 / 54.6
    13122: [9, 9, 9, 6, 3],  # 78.5 / 73.3
    13824: [16, 16, 9, 6],   # 84.9 / 72.4
    # a second round (the fourth sequence by cost, and the best one with one pass more)
    2160: [12, 12, 5, 3],    # 51.6 / 46.5
    14400: [20, 12, 12, 5],  # 66.2 / 57.1
    15360: [20, 12, 4, 4, 4],  # 78.7 / 69.2
    # leaves up to 1024, timed in both four-step roles (n = 256 L, 128 MiB), as rows and as 2D L x L
    720: [12, 12, 5],        # four-step 268 / 237, rows 51.9 / 45.2, 2D 120 / 101
    800: [20, 8, 5],         # four-step 273 / 257, rows 46.1 / 48.8, 2D 124 / 109
    # long-row leaves (SIP_GEN_BIG_RANK tuning builds; C2C rows, 256 MiB, from 256 rows up)
    19440: [16, 15, 9, 9],   # 187 / 148
    20480: [16, 16, 10, 8],  # 158 / 145
    20736: [16, 16, 9, 9],   # 158 / 148
    21600: [16, 15, 15, 6],  # 214 / 163
    25920: [16, 9, 9, 5, 4],  # 206 / 193
    30000: [10, 10, 10, 6, 5],  # 258 / 215
}
# (1000 = 10 x 10 x 10 was faster in the four-step roles, 305 / 283 us, but its 100 threads per
# transform halve the column tiles to 8 transforms, half-line HBM runs: 2D 1000^2 gained nothing.)

# Radices with a register butterfly (butterflies.h): prime, power-of-two and two-factor composites.
RADICES = [20, 16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2]
MAX_ELEMS = 24   # complex values per thread in one pass


def _sequences(n, maxr=20, depth=0):
    if n == 1:
        yield []
        return
    if depth > 7:
        return
    for r in RADICES:
        if r <= maxr and n % r == 0:
            for rest in _sequences(n // r, r, depth + 1):
                yield [r] + rest


def _cost(n, seq):
    """Passes (each an LDS round trip) plus idle thread-rounds of passes whose butterfly count is
    not a multiple of the thread count, plus the unused lanes of a partial last wave."""
    t = threads_per_transform(n, seq)
    waste, elems = 0.0, 0
    for r in seq:
        nbf = n // r
        nb = -(-nbf // t)
        waste += (nb * t - nbf) / nbf
        elems = max(elems, nb * r)
    if elems > MAX_ELEMS:
        return None
    waves = -(-t // 64)
    partial = (waves * 64 - t) / (waves * 64) if t >= 64 else 0.0
    return len(seq) + 0.3 * waste + 0.2 * partial


def radix_sequence(n):
    """Radix passes for length n. Powers of two: the exponent split as evenly as possible into
    radices <= 16. Other lengths: the sequence over RADICES (composites included) with the lowest
    _cost, ties to the larger leading radices. Largest radices first."""
    if n & (n - 1):
        if n in LEAF_SEQ:
            return list(LEAF_SEQ[n])
        ranked = []
        for seq in _sequences(n):
            c = _cost(n, seq)
            if c is not None:
                ranked.append((c, seq))
        if ranked:
            ranked.sort(key=lambda cs: cs[0])  # stable: ties keep the larger leading radices
            # tuning builds (SIP_GEN_SEQ_RANK=k) take the k-th sequence by cost among those with as
            # few passes as the first
            npass = len(ranked[0][1])
            # tuning builds vary the lengths in SIP_GEN_SEQ_RANGE ("lo,hi", default 1025..16384)
            lo, hi = (int(v) for v in os.environ.get("SIP_GEN_SEQ_RANGE", "1025,16384").split(","))
            tuned = lo <= n <= hi
            if tuned and os.environ.get("SIP_GEN_SEQ_EXTRA") == "1":
                # the best sequence with one pass more, where one exists
                more = [cs for cs in ranked if len(cs[1]) == npass + 1]
                if more:
                    return more[0][1]
            same = [cs for cs in ranked if len(cs[1]) == npass]
            rank = int(os.environ.get("SIP_GEN_SEQ_RANK", "0")) if tuned else 0
            return same[min(rank, len(same) - 1)][1]
    f = factor(n)
    seq = []
    a = f.get(2, 0)
    if a:
        npass = (a + 3) // 4
        bits = [a // npass + (1 if i < a % npass else 0) for i in range(npass)]
        seq += [2 ** b for b in sorted(bits, reverse=True)]
    for p in (13, 11, 7):
        seq += [p] * f.get(p, 0)
    seq += [5] * f.get(5, 0)
    seq += [3] * f.get(3, 0)
    # keep the biggest radix first
    seq.sort(key=lambda r: -r)
    return seq


def threads_per_transform(n, seq):
    """One butterfly of the largest radix per thread, within [1, 1024]; shrink when a smaller
    radix would need more than 32 elements per thread."""
    rmax = max(seq)
    t = max(1, n // rmax)
    while t > 1024:
        t //= 2
    return t


def elems_per_thread(n, seq, t):
    return max(((n // r + t - 1) // t) * r for r in seq)


# 2,3,5-smooth lengths above MAX_SMOOTH up to BIG_ROWS_MAX get only the single-plane contiguous-row
# kernel (one transform per workgroup of T <= 1024 threads; its plane, 4 (L + L/16 + 1) bytes, fits
# the 160 KiB LDS up to 32768): a one-pass leaf where the two-plane tile would not fit. Their radix
# sequences hold at most BIG_MAX_ELEMS values per thread (register budget of four waves per SIMD:
# 77-112 VGPRs, no scratch, with radix-15 and -20 passes as well); lengths with no such sequence
# (31104, 31250, 32000, 32400) stay four-step splits.
BIG_ROWS_MAX = 32768
BIG_RADICES = [20, 16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2]
BIG_MAX_ELEMS = 32


def big_lengths():
    out = []
    for a in range(16):
        for b in range(11):
            for c in range(8):
                n = 2 ** a * 3 ** b * 5 ** c
                if MAX_SMOOTH < n <= BIG_ROWS_MAX:
                    out.append(n)
    return sorted(out)


def big_threads(n, seq):
    """One butterfly of the largest radix per thread, at most 1024 threads."""
    return min(1024, n // max(seq))


def big_radix_sequence(n):
    """Fewest passes over BIG_RADICES within BIG_MAX_ELEMS values per thread, then the fewest idle
    butterfly rounds; largest radices first."""
    if n in LEAF_SEQ:
        return list(LEAF_SEQ[n])
    found = []

    def rec(m, maxr, seq):
        if m == 1:
            t = big_threads(n, seq)
            if elems_per_thread(n, seq, t) > BIG_MAX_ELEMS:
                return
            waste = sum((-(-(n // r) // t) * t - n // r) / (n // r) for r in seq)
            found.append(((len(seq), waste), list(seq)))
            return
        if len(seq) >= 8:
            return
        for r in BIG_RADICES:
            if r <= maxr and m % r == 0:
                rec(m // r, r, seq + [r])

    rec(n, 1 << 30, [])
    if not found:
        return None  # no sequence fits; the length stays a four-step split
    found.sort(key=lambda ks: ks[0])  # stable: ties keep the larger leading radices
    # tuning builds (SIP_GEN_BIG_RANK=k): the k-th sequence among those with the fewest passes
    same = [ks for ks in found if ks[0][0] == found[0][0][0]]
    rank = int(os.environ.get("SIP_GEN_BIG_RANK", "0"))
    return same[min(rank, len(same) - 1)][1]


def instances():
    res = []
    for n in smooth_lengths():
        seq = radix_sequence(n)
        t = threads_per_transform(n, seq)
        e = elems_per_thread(n, seq, t)
        assert e <= 40, (n, seq, t, e)
        assert all(r in RADICES for r in seq), (n, seq)
        res.append((n, t, seq))
    for n in big_lengths():
        seq = big_radix_sequence(n)
        if seq is None:
            continue
        t = big_threads(n, seq)
        assert t >= 32 and elems_per_thread(n, seq, t) <= BIG_MAX_ELEMS, (n, seq, t)
        res.append((n, t, seq))
    return res


# Contiguous-row kernels (rows.h) from ROWS_MIN points up, with three or more threads per transform: shorter
# rows, and leaves of fewer threads, are faster staged through LDS in line order (16: 5.3-6.0 TB/s staged,
# 4.1 from their own threads). Leaves of 16 to 31 threads already read and write HBM from their own threads on
# two planes; without a shape of their own one plane costs them its extra barriers (252 x 1 4.1 / 4.6 us, 351 x
# 1024 6.6 / 7.3, 16 MiB of 325 11.2 / 12.2; 64 MiB within 5 % on average), except 125, 256 and 400 (256 x 32768
# 27.7 / 21.7). Other lengths faster on the two-plane tile: 256 MiB of rows, single / two planes, 15625 268 / 240
# us, 15552 171 / 158; 8748 (512 rows 21.7 / 20.5, 700 rows 30.7 / 31.3).
ROWS_MIN, ROWS_MIN_THREADS = 24, 3
ROWS_TWO_PLANE = {8748, 15552, 15625}
# Leaves of fewer than 16 threads without a shape lose on one plane from 64 MiB on, where their narrow runs bound
# them: two planes in line order / one, 48 x 349525 57.3 / 68.8 us, x 1398101 193 / 252, 33 x 508400 61.3 / 72.5, 27, 28,
# 32, 39, 42, 44, 50 .. 56, 66, 75, 78, 84 and 128 3 to 28 %; below 48 MiB they win (48 x 21845 12.4 / 9.4).
ROWS_POINTS = {n: 6 << 20 for n in (27, 28, 32, 33, 39, 42, 44, 48, 50, 52, 54, 56, 66, 75, 78, 84, 128)}
ONE_PLANE_16 = {125, 256, 400}


def two_plane_threads(n, t):
    return 16 <= t < 32 and n not in ONE_PLANE_16


# longest leaf used for column tiles (the host's kColumnLeafMax); every leaf up to it gets a column
# kernel of its own (columns.h) with the shape measured for that role (column_shapes.py)
COLUMN_LEAF_MAX = 1024
# half lengths of the real transforms that get single-plane R2C / C2R row kernels: from REAL_ROWS_MIN to 8192
# with three or more threads (shorter ones are faster staged through LDS: 16 4.2 TB/s, from their own threads
# 3.7), and those above where the single plane measured faster than the two-plane fused kernel on MI355X (R2C +
# C2R of 256 MiB of reals, one box: 9216 155 / 211 us, 10000 161 / 226, 16384 131 / 173; it lost for most mixed
# lengths from 12000 up, e.g. 15000 241 / 218, 13824 225 / 212). Leaves of 16 to 31 threads without a shape take it
# from 48 MiB on (R2C / C2R, two planes / one: 702 x 64 7.8 / 9.0, 7.9 / 8.0 us; 16 MiB of 750 16.4 / 17.1, 16.6 /
# 17.7; 64 MiB of 750 43.7 / 39.4, 49.1 / 38.7).
REAL_ROWS_MIN = 30
REAL_ROWS_MAX = 8192
REAL_FROM_POINTS = 6 << 20
# as ROWS_POINTS (R2C / C2R, two planes / one: 66 x 508400 68.9 / 96.9, 70.3 / 91.3 us; 84 x 399457 1.11, 1.18)
REAL_POINTS = {n: 6 << 20 for n in (35, 42, 44, 50, 52, 54, 55, 56, 65, 66, 70, 75, 78, 84, 110, 112)}
REAL_POINTS.update({33: 2 << 20, 39: 2 << 20})
REAL_ROWS_LONG = {8640, 9000, 9216, 9375, 9600, 9720, 10000, 10125, 10240, 10368, 10800, 10935, 11250, 11664,
                  12288, 16384}
# lengths up to COLUMN_LEAF_MAX with two or more passes and at least this many threads per transform also get
# the rows-in / columns-out kernel of the second four-step stage
RC_MIN_THREADS = 3


def role_entry(role, n, t, seq, f, slot, names, start=0, points=0):
    """A RoleInstance initialiser whose kernels fill `slot` of the instance, used from `start` workgroups
    and up to `points` points (0: any number)."""
    slots = {"tile": "nullptr, nullptr", "rows": "nullptr, nullptr", "cols": "{nullptr, nullptr, nullptr, nullptr}",
             "real": "{nullptr, nullptr, nullptr, nullptr}", "rc": "{nullptr, nullptr}"}
    names = ", ".join(nm if nm == "nullptr" else f"(const void *)&{nm}" for nm in names)
    slots[slot] = names if slot == "rows" else "{" + names + "}"
    p = 1
    for r in seq:
        p *= r
    assert p == n and elems_per_thread(n, seq, t) <= 40 and (f or 1) * t <= 1024, (n, t, seq)
    rs = ", ".join(str(r) for r in seq)
    return f"    {{{role}, {f}, {start}, {points // n}, {{{n}, {t}, {len(seq)}, {{{rs}}}, {', '.join(slots.values())}}}}},"


def row_entries():
    for n, t, seq in instances():
        if n not in ROW_SHAPES and two_plane_threads(n, t):
            continue
        t, seq, w, f = ROW_SHAPES.get(n, (t, seq, 0, 0))
        if n < ROWS_MIN or t < ROWS_MIN_THREADS or n in ROWS_TWO_PLANE:
            continue
        rs = ", ".join(str(r) for r in seq)
        yield role_entry("ROLE_ROWS", n, t, seq, f, "rows", [f"stockham_rows_kernel<{w}, {n}, {t}, {sg}, {rs}>" for sg in (-1, 1)],
                         ROW_FROM.get(n, 0), ROWS_POINTS.get(n, 0))


# Split-plane rows up to this length go through LDS in line order (planes.h), on the leaf's threads but for these:
# 40 and 45 points on two and three threads spilled (116 and 48 bytes a lane; 40 x 4096 16.0 us, on eight threads
# 3.7), 33 and 39 took 97 and 115 registers (33 x 64 7.0 / 3.8). 65 and 66 points, also in line order, ran 64 MiB from
# their own five and six threads in 57.7 and 52.0 us.
PLANES_SMALL_MAX = 48
PLANES_SMALL_SHAPES = {33: (11, [11, 3]), 39: (13, [13, 3]), 40: (8, [8, 5]), 45: (9, [9, 5]), 52: (13, [13, 4]),
                       65: (13, [13, 5]), 66: (11, [11, 6])}


def plane_entries():
    for n, t, seq in instances():
        if n > MAX_SMOOTH:
            continue
        w, f = 0, 0
        small = n <= PLANES_SMALL_MAX or n in PLANES_SMALL_SHAPES
        if small:
            t, seq = PLANES_SMALL_SHAPES.get(n, (t, seq))
        else:
            t, seq, w, f = ROW_SHAPES.get(n, (t, seq, 0, 0))
        rs = ", ".join(str(r) for r in seq)
        name = f"planes_small_kernel<{n}, {t}, {rs}>" if small else f"planes_rows_kernel<{w}, {n}, {t}, {rs}>"
        yield role_entry("ROLE_PLANES", n, t, seq, f, "rows", [name, "nullptr"])


def real_row_entries():
    for n, t, seq in instances():
        start = REAL_FROM_POINTS // n if n not in REAL_SHAPES and two_plane_threads(n, t) else 0
        t, seq, w, f = REAL_SHAPES.get(n, (t, seq, 0, 0))
        if t >= 3 and (REAL_ROWS_MIN <= n <= REAL_ROWS_MAX or n in REAL_ROWS_LONG):
            rs = ", ".join(str(r) for r in seq)
            yield role_entry("ROLE_REAL_ROWS", n, t, seq, f, "real", [
                f"stockham_real_rows_kernel<{w}, {n}, {t}, {sg}, {m}, {rs}>" for m in (1, 2) for sg in (-1, 1)], start,
                             REAL_POINTS.get(n, 0))


# Odd lengths of the real transforms (real_odd.h), on the threads and radices of the row kernels, free registers and the
# default rows per workgroup. From 3 points up and at any count, two-plane full transform / this, R2C us:
# 3 x 3 2.82 / 1.80, 3 x 1398101 17.0 / 8.3, 11 x 381300 17.5 / 10.1, 375 x 699 9.3 / 5.5, 3645 x 3 9.0 / 6.2, 15625 x 268 63 / 50.
def real_odd_entries():
    for n, t, seq in instances():
        if n % 2 and 3 <= n <= MAX_SMOOTH:
            t, seq = ROW_SHAPES.get(n, (t, seq))[:2]
            rs = ", ".join(str(r) for r in seq)
            yield role_entry("ROLE_REAL_ODD", n, t, seq, 0, "real", [
                f"real_odd_kernel<{n}, {t}, {sg}, {m}, {rs}>" for m in (1, 2) for sg in (-1, 1)])


def column_entries():
    shapes = []
    for n, t, seq in instances():
        if n <= COLUMN_LEAF_MAX:
            shapes.append((n, False) + tuple(COLUMN_SHAPES.get(n, (t, seq, 0))) + (0,))
            shapes.append((n, True) + tuple(COLUMN_TW_SHAPES.get(n, (t, seq, 0))) + (0,))
    shapes += [(n, False) + shape for n, shape in LONG_COLUMN_SHAPES.items()]
    for n, tw, t, seq, w, f in shapes:
        rs = ", ".join(str(r) for r in seq)
        names = [f"stockham_cols_kernel<{w}, {n}, {t}, {sg}, {str(tw).lower()}, {rs}>" for sg in (-1, 1)]
        none = ["nullptr", "nullptr"]
        start = LONG_COLUMN_FROM.get(n, 128) if n in LONG_COLUMN_SHAPES else (COLUMN_TW_FROM if tw else COLUMN_FROM).get(n, 0)
        yield role_entry("ROLE_COLS_TW" if tw else "ROLE_COLS", n, t, seq, f, "cols", none + names if tw else names + none, start,
                         COLUMN_TW_POINTS.get(n, 0) if tw else 0)


def rc_entries():
    for n, t, seq in instances():
        t, seq, w = ROWS_COLS_SHAPES.get(n, (t, seq, 0))
        if n <= COLUMN_LEAF_MAX and len(seq) >= 2 and t >= RC_MIN_THREADS:
            rs = ", ".join(str(r) for r in seq)
            yield role_entry("ROLE_RC", n, t, seq, 0, "rc", [f"stockham_rc_kernel<{w}, {n}, {t}, {sg}, {rs}>" for sg in (-1, 1)],
                             ROWS_COLS_FROM.get(n, 0))


# role files: name, header, entries, parts
ROLE_FILES = [("rows", "rows.h", row_entries, 16), ("real_rows", "real_rows.h", real_row_entries, 16),
              ("columns", "columns.h", column_entries, 16), ("rows_cols", "rows_cols.h", rc_entries, 8),
              ("planes", "planes.h", plane_entries, 8), ("real_odd", "real_odd.h", real_odd_entries, 8)]


def write_roles(outdir):
    inc = ["// Generated by gen_instances.py (do not edit)."]
    for name, header, entries, parts in ROLE_FILES:
        items = list(entries())
        for k in range(parts):
            part = items[k::parts]
            text = ["// Generated by gen_instances.py (do not edit).", f'#include "{header}"', "namespace sip {",
                    f"extern const RoleInstance g_{name}_part_{k}[] = {{"] + part
            text += ["};", f"extern const int g_{name}_part_{k}_count = {len(part)};", "}  // namespace sip"]
            write_if_changed(os.path.join(outdir, f"{name}_part_{k}.hip"), "\n".join(text) + "\n")
            inc.append(f"SIP_ROLE_PART({name}_part_{k})")
    write_if_changed(os.path.join(outdir, "role_parts.inc"), "\n".join(inc) + "\n")
    rates = ["// Generated by gen_instances.py (do not edit): length, first and second four-step stage in GB/s."]
    rates += [f"{{{n}, {{{a}, {b}}}}}," for n, (a, b) in sorted(SPLIT_RATES.items())]
    write_if_changed(os.path.join(outdir, "split_rates.inc"), "\n".join(rates) + "\n")


# One-launch inverse short-time transforms (istft.h): every 2,3,5-smooth frame length in this range,
# with the leaf's radix sequence and threads.
ISTFT_MIN, ISTFT_MAX, ISTFT_PARTS = 24, 1499, 6
# Lengths whose kernel spilled 40 to 116 bytes a lane when held to 64 registers (two 1024-thread tiles per CU);
# within 73 to 91 it does not (64 MiB, held / free: 320, hop 40 68.8 / 46.5 us, 640, hop 160 64.5 / 39.2, 40, hop 5 65.2
# / 29.4). Others that spill less keep the limit (1000, hop 250 48.2 / 60.5; 500, hop 62 46.6 / 54.0).
ISTFT_FREE = {40, 45, 60, 160, 180, 192, 240, 320, 400, 640, 800}


def istft_instances():
    return [(n, t, seq) for n, t, seq in instances()
            if ISTFT_MIN <= n <= ISTFT_MAX and all(r not in (7, 11, 13) for r in seq)]


def write_if_changed(path, text):
    if not os.path.exists(path) or open(path).read() != text:
        with open(path, "w") as fh:
            fh.write(text)


def write_istft(outdir):
    inst = istft_instances()
    for k in range(ISTFT_PARTS):
        lines = ["// Generated by gen_instances.py: one-launch inverse short-time transforms (do not edit).",
                 '#include "istft.h"', "namespace sip {", f"extern const IstftInstance g_istft_part_{k}[] = {{"]
        items = inst[k::ISTFT_PARTS]
        for n, t, seq in items:
            rs = ", ".join(str(r) for r in seq)
            lines.append(f"    {{{n}, {t}, {len(seq)}, {{{rs}}}, (const void *)&istft_kernel<{0 if n in ISTFT_FREE else 8}, {n}, {t}, {rs}>}},")
        lines += ["};", f"extern const int g_istft_part_{k}_count = {len(items)};", "}  // namespace sip"]
        write_if_changed(os.path.join(outdir, f"istft_part_{k}.hip"), "\n".join(lines) + "\n")
    inc = ["// Generated by gen_instances.py (do not edit)."] + [f"SIP_ISTFT_PART({k})" for k in range(ISTFT_PARTS)]
    write_if_changed(os.path.join(outdir, "istft_parts.inc"), "\n".join(inc) + "\n")


def kernel_set(outdir):
    """Digest of every kernel source: the generated instances and the files beside this one."""
    here = os.path.dirname(os.path.abspath(__file__))
    h = hashlib.sha256()
    for d, ends in ((here, (".h", ".hip")), (outdir, (".hip", "_rates.inc"))):
        for name in sorted(os.listdir(d)):
            if name.endswith(ends):
                with open(os.path.join(d, name), "rb") as fh:
                    h.update(name.encode() + fh.read())
    return h.hexdigest()[:8]


def write_kernel_set(outdir):
    text = ["// Generated by gen_instances.py (do not edit): digest of the kernel sources.", f'"{kernel_set(outdir)}"']
    write_if_changed(os.path.join(outdir, "kernel_set.inc"), "\n".join(text) + "\n")


def main():
    outdir = sys.argv[1]
    nparts = int(sys.argv[2])
    os.makedirs(outdir, exist_ok=True)
    write_istft(outdir)
    write_roles(outdir)
    inst = [i for i in instances() if i[0] <= MAX_SMOOTH]  # longer leaves are row kernels only
    parts = [[] for _ in range(nparts)]
    # balance by estimated code size (passes x length)
    load = [0] * nparts
    for item in sorted(inst, key=lambda x: -len(x[2]) * x[0]):
        k = load.index(min(load))
        parts[k].append(item)
        load[k] += len(item[2]) * max(64, item[0] // 8)
    for k, items in enumerate(parts):
        items.sort()
        lines = [
            "// Generated by gen_instances.py: Stockham kernel instances (do not edit).",
            '#include "stockham_device.h"',
            "namespace sip {",
        ]
        tab = []
        for n, t, seq in items:
            rs = ", ".join(str(r) for r in seq)
            radix = ", ".join(str(r) for r in seq)
            kf = f"stockham_kernel<{n}, {t}, -1, {rs}>"
            ki = f"stockham_kernel<{n}, {t}, 1, {rs}>"
            lines.append(f"template __global__ void {kf}(const StockhamArgs);")
            lines.append(f"template __global__ void {ki}(const StockhamArgs);")
            tab.append(f"    {{{n}, {t}, {len(seq)}, {{{radix}}}, (const void *)&{kf}, (const void *)&{ki}, nullptr, nullptr, "
                       "{nullptr, nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr, nullptr}, {nullptr, nullptr}},")
        lines.append(f"extern const StockhamInstance g_stockham_part_{k}[] = {{")
        lines += tab
        lines.append("};")
        lines.append(f"extern const int g_stockham_part_{k}_count = {len(items)};")
        lines.append("}  // namespace sip")
        write_if_changed(os.path.join(outdir, f"stockham_part_{k}.hip"), "\n".join(lines) + "\n")
    inc = ["// Generated by gen_instances.py (do not edit)."]
    for k in range(nparts):
        inc.append(f"SIP_STOCKHAM_PART({k})")
    write_if_changed(os.path.join(outdir, "stockham_parts.inc"), "\n".join(inc) + "\n")
    write_kernel_set(outdir)
    print(f"{len(inst)} leaf lengths in {nparts} parts")


if __name__ == "__main__":
    main()
