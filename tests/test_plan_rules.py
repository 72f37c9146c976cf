"""Launch shapes that the planner's rules give (host only): what a rule promises about tiles, orders and
routes, read from the plan's description."""
import pytest

import sip_amd as S

C2C, FWD, VERT = S.ASCEND_FFT_C2C, S.ASCEND_FFT_FORWARD, S.ASCEND_FFT_VERTICAL


def columns(n, b):
    return S.describe_dry([n], C2C, FWD, b, VERT)


@pytest.mark.parametrize("n", [2, 3, 8, 16, 20, 27, 36, 40, 45, 48, 60, 64, 80, 100, 128, 200, 256, 512, 1000, 1024])
@pytest.mark.parametrize("b", [64, 100, 512, 2048])
def test_column_tiles_of_few_columns(n, b):
    """Tiles are narrowed to 8 columns only where 8 fill a wave, and then adjacent ones, which share every line,
    run on one XCD."""
    st = columns(n, b)["stages"][0]
    assert st["L"] == n
    if st["F"] == 8:
        assert st["block"] >= 64 and st["xcd_remap"] == 1
    else:
        assert st["F"] >= 16 and st["T"] < 8


@pytest.mark.parametrize("n,rows,cols", [(31, 1, 1), (1009, 1, 1), (8191, 1, 1), (9973, 12, 24), (12277, 16, 48), (16381, 24, 64)])
def test_bluestein_of_few_transforms(n, rows, cols, monkeypatch):
    """The longest convolutions stay stages below the measured number of transforms; SIP_FFT_FUSE=1 runs them
    in one launch all the same."""
    monkeypatch.delenv("SIP_FFT_FUSE", raising=False)
    for b, dim in ((rows, S.ASCEND_FFT_HORIZONTAL), (cols, VERT)):
        assert len(S.describe_dry([n], C2C, FWD, b, dim)["fused"]) == 1
        if b > 1:
            assert S.describe_dry([n], C2C, FWD, b - 1, dim)["fused"] == []
    monkeypatch.setenv("SIP_FFT_FUSE", "1")
    assert len(columns(n, 2)["fused"]) == 1


@pytest.mark.parametrize("n,b,grid", [(251, 32, 32), (509, 256, 256), (1009, 32, 32), (2039, 4, 4), (1009, 4096, 512)])
def test_bluestein_columns_fill_the_chip(n, b, grid):
    """Column tiles narrow until the launch has two workgroups per CU, down to one transform each."""
    assert columns(n, b)["fused"][0]["grid"] >= grid


@pytest.mark.parametrize("n,width", [(3, 64), (20, 64), (24, 32), (40, 32), (36, 16), (45, 16), (60, 16), (81, 16), (1000, 16)])
def test_column_tile_widths(n, width):
    """Many columns: whole waves for one or two threads per column, whole lines otherwise."""
    assert columns(n, 8192)["stages"][0]["F"] == width


def test_split_stages_cut_columns_alike():
    """A split axis of few-thread factors keeps one tile width in both launches, but in XCD order."""
    for n in (1080, 1200):
        st = S.describe_dry([n, 1024], C2C, FWD, 1)["stages"][1:]
        assert len(st) == 2 and [s["F"] for s in st] == [16, 16]
    st = S.describe_dry([1500, 162], C2C, FWD, 4)["stages"][1:]
    assert [s["F"] for s in st] == [64, 16] and [s["xcd_remap"] for s in st] == [1, 1]


@pytest.mark.parametrize("n,rows", [(12150, 257), (12960, 257), (14580, 257), (15000, 257), (16000, 320)])
def test_row_shapes_of_few_rows(n, rows):
    """Row shapes held to 64 registers need more workgroups than CUs; fewer rows run on the two-plane leaf."""
    at = [S.describe_dry([n], C2C, FWD, b)["stages"][0]["split_lds"] for b in (1, rows - 1, rows, 4 * rows)]
    assert at == [0, 0, 1, 1]


@pytest.mark.parametrize("n", [729, 864, 972])
def test_column_shapes_of_few_columns(n):
    """The same for column shapes, from 385 tiles of 16; both run the same radices."""
    few, last, many = (columns(n, b)["stages"][0] for b in (16, 6144, 6145))
    assert [s["split_lds"] for s in (few, last, many)] == [0, 0, 1]
    assert few["radices"] == last["radices"] == many["radices"]
    assert S.describe_dry([n, 64], C2C, FWD, 4)["stages"][1]["split_lds"] == 0


@pytest.mark.parametrize("n,first", [(1080, 128), (2048, 128), (1458, 320), (1728, 288), (1944, 320), (2025, 320)])
def test_long_columns_from(n, first):
    width = columns(n, 1 << 14)["fused"][0]["F"]
    assert [len(columns(n, width * t)["fused"]) for t in (first - 1, first)] == [0, 1]


@pytest.mark.parametrize("n", [2560, 3072, 4096])
def test_long_columns_in_two_passes(n):
    for b in (1024, 2048, 4096, 1 << 14):
        d = columns(n, b)
        assert d["fused"] == [] and len(d["stages"]) == 2


@pytest.mark.parametrize("n,one", [(162, 0), (252, 0), (288, 0), (360, 0), (375, 0), (8748, 0), (125, 1), (256, 1), (300, 1),
                                   (400, 1), (104, 1), (500, 1)])
def test_rows_on_one_or_two_planes(n, one):
    """Leaves of 16 to 31 threads keep the two-plane tile unless one plane was measured faster."""
    for b in (1, 64, 4096):
        assert S.describe_dry([n], C2C, FWD, b)["stages"][0]["split_lds"] == one


@pytest.mark.parametrize("n,start", [(250, 0), (324, (6 << 20) // 162), (750, (6 << 20) // 375), (512, 0), (4096, 0)])
def test_real_rows_on_one_or_two_planes(n, start):
    for t in (S.ASCEND_FFT_R2C, S.ASCEND_FFT_C2R):
        at = [S.describe_dry([n], t, FWD, b)["stages"][0]["split_lds"] for b in (1, max(1, start - 1), max(1, start))]
        assert at == ([0, 0, 1] if start else [1, 1, 1])


@pytest.mark.parametrize("dims,b,nt", [([1 << 20], 8, 1), ([1 << 20], 5, 0), ([1024000], 8, 1), ([65536], 128, 0), ([65536], 192, 0),
                                       ([65536], 193, 1), ([432000], 40, 1), ([40000], 400, 0),
                                       ([262144], 32, 0), ([40000], 220, 0), ([1000000], 8, 0), ([524288], 16, 0),
                                       ([1024, 1024], 16, 0), ([720, 1280], 16, 0), ([256, 256, 256], 2, 0)])
def test_streaming_inputs(dims, b, nt):
    """Below 512 MiB only first-stage columns in whole lines pass the last-level cache, short ones from 96 MiB of input."""
    assert S.describe_dry(dims, C2C, FWD, b)["stages"][0]["nt_in"] == nt


@pytest.mark.parametrize("n,points", [(27, 6 << 20), (48, 6 << 20), (50, 6 << 20), (128, 6 << 20), (64, 0), (100, 0), (104, 0)])
def test_short_rows_of_many(n, points):
    """Leaves of fewer than 16 threads that lose on one plane at large sizes leave it there."""
    for b in (1, 64, max(1, points // n) if points else 1 << 20):
        assert S.describe_dry([n], C2C, FWD, b)["stages"][0]["split_lds"] == 1
    if points:
        assert S.describe_dry([n], C2C, FWD, points // n + 1)["stages"][0]["split_lds"] == 0


@pytest.mark.parametrize("n,points", [(66, 2 << 20), (100, 6 << 20), (84, 6 << 20), (128, 0)])
def test_short_real_rows_of_many(n, points):
    for t in (S.ASCEND_FFT_R2C, S.ASCEND_FFT_C2R):
        b = points // (n // 2) if points else 1 << 20
        assert S.describe_dry([n], t, FWD, b)["stages"][0]["split_lds"] == 1
        if points:
            assert S.describe_dry([n], t, FWD, b + 1)["stages"][0]["split_lds"] == 0


@pytest.mark.parametrize("n,last", [(995328, 12), (1000000, 12), (1024000, 12)])
def test_long_first_stages_of_many(n, last):
    """972- and 1000-point first stages keep two tiles per CU up to 96 MiB."""
    at = [S.describe_dry([n], C2C, FWD, b)["stages"][0]["split_lds"] for b in (8, last, last + 1, 32)]
    assert at == [1, 1, 0, 0]


@pytest.mark.parametrize("dims,b,order", [([243, 60], 1150, [1, 1]), ([500, 1250], 26, [1, 1]), ([36, 96, 60], 80, [1, 1, 1]),
                                          ([243, 60], 288, [0, 1]), ([512, 1296], 25, [0, 0]), ([243, 60], 2300, [1, 1])])
def test_launches_of_one_array_in_one_order(dims, b, order):
    assert [s["xcd_remap"] for s in S.describe_dry(dims, C2C, FWD, b)["stages"]] == order
