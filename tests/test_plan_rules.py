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
    assert st["L"] == n and st["block"] >= 64
    if st["F"] == 8:
        assert st["T"] >= 8 and st["xcd_remap"] == 1
    else:
        assert st["F"] >= 16 and st["T"] < 8
