"""sfft_plan_get_info of chirp-z plans: what is reported is what runs.  One
launch (passes 1, the radices of the convolution length), three launches
(passes 3, the radices of the column length, which is the first launch), and
the launch sequence (two FFTs of the convolution length)."""
import math

import pytest

import fft_amd
from fft_amd import _lib as L

pytestmark = pytest.mark.gpu

COLUMNS = {16 * b: [16, b] for b in (8, 9, 10, 11, 12, 13, 15)}


@pytest.mark.parametrize("prec", [L.F32, L.F64])
@pytest.mark.parametrize("n", [17, 509, 1009, 4093])
def test_one_launch(n, prec):
    info = fft_amd.Plan(n, L.C2C, prec).info()
    assert info["passes"] == 1
    assert math.prod(info["radices"]) == info["chirp_length"] >= 2 * n - 1
    assert info["threads_per_transform"] * info["transforms_per_block"] <= 1024


@pytest.mark.parametrize("prec,n", [(L.F32, 9001), (L.F32, 100003), (L.F32, 1000003),
                                    (L.F64, 5003), (L.F64, 100003), (L.F64, 500009)])
def test_three_launches(n, prec):
    info = fft_amd.Plan(n, L.C2C, prec).info()
    assert info["passes"] == 3
    column = math.prod(info["radices"])
    assert info["radices"] == COLUMNS[column] and info["chirp_length"] % column == 0
    assert info["threads_per_transform"] * info["transforms_per_block"] <= 1024


def test_launch_sequence():
    info = fft_amd.Plan(1966081, L.C2C, L.F32).info()
    assert info["passes"] == 4 and info["chirp_length"] >= 2 * 1966081 - 1
