"""How many members share a block of the band solves (no device calls: runs without
a GPU): the number that sc_set_tuning asks for wherever a block's registers and LDS
hold them, as the header of the library lists it, and never more than the run has."""
import ctypes
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(os.path.join(ROOT, "shadow-channel_amd", "libshadowchannel.so"))


def members(lib, Ny, nrun, tuned):
    # sc::solve_columns_per_block(int), sc::solve_members(int, int, int, int)
    columns = getattr(lib, "_ZN2sc23solve_columns_per_blockEi")(Ny - 2)
    assert columns in (2, 4, 8)
    return getattr(lib, "_ZN2sc13solve_membersEiiii")(Ny - 2, columns, nrun, tuned)


def test_tuned_members_run(lib):
    for Ny in range(4, 515):
        four = Ny <= 130 or 179 <= Ny <= 274 or 355 <= Ny <= 450
        assert members(lib, Ny, 32, 4) == (4 if four else 2), Ny
        assert members(lib, Ny, 32, 2) == 2, Ny
        assert members(lib, Ny, 32, 1) == 1, Ny
        assert members(lib, Ny, 32, 0) == (1 if 147 <= Ny <= 178 or 291 <= Ny <= 354 else 2), Ny


@pytest.mark.parametrize("nrun,most", [(1, 1), (2, 2), (3, 2), (4, 4), (5, 4)])
def test_no_more_than_the_run_has(lib, nrun, most):
    for tuned in (0, 1, 2, 4):
        assert members(lib, 97, nrun, tuned) == min(most, tuned or 2)
