"""Host arrays about the size of a chunk of pinned memory (1 MB: just below, exactly,
just above), where their way back changes, and about 64 KB.  A run of no steps returns
its state and stores it, exactly; repeated, so that the chunks are used again.
"""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.c_destroy()


@pytest.mark.parametrize("Nx,Ny,Nz,size", [(16, 18, 16, 65536), (16, 19, 16, 69632), (32, 65, 32, 1032192),
                                           (32, 66, 32, 1048576), (32, 67, 32, 1064960)])
def test_round_trip(cc, Nx, Ny, Nz, size):
    print("case: host array sizes, %dx%dx%d" % (Nx, Ny, Nz), flush=True)
    assert cc.c_init(Nx, Ny, Nz, np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 0) == 0
    for seed in range(6):
        C0 = synthetic_state(Nx, Ny, Nz, np.pi, 0.5 * np.pi, 4.0 / 3.0, seed=seed, amp=0.1)
        assert C0.nbytes == size
        C0[Nz // 2] = 0                  # the Nyquist row holds no data
        C = C0.copy()
        cc.c_primal(0, C)
        np.testing.assert_array_equal(C, C0)
        np.testing.assert_array_equal(cc.c_getsoln(0), C0)
