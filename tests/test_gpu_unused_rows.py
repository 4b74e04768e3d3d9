"""The alpha rows dimQ and dimQ + 1 carry nothing in a column (kx, kz) != (0, 0):
values that are not finite there leave the physical fields and the other rows of
a primal step as they are with zeros, bit for bit.  Ny = 99 to 130, where the last
k-steps of the y-transform pass both bases' ends at different rows; Ny = 131 for
the kernel of longer bases."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.c_destroy()


@pytest.mark.parametrize("Ny", [99, 100, 101, 115, 129, 130, 131])
def test_unused_alpha_rows(cc, Ny):
    Nx, Nz = 12, 8
    print("case: unused rows, %dx%dx%d" % (Nx, Ny, Nz), flush=True)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
    nQ = Ny - 4
    out = []
    for fill in (0.0, np.nan, np.inf):
        C = synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=0, amp=0.05)
        mean = C[0, 0, nQ:, 0].copy()
        C[:, 0, nQ:, :] = fill
        C[0, 0, nQ:, 0] = mean
        flow = np.zeros((3, 3 * Nx // 2, 3 * Ny // 2, 3 * Nz // 2))
        cc.c_spec2phys(C.copy(), flow)
        cc.c_primal(0, C)
        C[:, 0, nQ:, 1:] = 0.0
        C[1:, 0, nQ:, 0] = 0.0
        out.append((flow, C))
    assert np.isfinite(out[0][0]).all() and np.isfinite(out[0][1]).all()
    for flow, C in out[1:]:
        assert np.array_equal(flow, out[0][0]) and np.array_equal(C, out[0][1])
