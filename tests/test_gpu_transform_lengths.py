"""The x/z transforms at every length with kernels of its own, and at lengths
without (the runtime-length kernels), through one primal, tangent and adjoint
step against the oracle.

Bound: 1e-10, the one-step bound of the parity tests.  The physical fields of a
mixed-precision context come from the FP64 kernels: equal bits."""
import numpy as np
import pytest

import pyorc
from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002

# (Nx, Nz): every fixed x length 3 Nx / 2 and z length 3 Nz / 2 once or more,
# planes shorter than a block's rows (Nz = 4, 10), the lengths 12, 216 and 6 of
# the runtime-length kernels
GRIDS = [(12, 10), (16, 12), (20, 18), (24, 16), (32, 20), (36, 24), (40, 30), (48, 32), (60, 36),
         (64, 40), (72, 48), (80, 50), (96, 54), (100, 60), (108, 64), (120, 72), (128, 80),
         (12, 90), (16, 96), (20, 100), (24, 108), (12, 120), (12, 128), (8, 12), (16, 144), (32, 4)]


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_precision(0)
    c_channel.c_destroy()


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("Nx,Nz", GRIDS)
def test_one_step(cc, Nx, Nz):
    Ny = 13
    print("case: one step, %dx%dx%d" % (Nx, Ny, Nz), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=seed, **kw)
    C0, d, a = st(0, amp=0.05), st(1, unit=True), st(2, unit=True)
    o = pyorc.Oracle(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1)
    C, I, A = C0.copy(), d.copy(), a.copy()
    flow = [np.zeros((3, 3 * Nx // 2, 3 * Ny // 2, 3 * Nz // 2)) for _ in range(2)]
    cc.sc_set_precision(1)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
    cc.c_spec2phys(C0.copy(), flow[1])
    cc.sc_set_precision(0)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
    cc.c_spec2phys(C0.copy(), flow[0])
    cc.c_primal(0, C)
    cc.c_tangent(0, 1, I, 0)
    cc.c_adjoint(1, 0, A, 0, 1.0)
    Co, Io, Ao = C0.copy(), d.copy(), a.copy()
    o.primal(0, Co)
    o.tangent(0, 1, Io, 0)
    o.adjoint(1, 0, Ao, 0, 1.0)
    for g, r in zip((C, I, A, flow[0]), (Co, Io, Ao, o.spec2phys(C0))):
        assert rel(g, r) < 1e-10
    assert np.array_equal(flow[0], flow[1])
    o.destroy()
