"""The y-transform to the Gauss points for 97 to 128 coefficients (Ny = 99 to 130:
a y-tile's whole basis in LDS) and the first Ny past it, against the oracle, one
solution and three members; grids whose kz rows do not divide over eight XCDs,
with one n-tile, and with a last n-tile partly empty.

Bounds: the physical fields are sums of at most 128 terms of unit size, whose
rounding is below 128 2^-53 times the largest partial sum (taken as 10 of the
result): 3e-13 with a margin of two.  A step has ten times the rounding floor of
the oracle on the grid (with and without FMA contraction, the largest of the three
directions).  Members equal the single run bit for bit."""
import numpy as np
import pytest

import pyorc
from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002
GRIDS = [(8, 99, 10, 2.4e-9), (12, 130, 8, 7.6e-9), (36, 115, 18, 2.1e-8), (4, 131, 4, 3.6e-9)]


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_members(1)
    c_channel.c_destroy()


@pytest.mark.parametrize("Nx,Ny,Nz,bound", GRIDS)
def test_fields_and_step(cc, Nx, Ny, Nz, bound):
    print("case: wide rebuild, %dx%dx%d" % (Nx, Ny, Nz), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=seed, **kw)
    X = (st(0, amp=0.05), st(1, unit=True), st(2, unit=True))
    o = pyorc.Oracle(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1)
    U = o.spec2phys(X[0])
    ref = [x.copy() for x in X]
    o.primal(0, ref[0])
    o.tangent(0, 1, ref[1], 0)
    o.adjoint(1, 0, ref[2], 0, 1.0)
    o.destroy()
    cc.sc_set_members(1)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
    flow = np.zeros(U.shape)
    cc.c_spec2phys(X[0].copy(), flow)
    assert np.linalg.norm(flow - U) / np.linalg.norm(U) < 3e-13
    got = [x.copy() for x in X]
    cc.c_primal(0, got[0])
    cc.c_tangent(0, 1, got[1], 0)
    cc.c_adjoint(1, 0, got[2], 0, 1.0)
    for g, r in zip(got, ref):
        assert np.linalg.norm(g - r) / np.linalg.norm(r) < bound
    cc.sc_set_members(3)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
    dev = [cc.DeviceArray(np.ascontiguousarray(np.stack([x] * 3))) for x in X]
    try:
        cc.sc_primal_members(0, dev[0])
        cc.sc_tangent_members(0, 1, dev[1], 0, False)
        cc.sc_adjoint_members(1, 0, dev[2], 1.0, False)
        for x, g in zip(dev, got):
            assert all(np.array_equal(y, g) for y in x.download())
    finally:
        for x in dev:
            x.free()
