"""The banded column solves at the edges of their block shapes: one primal,
tangent and adjoint step against the oracle, and five members for every choice
of members per block against the single run, bit for bit.

Ny - 2 rows in two parities give a worker 1, 2, 3 or 4 rows of an 8-column
block (up to Ny = 50, 98, 146 and 178), then 2 to 4 of a 4-column block, then 2
or 3 of a 2-column one.  The 4 x 10 columns, and 8 x 8 where the Nyquist row
ends on a block, leave the last block partly empty.

The bound of each Ny is ten times the rounding floor of the oracle there (one
step with and without FMA contraction, the largest of the three directions,
which grows with the conditioning of the Gram matrices), and 1e-13 at least."""
import numpy as np
import pytest

import pyorc
from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002

# Ny, Nz, ten floors
SHAPES = [(5, 10, 1e-13), (6, 8, 1e-13), (50, 10, 2.7e-10), (51, 8, 4.5e-10), (98, 10, 2.4e-9),
          (99, 8, 2.4e-9), (146, 10, 1.6e-8), (147, 10, 3.8e-8), (178, 10, 6.2e-8), (179, 8, 6.8e-8),
          (230, 10, 1.8e-6), (300, 8, 1.2e-5), (340, 10, 1.2e-5), (387, 10, 1.7e-5), (514, 8, 3.8e-4)]


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_tuning("solve_members_per_block", 0)
    c_channel.sc_set_members(1)
    c_channel.c_destroy()


@pytest.mark.parametrize("Ny,Nz,bound", SHAPES)
def test_one_step(cc, Ny, Nz, bound):
    Nx = 8
    print("case: solve shapes, %dx%dx%d" % (Nx, Ny, Nz), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=seed, **kw)
    C0, d, a = st(0, amp=0.05), st(1, unit=True), st(2, unit=True)
    o = pyorc.Oracle(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1)
    ref = [C0.copy(), d.copy(), a.copy()]
    o.primal(0, ref[0])
    o.tangent(0, 1, ref[1], 0)
    o.adjoint(1, 0, ref[2], 0, 1.0)
    o.destroy()
    cc.sc_set_members(1)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
    got = [C0.copy(), d.copy(), a.copy()]
    cc.c_primal(0, got[0])
    cc.c_tangent(0, 1, got[1], 0)
    cc.c_adjoint(1, 0, got[2], 0, 1.0)
    for g, r in zip(got, ref):
        assert np.linalg.norm(g - r) / np.linalg.norm(r) < bound
    nm = 5
    for mb in (1, 2, 4):
        cc.sc_set_tuning("solve_members_per_block", mb)
        cc.sc_set_members(nm)
        assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
        dev = [cc.DeviceArray(np.ascontiguousarray(np.stack([x] * nm))) for x in (C0, d, a)]
        try:
            cc.sc_primal_members(0, dev[0])
            cc.sc_tangent_members(0, 1, dev[1], 0, False)
            cc.sc_adjoint_members(1, 0, dev[2], 1.0, False)
            for x, g in zip(dev, got):
                assert all(np.array_equal(y, g) for y in x.download())
        finally:
            for x in dev:
                x.free()
