"""Members of different states against their own single runs, bit for bit, on grids
that take the other column counts and row slots of the band solves' blocks (8 columns
with 3 and 4 rows a thread, 4 with 2 and 3, 2 with 2), for every choice of members per
block, and the y-transform of 97 to 128 coefficients: five members, so that the last
group is not full."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

NX, NZ, LX, LZ, RE, FLUX, DT, NM = 8, 10, np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 5


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_tuning("solve_members_per_block", 0)
    c_channel.sc_set_members(1)
    c_channel.c_destroy()


@pytest.mark.parametrize("Ny", [50, 98, 115, 130, 161, 179, 201, 355])
def test_members_equal_their_single_runs(cc, Ny):
    print("case: distinct members, %dx%dx%d" % (NX, Ny, NZ), flush=True)
    st = lambda seed, **kw: synthetic_state(NX, Ny, NZ, LX, LZ, FLUX, seed=seed, **kw)
    X = [[st(m, amp=0.05), st(10 + m, unit=True), st(20 + m, unit=True)] for m in range(NM)]
    cc.sc_set_members(1)
    assert cc.c_init(NX, Ny, NZ, LX, LZ, RE, FLUX, DT, 1) == 0
    ref = []
    for m in range(NM):
        C, d, a = (x.copy() for x in X[m])
        cc.c_primal(0, C)
        cc.c_tangent(0, 1, d, 0)
        cc.c_adjoint(1, 0, a, 0, 1.0)
        ref.append((C, d, a))
        assert all(np.isfinite(x).all() for x in ref[m])
    for mb in (0, 1, 2, 4):
        cc.sc_set_tuning("solve_members_per_block", mb)
        cc.sc_set_members(NM)
        assert cc.c_init(NX, Ny, NZ, LX, LZ, RE, FLUX, DT, 1) == 0
        dev = [cc.DeviceArray(np.ascontiguousarray(np.stack([x[k] for x in X]))) for k in range(3)]
        try:
            cc.sc_primal_members(0, dev[0])
            cc.sc_tangent_members(0, 1, dev[1], 0, False)
            cc.sc_adjoint_members(1, 0, dev[2], 1.0, False)
            for k in range(3):
                got = dev[k].download()
                for m in range(NM):
                    np.testing.assert_array_equal(got[m], ref[m][k], err_msg="%d a block, member %d" % (mb, m))
        finally:
            for x in dev:
                x.free()
