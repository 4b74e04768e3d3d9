"""Tangent members along one trajectory, whose x transforms take the state's fields
once for all members, against the single runs, bit for bit: lengths 48, 60, 72, 96,
108 and 120, both precisions, member counts that split unevenly over the groups,
rows that do not fill the last block, the first stage's CFL check included; and a
length and a member count that keep the per-member kernel."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT, NY = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 9
CASES = [(32, 20, 4), (32, 20, 3), (40, 18, 5), (48, 30, 2), (64, 10, 7), (72, 12, 4), (80, 50, 3), (20, 18, 3)]


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_precision(0)
    c_channel.sc_set_members(1)
    c_channel.c_destroy()


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("Nx,Nz,nm", CASES)
def test_members_equal_single(cc, Nx, Nz, nm, mixed):
    print("case: shared rows, %dx%dx%d, %d members, mixed %d" % (Nx, NY, Nz, nm, mixed), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, NY, Nz, LX, LZ, FLUX, seed=seed, **kw)
    C0, D = st(0, amp=0.05), [st(10 + m, unit=True) for m in range(nm)]
    cc.sc_set_precision(mixed)
    cc.sc_set_members(nm)
    assert cc.c_init(Nx, NY, Nz, LX, LZ, RE, FLUX, DT, 2) == 0
    base = cc.DeviceArray(np.ascontiguousarray(np.stack([C0] * nm)))
    dev = cc.DeviceArray(np.ascontiguousarray(np.stack(D)))
    try:
        cc.sc_primal_members(0, base)
        cc.sc_tangent_members(0, 2, dev, 0b10, True)
        got = dev.download()
    finally:
        base.free()
        dev.free()
    cc.sc_set_members(1)
    assert cc.c_init(Nx, NY, Nz, LX, LZ, RE, FLUX, DT, 2) == 0
    cc.c_primal(0, C0.copy())
    for m in range(nm):
        d = D[m].copy()
        cc.c_tangent(0, 2, d, 1 if m == 1 else 0)
        assert np.isfinite(d).all()
        np.testing.assert_array_equal(got[m], d)
