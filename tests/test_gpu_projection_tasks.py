"""The y-projection with a task per wave (mixed precision, many tasks a block)
against two waves a task: members with few projection blocks, so that every block
has eight tasks or more, and the single run of each, whose blocks have fewer.
Both add the same halves in the same order, so the results are equal bits.

Ny at both ends of every k-step count of the kernels: up to 42, 85, 107 and 149
Gauss-point counts 3 Ny / 2 whose half domain fills 8, 16, 20 and 28 groups of
four points, and one far below."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002
NX, NZ, NM = 32, 16, 4


@pytest.fixture(scope="module")
def cc():
    import c_channel
    c_channel.sc_set_precision(1)
    c_channel.sc_set_tuning("force_blocks", 8)
    yield c_channel
    c_channel.sc_set_tuning("force_blocks", 0)
    c_channel.sc_set_precision(0)
    c_channel.sc_set_members(1)
    c_channel.c_destroy()


@pytest.mark.parametrize("Ny", [9, 42, 43, 85, 86, 107, 108, 149])
def test_members_equal_single(cc, Ny):
    print("case: projection tasks, %dx%dx%d, %d members" % (NX, Ny, NZ, NM), flush=True)
    st = lambda seed, **kw: synthetic_state(NX, Ny, NZ, LX, LZ, FLUX, seed=seed, **kw)
    X = [[st(m, amp=0.05) for m in range(NM)], [st(10 + m, unit=True) for m in range(NM)],
         [st(20 + m, unit=True) for m in range(NM)]]
    cc.sc_set_members(NM)
    assert cc.c_init(NX, Ny, NZ, LX, LZ, RE, FLUX, DT, 1) == 0
    dev = [cc.DeviceArray(np.ascontiguousarray(np.stack(x))) for x in X]
    try:
        cc.sc_primal_members(0, dev[0])
        cc.sc_tangent_members(0, 1, dev[1], 0, False)
        cc.sc_adjoint_members(1, 0, dev[2], 1.0, False)
        got = [x.download() for x in dev]
    finally:
        for x in dev:
            x.free()
    cc.sc_set_members(1)
    assert cc.c_init(NX, Ny, NZ, LX, LZ, RE, FLUX, DT, 1) == 0
    for m in range(NM):
        C, I, A = (x[m].copy() for x in X)
        cc.c_primal(0, C)
        cc.c_tangent(0, 1, I, 0)
        cc.c_adjoint(1, 0, A, 0, 1.0)
        for g, r in zip(got, (C, I, A)):
            assert np.isfinite(r).all()
            np.testing.assert_array_equal(g[m], r)
