"""An adjoint with cached fields (the first two stages' passes merged in one x kernel)
against one without: the same bits, but for the grids of 48 and 96 x points whose z
rows come in the groups of only one of the two kernels (4 of 8 rows, 2 of 4), where
the two round the first pass's twiddles in another order.

Bound there: ten times the difference of the oracle's two builds (with and without
FMA contraction) in one step of such grids, 2.2e-13."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT, NY = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 13


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_field_cache(1)
    c_channel.c_destroy()


@pytest.mark.parametrize("Nx,Nz,same", [(32, 16, True), (32, 20, True), (32, 24, False), (64, 16, True),
                                        (64, 20, False), (48, 20, True), (20, 18, True)])
def test_cached_adjoint(cc, Nx, Nz, same):
    print("case: cached adjoint, %dx%dx%d" % (Nx, NY, Nz), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, NY, Nz, LX, LZ, FLUX, seed=seed, **kw)
    out = []
    for cache in (1, 0):
        C, d, a = st(0, amp=0.05), st(1, unit=True), st(2, unit=True)
        cc.sc_set_field_cache(cache)
        assert cc.c_init(Nx, NY, Nz, LX, LZ, RE, FLUX, DT, 2) == 0
        assert cc.sc_field_cache_active() == cache
        cc.c_primal(0, C)
        cc.c_tangent(0, 2, d, 0)
        cc.c_adjoint(2, 0, a, 0, 1.0)
        out.append((C, d, a))
    for x, y in zip(out[0][:2 + same], out[1]):
        np.testing.assert_array_equal(x, y)
    assert np.linalg.norm(out[0][2] - out[1][2]) < 2.2e-12 * np.linalg.norm(out[1][2])
