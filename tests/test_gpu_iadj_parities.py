"""The incremental adjoint stage's band rows couple rows of one parity of one
column: an infinity in the first or last row of alpha or beta of one column leaves
the other parity's rows of that column, and every row of the other columns, as
they are without it, bit for bit (stage 0, whose explicit operator reads the given
coefficients, and whose next explicit part reads the solved ones)."""
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


@pytest.mark.parametrize("Ny", [9, 12, 33, 98])
def test_infinite_row(cc, Ny):
    Nx, Nz = 12, 8
    print("case: parities of the incremental stage, %dx%dx%d" % (Nx, Ny, Nz), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=seed, **kw)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
    cc.c_primal(0, st(0, amp=0.05))
    cc.c_tangent(0, 1, st(1, unit=True), 0)
    q, nR, nQ, Mx = 3 * Ny // 2, Ny - 2, Ny - 4, Nx // 2
    rng = np.random.default_rng(Ny)
    noise = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    IAC, IU, LIU, W = noise(Nz, 2, nR, Mx), noise(Nz, 5, q, Mx), noise(Nz, 5, q, Mx), noise(6, Nz, Mx)

    def stage(A):
        A = A.copy()
        cc.sc_increadjproject(0, 1, A, IU.copy(), LIU.copy(), W.copy())
        return A

    ref = stage(IAC)
    assert np.isfinite(np.delete(ref, Nz // 2, 0)).all()
    z, x = 2, 3
    for var, N in ((0, nQ), (1, nR)):
        for row in (0, 1, N - 2, N - 1):
            A = IAC.copy()
            A[z, var, row, x] = np.inf
            got = stage(A)
            assert not np.isfinite(got[z, var, row % 2:N:2, x]).all()
            other = np.arange(1 - row % 2, N, 2)
            assert np.array_equal(got[z, var, other, x], ref[z, var, other, x])
            got[z, var, :, x] = ref[z, var, :, x]
            assert np.array_equal(got[np.arange(Nz) != Nz // 2], ref[np.arange(Nz) != Nz // 2])
