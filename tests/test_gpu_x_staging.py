"""The mixed-precision x transforms at the lengths whose bins come into LDS first
(24, 48, 96, 144, 192 points) and one whose do not (30): a primal, tangent and
adjoint step against the FP64 context's on the same input, on grids whose rows do
not fill the last block.

Bound: the oracle's two rounding orders differ by 2.2e-13 at most in one step of
these grids, which is what FP64 rounding (2^-53) grows to; FP32 transforms round at
2^-24, so ten times 2.2e-13 2^29 = 1.2e-3."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT, NY = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 13
BOUND = 10 * 2.2e-13 * 2.0 ** 29


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_precision(0)
    c_channel.c_destroy()


@pytest.mark.parametrize("Nx,Nz", [(16, 12), (20, 18), (32, 20), (64, 40), (96, 54), (128, 80)])
def test_mixed_step(cc, Nx, Nz):
    print("case: x staging, %dx%dx%d" % (Nx, NY, Nz), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, NY, Nz, LX, LZ, FLUX, seed=seed, **kw)
    out = []
    for mixed in (0, 1):
        C, d, a = st(0, amp=0.05), st(1, unit=True), st(2, unit=True)
        cc.sc_set_precision(mixed)
        assert cc.c_init(Nx, NY, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
        cc.c_primal(0, C)
        cc.c_tangent(0, 1, d, 0)
        cc.c_adjoint(1, 0, a, 0, 1.0)
        out.append((C, d, a))
    for g, r in zip(out[1], out[0]):
        assert 0 < np.linalg.norm(g - r) / np.linalg.norm(r) < BOUND
