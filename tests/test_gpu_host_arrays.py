"""Host arrays through the library's pinned chunks: a run of no steps returns its
state and stores it, exactly, for arrays below one chunk (1 MB), of two chunks, and
of more than the four that are in flight together; from pageable and from pinned
memory.  The physical fields of the same state agree between the two."""
import ctypes

import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.c_destroy()


@pytest.fixture
def pinned(cc):
    """Arrays in pinned memory of the runtime that the library is linked to."""
    held = []

    def zeros(shape, dtype):
        n = int(np.prod(shape)) * np.dtype(dtype).itemsize
        p = ctypes.c_void_p()
        assert cc._L.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(n), ctypes.c_uint(0)) == 0
        held.append(p)
        a = np.frombuffer((ctypes.c_char * n).from_address(p.value), dtype=dtype).reshape(shape)
        a[...] = 0
        return a

    yield zeros
    for p in held:
        cc._L.hipHostFree(p)


@pytest.mark.parametrize("Nx,Ny,Nz", [(8, 9, 8), (32, 68, 32), (64, 97, 64)])
def test_round_trip(cc, pinned, Nx, Ny, Nz):
    print("case: host arrays, %dx%dx%d" % (Nx, Ny, Nz), flush=True)
    assert cc.c_init(Nx, Ny, Nz, np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 0) == 0
    C0 = synthetic_state(Nx, Ny, Nz, np.pi, 0.5 * np.pi, 4.0 / 3.0, seed=3, amp=0.1)
    C0[Nz // 2] = 0                      # the Nyquist row holds no data
    shape = (3, 3 * Nx // 2, 3 * Ny // 2, 3 * Nz // 2)
    Cp = pinned(C0.shape, np.complex128)
    Cp[...] = C0
    flows = [np.zeros(shape), pinned(shape, np.float64)]
    for C, flow in zip((C0.copy(), Cp), flows):
        cc.c_primal(0, C)
        np.testing.assert_array_equal(C, C0)
        np.testing.assert_array_equal(cc.c_getsoln(0), C0)
        cc.c_spec2phys(C, flow)
        assert np.isfinite(flow).all() and np.abs(flow).max() > 0
    np.testing.assert_array_equal(flows[0], flows[1])
