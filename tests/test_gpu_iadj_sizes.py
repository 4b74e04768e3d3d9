"""The incremental adjoint stage at the ends of its range of sizes, against the
oracle: 97 to 128 omega_y coefficients (seven and eight groups of preloaded factor
rows, up to 74 KB of LDS, 148 to 195 Gauss points, the y-transform with a whole basis
in LDS) and Ny = 5 and 6, where a parity of alpha has no or one row; Mx a multiple of
8 (factors of mirrored kz rows shared) and no multiple of 4.

Bounds: ten times the largest difference of the oracle's two builds (with and without
FMA contraction) over the stages and their three output arrays on the same inputs,
each after its own primal and tangent runs, and 1e-13 at least."""
import numpy as np
import pytest

import pyorc
from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT, NSTEPS = np.pi, 0.3 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 2
SIZES = [(16, 5, 12, 1e-13), (12, 6, 10, 1e-13), (12, 99, 10, 6.8e-9), (16, 99, 12, 7.1e-9), (16, 115, 12, 2.6e-8),
         (12, 115, 10, 2.1e-8), (12, 129, 10, 7.2e-8), (16, 130, 8, 1.4e-7), (12, 130, 10, 6.8e-8)]


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.c_destroy()


@pytest.mark.parametrize("Nx,Ny,Nz,bound", SIZES)
def test_stages(cc, Nx, Ny, Nz, bound):
    o = pyorc.Oracle(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, NSTEPS)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, NSTEPS) == 0
    for lib in (o, cc):
        C = synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=3, amp=0.02)
        I = synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=4, unit=True)
        (o.primal if lib is o else cc.c_primal)(0, C)
        (o.tangent if lib is o else cc.c_tangent)(0, NSTEPS, I, 0)
    for k in range(3):
        for force in (False, True):
            print("case: incremental stage sizes, %dx%dx%d, k=%d force=%d" % (Nx, Ny, Nz, k, force), flush=True)
            rng = np.random.default_rng(10 * k + force)
            noise = lambda s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
            IAC, IU, LIU = noise(o.cshape), noise(o.ushape), noise(o.ushape)
            W = noise((6, Nz, Nx // 2))
            F = noise((2, 2, Nz, Nx // 2, o.dimR)) if force else None
            ref = o.increadjproject(k, 5 - k, IAC, IU, LIU, W, F)
            got = IAC.copy()
            IAU, IAUb = cc.sc_increadjproject(k, 5 - k, got, IU, None if k == 2 else LIU, W, F)
            for g, r in zip((got, IAU, IAUb), ref):
                assert np.linalg.norm(g - r) / np.linalg.norm(r) < bound, (k, force)
    o.destroy()
