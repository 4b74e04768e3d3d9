"""Tangent members along one trajectory in groups: grids of so many blocks that a
block takes several members one after the other (the next one's bins fetched
meanwhile, the tile used again), all of them in one group and two or three groups of
unequal size, both precisions, against the single runs, bit for bit; and the same
launches recorded in a graph and replayed."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002

# rows of a block by x length, and 1024 blocks over all groups
ROWS = {48: 8, 72: 5, 96: 4, 120: 3}
# Nx, Ny, Nz, members, groups
CASES = [(32, 65, 32, 4, 1), (32, 43, 32, 5, 2), (48, 40, 20, 3, 2), (64, 50, 20, 3, 1), (64, 27, 20, 7, 3),
         (80, 30, 18, 3, 2)]


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_graphs(0)
    c_channel.sc_set_precision(0)
    c_channel.sc_set_members(1)
    c_channel.c_destroy()


def state(Nx, Ny, Nz, seed, **kw):
    return synthetic_state(Nx, Ny, Nz, LX, LZ, FLUX, seed=seed, **kw)


def groups(Nx, Ny, Nz, nm):
    blocks = -(-(3 * Ny // 2) * (3 * Nz // 2) // ROWS[3 * Nx // 2])
    return max(1, min(nm, 1024 // blocks))


def tangents(cc, C0, D, graphs):
    """Members' tangents along member 0's trajectory, once or (a graph) three times."""
    base = cc.DeviceArray(np.ascontiguousarray(np.stack([C0] * len(D))))
    out = []
    try:
        cc.sc_primal_members(0, base)
        cc.sc_set_graphs(graphs)
        for _ in range(3 if graphs else 1):
            dev = cc.DeviceArray(np.ascontiguousarray(np.stack(D)))
            try:
                cc.sc_tangent_members(0, 2, dev, 0b10, True)
                out.append(dev.download())
            finally:
                dev.free()
    finally:
        cc.sc_set_graphs(0)
        base.free()
    return out


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("Nx,Ny,Nz,nm,ng", CASES)
def test_groups_equal_single(cc, Nx, Ny, Nz, nm, ng, mixed):
    print("case: shared rows in groups, %dx%dx%d, %d members, mixed %d" % (Nx, Ny, Nz, nm, mixed), flush=True)
    assert groups(Nx, Ny, Nz, nm) == ng < nm
    C0, D = state(Nx, Ny, Nz, 0, amp=0.05), [state(Nx, Ny, Nz, 10 + m, unit=True) for m in range(nm)]
    cc.sc_set_precision(mixed)
    cc.sc_set_members(nm)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 2) == 0
    got = tangents(cc, C0, D, 0) + tangents(cc, C0, D, 1)
    cc.sc_set_members(1)
    assert cc.c_init(Nx, Ny, Nz, LX, LZ, RE, FLUX, DT, 2) == 0
    cc.c_primal(0, C0.copy())
    for m in range(nm):
        d = D[m].copy()
        cc.c_tangent(0, 2, d, 1 if m == 1 else 0)
        assert np.isfinite(d).all()
        for g in got:
            np.testing.assert_array_equal(g[m], d)
