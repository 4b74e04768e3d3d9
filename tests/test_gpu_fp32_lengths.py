"""The FP32 transforms at every x and z length with kernels of its own (and the
lengths 12, 216 and 6 without): a primal, tangent and adjoint step in mixed precision
against FP64, column by column (kz, kx).

A bin of the wrong value or place changes a column's increment over the step by the
order of that increment, whose smallest column has a thirtieth of the median or more
on these grids; FP32 rounding is far below.  Bounds, for the largest change of a
column, of the median increment:

* adjoint: the oracle's three adjoint stages on the same states with the products in
  plain numpy, once in FP64 and once with FP32 transforms and products, differ by the
  numbers of GRIDS (the forward transforms' rounding is the same in every bin and is
  then multiplied by the wavenumbers, so it is largest where those are and the states
  are small).  Ten times that, for the y-transform's FP32 products and another order.
* primal and tangent, whose products no wavenumber multiplies afterwards: with the
  fields and products of those stages rounded to FP32, but not the transforms, the
  change is 2e-6 to 1.2e-5 on ten of the grids; the transforms round some ten times
  more often, and as much again as a margin, 1e-3."""
import numpy as np
import pytest

from channel.synthetic import synthetic_state

pytestmark = pytest.mark.gpu

LX, LZ, RE, FLUX, DT, NY = np.pi, 0.5 * np.pi, 2000.0, 4.0 / 3.0, 0.002, 13

# Nx, Nz, the plain FP32 transforms' change of an adjoint column (of the median increment)
GRIDS = [(12, 10, 2.4e-05), (16, 12, 2.1e-05), (20, 18, 3.8e-05), (24, 16, 2.0e-05), (32, 20, 3.4e-05),
         (36, 24, 6.9e-05), (40, 30, 7.4e-05), (48, 32, 5.5e-05), (60, 36, 8.6e-05), (64, 40, 1.1e-04),
         (72, 48, 8.4e-05), (80, 50, 1.8e-04), (96, 54, 1.1e-04), (100, 60, 1.1e-04), (108, 64, 3.3e-04),
         (120, 72, 3.4e-04), (128, 80, 1.4e-04), (12, 90, 1.2e-03), (16, 96, 1.4e-03), (20, 100, 8.7e-04),
         (24, 108, 1.6e-03), (12, 120, 2.0e-03), (12, 128, 3.2e-03), (8, 12, 2.8e-05), (16, 144, 2.4e-03),
         (32, 4, 1.5e-05)]


@pytest.fixture(scope="module")
def cc():
    import c_channel
    yield c_channel
    c_channel.sc_set_precision(0)
    c_channel.c_destroy()


def columns(a, Nz):
    a = a[np.arange(Nz) != Nz // 2]
    return np.sqrt((np.abs(a) ** 2).sum(axis=(1, 2)))


@pytest.mark.parametrize("Nx,Nz,plain", GRIDS)
def test_mixed_step_by_column(cc, Nx, Nz, plain):
    print("case: FP32 lengths, %dx%dx%d" % (Nx, NY, Nz), flush=True)
    st = lambda seed, **kw: synthetic_state(Nx, NY, Nz, LX, LZ, FLUX, seed=seed, **kw)
    X0 = (st(0, amp=0.05), st(1, unit=True), st(2, unit=True))
    out = []
    for mixed in (0, 1):
        C, d, a = (x.copy() for x in X0)
        cc.sc_set_precision(mixed)
        assert cc.c_init(Nx, NY, Nz, LX, LZ, RE, FLUX, DT, 1) == 0
        cc.c_primal(0, C)
        cc.c_tangent(0, 1, d, 0)
        cc.c_adjoint(1, 0, a, 0, 0.0)
        out.append((C, d, a))
    for name, x0, r, g in zip(("primal", "tangent", "adjoint"), X0, *out):
        change, inc = columns(g - r, Nz), columns(r - x0, Nz)
        share = change.max() / np.median(inc)
        print("%s: %.1e of the median increment" % (name, share), flush=True)
        assert 0 < share < (10 * plain if name == "adjoint" else 1e-3), name
