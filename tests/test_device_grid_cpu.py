"""fft_deriv and intgrid_fields refuse a grid in HBM that does not hold the
doubles the library would read, before any of it is passed on.  The grids are
stand-ins with a device array's attributes; no GPU is used."""
import numpy as np
import pytest

from critic2_amd import _lib
from critic2_amd import bader as gb

N = (4, 5, 6)
NPTS = 120


class Grid:
    is_cuda = True

    def __init__(self, dtype="torch.float64", size=NPTS, contiguous=True, index=0):
        self.dtype, self.size, self.contiguous = dtype, size, contiguous
        self.device = type("device", (), {"index": index})()

    def data_ptr(self):
        raise AssertionError("the address of a refused grid was taken")

    def numel(self):
        return self.size

    def is_contiguous(self):
        return self.contiguous


class Ctx:
    device = 0

    def __getattr__(self, name):
        raise AssertionError(f"the context's {name} was used for a refused grid")


BAD = {"float32": (dict(dtype="torch.float32"), TypeError), "int64": (dict(dtype="torch.int64"), TypeError),
       "numpy float32": (dict(dtype=np.dtype("float32")), TypeError),
       "one short": (dict(size=NPTS - 1), ValueError), "strided": (dict(contiguous=False), TypeError),
       "another GPU": (dict(index=1), ValueError)}


@pytest.mark.parametrize("what", sorted(BAD))
def test_unfit_device_grids_are_refused(what):
    attrs, error = BAD[what]
    with pytest.raises(error):
        gb.fft_deriv(Ctx(), Grid(**attrs), N, np.eye(3), _lib.FT_LAP)
    bas = gb.BasinData(n=N, nattr=1, idg=np.ones(NPTS, dtype=np.int32))
    with pytest.raises(error):
        gb.intgrid_fields(Ctx(), bas, Grid(**attrs), np.eye(3), lap=True)


@pytest.mark.parametrize("grid", [Grid(), Grid(size=NPTS + 7), Grid(dtype=np.dtype("float64"))])
def test_fit_device_grids_pass(grid):
    gb._check_device_grid(Ctx(), grid, NPTS)
