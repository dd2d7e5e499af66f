"""The Fourier derivative grids over the edges at which their line transforms
change (radices, circulant edges, tile remainders, the longest line, the 3-D
transform beyond it) and over cell shapes, against the oracle's numpy FFT.

The fields are white noise, whose second derivatives are of the size of the
largest multiplier, so the round-off of either side is a few tens of 2.2e-16
of the largest value: 1e-12 of it is asserted.  The circulant edges are also
held to the 3-D transform's own round-off, on lines of atom-like peaks and of
noise, against 80-bit sums."""
import functools

import numpy as np
import pytest

from critic2_amd import _lib
from critic2_amd import bader as gb
from critic2_amd import nci as gn
from critic2_amd.synth import lattice_from_params
from oracle import oracle

pytestmark = pytest.mark.gpu

ORTHO = np.diag([7.0, 8.0, 9.0])
TRI = lattice_from_params(7.0, 8.0, 9.0, 80, 100, 110)
MONO = lattice_from_params(7.0, 8.0, 9.0, 90, 105, 90)
PERM = np.array([[0.0, 0.0, 9.0], [-7.0, 0.0, 0.0], [0.0, 8.0, 0.0]])  # axes along z, x (negative), y
CELLS = {"ortho": ORTHO, "ortho_angles": lattice_from_params(7.0, 8.0, 9.0, 90, 90, 90), "triclinic": TRI,
         "monoclinic": MONO, "permuted": PERM}
GRIDS = [
    (1, 2, 3), (2, 2, 2), (3, 1, 4), (5, 4, 7),   # the smallest edges
    (16, 15, 17), (17, 33, 31), (18, 49, 10),      # remainders of the 16-column tiles; primes
    (64, 9, 35), (11, 128, 22), (26, 13, 96),      # circulant edges, even and odd, on each axis
    (512, 6, 5), (3, 640, 4), (6, 5, 1024), (101, 4, 1001),  # fewer line pairs a workgroup
    (3375, 3, 2), (2, 3, 2048), (3391, 2, 3),      # 3375 = 5^3 3^3 needs too many threads: the 3-D transform
    (3500, 3, 2),                                  # the 3-D transform
    # one pair a workgroup: mixed radices with all 512 threads, and circulant
    # edges up to the longest, whose column tiles fill the LDS
    (2560, 3, 2), (3, 2560, 2), (3072, 2, 3), (2, 3, 3072), (2, 3391, 3), (3, 2, 3391), (3400, 2, 2), (2, 3400, 3),
    (3, 2, 3400),
    (2, 2625, 3), (3087, 2, 3),                    # the first with a factor 5, 3 past 512 threads: the 3-D transform
]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("cell", ["ortho_angles", "triclinic"])
def test_edges(ctx, cell, grid):
    print(f"[case] fourier {cell} {grid}", flush=True)
    f = np.random.default_rng(sum(grid)).normal(size=int(np.prod(grid)))
    for kind, name in ((_lib.FT_GRAD, "grad"), (_lib.FT_YY, "yy"), (_lib.FT_LAP, "lap")):
        g = gb.fft_deriv(ctx, f, grid, CELLS[cell], kind)
        o = oracle.fft_deriv(f, grid, CELLS[cell], name)
        assert np.abs(g - o).max() <= 1e-12 * max(np.abs(o).max(), 1e-3), name


@pytest.mark.parametrize("cell", sorted(CELLS))
@pytest.mark.parametrize("grid", [(12, 14, 18), (15, 20, 11), (21, 9, 25)])
def test_cells(ctx, cell, grid):
    """Every kind and nciplot's node values in both layouts."""
    print(f"[case] fourier {cell} {grid}", flush=True)
    f = 0.1 + np.random.default_rng(sum(grid)).uniform(size=int(np.prod(grid)))
    x2c = CELLS[cell]
    d = {}
    for kind, name in ((_lib.FT_GRAD, "grad"), (_lib.FT_XX, "xx"), (_lib.FT_YY, "yy"), (_lib.FT_ZZ, "zz"),
                       (_lib.FT_LAP, "lap")):
        d[name] = oracle.fft_deriv(f, grid, x2c, name)
        assert np.abs(gb.fft_deriv(ctx, f, grid, x2c, kind) - d[name]).max() <= 1e-12 * np.abs(d[name]).max(), name
    crho, s = gn.nciplot_grid(ctx, f, grid, x2c, zfast=False)
    ref = d["grad"] / (2 * (3 * np.pi ** 2) ** (1 / 3) * f ** (4 / 3))
    np.testing.assert_allclose(s, ref, rtol=1e-10, atol=1e-12 * ref.max())
    up = sum((d[q] > 0).astype(int) for q in ("xx", "yy", "zz"))
    clear = np.min([np.abs(d[q]) / np.abs(d[q]).max() for q in ("xx", "yy", "zz")], axis=0) > 1e-11
    assert np.array_equal(crho[clear], np.where(up >= 2, f, -f)[clear] * 100.0)
    cz, sz = gn.nciplot_grid(ctx, f, grid, x2c)
    for z, x in ((cz, crho), (sz, s)):
        assert np.array_equal(z.reshape(grid), x.reshape(grid[::-1]).transpose(2, 1, 0))


@pytest.mark.parametrize("cell", ["ortho", "triclinic"])
@pytest.mark.parametrize("grid", [(2560, 2, 3), (2, 3, 3072), (3, 3391, 2), (2, 3, 3400),   # the longest lines
                                  (3000, 2, 3), (2, 3, 3375), (3500, 3, 2)])                # the 3-D transform
def test_nci_of_long_edges(ctx, cell, grid):
    test_cells(ctx, cell, grid)


LD = np.longdouble


@functools.lru_cache(None)
def _circulant(n):
    """First columns, in 80 bits, of the matrices of d/dx and d2/dx2 on n
    points of a period 2 pi, summed from their definitions."""
    k = np.arange(n)
    pi = 4 * np.arctan(LD(1))
    sin, cos = np.sin(2 * pi * k / LD(n)), np.cos(2 * pi * k / LD(n))
    d, s = np.zeros(n, LD), np.zeros(n, LD)
    for m in range(1, (n + 1) // 2):
        mk = m * k % n
        d -= 2 * m * sin[mk]
        s -= 2 * m * m * cos[mk]
    if n % 2 == 0:
        s -= (n // 2) ** 2 * np.where(k % 2, LD(-1), LD(1))
    return d / n, s / n


def _apply(col, f):
    n = f.size
    out = np.zeros(n, LD)
    for j in range(n):
        out += np.roll(col, j) * f[j]
    return out


def _line(n, kind):
    rng = np.random.default_rng(n)
    if kind == "noise":
        return rng.normal(size=n)
    f, length = np.zeros(n), 0.19 * n  # bohr
    for x, z in zip(rng.uniform(size=max(2, n // 30)), rng.choice([1.0, 2.0, 3.0, 4.0], size=max(2, n // 30))):
        d = np.abs(np.arange(n) / n - x)
        d = np.minimum(d, 1 - d) * length
        f += z ** 3 * np.exp(-2 * z * np.sqrt(d * d + 0.01))
    return f


@pytest.mark.parametrize("kind", ["peaks", "noise"])
@pytest.mark.parametrize("n", [34, 127, 211, 509, 1408, 3391])
def test_circulant_edges_are_as_exact_as_the_3d_transform(ctx, n, kind):
    """The same line on each axis of a small grid, and beside an edge of 3500,
    which takes the 3-D transform.  The circulant sums are of 64 terms at a
    time, so their error is that of the entries, a few 2.2e-16 of the largest
    value for any n, and the transform's is 1e-15 to 3e-15: twice the
    transform's error is allowed, and 1e-15 in any case."""
    print(f"[case] circulant edge {n} {kind}", flush=True)
    f = _line(n, kind)
    col_d, col_s = _circulant(n)
    b = 2 * np.pi / 8.0
    want = {_lib.FT_GRAD: np.abs(_apply(col_d, f)) * b, _lib.FT_YY: _apply(col_s, f) * b * b}

    def error(grid, axis, kind):
        shape = [1, 1, 1]
        shape[2 - axis] = n  # x fastest
        full = np.broadcast_to(f.reshape(shape), grid[::-1])
        x2c = np.diag([8.0 if a == axis else 1e7 for a in range(3)])
        if kind == _lib.FT_YY:
            kind = (_lib.FT_XX, _lib.FT_YY, _lib.FT_ZZ)[axis]
            ref = want[_lib.FT_YY]
        else:
            ref = want[kind]
        got = gb.fft_deriv(ctx, full, grid, x2c, kind).reshape(grid[::-1])
        return float(np.abs(got - ref.reshape(shape)).max() / np.abs(ref).max())

    for kind_ in (_lib.FT_GRAD, _lib.FT_YY):
        allowed = max(2 * error((3500, n, 1), 1, kind_), 1e-15)
        for axis in range(3):
            grid = [2, 3, 4]
            grid[axis] = n
            assert error(tuple(grid), axis, kind_) <= allowed, (kind_, axis)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("cell", ["ortho", "permuted", "triclinic"])
@pytest.mark.parametrize("grid", [(12, 14, 18), (11, 9, 26)])
def test_non_finite_grids(ctx, cell, grid, value):
    """One NaN or infinity makes every derivative NaN and leaves crho the sign
    of no positive second derivative, as a 3-D transform does; the next call on
    a finite grid is as if that one had not been."""
    print(f"[case] fourier non-finite {cell} {grid} {value}", flush=True)
    x2c = CELLS[cell]
    f = 0.1 + np.random.default_rng(1).uniform(size=int(np.prod(grid)))
    kinds = (_lib.FT_GRAD, _lib.FT_XX, _lib.FT_YY, _lib.FT_ZZ, _lib.FT_LAP)
    before = [gb.fft_deriv(ctx, f, grid, x2c, k) for k in kinds] + list(gn.nciplot_grid(ctx, f, grid, x2c))
    for at in (0, f.size // 2 + 3, f.size - 1):
        bad = f.copy()
        bad[at] = value
        for k in kinds:
            assert np.isnan(gb.fft_deriv(ctx, bad, grid, x2c, k)).all(), (at, k)
        crho, s = gn.nciplot_grid(ctx, bad, grid, x2c, zfast=False)
        assert np.isnan(s).all()
        np.testing.assert_array_equal(crho, -np.abs(bad) * 100.0)
    after = [gb.fft_deriv(ctx, f, grid, x2c, k) for k in kinds] + list(gn.nciplot_grid(ctx, f, grid, x2c))
    for a, b in zip(before, after):
        np.testing.assert_array_equal(a, b)


def test_non_finite_grids_of_the_3d_transform(ctx):
    """The same from the 3-D transform itself."""
    grid = (3500, 3, 2)
    f = 0.1 + np.random.default_rng(2).uniform(size=int(np.prod(grid)))
    f[17] = np.nan
    assert np.isnan(gb.fft_deriv(ctx, f, grid, TRI, _lib.FT_LAP)).all()
    crho, s = gn.nciplot_grid(ctx, f, grid, TRI, zfast=False)
    assert np.isnan(s).all()
    np.testing.assert_array_equal(crho, -np.abs(f) * 100.0)
