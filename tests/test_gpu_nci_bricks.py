"""The node bricks of the promolecular and tricubic kernels at the edges of
their tiles, in both output orders, against the oracle; the tolerances are
those of tests/test_gpu_nci.py for the same quantities."""
import numpy as np
import pytest

from critic2_amd import nci as gn
from critic2_amd.radial import slater_grid1
from critic2_amd.synth import random_cell
from oracle import oracle

from helpers import images, node_points

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1, 1), (4, 8, 8), (8, 8, 4), (5, 9, 9), (3, 17, 7), (13, 2, 18)]


def _swap(a, n):
    """x-fastest values in z-fastest order."""
    return a.reshape(n[::-1]).transpose(2, 1, 0).reshape(-1)


@pytest.mark.parametrize("n", GRIDS)
@pytest.mark.parametrize("nat,edge", [(2, 5.0), (60, 9.0)])
def test_promol_bricks(ctx, n, nat, edge):
    """Few images, and more than the 512 staged at a time."""
    cell = random_cell(300 + nat, (edge, edge + 0.5, edge + 1.0), (85, 95, 100), nat, (1, 6, 7, 8), n,
                       min_sep_ang=1.2)
    print(f"[case] promol bricks n={n} atoms={nat}", flush=True)
    zs = sorted(set(int(z) for z in cell.zat))
    tables = [slater_grid1(z) for z in zs]
    species = np.array([zs.index(int(z)) for z in cell.zat], dtype=np.int32)
    pos, idx = images(cell.x2c, cell.xat, lim=3)
    ref = oracle.promol_nci_batch(node_points(cell.x2c, n), pos, species[idx],
                                  [oracle.Table(g.r, g.f, g.fp, g.fpp, g.cutrad) for g in tables])
    for prec, tol in (("fp64", 1e-12), ("fp32", 1e-5)):
        crho, s = gn.nciplot_promol(ctx, n, cell.x2c, tables, cell.xat, species, precision=prec)
        np.testing.assert_allclose(np.abs(crho), np.abs(ref[:, 3]), rtol=tol, atol=1e-10)
        assert np.mean(np.sign(crho) == np.sign(ref[:, 3])) > 0.99
        cx, sx = gn.nciplot_promol(ctx, n, cell.x2c, tables, cell.xat, species, precision=prec, zfast=False)
        assert np.array_equal(_swap(cx, n), crho) and np.array_equal(_swap(sx, n), s)
        if prec == "fp64":
            ok = ref[:, 0] > 1e-12
            np.testing.assert_allclose(s[ok], ref[ok, 2], rtol=1e-9)


@pytest.mark.parametrize("n", [(2, 2, 2), (3, 2, 5), (4, 8, 8), (8, 8, 4), (5, 9, 11), (13, 12, 17)])
def test_tricubic_bricks(ctx, n):
    print(f"[case] tricubic bricks n={n}", flush=True)
    cell = random_cell(310, (6.5, 7.5, 8.5), (75, 95, 115), 3, (1, 6, 7, 8), n)
    f = np.random.default_rng(sum(n)).uniform(0.5, 1.5, size=int(np.prod(n)))
    crho, s = gn.nciplot_grid(ctx, f, n, cell.x2c, interpolation="grid")
    cr_ref, s_ref = oracle.nci_grid_interp(f, n, cell.x2c)
    np.testing.assert_allclose(np.abs(crho), np.abs(cr_ref), rtol=1e-8)
    np.testing.assert_allclose(s, s_ref, rtol=1e-8, atol=1e-8)
    assert np.array_equal(np.sign(crho), np.sign(cr_ref))
    cx, sx = gn.nciplot_grid(ctx, f, n, cell.x2c, interpolation="grid", zfast=False)
    assert np.array_equal(_swap(cx, n), crho) and np.array_equal(_swap(sx, n), s)
