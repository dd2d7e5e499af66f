"""What bench.py says about kernels, against the kernels that are launched."""
import json

import numpy as np
import pytest

import bench
from critic2_amd import nci as gn
from critic2_amd.synth import lattice_from_params

pytestmark = pytest.mark.gpu


def test_copy_probe_runs_the_kernel_it_names(ctx):
    ctx.timing(True)
    probe = json.loads(json.dumps(bench.copy_probe(ctx)))
    launched = ctx.kernel_times()
    ctx.timing(False)
    assert launched[probe["copy_probe"]][1] == 1
    assert probe["bytes_read"] == probe["bytes_written"] == 4 * probe["points"]


@pytest.mark.parametrize("n", [(12, 10, 8), (3500, 3, 2)])
@pytest.mark.parametrize("angles", [(90, 90, 90), (80, 95, 105)])
@pytest.mark.parametrize("scheme", ["fourier", "grid"])
def test_grid_nci_kernels_are_known(ctx, scheme, angles, n):
    x2c = lattice_from_params(7.0, 8.0, 9.0, *angles)
    f = 0.1 + np.random.default_rng(0).uniform(size=int(np.prod(n)))
    ctx.timing(True)
    gn.nciplot_grid(ctx, f, n, x2c, interpolation=scheme)
    launched = ctx.kernel_times()
    ctx.timing(False)
    assert launched
    for name in launched:
        assert bench.compulsory_bytes_per_point(name) == 16, name
