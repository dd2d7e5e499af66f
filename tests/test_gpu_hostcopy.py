"""Large host transfers in chunks over several threads: every byte in its
place at the sizes where the path or the chunking changes, and cube files
written to a pipe."""
import os
import threading

import numpy as np
import pytest

from critic2_amd import cube as gc

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("nbytes", [1, 2 * MIB - 1, 2 * MIB, 2 * MIB + 1, 6 * MIB + 3, 12 * 4 * MIB + 5, 100 * MIB - 7])
def test_round_trip(ctx, nbytes):
    print(f"[case] hostcopy {nbytes}", flush=True)
    a = np.random.default_rng(nbytes).integers(0, 256, size=nbytes, dtype=np.uint8)
    d = ctx.to_device(a)
    assert np.array_equal(d.numpy(), a)
    d.free()


@pytest.mark.parametrize("nbytes", [7 * MIB - 1, 7 * MIB, 16 * MIB - 1, 16 * MIB, 16 * MIB + 1])
def test_round_trip_where_staging_begins(ctx, nbytes):
    test_round_trip(ctx, nbytes)


def test_cube_to_a_pipe(ctx, tmp_path):
    """A destination that cannot be written out of order gets the same bytes."""
    n = (40, 50, 60)
    f = np.random.default_rng(1).uniform(size=int(np.prod(n)))
    args = (n, (0.0, 0.0, 0.0), np.eye(3) * 0.1, [1], [[0.0, 0.0, 0.0]], f)
    gc.write_cube(ctx, str(tmp_path / "a.cube"), *args)
    want = (tmp_path / "a.cube").read_bytes()
    os.mkfifo(tmp_path / "pipe")
    got = []
    t = threading.Thread(target=lambda: got.append((tmp_path / "pipe").read_bytes()))
    t.start()
    gc.write_cube(ctx, str(tmp_path / "pipe"), *args)
    t.join(30)
    assert got and got[0] == want
    assert gc.format_body(ctx, f, n) == want[len(want) - len(gc.format_body(ctx, f, n)):]
