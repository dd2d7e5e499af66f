"""The sign of a Hessian's middle eigenvalue as the NCI kernels take it
(eig_mid_negative, nci_dev.hpp), compiled for the CPU, against its closed form
and against 64-bit eigenvalues."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def signs(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("eig") / "eig_check")
    tests = os.path.join(ROOT, "tests")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(tests, "hip_stub"),
                    os.path.join(tests, "eig_check.cpp"), "-o", exe], check=True)

    def run(h, dtype):
        """(negative by the kernels' rule, negative by the closed form)"""
        h = np.ascontiguousarray(h, dtype=dtype)
        out = subprocess.run([exe, "float" if dtype == np.float32 else "double"], input=h.tobytes(),
                             stdout=subprocess.PIPE, check=True).stdout
        return np.frombuffer(out, dtype=np.int8).reshape(-1, 2).T.astype(bool)

    return run


def _matrices(n, seed):
    """h00 h11 h22 h01 h02 h12: random, nearly a multiple of 1, uniaxial (one
    atom's Hessian) and nearly uniaxial."""
    rng = np.random.default_rng(seed)
    near = rng.normal(size=(n, 6)) * 10.0 ** rng.uniform(-9, -1, size=(n, 1))
    near[:, :3] += rng.normal(size=(n, 1))
    v = rng.normal(size=(n, 3))
    v /= np.linalg.norm(v, axis=1)[:, None]
    uni = np.stack([v[:, 0] ** 2, v[:, 1] ** 2, v[:, 2] ** 2, v[:, 0] * v[:, 1], v[:, 0] * v[:, 2], v[:, 1] * v[:, 2]], 1)
    uni *= rng.normal(size=(n, 1)) * 10.0 ** rng.uniform(-3, 3, size=(n, 1))
    uni[:, :3] += rng.normal(size=(n, 1))
    return np.concatenate([rng.normal(size=(n, 6)), near, uni, uni + 1e-3 * rng.normal(size=(n, 6))])


def _eigenvalues(h):
    full = np.zeros((len(h), 3, 3))
    for k, (i, j) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
        full[:, i, j] = full[:, j, i] = h[:, k]
    return np.linalg.eigvalsh(full)


@pytest.mark.parametrize("dtype,scale", [(np.float32, s) for s in (-24, -20, -15, -8, 0, 8, 15, 20, 25)] +
                         [(np.float64, s) for s in (-165, -140, 0, 140, 160)])
def test_sign_of_the_middle_eigenvalue(signs, dtype, scale):
    """Where the eigenvalues are clear of zero the sign is theirs at any scale.
    Where the closed form's squares (of the entries, and of the traceless part
    that it divides by) are normal numbers the answer is its own, clear or
    not."""
    h = (_matrices(50000, 100 + abs(scale)) * 10.0 ** scale).astype(dtype)
    rule, closed = signs(h, dtype)
    e = _eigenvalues(h.astype(np.float64) / 10.0 ** scale)
    clear = np.abs(e).min(axis=1) > 1e-2 * np.sqrt((e * e).sum(axis=1))
    assert clear.mean() > 0.8
    np.testing.assert_array_equal(rule[clear], e[clear, 1] < 0)
    traceless = np.std(e, axis=1) * np.sqrt(3.0) * 10.0 ** scale
    end = 1e18 if dtype == np.float32 else 1e152
    normal = (traceless > 1 / end) & (np.abs(h).max(axis=1) < end)
    assert normal.any() or abs(scale) > 18
    np.testing.assert_array_equal(rule[normal], closed[normal])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_zeros_infinities_and_nan(signs, dtype):
    """The closed form's answer, whatever it is."""
    v = np.array([0.0, -0.0, 1.0, -1.0, np.inf, -np.inf, np.nan], dtype=dtype)
    h = np.stack(np.meshgrid(v, v, v, v, v, v, indexing="ij"), -1).reshape(-1, 6)
    special = ~np.isfinite(h).all(axis=1) | (h == 0).all(axis=1)
    rule, closed = signs(h[special], dtype)
    np.testing.assert_array_equal(rule, closed)
