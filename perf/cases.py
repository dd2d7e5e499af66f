"""Measured workloads of this repository, through its public entry points.

Each case is a call (or the short sequence of calls) that a user of the
BADER, NCIPLOT, YT and cube keywords makes on one density.  Grids are FP64
Slater-sum densities of seeded random cells at crystal-like atom densities
(about 8 atoms per 1000 cubic angstrom) and grid spacings of 0.06-0.16
angstrom; batches and nciplot boxes use the dimer cells of synth.batch_cells.
Grids stay resident on the GPU, except in the "keyword" cases, which take
host arrays as critic2 itself holds them, and in the cube cases, which start
from a file or end in host text.
"""
from __future__ import annotations

import functools
import math
import os
import tempfile
import weakref

import numpy as np
import torch

from critic2_amd import _lib, synth
from critic2_amd import bader as gb
from critic2_amd import batch as gq
from critic2_amd import cube as gc
from critic2_amd import nci as gn
from critic2_amd import yt as gy
from critic2_amd.radial import BOHR_PER_ANG, slater_grid1

ZSET = (1, 6, 7, 8)
DEV = "cuda"


def _case(name, kind, n, h=None, edges=None, angles=(90.0, 90.0, 90.0), nat=None, **more):
    """A crystal case: grid n, cell edges in angstrom (or the grid spacing h)."""
    e = tuple(edges) if edges else tuple(max(4.0, h * v) for v in n)
    al, be, ga = (math.cos(math.radians(t)) for t in angles)
    vol = e[0] * e[1] * e[2] * math.sqrt(1 - al * al - be * be - ga * ga + 2 * al * be * ga)
    c = {"kind": kind, "n1": n[0], "n2": n[1], "n3": n[2], "a": e[0], "b": e[1], "c": e[2],
         "alpha": angles[0], "beta": angles[1], "gamma": angles[2],
         "nat": nat or max(2, min(216, round(0.008 * vol))), "volume": vol, **more}
    return {"name": name, **c} if name else c


def listed():
    tri = (77.0, 95.0, 104.0)
    return [
        # BADER on the smallest grid in use: latency and launches count
        _case("bader_64", "bader", (64, 64, 64), edges=(10.0, 10.0, 10.0), nat=8, mode="default"),
        # BADER as the benchmark runs it: labels and Volume/Pop of a large cell
        _case("bader_512", "bader", (512, 512, 512), edges=(30.0, 30.0, 30.0), nat=216, mode="default"),
        # critic2's own call order on host arrays: BADER with the Laplacian
        # integrated, then INTEGRABLE ... MULTIPOLE
        _case("keyword_host_150x135x128", "keyword", (150, 135, 128), h=0.11, lmax=5),
        # NCIPLOT on the promolecular density, mixed precision, the benchmark's grid
        _case("promol_fp32_512", "promol", (512, 512, 512), edges=(30.0, 30.0, 30.0), nat=216, precision="fp32"),
        # NCIPLOT with two FRAGMENTs in the box around a dimer, FP64: density,
        # fragment densities, cutoffs and the .dat text
        {"name": "nciplot_box_161x143x178", "kind": "box", "n1": 161, "n2": 143, "n3": 178},
        # NCIPLOT on a loaded grid, the default Fourier scheme
        _case("nci_fourier_256", "fourier", (256, 256, 256), edges=(20.0, 20.0, 24.0), nat=64),
        # the same on a triclinic cell with a ragged grid
        _case("nci_fourier_135x120x98_triclinic", "fourier", (135, 120, 98), h=0.12, angles=tri),
        # NCIPLOT with INTERPOLATION GRID
        _case("nci_tricubic_192x180x160_triclinic", "tricubic", (192, 180, 160), h=0.10, angles=tri),
        # YT with Pop and MULTIPOLE
        _case("yt_200x192x240", "yt", (200, 192, 240), h=0.10, lmax=5),
        # LOAD of a cube file into HBM
        _case("cube_read_200x180x192", "cube_read", (200, 180, 192), h=0.10, style=_lib.CUBE_E22_14),
        # the body of a cube file written from HBM
        _case("cube_format_256x250x243", "cube_format", (256, 250, 243), h=0.08, style=_lib.CUBE_E22_14),
        # many small molecules in one call
        {"name": "batch_16_dimers", "kind": "batch", "cells": 16, "first": 0},
    ]


#: kind: (smallest edge, largest edge, most points) of drawn cases
RANGES = {"bader": (48, 512, 512 ** 3), "keyword": (40, 200, 160 ** 3), "promol": (48, 512, 512 ** 3),
          "box": (40, 200, 180 ** 3), "fourier": (24, 320, 256 ** 3), "tricubic": (24, 320, 256 ** 3),
          "yt": (40, 256, 210 ** 3), "cube_read": (24, 256, 200 ** 3), "cube_format": (24, 320, 256 ** 3),
          "batch": (2, 18, 0)}


def _smooth(v):
    while any(v % p == 0 for p in (2, 3, 5, 7)):
        for p in (2, 3, 5, 7):
            v = v // p if v % p == 0 else v
    return v == 1


def draw(rng):
    kind = rng.choice(sorted(RANGES))
    lo, hi, most = RANGES[kind]
    if kind == "batch":
        return {"kind": "batch", "cells": rng.randint(lo, hi), "first": 16 * rng.randint(1, 30)}
    while True:
        # one size for the grid, each edge up to a third off it
        size = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        n = tuple(min(hi, max(lo, round(size * math.exp(rng.uniform(-0.3, 0.3))))) for _ in range(3))
        if n[0] * n[1] * n[2] <= most:
            break
    if kind == "box":
        return {"kind": "box", "n1": n[0], "n2": n[1], "n3": n[2]}
    if kind == "fourier" and rng.random() < 0.75:  # plane-wave codes choose edges with small factors
        n = tuple(next(w for w in range(v, 2 * v) if _smooth(w)) for v in n)
    more = {}
    if kind == "bader":
        more["mode"] = rng.choice(("default", "default", "nnm", "noatoms"))
    if kind in ("keyword", "yt"):
        more["lmax"] = rng.choice((2, 4, 5))
    if kind == "promol":
        more["precision"] = rng.choice(("fp32", "fp64"))
    if kind == "cube_read":
        more["style"] = rng.choice((_lib.CUBE_E22_14, _lib.CUBE_1P_E12_5))
    if kind == "cube_format":
        more["style"] = rng.choice((_lib.CUBE_E22_14, _lib.CUBE_1P_E12_5, _lib.CUBE_1P_E13_5))
    angles = tuple(rng.uniform(70.0, 110.0) for _ in range(3)) if rng.random() < 0.5 else (90.0, 90.0, 90.0)
    return _case(None, kind, n, h=rng.uniform(0.06, 0.12 if max(n) > 256 else 0.16), angles=angles, **more)


# ------------------------------------------------------------------ inputs


@functools.lru_cache(None)
def _ctx():
    return _lib.Context(0)


@functools.lru_cache(None)
def _tables():
    return [slater_grid1(z) for z in ZSET]


def _n(case):
    return case["n1"], case["n2"], case["n3"]


def _npts(case):
    return case["n1"] * case["n2"] * case["n3"]


def _species(zat):
    return np.array([ZSET.index(int(z)) for z in zat], dtype=np.int32)


def _crystal(case, seed):
    return synth.random_cell(1 + seed, (case["a"], case["b"], case["c"]),
                             (case["alpha"], case["beta"], case["gamma"]), case["nat"], ZSET, _n(case))


def _empty(npts, dtype):
    return torch.empty(npts, dtype=dtype, device=DEV)


def _density(cell):
    rho = _empty(cell.npts, torch.float64)
    gb.synth_slater(_ctx(), cell, device_out=rho)
    return rho


def _monomers(cell):
    """Atom indices of the two molecules of a dimer cell (bonds below 2 A)."""
    xyz = cell.xat @ cell.x2c.T
    near = np.linalg.norm(xyz[:, None] - xyz[None], axis=2) < 2.0 * BOHR_PER_ANG
    first = np.zeros(len(xyz), dtype=bool)
    first[0] = True
    for _ in range(len(xyz)):
        first |= near[first].any(axis=0)
    return xyz, [m for m in (np.flatnonzero(first), np.flatnonzero(~first)) if m.size]


class _Held:
    """A library-owned device array seen as a torch tensor."""

    def __init__(self, d):
        self.held = d
        self.__cuda_array_interface__ = {"shape": d.shape, "typestr": d.dtype.str, "data": (d.data_ptr(), False),
                                         "version": 3}


def _tensor(d):
    return torch.as_tensor(_Held(d), device=DEV)


class _File:
    """A file that goes with the object."""

    def __init__(self):
        fd, self.path = tempfile.mkstemp(suffix=".cube")
        os.close(fd)
        weakref.finalize(self, os.unlink, self.path)


def prepare(case, seed):
    kind, ctx = case["kind"], _ctx()
    if kind == "batch":
        # snapshots of the same molecules: the atoms 0.05 A about their places
        cells = synth.batch_cells(case["cells"], base_seed=1000 + case["first"])
        rng = np.random.default_rng(seed)
        for c in cells:
            c.xat = c.xat + rng.normal(scale=0.05 * BOHR_PER_ANG, size=c.xat.shape) / np.diag(c.x2c)
        return {"kind": kind, "cells": cells, "grids": [_density(c) for c in cells],
                "species": [_species(c.zat) for c in cells]}
    npts = _npts(case)
    if kind == "box":
        cell = synth.batch_cells(1, base_seed=70000 + seed)[0]
        sp = _species(cell.zat)
        xyz, mono = _monomers(cell)
        frags = [(xyz[m], sp[m]) for m in mono]
        return {"kind": kind, "cell": cell, "species": sp, "frags": frags,
                "nodes": gn.fragment_box(frags, nstep=_n(case)),
                "outs": tuple(_empty(npts, torch.float64) for _ in range(3)),
                "dat": np.zeros(31 * npts, dtype=np.uint8),  # a text buffer for the most rows there can be
                "rhofrag": torch.empty((len(frags), npts), dtype=torch.float64, device=DEV)}
    cell = _crystal(case, seed)
    s = {"kind": kind, "cell": cell, "case": case}
    if kind == "promol":
        dt = torch.float32 if case["precision"] == "fp32" else torch.float64
        s.update(species=_species(cell.zat), outs=tuple(_empty(npts, dt) for _ in range(2)))
        return s
    s["rho"] = _density(cell)
    if kind == "bader":
        s["labels"] = _empty(npts, torch.int32)
    elif kind == "keyword":
        s["rho"] = s["rho"].cpu().numpy()
    elif kind in ("fourier", "tricubic"):
        s["outs"] = tuple(_empty(npts, torch.float64) for _ in range(2))
    elif kind == "cube_read":
        s["file"] = _File()
        gc.write_cube(ctx, s["file"].path, cell.n, (0.0, 0.0, 0.0), cell.x2c / np.array(cell.n), cell.zat,
                      cell.xat @ cell.x2c.T, s.pop("rho"), case["style"])
    return s


# ------------------------------------------------------------------ one pass


def run(s):
    kind, ctx = s["kind"], _ctx()
    if kind == "batch":
        res, _ = gq.batch_run(ctx, s["cells"], s["grids"], _tables(), s["species"])
        return {"cells": [{k: _tensor(r[k]) for k in ("labels", "crho", "cgrad")} for r in res],
                "counts": np.concatenate([r["counts"] for r in res]), "sums": np.concatenate([r["sums"] for r in res])}
    cell = s["cell"]
    if kind == "box":
        crho, cgrad, rhoat = gn.promol_nodes(ctx, s["nodes"], cell.x2c, _tables(), cell.xat, s["species"],
                                             precision="fp64", outs=s["outs"])
        rhofrag = gn.fragments(ctx, s["nodes"], _tables(), s["frags"], precision="fp64", out=s["rhofrag"])
        dat, sums = gn.cutoffs(ctx, crho, cgrad, rhoat=rhoat, rhofrag=rhofrag)
        s["dat"][:len(dat)] = np.frombuffer(dat, dtype=np.uint8)
        return {"crho": crho, "cgrad": cgrad, "rhoat": rhoat, "rhofrag": rhofrag, "dat": s["dat"], "sums": sums}
    if kind == "promol":
        crho, cgrad = gn.nciplot_promol(ctx, cell.n, cell.x2c, _tables(), cell.xat, s["species"],
                                        precision=s["case"]["precision"], outs=s["outs"])
        return {"crho": crho, "cgrad": cgrad}
    if kind == "bader":
        mode = s["case"]["mode"]
        bas = gb.bader_integrate(ctx, s["rho"], cell.n, cell.x2c, cell.xat, nnm=mode == "nnm",
                                 noatoms=mode == "noatoms", labels_out=s["labels"])
        props = gb.intgrid_fields(ctx, bas, s["rho"], cell.x2c, lap=False)
        return {"labels": bas.idg, "xattr": bas.xattr, **props}
    if kind == "keyword":
        bas, props = gb.bader(ctx, s["rho"], cell.n, cell.x2c, cell.xat)
        mp = gb.multipoles(ctx, bas.idg, s["rho"], cell.n, cell.x2c, bas.xattr, s["case"]["lmax"])
        return {"labels": bas.idg, "xattr": bas.xattr, "multipoles": mp, **props}
    if kind in ("fourier", "tricubic"):
        crho, cgrad = gn.nciplot_grid(ctx, s["rho"], cell.n, cell.x2c, outs=s["outs"],
                                      interpolation="fourier" if kind == "fourier" else "grid")
        return {"crho": crho, "cgrad": cgrad}
    if kind == "yt":
        r = gy.yt_integrate(ctx, s["rho"], cell.n, cell.x2c, cell.xat, fields=[s["rho"]])
        mp = gy.yt_multipoles(ctx, r["labels"], s["rho"], cell.n, cell.x2c, r["xattr"], s["case"]["lmax"])
        return {"labels": _tensor(r["labels"]), "xattr": r["xattr"], "vol": r["vol"], "sums": r["sums"],
                "multipoles": mp}
    if kind == "cube_read":
        hdr, f = gc.read_cube(ctx, s["file"].path, device=True)
        return {"f": _tensor(f), "step": hdr["step"]}
    if kind == "cube_format":
        return np.frombuffer(gc.format_body(ctx, s["rho"], cell.n, s["case"]["style"]), dtype=np.uint8)
    raise ValueError(kind)


# ------------------------------------------------------------------ compulsory work


def _reach():
    """Mean volume (bohr^3) of the sphere an atom's table covers."""
    return float(np.mean([4.0 / 3.0 * math.pi * min(t.cutrad, t.rmax) ** 3 for t in _tables()]))


def work(case):
    kind = case["kind"]
    if kind == "batch":
        like = synth.batch_cells(case["cells"], base_seed=1000 + case["first"])
        npts = sum(c.npts for c in like)
        # grid in; labels and FP32 crho, cgrad out; an atom term is about 60 operations
        pairs = sum(c.npts * len(c.zat) / (c.omega) * _reach() for c in like)
        return {"bytes": 20 * npts, "flops": 60 * pairs + 60 * npts}
    npts = _npts(case)
    per_atom = {"box": 0.0, "promol": case.get("nat", 0) / (case.get("volume", 1.0) * BOHR_PER_ANG ** 3) * _reach()}
    logn = math.log2(npts)
    nlm = (case.get("lmax", 0) + 1) ** 2
    width = {_lib.CUBE_E22_14: 23, _lib.CUBE_1P_E12_5: 13, _lib.CUBE_1P_E13_5: 14}.get(case.get("style"), 0)
    b, f = {
        # grid in, labels out; the 26 slopes of a point
        "bader": (12, 60),
        # as bader, and one forward and one backward real transform and the harmonics
        "keyword": (12, 60 + 5 * logn + 6 * nlm),
        # FP32 or FP64 crho and cgrad out
        "promol": (8 if case.get("precision") == "fp32" else 16, 60 * per_atom["promol"]),
        # crho, cgrad, rhoat, two fragment densities; about 20 atoms per node, twice
        "box": (40, 2 * 60 * 20),
        # grid in, crho and cgrad out; one forward and six backward real transforms
        "fourier": (24, 17.5 * logn),
        # grid in, crho and cgrad out; ten contractions of the 64-point stencil
        "tricubic": (24, 300),
        # grid in, labels out; 14 facet weights and the harmonics
        "yt": (12, 14 * 4 + 6 * nlm),
        "cube_read": (width + 8, 40),
        "cube_format": (width + 8, 40),
    }[kind]
    return {"bytes": b * npts, "flops": f * npts}


# ------------------------------------------------------------------ the same in 64 bits


def _images(cell, reach):
    """Atoms of the cell and their lattice repeats within `reach` bohr of it."""
    inv = np.linalg.inv(cell.x2c)
    far = reach * np.linalg.norm(inv, axis=1)  # in fractions of each lattice vector
    lo, hi = np.floor(-far).astype(int), np.ceil(1 + far).astype(int)
    t = np.stack(np.meshgrid(*(np.arange(l - 1, h + 1) for l, h in zip(lo, hi)), indexing="ij"), -1).reshape(-1, 3)
    for x, z in zip(cell.xat - np.floor(cell.xat), cell.zat):
        for f in x + t[((x + t >= -far) & (x + t <= 1 + far)).all(axis=1)]:
            yield cell.x2c @ f, int(z)


def _radial(tab, r):
    """grid1's 4-point Lagrange interpolation of the table's three columns."""
    at = (torch.floor(torch.log(r / tab["a"]) / tab["b"]).long() + 1).clamp(2, tab["r"].numel() - 2)
    cols = [torch.zeros_like(r) for _ in range(3)]
    for p in range(4):
        w = torch.ones_like(r)
        for q in range(4):
            if p != q:
                w *= (r - tab["r"][at - 2 + q]) / (tab["r"][at - 2 + p] - tab["r"][at - 2 + q])
        for c, col in zip(cols, tab["cols"]):
            c += col[at - 2 + p] * w
    return cols


def _promol_exact(images, n, x0, axes):
    """crho, cgrad and density of the atom sum on the nodes x0 + i a1 + j a2 +
    k a3 (axes: a1, a2, a3 as columns, bohr), z fastest."""
    tabs = {}
    for z, t in zip(ZSET, _tables()):
        col = lambda v: torch.as_tensor(np.asarray(v), dtype=torch.float64, device=DEV)  # noqa: E731
        tabs[z] = {"a": t.a, "b": t.b, "r": col(t.r), "cols": [col(t.f), col(t.fp), col(t.fpp)],
                   "rc": min(t.cutrad, t.rmax), "rmax": t.rmax}
    inv = np.linalg.inv(axes)
    acc = [torch.zeros(n, dtype=torch.float64, device=DEV) for _ in range(10)]
    nuc = torch.zeros(n, dtype=torch.bool, device=DEV)
    for pos, z in images:
        t = tabs[z]
        mid, far = inv @ (pos - x0), t["rc"] * np.linalg.norm(inv, axis=1)
        lo = np.maximum(np.ceil(mid - far).astype(int), 0)
        hi = np.minimum(np.floor(mid + far).astype(int) + 1, n)
        if (hi <= lo).any():
            continue
        at = tuple(slice(int(a), int(b)) for a, b in zip(lo, hi))
        ijk = [torch.arange(int(a), int(b), dtype=torch.float64, device=DEV) for a, b in zip(lo, hi)]
        d = [float(x0[c] - pos[c]) + float(axes[c, 0]) * ijk[0][:, None, None]
             + float(axes[c, 1]) * ijk[1][None, :, None] + float(axes[c, 2]) * ijk[2][None, None, :] for c in range(3)]
        r = torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
        nuc[at] |= r <= 1e-5
        inside = (r <= t["rc"]) & (r < t["rmax"])
        r = r.clamp_min(float(t["r"][0]))
        f, fp, fpp = (torch.where(inside, v, torch.zeros_like(v)) for v in _radial(t, r))
        acc[0][at] += f.clamp_min(0.0)
        g1 = fp / r
        g2 = (fpp - g1) / r ** 2
        for q in range(3):
            acc[1 + q][at] += d[q] * g1
            acc[4 + q][at] += g1 + g2 * d[q] ** 2
            acc[7 + q][at] += g2 * d[q] * d[(q + 1) % 3]  # xy, yz, zx
    rho, gx, gy_, gz, xx, yy, zz, xy, yz, zx = acc
    # the middle eigenvalue's sign: the roots of the characteristic cubic are
    # real, so its positive roots are its sign changes
    m = xx * yy + xx * zz + yy * zz - xy ** 2 - yz ** 2 - zx ** 2
    det = xx * (yy * zz - yz ** 2) - xy * (xy * zz - yz * zx) + zx * (xy * yz - yy * zx)
    tr = xx + yy + zz
    seq = torch.stack([-tr.sign(), m.sign(), -det.sign()])
    last, changes = torch.ones_like(tr), torch.zeros_like(tr)
    for v in seq:
        changes += (v * last < 0).to(tr.dtype)
        last = torch.where(v != 0, v, last)
    positive = (changes >= 2) | ((seq == 0).sum(0) >= 2) & (changes == 1) | (seq == 0).all(0)
    g = torch.sqrt(gx ** 2 + gy_ ** 2 + gz ** 2)
    g[nuc] = 0.0
    crho = torch.where(positive, rho, -rho) * 100.0
    return crho.reshape(-1), _rdg(rho, g).reshape(-1), rho.reshape(-1)


def _rdg(rho, grad):
    return grad / (2.0 * (3.0 * math.pi ** 2) ** (1.0 / 3.0) * rho.clamp_min(1e-80) ** (4.0 / 3.0))


def _fourier_exact(rho, n, x2c):
    f = torch.fft.fftn(rho.reshape(n[::-1]).permute(2, 1, 0).to(torch.complex128))
    b = 2.0 * math.pi * np.linalg.inv(x2c)  # rows: reciprocal vectors
    idx = [torch.tensor([i if i <= v // 2 else i - v for i in range(v)], dtype=torch.float64) for v in n]
    gsq, up = 0.0, 0
    for c in range(3):
        g = (float(b[0, c]) * idx[0][:, None, None] + float(b[1, c]) * idx[1][None, :, None]
             + float(b[2, c]) * idx[2][None, None, :])
        gsq = gsq + torch.fft.ifftn(1j * g * f).real ** 2
        up = up + (torch.fft.ifftn(-(g * g) * f).real > 0.0).to(torch.int8)
    rho = rho.reshape(n[::-1]).permute(2, 1, 0)
    crho = torch.where(up >= 2, rho.abs(), -rho.abs()) * 100.0
    return crho.reshape(-1), _rdg(rho, torch.sqrt(gsq)).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    # Basin sums and weights follow from the basins of a serial sweep over the
    # grid, and the tricubic's cell from how a coordinate rounds: no 64-bit value
    if kind in ("bader", "keyword", "tricubic", "yt", "cube_format"):
        return None
    s = prepare(case, seed)
    reach = max(min(t.cutrad, t.rmax) for t in _tables())
    if kind == "batch":
        out = []
        for c in s["cells"]:
            crho, cgrad, _ = _promol_exact(_images(c, reach), c.n, np.zeros(3), c.x2c / np.array(c.n))
            out.append({"labels": None, "crho": crho, "cgrad": cgrad})
        return {"cells": out, "counts": None, "sums": None}
    cell = s["cell"]
    if kind == "promol":
        crho, cgrad, _ = _promol_exact(_images(cell, reach), cell.n, np.zeros(3), cell.x2c / np.array(cell.n))
        return {"crho": crho, "cgrad": cgrad}
    if kind == "fourier":
        crho, cgrad = _fourier_exact(s["rho"].cpu(), cell.n, cell.x2c)
        return {"crho": crho, "cgrad": cgrad}
    if kind == "box":
        nd = s["nodes"]
        x0, axes = np.array(list(nd.x0)), np.array(list(nd.xmat)).reshape(3, 3).T
        # repeats that reach the box, wherever it lies
        far = float(np.linalg.norm(axes @ np.array(_n(case)))) + reach
        crho, cgrad, rhoat = _promol_exact(_images(cell, far), _n(case), x0, axes)
        each = [_promol_exact([(p, ZSET[q]) for p, q in zip(xyz, sp)], _n(case), x0, axes)[2]
                for xyz, sp in s["frags"]]
        # critic2's defaults: s is masked where |rho| > rhoplot = 0.1, or where
        # the fragments hold too little of the density or one holds it alone
        total = sum(each)
        masked = (crho.abs() / 100.0 > 0.1) | (total < 0.75 * rhoat)
        for e in each:
            masked |= e > 0.95 * total
        return {"crho": crho, "cgrad": torch.where(masked, 100.0, cgrad), "rhoat": rhoat,
                "rhofrag": torch.stack(each), "dat": None, "sums": None}
    # cube_read: each token's value is the correctly rounded one
    hdr = 6 + len(cell.zat)
    with open(s["file"].path, "rb") as fh:
        body = fh.read().split(b"\n", hdr)[hdr]
    v = np.array(body.split(), dtype=np.float64).reshape(cell.n)
    return {"f": torch.from_numpy(v.transpose(2, 1, 0).reshape(-1).copy()), "step": cell.x2c / np.array(cell.n)}
