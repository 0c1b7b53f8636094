"""Cell-order images (host builder): which lattices step in place, which cells are
LINKS, and that every lattice that steps in place may: each element of the nine
planes is one slot's and no other's, and every streamed slot has its partner."""
import os
import subprocess

import numpy as np
import pytest

from mantiis_amd import geometry as G
from test_gpu_step_shapes import DIAGONAL, cut

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def images(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("compact") / "compact")
    csrc = os.path.join(ROOT, "mantiis_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I" + csrc, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "drivers", "compact_driver.cpp"), os.path.join(csrc, "mts_grid.cpp"),
                    "-o", exe], check=True, timeout=600)

    def run(lattices):
        text = "\n".join(f"{p.shape[1]} {p.shape[0]} {int(t)}\n" + " ".join(map(str, p.reshape(-1))) for p, t in lattices)
        lines = subprocess.run([exe], input=text, check=True, capture_output=True, text=True, timeout=600).stdout.split("\n")
        out = []
        for line in lines[:-1]:
            f = line.split()
            out.append(None if f[0] == "error" else dict(cells=int(f[0]), raw=int(f[1]), links=int(f[2]),
                                                         inplace=int(f[3]), bad=f[4]))
        assert len(out) == len(lattices)
        return out

    return run


def test_step_shapes_run_in_place(images):
    """The lattices of test_gpu_step_shapes.py take the paths they are there for."""
    pores = [np.ones((4, 4), np.int32), np.ones((5, 5), np.int32)] + [cut(n, 11)[0] for n in (17, 33, 64)]
    pores += [G.disk_packing(n, 0.65, 3, 7, seed=5) for n in (65, 100)]
    for i, im in enumerate(images([(p, True) for p in pores])):
        assert im["raw"] == 0 and im["inplace"] == 1 and im["bad"] == "-", (pores[i].shape, im)
    corner = np.ones((48, 48), np.int32)
    corner[16:31, 16:31] = np.array([[int(ch) for ch in row] for row in DIAGONAL.split()])
    corner = np.ascontiguousarray(G.sanitize(corner), np.int32)
    (im,) = images([(corner, True)])
    assert im["raw"] == 0 and im["inplace"] == 1 and im["links"] == 2 and im["bad"] == "-"


def test_default_seam_steps_between_copies(images):
    """The default seam rule overwrites wall contributions at the x-seam: its
    columns are RAW and nothing runs in place; without fluid there, it does."""
    open_ = cut(64, 7)[0]
    open_[0] = open_[-1] = 0
    closed = cut(64, 7)[0]
    closed[0] = closed[-1] = closed[:, 0] = closed[:, -1] = 0
    open_, closed = (np.ascontiguousarray(G.sanitize(p), np.int32) for p in (open_, closed))
    a, b = images([(open_, False), (closed, False)])
    assert a["raw"] > 0 and a["inplace"] == 0
    assert b["raw"] == 0 and b["inplace"] == 1 and b["bad"] == "-"


@pytest.mark.parametrize("torus", [False, True])
def test_every_in_place_lattice_may(images, torus):
    rng = np.random.default_rng(17 + torus)
    lattices = []
    for k in range(700):
        ny, nx = rng.integers(1, 25, 2)
        p = (rng.uniform(size=(ny, nx)) < rng.uniform(0.4, 1.0)).astype(np.int32)
        if k % 3 == 0:  # smoother shapes
            p = ((p + np.roll(p, 1, 0) + np.roll(p, 1, 1) + np.roll(p, (1, 1), (0, 1))) >= 2).astype(np.int32)
        if not torus and k % 2:
            p[0] = p[-1] = p[:, 0] = p[:, -1] = 0
        lattices.append((np.ascontiguousarray(G.sanitize(p), np.int32), torus))
    ims = images(lattices)
    got = [im for im in ims if im]
    assert all(im["bad"] == "-" for im in got)
    assert sum(im["inplace"] and im["cells"] > 0 for im in got) > 50  # both kinds are there
    if not torus:
        assert sum(not im["inplace"] for im in got) > 50
