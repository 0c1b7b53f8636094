"""Fused steps at the sizes where a tile, a block or a row ends: one site over
and under, ragged sides, lattices smaller than one tile -- against the oracle."""
import numpy as np
import pytest

import _oracle as O
from _gpu_util import banner, rel_l2
from mantiis_amd import geometry as G
from mantiis_amd.hip import Lattice

pytestmark = pytest.mark.gpu
MFP_DX = 0.7730846760658538


def cut(n, seed):
    """A disk packing cut to n x n sites (the oracle takes squares)."""
    pore = G.sanitize(np.ascontiguousarray(G.disk_packing(64, 0.7, 2, 5, seed=seed)[:n, :n]))
    kn, lp = G.uniform_kn(pore, 0.1, MFP_DX)
    return pore, kn, lp


# the Shan-Chen tile has 14 x 14 sites and a ring around it
@pytest.mark.parametrize("n", [12, 13, 14, 15, 28, 29, 57])
@pytest.mark.parametrize("kind,coll,wall", [("adsorption", 1, 0), ("coupled", 2, 2)])
def test_shan_chen_fp64_tile_edges(n, kind, coll, wall):
    banner(f"{kind} FP64 {n} x {n}, 12 steps")
    pore, kn, lp = cut(n, 7)
    par = dict(dx=12e-9, Fbody=1e-8, periodic_y=True)
    o = O.Oracle(pore, kn, lp, **par)
    o.set_operators(coll, wall)
    g = Lattice(pore, kn, lp, precision="fp64", collision=coll, wall=wall, dx=12e-9, Fbody=1e-8, periodic_y=1)
    if kind == "adsorption":
        o.run("adsorption", 12, 0.0)
    else:  # the oracle's coupled run starts with 100 adsorption steps at F = 0
        o.run("coupled", 12, 0.0)
        g.set_body_force(0.0)
        g.step("adsorption", 100)
        g.set_body_force(1e-8)
    g.step(kind, 12)
    # same operations in the same order: FP64 rounding of 12 (112) steps
    for name in ("f", "rho", "ux", "uy"):
        assert rel_l2(g.get(name), o.get(name)) <= 1e-12, name
