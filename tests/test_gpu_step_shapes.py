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


# FP32 steps run in pairs that write where they read; odd counts start with a
# pass to the other copy.  f deviates from w rho0 by what 16 roundings of 2^-24
# per step can add up to (times 4: the sums of nine).
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("n,coll,wall,pairs", [(4, 2, 2, 1), (5, 2, 0, 1), (17, 0, 2, 2), (33, 1, 2, 1), (64, 2, 2, 3),
                                               (65, 2, 2, 1), (100, 1, 0, 1)])
def test_fp32_transport_in_place(n, coll, wall, pairs, steps):
    banner(f"FP32 in-place transport {n} x {n}, collision {coll}, wall {wall}, {pairs} pairs, {steps} steps")
    if n < 12:
        pore = np.ones((n, n), np.int32)  # no wall: every slot streams over the seams
    else:
        pore = cut(n, 11)[0] if n <= 64 else G.disk_packing(n, 0.65, 3, 7, seed=5)
    kn, lp = G.uniform_kn(pore, 0.1, MFP_DX)
    for k in range(1, pairs):  # vertical bands of other Knudsen numbers
        kn[:, k::pairs] *= 1 + 0.5 * k
        lp[:, k::pairs] /= 1 + 0.5 * k
    par = dict(dx=1e-9, Fbody=1e-6)
    o = O.Oracle(pore, kn, lp, periodic_y=True, **par)
    o.set_operators(coll, wall)
    o.run("transport", steps, 0.0)
    g = Lattice(pore, kn, lp, precision="fp32dev", collision=coll, wall=wall, periodic_y=1, **par)
    g.step("transport", steps)
    w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
    rho0 = 0.235554544075989  # default gas state
    a, b = (np.asarray(x.get("f")).reshape(-1, 9) - w * rho0 for x in (g, o))
    assert rel_l2(a, b) <= 4 * 16 * 2.0**-24 * (steps + 1)
    g.step("transport", steps)  # a second call goes on from the canonical state
    o.run("transport", steps, 0.0)
    a, b = (np.asarray(x.get("f")).reshape(-1, 9) - w * rho0 for x in (g, o))
    assert rel_l2(a, b) <= 4 * 16 * 2.0**-24 * (2 * steps + 2)


# a channel of two cells' width across a corner: two of its cells have wall
# links whose specular slot streams, so their rule does not fit the per-type table
DIAGONAL = """
000001111111111
000001111111111
000001111111111
000011111111111
000011111110000
000001111100000
000000111000000
000000011000000
000000110000000
000001111000000
000011111000000
000011111000000
000001111110000
000000111111111
000000001111111
"""


@pytest.mark.parametrize("steps", [1, 2, 3, 6])
@pytest.mark.parametrize("coll,wall", [(2, 2), (1, 2), (0, 2), (2, 0)])
def test_fp32_links_cells(coll, wall, steps):
    from mantiis_amd.hip import Batch
    banner(f"FP32 transport with shared specular slots, collision {coll}, wall {wall}, {steps} steps")
    pore = np.ones((48, 48), np.int32)
    pore[16:31, 16:31] = np.array([[int(ch) for ch in row] for row in DIAGONAL.split()])
    pore = np.ascontiguousarray(G.sanitize(pore), np.int32)
    kn, lp = G.uniform_kn(pore, 0.1, MFP_DX)
    par = dict(dx=1e-9, Fbody=1e-6)
    o = O.Oracle(pore, kn, lp, periodic_y=True, **par)
    o.set_operators(coll, wall)
    o.run("transport", 40 + steps, 0.0)
    g = Lattice(pore, kn, lp, precision="fp32dev", collision=coll, wall=wall, periodic_y=1, **par)
    g.step("transport", 40)
    g.step("transport", steps)
    w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
    rho0 = 0.235554544075989  # default gas state
    a, b = (np.asarray(x.get("f")).reshape(-1, 9) - w * rho0 for x in (g, o))
    assert rel_l2(a, b) <= 4 * 16 * 2.0**-24 * (40 + steps + 2)
    # the batch (tuned: the tuner's steps must leave nothing behind)
    bt = Batch([(pore, kn, lp)], collision=coll, wall=wall, **par)
    bt.run(40, check_every=40, tol=1e-300)
    bt.step(steps)
    bt.run(2, check_every=2, tol=1e-300)
    o = O.Oracle(pore, kn, lp, periodic_y=True, **par)
    o.set_operators(coll, wall)
    o.run("transport", 40 + steps + 2, 0.0)
    for got, want in zip(bt.fields(0)[1:], o.complete_domain()[:2]):
        assert rel_l2(np.asarray(got).reshape(-1), want) <= 4 * 16 * 2.0**-24 * (40 + steps + 3) * 10
