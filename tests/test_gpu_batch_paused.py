"""A lattice taken out of a batch's queue keeps its state, whatever the others
run meanwhile: put back, it goes on bit for bit where it stopped."""
import numpy as np
import pytest

from _gpu_util import banner
from mantiis_amd import geometry as G

pytestmark = pytest.mark.gpu

# two cells' wall links whose specular slot streams (see test_gpu_step_shapes.py)
CORNER = """
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


def geoms():
    a = np.ones((64, 64), np.int32)
    a[16:31, 16:31] = np.array([[int(ch) for ch in row] for row in CORNER.split()])
    out = []
    for i, p in enumerate((a, G.disk_packing(64, 0.7, 2, 5, seed=7), G.disk_packing(128, 0.6, 3, 8, seed=9))):
        p = np.ascontiguousarray(G.sanitize(p), np.int32)
        out.append((p,) + tuple(G.uniform_kn(p, 0.1 * (i + 1), 0.7730846760658538)))
    return out


# one-step kernel: in place (BB, SRBB) and between two copies (MDBB); tile kernels
@pytest.mark.parametrize("coll,wall,steps", [(2, 2, 1), (1, 0, 1), (2, 1, 1), (2, 2, 2)])
@pytest.mark.parametrize("pause", [[1], [2], [3], [1, 1], [3, 2, 2]])
def test_paused_lattice_goes_on_where_it_stopped(coll, wall, steps, pause):
    from mantiis_amd.hip import Batch
    banner(f"batch with lattices out of the queue for {pause} steps, collision {coll}, wall {wall}, {steps} per launch")

    def fields(pause):
        b = Batch(geoms(), collision=coll, wall=wall, dx=1e-9, Fbody=1e-6, batch_steps=steps)
        assert b.kernel()[0] == steps
        b.step(4)
        for k, n in enumerate(pause):
            b.activate([0, 1, k % 2])  # lattice 2 comes and goes
            b.step(n)
        b.activate([1, 0, 0])
        b.run(2, check_every=2, tol=1e-300)
        return b.fields(0)

    for name, got, want in zip(("rho", "ux", "uy"), fields(pause), fields([])):
        assert np.array_equal(got, want), name


@pytest.mark.parametrize("wall", [1, 2])
def test_state_given_to_a_paused_lattice(wall):
    """Populations set while a lattice is out of the queue are the ones it goes
    on from."""
    from mantiis_amd.hip import Batch
    banner(f"batch: state set on a lattice out of the queue, wall {wall}")
    gs = geoms()
    w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
    rng = np.random.default_rng(3)
    f = (w[:, None] * 0.2355 * (1 + 1e-3 * rng.normal(size=gs[0][0].size))[None, :]) * gs[0][0].reshape(-1)[None, :]

    def fields(paused):
        b = Batch(gs, collision=2, wall=wall, dx=1e-9, Fbody=1e-6)
        b.step(2)
        if paused:
            b.activate([0, 1, 1])
            b.step(1)
        b.set_state(0, f.reshape(-1))
        if paused:
            b.step(3)
            b.activate([1, 1, 1])
        b.run(2, check_every=2, tol=1e-300)
        return b.fields(0)

    for got, want in zip(fields(True), fields(False)):
        assert np.array_equal(got, want)
