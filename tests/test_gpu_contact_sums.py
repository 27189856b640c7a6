"""Volume, displacement and volume gradient that a contact extrapolates of uGIMP and classic particles, node
by node against the oracle, at the scatters' edges: cells of 1 to 131 particles, unequal sizes, particles
outside the element they were uploaded with, before and after the particle update (whose sums take the new
positions). A sum has at most 64 cells of 131 terms, so the order of summation changes it by less than
1e-12 of the sum of magnitudes, which is at most that of the particles in reach of a node: 64 times the
largest node's, and for a gradient over the cell's size."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
import oracle as orc
from test_gpu_scatter_edges import crowded

pytestmark = pytest.mark.gpu

F = nm.F
CASES = {
    "2D": (2, lambda: configs.contact_blocks_2d(w=4, h=6, gap=0., vx=3000., vy=2000.), False, False),
    "2D sizes": (2, lambda: configs.contact_blocks_2d(w=4, h=6, gap=0., vx=3000., vy=2000.), True, False),
    "2D classic": (2, lambda: configs.contact_blocks_2d(w=4, h=6, gap=0., vx=3000.).replace('"uGIMP"', '"Classic"'), False, False),
    "3D": (3, lambda: configs.contact_cylinders_3d(cells=16, radius=3., length=4., gap=0., shape="uGIMP", friction=0.2), False, False),
    "3D sizes, strayed": (3, lambda: configs.contact_cylinders_3d(cells=16, radius=3., length=4., gap=0., shape="uGIMP"), True, True),
    "3D classic": (3, lambda: configs.contact_cylinders_3d(cells=16, radius=3., length=4., gap=0., shape="Classic"), False, False),
}


@pytest.mark.parametrize("tile_shape", [0, 1])
@pytest.mark.parametrize("name", CASES)
def test_contact_extrapolations(name, tile_shape):
    print("case: contact extrapolations,", name, "tile shape", tile_shape, flush=True)
    dim, make, sizes, strayed = CASES[name]
    g, mats, run, d, i = crowded(nm.Problem.from_xml(make()), dim, sizes, strayed)
    rng = np.random.default_rng(4)
    for a in "xyz"[:dim]:
        d[F["orig_" + a]] -= 0.1 * rng.uniform(0.2, 1., d.shape[1])
    for c in ("ep_xx", "ep_yy", "ep_xy"):
        d[F[c]] = 0.02 * rng.uniform(-1., 1., d.shape[1])
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    sim.set_tile_shape(tile_shape)
    ora = orc.Oracle(g, mats, run, d, i)
    for t, task in enumerate(nm.TASKS):
        sim.run_task(t)
        ora.run_task(t)
        if task not in ("Post Extrapolation Tasks", "Update Strains Last with Extrapolation"):
            continue
        got, want = sim.contact_values(), ora.contact_values()
        vol, mass = want[0].max(), ora.grid_fields()[0].max()
        move = max(np.abs(d[F["pos_" + a]] - d[F["orig_" + a]]).max() for a in "xyz"[:dim])
        for x, y, scale in zip(got, want, (vol, mass * 2. * move, vol / g.dx)):
            assert np.abs(y).max() > 0.
            err = np.abs(x - y).max() / (64. * scale)
            print(task, f"{err:.1e}", flush=True)
            assert err <= 1e-12, (task, err)
    sim.close()
