"""Whole steps, whose first strain half step and internal forces are one pass for uGIMP and classic
particles, against the same steps taken task by task, whose passes are separate: bit for bit, for each
material law, a mixture of laws, both dimensions and tile shapes, contact, XPIC, crowded cells and elastic
particles uploaded with a pressure (which no elastic step changes); and with loads and lCPDI, which take
the separate passes either way."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
from test_gpu_scatter_edges import crowded, block

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I

MOONEY = configs.mooney_material_xml(G1=300., G2=100., K=2000., rho=1.0)
CASES = {
    "2D elastic": (2, lambda: block(2, "uGIMP")),
    "2D J2": (2, lambda: configs.j2_block_2d(cells=24, block=11)),
    "2D Mooney": (2, lambda: configs.elastic_block_2d(cells=21, block=11, material_xml=MOONEY)),
    "2D contact": (2, lambda: configs.contact_blocks_2d(w=4, h=6, gap=0., vx=3000., vy=2000.)),
    "2D classic": (2, lambda: block(2, "Classic")),
    "3D J2": (3, lambda: configs.j2_block_3d(cells=14, lo=4, hi=9, vx=2e5)),
    "3D neo-Hookean": (3, lambda: block(3, "uGIMP")),
    "3D Mooney": (3, lambda: configs.neohookean_block_3d(cells=14, lo=4, hi=9, material_xml=configs.mooney_material_xml())),
    "3D contact, two materials": (3, lambda: configs.contact_cylinders_3d(cells=16, radius=3., length=4., gap=0., shape="uGIMP",
                                                                         law_type=61, friction=0.2)),
    "3D XPIC(2)": (3, lambda: configs.periodic_xpic(block(3, "uGIMP"), order=2)),
    "3D lCPDI": (3, lambda: block(3, "lCPDI")),
    "2D with loads": (2, lambda: configs.particle_bcs(block(2, "uGIMP"), [
        ("BCLine", {"x1": 5, "y1": 15.75, "x2": 16, "y2": 15.75, "tolerance": 0.3}, ["net", {"dir": 1, "style": 2, "load": 0.5, "ftime": 0.}])])),
}


@pytest.mark.parametrize("tile_shape", [0, 1])
@pytest.mark.parametrize("name", CASES)
def test_step_equals_its_tasks(name, tile_shape):
    print("case: step against its tasks,", name, "tile shape", tile_shape, flush=True)
    dim, make = CASES[name]
    prob = nm.Problem.from_xml(make())
    if "loads" in name:
        sims = [nm.Simulation.from_problem(prob) for _ in range(2)]
    else:
        g, mats, run, d, i = crowded(prob, dim, False, False)
        if name == "2D elastic":
            d[F["pressure"]] = np.linspace(-1., 1., d.shape[1])
        sims = [nm.Simulation(g, mats, run) for _ in range(2)]
        for s in sims:
            s.upload(d, i)
    a, b = sims
    a.set_tile_shape(tile_shape)
    b.set_tile_shape(tile_shape)
    start = a.particles()[0]
    a.step(5)
    for _ in range(5):
        for t in range(len(nm.TASKS)):
            b.run_task(t)
    x, y = a.particles(), b.particles()
    assert not np.array_equal(x[0], start)
    assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])


def test_mixed_types_in_one_batch():
    print("case: batch of an elastic, a J2 and a Mooney instance against each alone", flush=True)
    probs = [nm.Problem.from_xml(x) for x in (configs.elastic_block_2d(cells=21, block=11), configs.j2_block_2d(cells=24, block=11),
                                              configs.elastic_block_2d(cells=21, block=9, material_xml=MOONEY))]
    batch = nm.Batch(probs)
    batch.step(6)
    got = batch.particles()
    at = 0
    for p in probs:
        s = nm.Simulation.from_problem(p)
        s.step(6)
        want = s.particles()[0]
        n = want.shape[1]
        assert np.array_equal(got[0][:, at:at + n], want)
        at += n
