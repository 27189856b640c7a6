"""Particles of three laws (neo-Hookean, J2 and elastic, the elastic ones uploaded with a pressure that no
elastic step changes) among one another in the same cells, whose strain updates and one-pass internal forces
take the kernels with every law: whole steps against the same steps task by task, bit for bit, and against
the oracle; and in batches beside instances of one law each, whose tiles take the kernels of their law."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
import oracle as orc
from helpers import compare

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I
TOL = 1e-9
STEPS = 6

LAWS = """  <Material Type="28" Name="rubber">
    <rho>1.1</rho>
    <G>10.0</G>
    <K>50.0</K>
  </Material>
  <Material Type="9" Name="J2">
    <rho>1.1</rho>
    <E>60.0</E>
    <nu>0.3</nu>
    <yield>0.2</yield>
    <Ep>2.0</Ep>
  </Material>
  <Material Type="1" Name="elastic">
    <rho>1.1</rho>
    <E>60.0</E>
    <nu>0.3</nu>
  </Material>
"""


def problem(dim):
    if dim == 2:
        return nm.Problem.from_xml(configs.elastic_block_2d(cells=24, block=11, vmax=20000., material_xml=LAWS))
    return nm.Problem.from_xml(configs.neohookean_block_3d(cells=14, lo=4, hi=9, vx=10000., material_xml=LAWS))


def mixed(prob, laws=(0, 1, 2), seed=2):
    d, i = prob.particles()
    rng = np.random.default_rng(seed)
    i[I["mat"]] = rng.choice(laws, d.shape[1])
    d[F["pressure"]] = np.where(i[I["mat"]] == 2, rng.uniform(-0.1, 0.1, d.shape[1]), 0.)
    return np.ascontiguousarray(d), np.ascontiguousarray(i)


def alone(prob, d, i, steps=STEPS, by_task=False, tile_shape=0):
    g, mats, run, _, _ = prob.describe()
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    sim.set_tile_shape(tile_shape)
    if by_task:
        for _ in range(steps):
            for t in range(len(nm.TASKS)):
                sim.run_task(t)
    else:
        sim.step(steps)
    out = sim.particles()
    sim.close()
    return out


@pytest.mark.parametrize("tile_shape", [0, 1])
@pytest.mark.parametrize("dim", [2, 3])
def test_laws_in_one_context(dim, tile_shape):
    print(f"case: three laws in one {dim}D context, tile shape {tile_shape}", flush=True)
    prob = problem(dim)
    d, i = mixed(prob)
    a, b = alone(prob, d, i, tile_shape=tile_shape), alone(prob, d, i, by_task=True, tile_shape=tile_shape)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    elastic = i[I["mat"]] == 2
    assert np.array_equal(a[0][F["pressure"], elastic], d[F["pressure"], elastic])
    assert (a[0][F["hist0"], i[I["mat"]] == 1] > 0.).any()              # some of the J2 particles yielded
    g, mats, run, _, _ = prob.describe()
    ora = orc.Oracle(g, mats, run, d, i)
    ora.step(STEPS)
    err = compare(a[0], ora.particles()[0], dim)
    assert max(err.values()) <= TOL, err


@pytest.mark.parametrize("dim", [2, 3])
def test_laws_in_one_batch(dim):
    print(f"case: {dim}D batch of one instance of three laws and one of each", flush=True)
    probs = [problem(dim) for _ in range(4)]
    parts = [mixed(p, laws) for p, laws in zip(probs, [(1,), (0, 1, 2), (2,), (0,)])]
    batch = nm.Batch(probs, parts)
    batch.step(STEPS)
    for k, (p, (d, i)) in enumerate(zip(probs, parts)):
        got, want = batch.instance_particles(k), alone(p, d, i)
        assert np.array_equal(got[0], want[0])
    batch.close()
