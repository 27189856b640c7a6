"""Static-scratch solves that reorder the caller's rows while they step (65,536 particles and more, 16
steps and more) against the context path, and against the same solve just below either limit's path: the
rows in a shuffled order, odd and even step counts, past one and two renewals of the order (every 50
steps), 2D and 3D, and a run that stops on the device. Results do not depend on the order, so they are
compared bit for bit."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I


def _shuffled(prob, n=None):
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    at = np.random.default_rng(5).permutation(d.shape[1])[:n]
    return g, mats, run, np.ascontiguousarray(d[:, at]), np.ascontiguousarray(i[:, at])


def _static(hip, g, mats, run, d, i, steps):
    dd, di = hip.upload(d), hip.upload(i)
    error = None
    try:
        nm.solve_static(g, mats, run, d.shape[1], dd, di, steps)
    except nm.MPMError as e:
        error = str(e)
    out = hip.download(dd, d), hip.download(di, i)
    hip.free(dd)
    hip.free(di)
    return out, error


def _context(g, mats, run, d, i, steps):
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    error = None
    try:
        sim.step(steps)
        sim.sync()
    except nm.MPMError as e:
        error = str(e)
    out = sim.particles()
    sim.close()
    return out, error


def _check(a, b):
    assert a[1] == b[1], (a[1], b[1])
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("dim,n,steps", [(2, 65536, 15), (2, 65535, 17), (2, 65536, 16), (2, 65536, 53), (3, None, 17),
                                         (3, None, 104)])
def test_ordered_solve_equals_context(dim, n, steps):
    print(f"case: static solve {dim}D, {n} particles, {steps} steps", flush=True)
    xml = configs.j2_block_2d(cells=144, block=128) if dim == 2 else configs.j2_block_3d(cells=28, lo=3, hi=24, vx=2e5)
    case = _shuffled(nm.Problem.from_xml(xml), n)
    assert case[3].shape[1] >= 65535
    _check(_static(_Hip(), *case, steps), _context(*case, steps))


def test_stopped_run_gives_its_rows_back():
    print("case: static solve stopped by a particle that has left the grid", flush=True)
    g, mats, run, d, i = _shuffled(nm.Problem.from_xml(configs.j2_block_3d(cells=28, lo=3, hi=24, vx=2e5)))
    run.maxLeaving, run.deleteLeaving = 1, 0
    d[F["vel_x"]] += 0.2 * g.dx / run.timestep
    a = _static(_Hip(), g, mats, run, d, i, 60)
    assert a[1] and "left the grid" in a[1]
    assert np.array_equal(a[0][1][I["id"]], i[I["id"]]) and np.array_equal(a[0][0][F["orig_x"]], d[F["orig_x"]])
    b = _context(g, mats, run, d, i, 60)
    assert b[1] == a[1]
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)
