"""Particles come back exactly as they were uploaded, in upload order: one particle, sizes at which a
2 MiB chunk of the result ends in a double row, at the end of the double rows or between them and the
int rows, and one that takes several chunks and threads; twice, and after the rows were sorted."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I
WORDS = 2 * 2 ** 20 // 8
NF, NI = nm.NUM_FIELDS, nm.NUM_IFIELDS
SIZES = sorted({1, 2, 63, WORDS // (NF + NI // 2), WORDS // (NF + NI // 2) + 1, WORDS // NF, WORDS // NF + 1, 100003, 400000})


@pytest.mark.parametrize("n", SIZES)
def test_round_trip(n):
    print("case: download of", n, "particles", flush=True)
    prob = nm.Problem.from_xml(configs.elastic_block_2d(cells=24, block=12))
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    rng = np.random.default_rng(n)
    pick = rng.integers(0, d.shape[1], n)
    d, i = np.ascontiguousarray(d[:, pick]), np.ascontiguousarray(i[:, pick])
    d[F["hist1"]] = rng.standard_normal(n)
    d[F["orig_z"]] = np.arange(n)
    i[I["id"]] = rng.permutation(n)
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    for _ in range(2):
        a, b = sim.particles()
        assert np.array_equal(a, d) and np.array_equal(b, i)
    sim.set_sort_interval(1)
    sim.step(1)
    a, b = sim.particles()
    for f in ("mass", "hist1", "orig_x", "orig_z", "lp_x"):
        assert np.array_equal(a[F[f]], d[F[f]]), f
    assert np.array_equal(b[I["id"]], i[I["id"]])
