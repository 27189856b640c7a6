"""The binning's scan and tile list over grids of one tile, of exactly one scan block of 32,768 keys and of
one key more or less than whole tiles, and of more blocks than one look-back window (256), with particles
at both ends of the grid and in its middle, against the oracle. The steps are the parity tests' and so
is the bound, 1e-9: a wrong cell start or a missing tile loses whole particles from the sums."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
import oracle as orc
from helpers import compare

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I


@pytest.mark.parametrize("nx,ny", [(8, 8), (256, 128), (257, 128), (264, 120), (70000, 128)])
def test_particles_across_the_grid(nx, ny):
    print("case: binning of", nx, "by", ny, "cells", flush=True)
    prob = nm.Problem.from_xml(configs.elastic_block_2d(cells=8, block=4, vmax=3000.))
    g, mats, run, _, _ = prob.describe()
    d0, i0 = prob.particles()
    x, y = (d0[F["pos_x"]] - g.xmin) / g.dx, (d0[F["pos_y"]] - g.ymin) / g.dy
    # the 4 by 4 cells of particles, moved to start at these cells
    spots = {(1, 1), (nx - 5, ny - 5), (nx // 2, ny // 2), (nx - 5, 1)} if nx > 8 else {(2, 2)}
    d, i = [], []
    for sx, sy in sorted(spots):
        a, b = d0.copy(), i0.copy()
        for f, s, low, size in (("x", sx, x.min(), g.dx), ("y", sy, y.min(), g.dy)):
            for row in ("pos_", "orig_"):
                a[F[row + f]] += (s - np.floor(low)) * size
        b[I["elem"]] = (np.floor((a[F["pos_y"]] - g.ymin) / g.dy) * nx + np.floor((a[F["pos_x"]] - g.xmin) / g.dx))
        d.append(a)
        i.append(b)
    d, i = np.concatenate(d, 1), np.concatenate(i, 1)
    i[I["id"]] = np.arange(d.shape[1])
    g.nx, g.ny = nx, ny
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    ora = orc.Oracle(g, mats, run, d, i)
    for n in (1, 2):
        sim.step(n)
        ora.step(n)
        got, ref = sim.particles()[0], ora.particles()[0]
        errs = compare(got, ref, 2)
        disp = ref[F["pos_x"]:F["pos_x"] + 2] - ref[F["orig_x"]:F["orig_x"] + 2]
        rounding = 3 * np.spacing(nx * g.dx) / np.sqrt(np.mean(np.sum(disp ** 2, 0)))
        print({k: f"{v:.2e}" for k, v in errs.items()}, flush=True)
        for k, v in errs.items():
            assert v <= 1e-9 + (rounding if k == "disp" else 0.), (nx, ny, k, v)
    sim.close()
