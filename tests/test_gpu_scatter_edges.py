"""Particle-to-grid sums at the edges of the matrix-core scatters, against the oracle: cells that hold
one to 131 particles (incomplete groups of four records, a cell over several rounds of 32 and 64, empty
cells between), particles on cell edges, centres and support edges, unequal particle sizes, and
particles a little outside the element they were uploaded with, for each shape function, dimension and
tile shape, with XPIC and contact. A node's sum has at most 4^3 cells of 131 terms, so the order of
summation changes it by less than 1e4 rounding errors, 1e-12 relative to the sum of magnitudes; the
bound on each particle field is the parity tests' 1e-9."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
import oracle as orc
from helpers import compare

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I
TOL = 1e-9
COUNTS = (1, 2, 3, 4, 5, 7, 8, 9, 31, 32, 33, 63, 65, 131, 0, 0)


def crowded(prob, dim, sizes, strayed):
    """The problem's block with its particles redrawn: COUNTS particles per cell in turn"""
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    rng = np.random.default_rng(11)
    elem = i[I["elem"]]
    dd, ii = [], []
    ax = "xyz"[:dim]
    org = dict(zip("xyz", (g.xmin, g.ymin, g.zmin)))
    size = dict(zip("xyz", (g.dx, g.dy, g.dz)))
    for k, e in enumerate(np.unique(elem)):
        n = COUNTS[k % len(COUNTS)] if k < 60 else 2
        src = np.flatnonzero(elem == e)
        cell = dict(zip("xyz", (e % g.nx, e // g.nx % g.ny, e // (g.nx * g.ny))))
        for j in range(n):
            s = src[j % len(src)]
            c, ci = d[:, s].copy(), i[:, s].copy()
            for a in ax:
                # quarter points are centres of particles of the usual size: support and cell edges
                u = rng.integers(0, 4) / 4. if j % 3 == 0 else rng.uniform(0.01, 0.99)
                if strayed and j % 5 == 1:
                    u = 1.03 + 0.05 * rng.uniform()
                c[F["pos_" + a]] = c[F["orig_" + a]] = org[a] + (cell[a] + u) * size[a]
                if sizes:
                    c[F["lp_" + a]] *= rng.uniform(0.6, 1.)
            dd.append(c)
            ii.append(ci)
    d, i = np.stack(dd, 1), np.stack(ii, 1)
    order = rng.permutation(d.shape[1])
    return g, mats, run, np.ascontiguousarray(d[:, order]), np.ascontiguousarray(i[:, order])


def block(dim, shape):
    if dim == 2:
        return configs.elastic_block_2d(cells=21, block=11, vmax=3000., shape=shape)
    return configs.neohookean_block_3d(cells=14, lo=4, hi=9, vx=2000., shape=shape)


CASES = [(f"{dim}D {shape}{', sizes' if sizes else ''}{', strayed' if strayed else ''}", dim,
          lambda dim=dim, shape=shape: block(dim, shape), sizes, strayed)
         for dim in (2, 3)
         for shape, sizes, strayed in (("uGIMP", False, False), ("uGIMP", True, False), ("uGIMP", False, True),
                                       ("Classic", False, False), ("lCPDI", False, False), ("lCPDI", True, False))]
CASES += [
    ("2D XPIC(3)", 2, lambda: configs.periodic_xpic(block(2, "uGIMP"), order=3), False, False),
    ("3D XPIC(3) lCPDI", 3, lambda: configs.periodic_xpic(block(3, "lCPDI"), order=3), False, False),
    ("2D contact", 2, lambda: configs.contact_blocks_2d(w=4, h=6, gap=0., vx=3000., vy=2000.), False, False),
    ("3D contact", 3, lambda: configs.contact_cylinders_3d(cells=16, radius=3., length=4., gap=0., shape="uGIMP",
                                                           law_type=61, friction=0.2), False, False),
]


@pytest.mark.parametrize("tile_shape", [0, 1])
@pytest.mark.parametrize("label,dim,make,sizes,strayed", CASES, ids=[c[0] for c in CASES])
def test_crowded_and_sparse_cells(label, dim, make, sizes, strayed, tile_shape):
    print("case:", label, "tile shape", tile_shape, flush=True)
    g, mats, run, d, i = crowded(nm.Problem.from_xml(make()), dim, sizes, strayed)
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    sim.set_tile_shape(tile_shape)
    ora = orc.Oracle(g, mats, run, d, i)
    done = 0
    for target in (1, 6):
        sim.step(target - done)
        ora.step(target - done)
        done = target
        errs = compare(sim.particles()[0], ora.particles()[0], dim)
        print(target, {k: f"{v:.2e}" for k, v in errs.items()}, flush=True)
        for k, v in errs.items():
            assert v <= TOL, (label, target, k, v)
