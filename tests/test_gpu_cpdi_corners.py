"""lCPDI particles whose corners lie at infinity: an error that names the corners, as for any corner beyond
the grid, in every cell, the first two of an axis (which a corner taken for cell 0 would pass for a
neighbour of) among them."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I


@pytest.mark.parametrize("cell", [0, 1, 2, 9])
@pytest.mark.parametrize("dim,axis", [(2, 0), (2, 1), (3, 0), (3, 1), (3, 2)])
def test_infinite_corners(dim, axis, cell):
    print(f"case: {dim}D lCPDI corners at infinity, axis {axis}, cell {cell}", flush=True)
    prob = nm.Problem.from_xml(configs.elastic_block_2d(cells=16, block=2, shape="lCPDI") if dim == 2 else
                               configs.neohookean_block_3d(cells=16, lo=7, hi=9, shape="lCPDI"))
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    d, i = np.ascontiguousarray(d[:, :1]), np.ascontiguousarray(i[:, :1])
    at = [cell if a == axis else 6 for a in range(dim)]
    org, size, elem = (g.xmin, g.ymin, g.zmin), (g.dx, g.dy, g.dz), 0
    for a in range(dim):
        d[F["pos_" + "xyz"[a]]] = d[F["orig_" + "xyz"[a]]] = org[a] + (at[a] + 0.5) * size[a]
        elem += at[a] * (1, g.nx, g.nx * g.ny)[a]
    i[I["elem"]] = elem
    d[F["ep_" + 2 * "xyz"[axis]]] = np.inf
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    sim.run_task(0)
    sim.run_task(1)
    with pytest.raises(nm.MPMError, match="CPDI particle domain node has left the grid"):
        sim.sync()
    sim.close()
