"""Which nodes an lCPDI particle reaches, against the oracle: the reference leaves a corner's node out when
the corner's function there is below 1e-15, so a corner about 1e-8 from two edges of its element gives the
node across both nothing, and the node across one a weight of that size. Every node must have mass in both
or in neither, and the contact of two materials must not see a third whose corner ends so near a node."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
import oracle as orc
from helpers import compare

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I
MASS_TASK, MOMENTA_TASK = nm.TASKS.index("Extrapolate Mass and Momentum"), nm.TASKS.index("Update Momenta")


def scattered(dim, seed):
    """Particles of half a cell, far apart, whose corners end 1e-16 to 1e-3 beyond or before the edges of
    their cells on each axis in turn and together"""
    make = configs.elastic_block_2d if dim == 2 else configs.neohookean_block_3d
    prob = nm.Problem.from_xml(make(cells=64, block=2, shape="lCPDI") if dim == 2 else make(cells=40, lo=4, hi=6, shape="lCPDI"))
    g, mats, run, _, _ = prob.describe()
    d0, i0 = prob.particles()
    rng = np.random.default_rng(seed)
    ax = "xyz"[:dim]
    dd, ii = [], []
    n = (g.nx, g.ny, g.nz if dim == 3 else 1)
    org, size = (g.xmin, g.ymin, g.zmin), (g.dx, g.dy, g.dz)
    cells = [range(4, k - 4, 4) for k in n[:dim]]
    for c in np.stack(np.meshgrid(*cells, indexing="ij"), -1).reshape(-1, dim):
        p, q = d0[:, 0].copy(), i0[:, 0].copy()
        e = 0
        for a in range(dim):
            off = 10. ** rng.uniform(-16., -3.) * rng.choice((0., 1., 1., 1., -1.))
            low = rng.integers(2)                                  # the corner at the cell's low edge, or high
            x = org[a] + (c[a] + (0.25 - off if low else 0.75 + off)) * size[a]
            p[F["pos_" + ax[a]]] = p[F["orig_" + ax[a]]] = x
            e += int(c[a]) * (1, g.nx, g.nx * g.ny)[a]
        q[I["elem"]] = e
        q[I["id"]] = len(ii)
        dd.append(p)
        ii.append(q)
    return g, mats, run, np.ascontiguousarray(np.stack(dd, 1)), np.ascontiguousarray(np.stack(ii, 1))


@pytest.mark.parametrize("tile_shape", [0, 1])
@pytest.mark.parametrize("dim", [2, 3])
def test_nodes_with_mass(dim, tile_shape):
    print(f"case: nodes with mass, {dim}D lCPDI, tile shape {tile_shape}", flush=True)
    g, mats, run, d, i = scattered(dim, 3)
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    sim.set_tile_shape(tile_shape)
    ora = orc.Oracle(g, mats, run, d, i)
    for t in range(MASS_TASK + 1):
        sim.run_task(t)
        ora.run_task(t)
    m, r = sim.grid_fields()[0], ora.grid_fields()[0]
    # the same functions from the same operations, at most 8 corners of one particle a node: rounding alone
    assert np.array_equal(m > 0., r > 0.)
    assert np.allclose(m, r, rtol=1e-12, atol=0.)
    assert 0. < r[r > 0.].min() < 1e-12 * r.max()
    sim.close()


def three_blocks(normals):
    """Two blocks in contact along x = 11, and a third a cell away whose corner lies 1e-8 beyond (10, 10)"""
    xml = configs.contact_cylinders_3d(cells=20, radius=2., length=4., gap=0., friction=0.3, normals=normals)
    lo = xml.index("  <MaterialPoints>")
    hi = xml.index("</MaterialPoints>") + len("</MaterialPoints>\n")
    box = ('    <Body mat="{}" vx="{}" vy="{}" vz="0">\n      <Box xmin="{}" xmax="{}" ymin="{}" ymax="{}" zmin="8" zmax="12"/>\n'
           "    </Body>\n")
    bodies = box.format(1, 2000, 0, 8, 11, 11, 14) + box.format(2, -2000, 300, 11, 14, 11, 14) + box.format(3, 0, 0, 7, 10, 7, 10)
    body = xml[:lo] + "  <MaterialPoints>\n" + bodies + "  </MaterialPoints>\n" + xml[hi:]
    # the law becomes material 4, a copy of the second cylinder's material 3
    a = body.index('  <Material Type="28" Name="cylinder 2">')
    b = body.index('  <Material Type="61"')
    body = body[:b] + body[a:b].replace("cylinder 2", "corner") + body[b:]
    prob = nm.Problem.from_xml(body.replace('<Friction law="3"/>', '<Friction law="4"/>'))
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    third = i[I["mat"]] == 2
    assert third.sum() == 8 * 3 * 3 * 4
    for a in "xy":
        d[F["pos_" + a], third] += 1e-8
    return g, mats, run, np.ascontiguousarray(d), i


@pytest.mark.parametrize("normals", [0, 2, 5, 6])
def test_corner_beside_a_contact_node(normals):
    print(f"case: third material's corner 1e-8 from two edges beside a contact, normals {normals}", flush=True)
    g, mats, run, d, i = three_blocks(normals)
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    ora = orc.Oracle(g, mats, run, d, i)
    for t in range(MOMENTA_TASK + 1):
        sim.run_task(t)
        ora.run_task(t)
    m, r = sim.grid_fields()[0], ora.grid_fields()[0]
    assert np.array_equal(m > 0., r > 0.)
    # no volume, displacement, gradient or force where there is no mass
    none = m == 0.
    v, u, n = sim.contact_values()
    assert not v[none].any()
    for rows in (sim.grid_fields()[2], u, n):
        assert not rows.transpose(0, 2, 1)[none].any()
    sim.upload(d, i)
    ora = orc.Oracle(g, mats, run, d, i)
    sim.step(3)
    ora.step(3)
    got, want = sim.particles()[0], ora.particles()[0]
    err = compare(got, want, 3)
    assert max(err.values()) <= 1e-9, err
    sim.close()
