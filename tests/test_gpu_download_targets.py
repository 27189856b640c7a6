"""Rows downloaded into device memory, as into the host's: into arrays of the device that the caller owns,
the double rows and the int rows in either kind of memory, for one chunk and for several."""
import ctypes

import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 101, 60001])
@pytest.mark.parametrize("doubles,ints", [("device", "device"), ("device", "host"), ("host", "device"), ("device", None)])
def test_rows_into_device_memory(n, doubles, ints):
    print(f"case: download of {n} particles, double rows to the {doubles}, int rows to {ints}", flush=True)
    prob = nm.Problem.from_xml(configs.elastic_block_2d(cells=24, block=12))
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    pick = np.random.default_rng(n).integers(0, d.shape[1], n)
    d, i = np.ascontiguousarray(d[:, pick]), np.ascontiguousarray(i[:, pick])
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    hip = _Hip()
    a, b = np.zeros_like(d), np.zeros_like(i)
    pa = hip.upload(a) if doubles == "device" else a.ctypes.data
    pb = hip.upload(b) if ints == "device" else b.ctypes.data if ints else None
    get = nm.library().mpmgpu_download_particles
    assert get(sim._h, ctypes.cast(pa, get.argtypes[1]), ctypes.cast(pb, get.argtypes[2]) if pb else None) == 0
    if doubles == "device":
        a = hip.download(pa, a)
        hip.free(pa)
    if ints == "device":
        b = hip.download(pb, b)
        hip.free(pb)
    assert np.array_equal(a, d)
    assert np.array_equal(b, i) if ints else not b.any()
    sim.close()


def test_collect_after_an_unread_error():
    print("case: server collect after an unread error of the runtime", flush=True)
    prob = nm.Problem.from_xml(configs.elastic_block_2d(cells=24, block=12))
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    srv = nm.Server(nm.PLANE_STRAIN, nm.SHAPE_UGIMP)
    rid = srv.submit(g, mats, run, d, i, 4)
    while srv.info(rid)["state"] < 2:
        srv.advance(4)
    hip = _Hip()
    assert hip.lib.hipMemcpy(None, d.ctypes.data, 8, hip.D2H) != 0          # refused, and kept as the last error
    a, b = srv.collect(rid)
    assert np.array_equal(a[nm.F["orig_x"]], d[nm.F["orig_x"]]) and np.array_equal(b[nm.I["id"]], i[nm.I["id"]])
    hip.lib.hipGetLastError()
    srv.close()
