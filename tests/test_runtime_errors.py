"""What the library does when a call of the HIP runtime fails, on the CPU: a stand-in for the runtime
(native/hip_stand_in.cpp) takes its calls and fails the one that a test names. Each case runs in a process
of its own, which loads the stand-in before the library."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {package!r})
fake = ctypes.CDLL({stand_in!r}, mode=ctypes.RTLD_GLOBAL)
fake.stand_in_count.restype = ctypes.c_long
fake.stand_in_fail.argtypes = [ctypes.c_char_p, ctypes.c_long, ctypes.c_int]
fail = lambda what, nth=0, error=1: fake.stand_in_fail(what.encode(), nth, error)     # 1: hipErrorInvalidValue
count = lambda part: fake.stand_in_count(part.encode())
import numpy as np
import nairnmpm as nm
from nairnmpm import configs
lib = nm.library()
prob = nm.Problem.from_xml(configs.elastic_block_2d(cells=16, block=8))
g, mats, run, n, _ = prob.describe()
d, i = prob.particles()
def message(call):
    try:
        call()
    except nm.MPMError as e:
        return str(e)
    return None
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    out = tmp_path_factory.mktemp("hip") / "libhip_stand_in.so"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I" + rocm + "/include",
                    os.path.join(HERE, "native", "hip_stand_in.cpp"), "-o", str(out)], check=True)
    return str(out)


def _run(stand_in, body):
    text = PRELUDE.format(package=os.path.join(ROOT, "nairn-mpm-fea_amd"), stand_in=stand_in) + body + "\nprint('done')\n"
    r = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), (r.returncode, r.stdout, r.stderr)


def test_download_without_rows_is_an_error(stand_in):
    _run(stand_in, """
sim = nm.Simulation(g, mats, run)
sim.upload(d, i)
assert lib.mpmgpu_download_particles(sim._h, None, None) != 0
assert lib.mpmgpu_last_error(sim._h)
a, b = sim.particles()
assert a.shape == d.shape and b.shape == i.shape
""")


@pytest.mark.parametrize("what,expect", [("hipEventRecord", "result download failed"), ("k_result_words", "result download failed"),
                                         ("places", "left its range"), (None, None)])
def test_message_of_a_failed_collect(stand_in, what, expect):
    _run(stand_in, f"""
what, expect = {what!r}, {expect!r}
srv = nm.Server(nm.PLANE_STRAIN, nm.SHAPE_UGIMP)
rid = srv.submit(g, mats, run, d, i, 4)
for _ in range(10):
    srv.advance(4)
assert srv.info(rid)["state"] == 2
if what == "places":
    fake.stand_in_places_outside(1)
elif what:
    fail(what)                       # with hipErrorInvalidValue
m = message(lambda: srv.collect(rid))
assert (m is None) == (expect is None) and (m is None or expect in m), m
""")


@pytest.mark.parametrize("what,nth", [("k_p2g_mass", 3), ("k_reorder_rows", 20), ("hipStreamSynchronize", 1), ("hipMemcpyAsync", 6),
                                      ("k_reorder_rowsIdLb1", 2), ("k_copy_unless", -2)])
def test_static_solve_puts_the_rows_back(stand_in, what, nth):
    """a solve that orders the caller's rows: one that fails orders them back, and says so if that fails"""
    _run(stand_in, f"""
what, nth = {what!r}, {nth}
prob = nm.Problem.from_xml(configs.j2_block_2d(cells=144, block=128))
g, mats, run, n, _ = prob.describe()
d, i = prob.particles()
d, i = np.ascontiguousarray(d), np.ascontiguousarray(i)
solve = lambda: nm.solve_static(g, mats, run, n, d.ctypes.data, i.ctypes.data, 16)
assert n >= 65536 and message(solve) is None
back = count("k_reorder_rowsIdLb1") + count("k_reorder_rowsIiLb1")
assert back == -(-nm.NUM_FIELDS // 3) + 1
fail(what, nth if nth >= 0 else count(what) + nth)
assert message(solve)
assert count("k_reorder_rowsIdLb1") + count("k_reorder_rowsIiLb1") == 2 * back
""")


def test_unread_error_before_a_collect(stand_in):
    """an error of the caller's own that nobody has read fails no collect and stays for its caller; a context's
    download reports it, with the rows"""
    _run(stand_in, """
def unread():
    assert fake.hipMemcpy(None, None, 8, 0) != 0
srv = nm.Server(nm.PLANE_STRAIN, nm.SHAPE_UGIMP)
rid = srv.submit(g, mats, run, d, i, 4)
for _ in range(10):
    srv.advance(4)
assert srv.info(rid)["state"] == 2
unread()
a, b = srv.collect(rid)
assert a.shape == d.shape
assert fake.hipGetLastError() == 1
sim = nm.Simulation(g, mats, run)
sim.upload(d, i)
unread()
before = count("k_result_words")
assert "invalid argument" in message(sim.particles)
assert count("k_result_words") > before
assert message(sim.particles) is None
""")


def test_download_with_less_pinned_memory(stand_in):
    """slots that cannot be pinned are done without, down to one"""
    _run(stand_in, """
prob = nm.Problem.from_xml(configs.j2_block_2d(cells=144, block=128))
g, mats, run, n, _ = prob.describe()
d, i = prob.particles()
for refused in (1, 2, 3, 4):
    sim = nm.Simulation(g, mats, run)
    sim.upload(d, i)
    fake.stand_in_refuse_pinned(refused)
    m = message(sim.particles)
    assert (m is None) == (refused < 4), (refused, m)
    fake.stand_in_refuse_pinned(0)
    assert message(sim.particles) is None
""")
