"""A static-scratch solve that finds an earlier error of the runtime still unread reports it, as it did, and
the rows that it ordered while it stepped are in the caller's order again."""
import numpy as np
import pytest

import nairnmpm as nm
from nairnmpm import configs
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu

F, I = nm.F, nm.I


def test_rows_after_an_unread_error():
    print("case: static solve after an unread error of the runtime", flush=True)
    prob = nm.Problem.from_xml(configs.j2_block_2d(cells=144, block=128))
    g, mats, run, _, _ = prob.describe()
    d, i = prob.particles()
    at = np.random.default_rng(5).permutation(d.shape[1])
    d, i = np.ascontiguousarray(d[:, at]), np.ascontiguousarray(i[:, at])
    hip = _Hip()
    dd, di = hip.upload(d), hip.upload(i)
    assert hip.lib.hipMemcpy(None, dd, 8, hip.D2H) != 0          # refused, and kept as the last error
    with pytest.raises(nm.MPMError, match="invalid argument"):
        nm.solve_static(g, mats, run, d.shape[1], dd, di, 16)
    a, b = hip.download(dd, d), hip.download(di, i)
    assert np.array_equal(b[I["id"]], i[I["id"]]) and np.array_equal(a[F["orig_x"]], d[F["orig_x"]])
    # the next solve does not see it
    nm.solve_static(g, mats, run, d.shape[1], dd, di, 16)
    hip.free(dd)
    hip.free(di)
