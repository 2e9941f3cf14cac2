"""The coarsest operator's inverse of the AMG set-up: by the device kernel, and by
the host where that kernel leaves it (a pivot that is not clearly positive; forced
here by a switch).  The two inverses of one operator differ by FP64 rounding before both
are stored in FP32, so the preconditioner is the same to FP32 rounding: the same
iterations within one, and both solutions meet the residual that was asked for."""
import numpy as np
import pytest
import scipy.sparse as sp

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


def _solve(ctx, coords, etype, conn, fixed):
    dev = _lib.DeviceMesh(ctx, coords, etype, conn)
    val, _ = dev.assemble(_lib.OP_STIFFNESS, R.rule_tables(etype, 3), E=1.0)
    cp, rv = dev.pattern()
    n = 3 * len(coords)
    K = sp.csc_matrix((val, rv, cp), shape=(n, n))
    f = np.random.default_rng(n).uniform(-1.0, 1.0, n)
    u, st = dev.solve(f, fixed, method=_lib.PCG_AMG_RELIABLE, reltol=1e-10)
    u2, st2 = dev.solve(f, fixed, method=_lib.PCG_AMG_RELIABLE, reltol=1e-10)
    assert np.array_equal(u, u2) and st.iterations == st2.iterations
    dev.close()
    r = K @ u - f
    r[fixed] = 0.0
    f[fixed] = 0.0
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(f)
    return u, st.iterations


# every level in the tail kernel; a level outside it; two outside it
@pytest.mark.parametrize("kw", [dict(n=4), dict(n=9), dict(n=6, elem="tet", order=2), dict(n=30)],
                         ids=["125", "1000", "tet10", "29791"])
def test_left_to_the_host(gpu_ctx, monkeypatch, kw):
    m = M.structured_box_mesh(**kw)
    left = m.nodes_on("left")
    fixed = (3 * left[:, None] + np.arange(3)).ravel()
    u, its = _solve(gpu_ctx, m.coords, m.etype, m.conn, fixed)
    monkeypatch.setenv("LLFEM_AMG_HOST_INVERSE", "1")
    v, host_its = _solve(gpu_ctx, m.coords, m.etype, m.conn, fixed)
    assert abs(its - host_its) <= 1
    assert np.linalg.norm(u - v) <= 1e-6 * np.linalg.norm(u)
