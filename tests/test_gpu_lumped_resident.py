"""Lumped mass kept on the device (no target on the host: the launches stay on one
stream and its side streams) and with one (they leave the stream to the copy):
the same sums and the same consistent values, in any order of the two calls."""
import numpy as np
import pytest

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("elem,order,n", [("hex", 1, 1), ("tet", 1, 9), ("tet", 2, 12), ("hex", 2, 5)])
@pytest.mark.parametrize("streams", ["1", "2", "3"])
def test_with_and_without_a_target(gpu_ctx, monkeypatch, elem, order, n, streams):
    monkeypatch.setenv("LLFEM_PANEL_STREAMS", streams)
    m = M.structured_box_mesh(n=n, elem=elem, order=order)
    tab = R.rule_tables(m.etype, 2 * order + 1)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    for first, second in ((False, True), (True, False)):
        got = []
        for target in (first, second):
            out, _ = dev.assemble(_lib.OP_MASS, tab, rho=2.5, lumped=True, copy_out=target)
            got.append((dev.values(_lib.OP_MASS, lumped=True), dev.values(_lib.OP_MASS)))
            if target:
                assert np.array_equal(out, got[-1][0])
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
        assert abs(got[0][0].sum() - got[0][1].sum()) <= 1e-12 * got[0][1].sum()
    dev.close()
