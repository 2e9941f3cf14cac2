"""Large assemblies are launched in parts while the values of the parts before
leave for the host.  Whole and in parts, the same waves sum the same terms in
the same order: the values that arrive equal the resident ones, which a call
without a host target wrote in one part, bit for bit."""
import numpy as np
import pytest

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


# values of 41, 51 (curved: 48 MB) and 97 and 104 MB (affine: 96 MB), one and two side streams; consistent mass 75 MB
@pytest.mark.parametrize("streams", ["1", "2", "3"])
@pytest.mark.parametrize("op,elem,order,n,perturb", [("K", "hex", 1, 28, 0.2), ("K", "hex", 1, 30, 0.2),
                                                     ("K", "hex", 1, 37, 0.0), ("K", "hex", 1, 38, 0.0),
                                                     ("K", "tet", 2, 17, 0.02), ("K", "prism", 1, 34, 0.1),
                                                     ("K", "hex", 2, 12, 0.1), ("M", "tet", 2, 24, 0.02)])
def test_values_in_parts(gpu_ctx, monkeypatch, op, elem, order, n, perturb, streams):
    monkeypatch.setenv("LLFEM_PANEL_STREAMS", streams)
    m = M.structured_box_mesh(n=n, elem=elem, order=order, perturb=perturb, seed=3)
    tab = R.rule_tables(m.etype, 2 * order + 1)
    op = _lib.OP_STIFFNESS if op == "K" else _lib.OP_MASS
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    dev.assemble(op, tab, copy_out=False)
    whole = dev.values(op)
    out = np.full(whole.size, np.nan)
    for _ in range(2):
        out[:] = np.nan
        _, st = dev.assemble(op, tab, out=out)
        assert np.array_equal(out, whole)
        assert st.kernel_ms >= st.main_kernel_ms > 0.0
    assert np.array_equal(dev.values(op), whole)
    # two groups, the second added: the sum of the groups' own values
    sc = (np.arange(m.E) % 2).astype(np.float64)
    a, _ = dev.assemble(op, tab, element_scale=1.0 - sc, copy_out=True)
    out[:] = np.nan
    dev.assemble(op, tab, element_scale=sc, accumulate=True, out=out)
    both = dev.values(op)
    assert np.array_equal(out, both)
    b, _ = dev.assemble(op, tab, element_scale=sc, copy_out=True)
    assert np.array_equal(both, a + b)
    dev.close()


# node numbers in random order: parts cut the launches anywhere
def test_parts_of_a_shuffled_mesh(gpu_ctx):
    m = M.structured_box_mesh(n=31, perturb=0.2, seed=3)
    perm = np.random.default_rng(4).permutation(m.N)
    inv = np.empty(m.N, np.int64)
    inv[perm] = np.arange(m.N)
    tab = R.rule_tables(m.etype, 3)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords[perm], m.etype, inv[np.asarray(m.conn) - m.conn.min()] + m.conn.min())
    dev.assemble(_lib.OP_STIFFNESS, tab, copy_out=False)
    out, _ = dev.assemble(_lib.OP_STIFFNESS, tab)
    assert np.array_equal(out, dev.values(_lib.OP_STIFFNESS))
    dev.close()
