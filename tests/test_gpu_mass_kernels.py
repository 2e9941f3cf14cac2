"""Mass with packed geometry and the direct lumped sums, against the CPU
oracle: affine and curved elements, node counts that do not fill a block,
per-element factors, a stiffness before and after the mass on one mesh (the
two operators write different geometry), and the same items in a batch.
Entries are FP64 sums of some ten to some hundred terms: 1e-13 of the largest
entry."""
import numpy as np
import pytest

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [("hex", 1, (1, 1, 1), 0.0, 3), ("hex", 1, (5, 4, 7), 0.2, 3), ("tet", 1, (3, 2, 4), 0.0, 3),
         ("tet", 2, (3, 3, 3), 0.0, 5), ("tet", 2, (2, 2, 2), 0.05, 5), ("prism", 1, (4, 3, 3), 0.15, 3),
         ("hex", 2, (2, 3, 2), 0.0, 5), ("hex", 2, (2, 2, 3), 0.1, 5), ("hex", 3, (2, 2, 2), 0.03, 7)]


@pytest.mark.parametrize("elem,order,cells,perturb,deg", CASES)
def test_mass(gpu_ctx, elem, order, cells, perturb, deg):
    m = M.structured_box_mesh(cells=cells, elem=elem, order=order, perturb=perturb, seed=5)
    tab = R.rule_tables(m.etype, deg)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)

    def close(a, b):
        assert np.abs(a - b).max() <= 1e-13 * np.abs(b).max()

    K0, _ = dev.assemble(_lib.OP_STIFFNESS, tab)
    ref = O.mass_legacy(m, tab, rho=2.5)
    refl = O.mass_legacy(m, tab, rho=2.5, lumped=True).diagonal()
    Mc, _ = dev.assemble(_lib.OP_MASS, tab, rho=2.5)
    close(Mc, ref.data)
    Ml, _ = dev.assemble(_lib.OP_MASS, tab, rho=2.5, lumped=True)
    close(Ml, refl)
    assert np.array_equal(dev.values(_lib.OP_MASS), Mc)          # the consistent mass is kept beside it
    K1, _ = dev.assemble(_lib.OP_STIFFNESS, tab)
    assert np.array_equal(K0, K1)
    sc = np.random.default_rng(6).uniform(0.0, 2.0, m.E)
    a, _ = dev.assemble(_lib.OP_MASS, tab, rho=2.5, lumped=True, element_scale=sc)
    b, _ = dev.assemble(_lib.OP_MASS, tab, rho=2.5, lumped=True, element_scale=2.0 - sc)
    close(a + b, 2.0 * refl)
    if m.npe <= 10:
        _lib.assemble_batch([(dev, _lib.OP_MASS, tab, dict(rho=2.5, lumped=True))])
        close(dev.values(_lib.OP_MASS, lumped=True), refl)
        _lib.assemble_batch([(dev, _lib.OP_STIFFNESS, tab, {}), (dev, _lib.OP_MASS, tab, dict(rho=2.5, lumped=True))])
        close(dev.values(_lib.OP_MASS, lumped=True), refl)
        close(dev.values(_lib.OP_STIFFNESS), K0)


# the lumped sums leave for the host while the panel launches run on one or two
# side streams: the values written by them are whole for the call that follows
@pytest.mark.parametrize("streams", ["1", "2", "3"])
@pytest.mark.parametrize("elem,order,n", [("hex", 1, 1), ("tet", 2, 12), ("hex", 2, 6)])
def test_lumped_beside_panels(gpu_ctx, monkeypatch, elem, order, n, streams):
    m = M.structured_box_mesh(n=n, elem=elem, order=order)
    tab = R.rule_tables(m.etype, 2 * order + 1)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    ref, _ = dev.assemble(_lib.OP_MASS, tab, rho=2.5)
    monkeypatch.setenv("LLFEM_PANEL_STREAMS", streams)
    refl = O.mass_legacy(m, tab, rho=2.5, lumped=True).diagonal()
    for _ in range(3):
        lum, st = dev.assemble(_lib.OP_MASS, tab, rho=2.5, lumped=True)
        assert np.abs(lum - refl).max() <= 1e-13 * np.abs(refl).max()
        assert st.kernel_ms >= st.main_kernel_ms > 0.0
        twice, _ = dev.assemble(_lib.OP_MASS, tab, rho=2.5, accumulate=True)
        assert np.array_equal(twice, 2.0 * ref)
    dev.close()
