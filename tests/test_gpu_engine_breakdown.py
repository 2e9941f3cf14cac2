"""PCG engine, breakdown: an operator that is indefinite on the free DoFs has a
direction with p.Kp <= 0, where the recursion stops and the solution so far is
kept.  An isotropic K with mu = 1 and lambda between -2 mu and -2/3 mu has a
positive diagonal, and with one clamped face negative directions; CG meets one
within a few iterations.  maxiter=1 ends the solve at that update.

The reference is the same Jacobi-CG in FP64 on the host up to its breakdown.
Its products p.Kp are at least 5 % of |p||Kp| here on either side of the
breakdown, so an FP32 operator (2^-24 an entry) moves alpha by about 20 times
its rounding an iteration: 1e-5 of x in five iterations, 1e-4 asked for.  One
iteration more or less changes x by its own size.
Every block of a launch has to find the breakdown alike, so repeats and systems
among others agree bit for bit."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

from lowlevelfem import _lib
from lowlevelfem import mesh as M
from lowlevelfem import refelem as R

pytestmark = pytest.mark.gpu


def _material(lam):
    return (3 * lam + 2) / (lam + 1), lam / (2 * (lam + 1))   # E, nu of mu = 1


def _fixed(m):
    left = m.nodes_on("left")
    return (3 * left[:, None] + np.arange(3)).ravel()


def _solve(dev, f, fixed, method):
    u, st = np.empty_like(f), _lib.Stats()
    code = dev.ctx.lib.llfem_solve(dev.h, _lib.ptr(f), _lib.ptr(fixed), fixed.size, 0, None, method, 1e-10, 1,
                                   _lib.ptr(u), C.byref(st))
    with pytest.raises(_lib.LLFEMError, match="maxiter"):
        _lib.check(code)
    return u, st.iterations


def _host_cg(K, f, fixed):
    d = 1.0 / K.diagonal()
    d[fixed] = 0.0
    r = f.copy()
    r[fixed] = 0.0
    x = np.zeros_like(r)
    z = d * r
    p, rho, r0 = z.copy(), r @ z, r @ r
    for k in range(100):
        q = K @ p
        q[fixed] = 0.0
        if p @ q <= 0.0:
            assert p @ q < -0.05 * np.linalg.norm(p) * np.linalg.norm(q)
            return x, k
        assert p @ q > 0.05 * np.linalg.norm(p) * np.linalg.norm(q)
        a = rho / (p @ q)
        x += a * p
        r -= a * q
        assert r @ r > 0.02 * r0   # no FP64 update before the breakdown
        z = d * r
        p, rho = z + (r @ z / rho) * p, r @ z
    raise AssertionError("no breakdown")


# 64 to 4,913 nodes: one vector block to twenty, four product blocks to 308
@pytest.mark.parametrize("method", [_lib.PCG_MIXED_RELIABLE, _lib.PCG_F32OP_RELIABLE])
@pytest.mark.parametrize("elem,order,n,lam", [("hex", 1, 3, -1.5), ("hex", 1, 6, -1.2), ("hex", 1, 9, -1.2),
                                              ("tet", 2, 4, -1.2), ("hex", 1, 16, -0.9)])
def test_stops_at_the_breakdown(gpu_ctx, elem, order, n, lam, method):
    m = M.structured_box_mesh(n=n, elem=elem, order=order)
    E, nu = _material(lam)
    dev = _lib.DeviceMesh(gpu_ctx, m.coords, m.etype, m.conn)
    val, _ = dev.assemble(_lib.OP_STIFFNESS, R.rule_tables(m.etype, 3), E=E, nu=nu)
    cp, rv = dev.pattern()
    K = sp.csc_matrix((val, rv, cp), shape=(3 * m.N, 3 * m.N))
    f = np.random.default_rng(n).uniform(-1.0, 1.0, 3 * m.N)
    fixed = _fixed(m)
    x, its = _host_cg(K, f, fixed)
    u, st_its = _solve(dev, f, fixed, method)
    assert st_its == its
    assert np.linalg.norm(u - x) <= 1e-4 * np.linalg.norm(x)
    u2, _ = _solve(dev, f, fixed, method)
    assert np.array_equal(u, u2)
    dev.close()


# nine systems of 68,921 nodes in one launch: 2,430 vector blocks, more than the device holds at once, so the last
# ones start after the first have found the breakdown; 4,308 product blocks each, folded
def test_alone_equals_mix():
    m = M.structured_box_mesh(n=40)
    tab, face = R.rule_tables(m.etype, 3), m.faces["right"]
    ftab = R.rule_tables(face.etype, 3)
    mats = [_material(lam) for lam in (-1.5, -1.2, -0.9)]

    def run(together):
        srv, out, ids = _lib.Server(), [], []

        def take():
            rid = ids.pop(0)
            u = srv._keep[rid][8]
            with pytest.raises(_lib.LLFEMError, match="maxiter"):
                srv.wait(rid)
            out.append(u)

        for k in range(9):
            E, nu = mats[k % 3]
            ids.append(srv.submit(m, tab, ftab, face, [0.0, 1.0, 0.1 * k], _fixed(m), E=E, nu=nu, maxiter=1))
            if not together:
                take()
        while ids:
            take()
        srv.close()
        return out

    alone = run(False)
    assert all(np.isfinite(u).all() and np.abs(u).max() > 0 for u in alone)
    for a, b in zip(alone, run(True)):
        assert np.array_equal(a, b)
