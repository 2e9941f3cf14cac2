"""Workloads of the assembly library as a user's program runs them.

Each case is a dict of plain values.  ``listed()`` gives the standing ones,
``draw(rng)`` one more of the same ranges, ``prepare(case, seed)`` what a
program holds before the call (mesh on the device, rule tables, host arrays
that receive results), ``run(state)`` one pass through the public entry
points, ``work(case)`` the bytes and operations the pass cannot do without
and ``exact(case, seed)`` the same outputs in 64-bit torch.

Kinds:

* ``stiffness``: stiffnessMatrix of one mesh into CSC values on the host
  (llfem_assemble with an output array), one or several material groups,
  straight-sided or perturbed (curved) elements, every precision;
* ``mass``: massMatrix, lumped (the default) or consistent;
* ``load``: loadVector with a body force, a traction or a pressure;
* ``solve``: assembly left on the device, then solveDisplacement on it;
* ``device-solve``: the allocation-free solve on device arrays of the caller;
* ``batch``: K and consistent M of several uneven problems in one call;
* ``serve``: a group of assemble-and-solve requests to the server.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lowlevelfem.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from lowlevelfem import _lib, mesh as M, refelem as R, workloads as W  # noqa: E402

# element name -> (structured_box_mesh family, order)
ELEMS = {"hex8": ("hex", 1), "hex27": ("hex", 2), "hex125": ("hex", 4), "tet4": ("tet", 1), "tet10": ("tet", 2),
         "wedge6": ("prism", 1)}
PREC = {"fp64": _lib.FP64, "fp32": _lib.FP32_INT_FP64_SUM, "bf16x3": _lib.BF16X3}
METHOD = {"jacobi": _lib.PCG_JACOBI_FP64, "mixed": _lib.PCG_MIXED_RELIABLE, "amg": _lib.PCG_AMG_RELIABLE}


def _case(kind, elem="hex8", cells=(8, 8, 8), **kw):
    c = {"kind": kind, "elem": elem, "nx": cells[0], "ny": cells[1], "nz": cells[2]}
    c.update(kw)
    return c


def _stiffness(elem, cells, perturb=0.0, degree=None, precision="fp64", groups=1):
    fam, order = ELEMS[elem]
    return _case("stiffness", elem, cells, perturb=perturb, degree=degree or 2 * order + 1, precision=precision,
                 groups=groups)


def listed():
    return [
        # the smallest call: a coupon of a few hundred elements, reassembled in a parameter sweep
        dict(_stiffness("hex8", (6, 5, 7)), name="stiffness-hex8-small"),
        # the quadratic-tet beam at an ordinary size, K handed to the host
        dict(_stiffness("tet10", (20, 20, 80), degree=2), name="stiffness-tet10"),
        # an unstructured (mesher-made) hexahedral part of two materials: curved elements, one call per group
        dict(_stiffness("hex8", (40, 36, 44), perturb=0.2, groups=2), name="stiffness-hex8-curved-2mat"),
        # curved quadratic hexahedra
        dict(_stiffness("hex27", (15, 13, 17), perturb=0.1), name="stiffness-hex27-curved"),
        # order-4 hexahedra on the matrix cores
        dict(_stiffness("hex125", (8, 7, 9), perturb=0.02, degree=9), name="stiffness-hex125"),
        # the default massMatrix (lumped) of the largest configuration, the 40x40x160 tet10 beam
        _case("mass", "tet10", (40, 40, 160), perturb=0.0, degree=5, lumped=True, name="mass-lumped-tet10-beam"),
        # self-weight of a tet10 part
        _case("load", "tet10", (24, 24, 96), perturb=0.0, load="body", name="load-body-tet10"),
        # the default solve (FP64 Jacobi-PCG to 1e-12) of a part of ordinary size
        _case("solve", "tet10", (12, 11, 40), perturb=0.0, method="jacobi", tol=1e-12, name="solve-jacobi-tet10"),
        # the large solve: assembly and AMG-preconditioned CG of the 6.3 M-DoF beam
        _case("solve", "tet10", (40, 40, 160), perturb=0.0, method="amg", tol=1e-10, name="solve-amg-tet10-beam"),
        # small systems solved back to back without allocation
        _case("device-solve", "hex8", (9, 8, 19), tol=1e-10, name="device-solve-hex8"),
        # K and M of a set of uneven hex8 / tet10 / wedge6 parts
        {"kind": "batch", "shapes": 2024, "count": 10, "dofs": 60000, "name": "batch-10"},
        # a group of requests arriving together
        {"kind": "serve", "shapes": 7, "count": 8, "meshes": 4, "dofs": 250000, "tol": 1e-10, "name": "serve-8"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, cells):
    """Three edge counts of about `cells` cells in all, aspect up to about 1:1:4."""
    e = (cells / rng.uniform(1.0, 4.0)) ** (1.0 / 3.0)
    nx = max(2, int(round(e * rng.uniform(0.85, 1.15))))
    ny = max(2, int(round(e * rng.uniform(0.85, 1.15))))
    return nx, ny, max(2, int(round(cells / (nx * ny))))


def draw(rng):
    kind = rng.choice(["stiffness"] * 4 + ["mass"] * 2 + ["load"] * 2 + ["solve"] * 2
                      + ["device-solve", "batch", "serve"])
    if kind == "stiffness":
        elem = rng.choice(["hex8", "tet10", "tet4", "wedge6", "hex27", "hex125"])
        most = {"hex8": 90000, "tet10": 30000, "tet4": 60000, "wedge6": 60000, "hex27": 3400, "hex125": 500}[elem]
        cells = _box(rng, _log_int(rng, 40 if elem == "hex125" else 150, most))
        if elem == "hex125":
            return _stiffness(elem, cells, 0.02, 9, rng.choice(["fp64", "fp64", "bf16x3"]))
        perturb = 0.1 if elem == "hex27" else rng.choice([0.0, 0.15]) if elem in ("hex8", "wedge6") else 0.0
        return _stiffness(elem, cells, perturb, 2 if elem == "tet10" and rng.random() < 0.5 else None,
                          rng.choice(["fp64", "fp64", "fp64", "fp32"]), rng.choice([1, 1, 2, 3]))
    if kind == "mass":
        elem = rng.choice(["hex8", "tet10", "wedge6", "hex27"])
        most = {"hex8": 400000, "tet10": 200000, "wedge6": 300000, "hex27": 20000}[elem]
        perturb = 0.0 if elem == "tet10" else rng.choice([0.0, 0.1])
        lumped = rng.random() < 0.7
        if not lumped:
            most //= 6
        return _case("mass", elem, _box(rng, _log_int(rng, 200, most)), perturb=perturb,
                     degree=2 * ELEMS[elem][1] + 1, lumped=lumped)
    if kind == "load":
        elem = rng.choice(["hex8", "tet10", "hex27"])
        most = {"hex8": 300000, "tet10": 50000, "hex27": 30000}[elem]
        return _case("load", elem, _box(rng, _log_int(rng, 200, most)), perturb=rng.choice([0.0, 0.1]),
                     load=rng.choice(["body", "body", "traction", "pressure"]))
    if kind == "solve":
        elem = rng.choice(["hex8", "tet10", "wedge6"])
        method = rng.choice(["jacobi", "mixed", "amg"])
        most = {"hex8": 60000, "tet10": 8000, "wedge6": 60000}[elem] * (4 if method == "amg" else 1)
        return _case("solve", elem, _box(rng, _log_int(rng, 300, most)), perturb=0.0, method=method,
                     tol=1e-12 if method == "jacobi" else 1e-10)
    if kind == "device-solve":
        elem = rng.choice(["hex8", "tet10"])
        return _case("device-solve", elem, _box(rng, _log_int(rng, 60, 12000 if elem == "hex8" else 1500)), tol=1e-10)
    if kind == "batch":
        return {"kind": "batch", "shapes": rng.randrange(1 << 20), "count": rng.randrange(4, 13),
                "dofs": _log_int(rng, 8000, 60000)}
    return {"kind": "serve", "shapes": rng.randrange(1 << 20), "count": rng.randrange(3, 9), "meshes": 3,
            "dofs": _log_int(rng, 20000, 250000), "tol": 1e-10}


# ---- inputs ----------------------------------------------------------------

def _mesh(case, rng, seed):
    """A box of the case's cells whose edge lengths come from the seed."""
    fam, order = ELEMS[case["elem"]]
    cells = (case["nx"], case["ny"], case["nz"])
    h = rng.uniform(0.02, 0.03, size=3)
    return M.structured_box_mesh(lx=h[0] * cells[0], ly=h[1] * cells[1], lz=h[2] * cells[2], cells=cells, elem=fam,
                                 order=order, perturb=case.get("perturb", 0.0), seed=seed)


def _materials(rng, n):
    return [(float(rng.uniform(1e5, 3e5)), float(rng.uniform(0.2, 0.45))) for _ in range(n)]


def _group_scales(mesh, groups):
    """Per material group 1 on its elements and 0 elsewhere (slabs in z, as
    cut volumes of one part are), or [None] for a single material."""
    if groups == 1:
        return [None]
    z = mesh.coords[mesh.conn, 2].mean(axis=1)
    g = np.minimum((groups * (z - z.min()) / (z.max() - z.min() + 1e-300)).astype(int), groups - 1)
    return [(g == k).astype(np.float64) for k in range(groups)]


def _clamp(mesh):
    left = mesh.nodes_on("left")
    return (3 * left[:, None] + np.arange(3)[None, :]).ravel()


def _stiffness_degree(elem):
    return 2 if elem == "tet10" else 2 * ELEMS[elem][1] + 1


def _serve_requests(case, seed):
    rng = np.random.default_rng(seed)
    reqs = W.serving_requests(seed=case["shapes"], count=case["count"], dof_range=(5_000, case["dofs"]),
                              distinct_meshes=case["meshes"])
    meshes, out = {}, []
    for r in reqs:
        key = (r.kind, r.cells)
        if key not in meshes:
            h = rng.uniform(0.02, 0.03, size=3)
            fam, order = W.KINDS[r.kind]
            meshes[key] = M.structured_box_mesh(lx=h[0] * r.cells[0], ly=h[1] * r.cells[1], lz=h[2] * r.cells[2],
                                                cells=r.cells, elem=fam, order=order)
        (E, nu), = _materials(rng, 1)
        out.append((r.kind, meshes[key], E, nu, float(rng.uniform(0.2, 1.0))))
    return out


def _inputs(case, seed):
    """Host-side inputs of a case: what prepare() uploads and exact() works from."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "batch":
        probs = W.batched_problems(seed=case["shapes"], count=case["count"], dof_range=(2_000, case["dofs"]))
        items = []
        for p in probs:
            fam, order = W.KINDS[p.kind]
            h = rng.uniform(0.02, 0.03, size=3)
            m = M.structured_box_mesh(lx=h[0] * p.cells[0], ly=h[1] * p.cells[1], lz=h[2] * p.cells[2],
                                      cells=p.cells, elem=fam, order=order)
            (E, nu), = _materials(rng, 1)
            items.append((p.kind, m, E, nu, float(rng.uniform(2e-9, 8e-9))))
        return items
    if kind == "serve":
        return _serve_requests(case, seed)
    m = _mesh(case, rng, seed)
    if kind == "stiffness":
        return m, R.rule_tables(m.etype, case["degree"]), _materials(rng, case["groups"])
    if kind == "mass":
        return m, R.rule_tables(m.etype, case["degree"]), float(rng.uniform(2e-9, 8e-9))
    if kind == "load":
        return m, rng.uniform(-1.0, 1.0, size=3)
    # solve, device-solve: the box clamped on one side and loaded on the other
    return m, R.rule_tables(m.etype, _stiffness_degree(case["elem"])), _materials(rng, 1)[0], \
        rng.uniform(-1.0, 1.0, size=3)


def prepare(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    ctx = _lib.default_context()
    if kind == "stiffness":
        m, tab, mats = inp
        dev = _lib.DeviceMesh(ctx, m.coords, m.etype, m.conn)
        out = np.empty(dev.pattern(_lib.OP_STIFFNESS, with_arrays=False))
        out[::512] = 0.0
        return case, dev, tab, mats, _group_scales(m, case["groups"]), out
    if kind == "mass":
        m, tab, rho = inp
        dev = _lib.DeviceMesh(ctx, m.coords, m.etype, m.conn)
        out = np.empty(3 * m.N if case["lumped"] else dev.pattern(_lib.OP_MASS, with_arrays=False))
        out[::512] = 0.0
        return case, dev, tab, rho, out
    if kind == "load":
        m, g = inp
        dev = _lib.DeviceMesh(ctx, m.coords, m.etype, m.conn)
        face = m.faces["right"]
        return case, dev, R.rule_tables(m.etype, 2 * ELEMS[case["elem"]][1] + 1), face, \
            R.rule_tables(face.etype, 2 * ELEMS[case["elem"]][1] + 1), g
    if kind in ("solve", "device-solve"):
        m, tab, mat, t = inp
        dev = _lib.DeviceMesh(ctx, m.coords, m.etype, m.conn)
        face = m.faces["right"]
        f = dev.traction(face.etype, face.conn, R.rule_tables(face.etype, 2 * ELEMS[case["elem"]][1] + 1), t)
        fixed = _clamp(m)
        if kind == "solve":
            return case, dev, tab, mat, f, fixed
        val, _ = dev.assemble(_lib.OP_STIFFNESS, tab, E=mat[0], nu=mat[1])
        cp, rv = dev.pattern(_lib.OP_STIFFNESS)
        mask = np.zeros(f.size, np.uint8)
        mask[fixed] = 1
        d = [torch.from_numpy(x).cuda() for x in (cp, rv.astype(np.int32), val, f, mask)]
        return (case, ctx, *d, torch.empty(f.size, dtype=torch.float64, device="cuda"))
    if kind == "batch":
        items, devs = [], []
        for k, m, E, nu, rho in inp:
            dev = _lib.DeviceMesh(ctx, m.coords, m.etype, m.conn)
            tk, tm = W.rules(k)
            items += [(dev, _lib.OP_STIFFNESS, tk, dict(E=E, nu=nu)), (dev, _lib.OP_MASS, tm, dict(rho=rho))]
            devs.append(dev)
        return case, _lib.Batch(items), devs
    srv = _lib.Server(max_active=64)
    args = []
    for k, m, E, nu, fy in inp:
        face = m.faces["right"]
        args.append((m, R.rule_tables(m.etype, _stiffness_degree(k)),
                     R.rule_tables(face.etype, 2 * W.KINDS[k][1] + 1), face, [0.0, fy, 0.0], _clamp(m), E, nu))
    return case, srv, args


def run(state):
    case = state[0]
    kind = case["kind"]
    if kind == "stiffness":
        _, dev, tab, mats, scales, out = state
        last = len(mats) - 1
        for i, ((E, nu), sc) in enumerate(zip(mats, scales)):
            dev.assemble(_lib.OP_STIFFNESS, tab, E=E, nu=nu, precision=PREC[case["precision"]], element_scale=sc,
                         accumulate=i > 0, copy_out=False, out=out if i == last else None)
        return out
    if kind == "mass":
        _, dev, tab, rho, out = state
        dev.assemble(_lib.OP_MASS, tab, rho=rho, lumped=case["lumped"], out=out)
        return out
    if kind == "load":
        _, dev, tab, face, ftab, g = state
        if case["load"] == "body":
            return dev.body(tab, g=g)
        if case["load"] == "traction":
            return dev.traction(face.etype, face.conn, ftab, g)
        dNn = R.basis(face.etype, R.node_coords(face.etype))[1]
        return dev.pressure(face.etype, face.conn, ftab, dNn, p=g[0])
    if kind == "solve":
        _, dev, tab, (E, nu), f, fixed = state
        dev.assemble(_lib.OP_STIFFNESS, tab, E=E, nu=nu, copy_out=False)
        u, _ = dev.solve(f, fixed, method=METHOD[case["method"]], reltol=case["tol"], maxiter=200000)
        return u
    if kind == "device-solve":
        _, ctx, cp, rv, val, f, mask, u = state
        _lib.solve_csc_noalloc(ctx, f.numel(), cp.data_ptr(), rv.data_ptr(), val.data_ptr(), f.data_ptr(),
                               mask.data_ptr(), None, u.data_ptr(), reltol=case["tol"], maxiter=200000)
        return u
    if kind == "batch":
        _, batch, devs = state
        batch.run()
        return [{"K": d.values(_lib.OP_STIFFNESS), "M": d.values(_lib.OP_MASS)} for d in devs]
    _, srv, args = state
    ids = [srv.submit(m, tab, ftab, face, t, fixed, E=E, nu=nu, method=_lib.PCG_AMG_RELIABLE, reltol=case["tol"],
                      maxiter=200000) for m, tab, ftab, face, t, fixed, E, nu in args]
    return [srv.wait(i)[0] for i in ids]


# ---- bytes and operations ----------------------------------------------------

def _counts(elem, cells):
    """(elements, nodes, node pairs that share an element, nodes per element) of a box."""
    nx, ny, nz = cells
    fam, p = ELEMS[elem]
    C = nx * ny * nz
    N = (p * nx + 1) * (p * ny + 1) * (p * nz + 1)
    if fam == "hex":
        pairs = math.prod(n * (p + 1) ** 2 - (n - 1) for n in cells)
        return C, N, pairs, (p + 1) ** 3
    if fam == "prism":
        edges = nx * (ny + 1) + ny * (nx + 1) + nx * ny
        return 2 * C, N, ((nx + 1) * (ny + 1) + 2 * edges) * (3 * nz + 1), 6
    T = 6 * C
    F = (4 * T + 4 * (nx * ny + ny * nz + nx * nz)) // 2
    V = (nx + 1) * (ny + 1) * (nz + 1)
    edges = V + F - T - 1
    if p == 1:
        return T, N, N + 2 * edges, 4
    return T, N, N + 2 * (3 * edges + 6 * F + 3 * T), 10


def _work_one(elem, cells, blk, q=0):
    E, N, pairs, npe = _counts(elem, cells)
    # curved elements cannot use per-element reference integrals: the symmetric point sum
    flops = E * (q * 9.0 * npe * (npe + 1) if q and blk == 9 else q * npe * (npe + 1.0) if q else 60.0 * npe * npe)
    return 24.0 * N + 4.0 * npe * E + 8.0 * blk * pairs, flops


def work(case):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        if kind == "batch":
            shapes = [(p.kind, p.cells) for p in W.batched_problems(seed=case["shapes"], count=case["count"],
                                                                    dof_range=(2_000, case["dofs"]))]
        else:
            shapes = [(r.kind, r.cells) for r in W.serving_requests(seed=case["shapes"], count=case["count"],
                                                                    dof_range=(5_000, case["dofs"]),
                                                                    distinct_meshes=case["meshes"])]
        b, f = map(sum, zip(*[_work_one(k, c, 12 if kind == "batch" else 9) for k, c in shapes]))
        return {"bytes": b, "flops": f}
    elem, cells = case["elem"], (case["nx"], case["ny"], case["nz"])
    E, N, pairs, npe = _counts(elem, cells)
    if kind in ("stiffness", "mass"):
        q = len(R.rule_tables(_etype(elem), case["degree"]).weights) if case["perturb"] else 0
        blk = 9 if kind == "stiffness" else 3
        b, f = _work_one(elem, cells, blk, q)
        if kind == "mass" and case["lumped"]:
            b += 24.0 * N - 8.0 * blk * pairs
        if elem == "hex125":
            f = E * 3.0 * npe * (3.0 * npe + 1.0) * q
        return {"bytes": b, "flops": f * case.get("groups", 1)}
    if kind == "load":
        return {"bytes": 48.0 * N + (4.0 * npe * E if case["load"] == "body" else 0.0), "flops": 30.0 * npe * E}
    # a solve: the operator formed once, the load in, the displacement out
    b, f = _work_one(elem, cells, 9)
    return {"bytes": b + 48.0 * N, "flops": f + 18.0 * pairs}


def _etype(elem):
    fam, order = ELEMS[elem]
    return {"prism": 6, "tet": 4 if order == 1 else 11}.get(fam) or R.HEX_TYPE_BY_ORDER[order]


# ---- the same outputs in 64-bit torch ----------------------------------------

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=_dev())


def _pattern(conn, N):
    """Node adjacency in column order: (pairs, first pair of each column,
    pair index of (element, column node, row node))."""
    c = _t(conn, torch.int64)
    uniq, inv = torch.unique((c[:, :, None] * N + c[:, None, :]).reshape(-1), return_inverse=True)
    ptr = torch.searchsorted(uniq, torch.arange(N + 1, device=c.device) * N)
    return uniq, ptr, inv.reshape(c.shape[0], c.shape[1], c.shape[1])


def _geometry(x, dN):
    """Physical gradients [e][q][a][c] and det J [e][q] of elements with node coordinates x [e][a][3]."""
    rel = x - x[:, :1]
    J = torch.einsum("eac,qad->eqcd", rel, dN)
    return torch.einsum("qad,eqdc->eqac", dN, torch.linalg.inv(J)), torch.linalg.det(J)


def _stiffness_values(m, tab, mats, scales):
    conn, N, n = m.conn, m.N, m.npe
    uniq, ptr, inv = _pattern(conn, N)
    col = uniq // N
    R3 = 3 * (ptr[1:] - ptr[:-1])
    base = 9 * ptr[col] + 3 * (torch.arange(uniq.numel(), device=uniq.device) - ptr[col])
    out = torch.zeros(9 * uniq.numel(), dtype=torch.float64, device=uniq.device)
    xyz, dN, w = _t(m.coords), _t(tab.dN), _t(tab.weights)
    cc = torch.arange(3, device=uniq.device)
    step = max(1, 200_000_000 // (9 * n * n * 8))
    for e0 in range(0, m.E, step):
        c = _t(conn[e0:e0 + step], torch.int64)
        ne = c.shape[0]
        g, det = _geometry(xyz[c], dN)
        wd = det.abs() * w
        Z = (g * wd.sqrt()[:, :, None, None]).reshape(ne, -1, 3 * n)
        G = torch.bmm(Z.transpose(1, 2).contiguous(), Z).reshape(ne, n, 3, n, 3)
        tr = G.diagonal(dim1=2, dim2=4).sum(-1)
        K = torch.zeros_like(G)
        for (E, nu), sc in zip(mats, scales):
            mu = E / (2 * (1 + nu))
            lam = 2 * mu * nu / (1 - 2 * nu)
            Kg = lam * G + mu * G.transpose(2, 4)
            for d in range(3):
                Kg[:, :, d, :, d] += mu * tr
            K += Kg if sc is None else Kg * _t(sc[e0:e0 + step])[:, None, None, None, None]
        p = inv[e0:e0 + step]                                # [e][column a][row b]
        pos = base[p][..., None, None] + cc[:, None] * R3[c][:, :, None, None, None] + cc
        out.index_add_(0, pos.reshape(-1), K.permute(0, 3, 1, 4, 2).reshape(-1))   # [e][a][b][c][d]
    return out, uniq, ptr


def _mass_values(m, tab, rho, lumped):
    N, n = m.N, m.npe
    xyz, dN, w, Nr = _t(m.coords), _t(tab.dN), _t(tab.weights), _t(tab.N)
    if lumped:
        acc = torch.zeros(N, dtype=torch.float64, device=xyz.device)
        rows = Nr * Nr.sum(1, keepdim=True)                  # sum over the row's columns
    else:
        uniq, ptr, inv = _pattern(m.conn, N)
        acc = torch.zeros(uniq.numel(), dtype=torch.float64, device=xyz.device)
        prod = Nr[:, :, None] * Nr[:, None, :]
    step = max(1, 200_000_000 // (n * max(n, 9 * tab.q) * 8))
    for e0 in range(0, m.E, step):
        c = _t(m.conn[e0:e0 + step], torch.int64)
        x = xyz[c]
        det = torch.linalg.det(torch.einsum("eac,qad->eqcd", x - x[:, :1], dN)).abs() * w * rho
        if lumped:
            acc.index_add_(0, c.reshape(-1), (det @ rows).reshape(-1))
        else:
            acc.index_add_(0, inv[e0:e0 + step].reshape(-1), torch.einsum("eq,qab->eab", det, prod).reshape(-1))
    if lumped:
        return acc.repeat_interleave(3)
    col = uniq // N
    Rn = (ptr[1:] - ptr[:-1])[col]
    s = torch.arange(uniq.numel(), device=uniq.device) - ptr[col]
    out = torch.empty(3 * uniq.numel(), dtype=torch.float64, device=uniq.device)
    for k in range(3):
        out[3 * ptr[col] + k * Rn + s] = acc
    return out


def _face_load(m, face, tab, t_nodes):
    """Sum over faces of N_a t |t1 x t2| w, the traction interpolated from its nodal values [f][a][3]."""
    x, dN, Nr, w = _t(m.coords[face.conn]), _t(tab.dN), _t(tab.N), _t(tab.weights)
    J = torch.einsum("eac,qad->eqcd", x, dN)
    ja = torch.linalg.cross(J[..., 0], J[..., 1]).norm(dim=-1) * w
    tq = torch.einsum("qa,eac->eqc", Nr, t_nodes)
    f = torch.zeros(m.N, 3, dtype=torch.float64, device=x.device)
    f.index_add_(0, _t(face.conn, torch.int64).reshape(-1),
                 torch.einsum("qa,eqc,eq->eac", Nr, tq, ja).reshape(-1, 3))
    return f.reshape(-1)


def _load_values(case, m, g):
    order = ELEMS[case["elem"]][1]
    if case["load"] == "body":
        tab = R.rule_tables(m.etype, 2 * order + 1)
        xyz, dN, Nr, w, gt = _t(m.coords), _t(tab.dN), _t(tab.N), _t(tab.weights), _t(g)
        acc = torch.zeros(m.N, dtype=torch.float64, device=xyz.device)
        step = max(1, 200_000_000 // (9 * tab.q * 8 * 4))
        for e0 in range(0, m.E, step):
            c = _t(m.conn[e0:e0 + step], torch.int64)
            x = xyz[c]
            det = torch.linalg.det(torch.einsum("eac,qad->eqcd", x - x[:, :1], dN))
            acc.index_add_(0, c.reshape(-1), ((det * w) @ Nr).reshape(-1))
        return (acc[:, None] * gt).reshape(-1)
    face = m.faces["right"]
    tab = R.rule_tables(face.etype, 2 * order + 1)
    conn = _t(face.conn, torch.int64)
    if case["load"] == "traction":
        return _face_load(m, face, tab, _t(g).expand(conn.shape[0], conn.shape[1], 3))
    # the average over a node's faces of the unit normals there, times -p
    dNn = _t(R.basis(face.etype, R.node_coords(face.etype))[1])
    J = torch.einsum("eac,kad->ekcd", _t(m.coords[face.conn]), dNn)
    nrm = torch.linalg.cross(J[..., 0], J[..., 1])
    nrm = -float(g[0]) * nrm / nrm.norm(dim=-1, keepdim=True)
    acc = torch.zeros(m.N, 3, dtype=torch.float64, device=nrm.device)
    cnt = torch.zeros(m.N, dtype=torch.float64, device=nrm.device)
    acc.index_add_(0, conn.reshape(-1), nrm.reshape(-1, 3))
    cnt.index_add_(0, conn.reshape(-1), torch.ones(conn.numel(), dtype=torch.float64, device=nrm.device))
    return _face_load(m, face, tab, (acc / cnt.clamp(min=1.0)[:, None])[conn])


def _solution(m, tab, mat, t, face, ftab):
    """K_ff u = f_f by Jacobi-CG in 64 bits, run until its residual stops falling."""
    val, uniq, ptr = _stiffness_values(m, tab, [mat], [None])
    N = m.N
    col, row = uniq // N, uniq % N
    R3 = 3 * (ptr[1:] - ptr[:-1])
    crow = torch.zeros(3 * N + 1, dtype=torch.int64, device=val.device)
    crow[1:] = R3.repeat_interleave(3).cumsum(0)
    s = torch.arange(uniq.numel(), device=val.device) - ptr[col]
    idx = torch.empty(val.numel(), dtype=torch.int64, device=val.device)
    diag = torch.empty(3 * N, dtype=torch.float64, device=val.device)
    on = col == row
    for c in range(3):
        for d in range(3):
            pos = 9 * ptr[col] + c * R3[col] + 3 * s + d
            idx[pos] = 3 * row + d
            if c == d:
                diag[3 * col[on] + c] = val[pos[on]]
    K = torch.sparse_csr_tensor(crow, idx, val, size=(3 * N, 3 * N))   # K is symmetric: columns serve as rows
    f = _face_load(m, face, ftab, _t(t).expand(face.conn.shape[0], face.conn.shape[1], 3))
    free = torch.ones(3 * N, dtype=torch.float64, device=val.device)
    free[_t(_clamp(m), torch.int64)] = 0.0
    u = torch.zeros_like(f)
    for _ in range(2):                                       # a restart from the true residual
        r = free * (f - K @ u)
        z = free * r / diag
        p, rho = z.clone(), torch.dot(r, z)
        stop = 1e-30 * float(torch.dot(f, f))
        for it in range(20000):
            q = free * (K @ p)
            a = rho / torch.dot(p, q)
            u += a * p
            r -= a * q
            if it % 25 == 0 and float(torch.dot(r, r)) <= stop:
                break
            z = r / diag
            new = torch.dot(r, z)
            p = z + (new / rho) * p
            rho = new
    return u


def exact(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind == "stiffness":
        m, tab, mats = inp
        return _stiffness_values(m, tab, mats, _group_scales(m, case["groups"]))[0]
    if kind == "mass":
        return _mass_values(*inp, case["lumped"])
    if kind == "load":
        return _load_values(case, *inp)
    if kind == "batch":
        out = []
        for k, m, E, nu, rho in inp:
            tk, tm = W.rules(k)
            out.append({"K": _stiffness_values(m, tk, [(E, nu)], [None])[0], "M": _mass_values(m, tm, rho, False)})
        return out
    if kind == "serve":
        got = []
        for k, m, E, nu, fy in inp:
            face = m.faces["right"]
            got.append(_solution(m, R.rule_tables(m.etype, _stiffness_degree(k)), (E, nu), [0.0, fy, 0.0], face,
                                 R.rule_tables(face.etype, 2 * W.KINDS[k][1] + 1)) if m.N < 60000 else None)
        return got
    m, tab, mat, t = inp
    if m.N > 150000:
        return None                                          # minutes of Jacobi-CG
    face = m.faces["right"]
    return _solution(m, tab, mat, t, face, R.rule_tables(face.etype, 2 * ELEMS[case["elem"]][1] + 1))
