"""The work that a user of this library has it do, as timed cases.

Every case calls the library through ``ngsxfem_amd._abi`` (``Context`` and
``Batch``, the binding of the C ABI in include/xg_abi.h) on device tensors, the
way a solver step does: mark the elements of a level set, build cut rules,
integrate, form element matrices, assemble.

Kinds:
  step       one small whole step: marking, then the matrices of the cut elements
  mark       marking of a mesh (domains, cut ratios, bit arrays, cut list)
  integrate  a straight cut rule on the whole mesh and an integral on it
  form       fused cut rule + element matrices, moment form or MFMA contraction
  cf         rule, coefficient function on its points, matrices and vectors
  subdiv     subdivision rule of a P2 level set + element matrices
  assemble   matrix graph, element matrices, global CSR values
  hex        quadrilateral / hexahedral cut rule + Q1 matrices
  batch      many meshes of uneven size and order in one captured sequence
"""
import itertools
import math

import numpy as np
import torch

from ngsxfem_amd import _abi

NEG, POS, IF = 0, 1, 2
DTS = {"neg": [NEG], "pos": [POS], "if": [IF], "neg+if": [NEG, IF], "neg+pos+if": [NEG, POS, IF]}
PREC = {"fp64": _abi.XG_PREC_FP64, "fp32": _abi.XG_PREC_FP32, "bf16x3": _abi.XG_PREC_BF16X3}
TERMS = [(1.0, (0, 0, 0)), (0.5, (1, 1, 0)), (2.0, (0, 2, 0))]
BALLS = 64  # spheres of the large mixed workload


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one time step of the reference's two-dimensional circle example
        {"name": "step_tri_60", "kind": "step", "D": 2, "nx": 60, "ny": 60, "nz": 0, "p": 1, "prec": "fp64"},
        # marking alone, on the largest mesh that the benchmark uses (12.6 million tetrahedra)
        {"name": "mark_tet_128", "kind": "mark", "D": 3, "nx": 128, "ny": 128, "nz": 128},
        # Integrate over the inside of a level set, order 4, 64^3 cells
        {"name": "integrate_tet_64", "kind": "integrate", "D": 3, "nx": 64, "ny": 64, "nz": 64, "dom": "neg",
         "order": 4},
        # the 3D benchmark: P2 mass + stiffness on the inside and on the interface
        {"name": "form_tet_p2_64", "kind": "form", "D": 3, "nx": 64, "ny": 64, "nz": 64, "p": 2, "order": 4,
         "dom": "neg+if", "mask": 3, "prec": "fp32", "moments": True},
        # cubic elements on the largest mesh
        {"name": "form_tet_p3_128", "kind": "form", "D": 3, "nx": 128, "ny": 128, "nz": 128, "p": 3, "order": 6,
         "dom": "neg+if", "mask": 3, "prec": "fp32", "moments": True},
        # the same matrices by the MFMA contraction (the Python surface's default arithmetic), ragged mesh
        {"name": "form_tet_mfma_p2", "kind": "form", "D": 3, "nx": 61, "ny": 53, "nz": 67, "p": 2, "order": 4,
         "dom": "neg+if", "mask": 3, "prec": "fp32", "moments": False},
        # c u v and f v with a coefficient function on all elements with an inside part
        {"name": "cf_tet_p2_40", "kind": "cf", "D": 3, "nx": 40, "ny": 40, "nz": 40, "p": 2, "order": 6, "dom": "neg",
         "prec": "fp32"},
        # a curved (P2) level set on a small mesh
        {"name": "subdiv_p2_l3_20", "kind": "subdiv", "nx": 20, "p": 2, "L": 3, "dom": "neg+if", "mask": 3,
         "prec": "fp32"},
        # the default benchmark: 128^3 cells, union of 64 spheres, P3, level-4 subdivision
        {"name": "subdiv_p3_l4_128", "kind": "subdiv", "nx": 128, "p": 3, "L": 4, "dom": "neg+if", "mask": 3,
         "prec": "fp32"},
        # BilinearForm.Assemble: P2 graph of the mesh, matrices of the elements inside, CSR values
        {"name": "assemble_tet_p2_32", "kind": "assemble", "D": 3, "nx": 32, "ny": 32, "nz": 32, "p": 2, "dom": "neg",
         "prec": "fp64"},
        # hexahedra: tensor-product cut rule and Q1 matrices of the cut elements
        {"name": "hex_48", "kind": "hex", "D": 3, "nx": 48, "ny": 48, "nz": 48, "order": 4, "dom": "neg", "policy": 1,
         "prec": "fp64"},
        # many meshes of uneven size and order, one graph launch
        {"name": "batch_64", "kind": "batch", "meshes": 64, "nmin": 8, "nmax": 48, "dom": "neg+if", "mask": 3},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def _cells(rng, D, lo, hi):
    n = _log(rng, lo, hi)
    m = [max(2, int(round(n * rng.uniform(0.7, 1.0)))) for _ in range(3)]
    return {"nx": m[0], "ny": m[1], "nz": m[2] if D == 3 else 0}


def draw(rng):
    kind = rng.choice(["step", "mark", "integrate", "form", "form", "cf", "subdiv", "subdiv", "assemble", "hex",
                       "batch"])
    D = rng.choice([2, 3, 3])
    p = rng.choice([1, 2, 3])
    if kind == "step":
        return dict({"kind": kind, "D": D, "p": p, "prec": rng.choice(["fp64", "fp32"])},
                    **_cells(rng, D, 6, 400 if D == 2 else 24))
    if kind == "mark":
        return dict({"kind": kind, "D": D}, **_cells(rng, D, 6, 1500 if D == 2 else 128))
    if kind == "integrate":
        return dict({"kind": kind, "D": D, "dom": rng.choice(["neg", "neg", "pos", "if"]),
                     "order": rng.choice([2, 3, 4, 5, 6])}, **_cells(rng, D, 8, 800 if D == 2 else 64))
    if kind == "form":
        c = {"kind": kind, "D": D, "p": p, "order": 2 * p + rng.choice([0, 0, 1, 2]), "mask": rng.choice([1, 2, 3, 3]),
             "dom": rng.choice(["neg", "pos", "if", "neg+if", "neg+pos+if"])}
        how = rng.choice(["moments", "moments", "mfma", "bf16x3"])
        c["moments"] = how == "moments"
        c["prec"] = rng.choice(["fp32", "fp64"]) if how == "moments" else ("fp32" if how == "mfma" else "bf16x3")
        return dict(c, **_cells(rng, D, 8, 800 if D == 2 else (96 if how == "moments" else 48)))
    if kind == "cf":
        return dict({"kind": kind, "D": D, "p": p, "order": 2 * p + 2, "dom": rng.choice(["neg", "neg", "if"]),
                     "prec": rng.choice(["fp32", "fp64"])}, **_cells(rng, D, 6, 300 if D == 2 else 32))
    if kind == "subdiv":
        return {"kind": kind, "nx": _log(rng, 8, 96), "p": p, "L": rng.choice([1, 2, 3, 4, 4]),
                "dom": rng.choice(["neg", "if", "pos", "neg+if", "neg+if"]), "mask": rng.choice([1, 2, 3, 3]),
                "prec": rng.choice(["fp32", "fp32", "fp64"])}
    if kind == "assemble":
        return dict({"kind": kind, "D": D, "p": rng.choice([1, 2]), "dom": rng.choice(["neg", "pos", "if"]),
                     "prec": rng.choice(["fp32", "fp64"])}, **_cells(rng, D, 6, 300 if D == 2 else 36))
    if kind == "hex":
        return dict({"kind": kind, "D": D, "order": rng.choice([2, 3, 4, 5]), "dom": rng.choice(["neg", "pos", "if"]),
                     "policy": rng.choice([0, 1, 1, 2]), "prec": rng.choice(["fp32", "fp64"])},
                    **_cells(rng, D, 6, 300 if D == 2 else 48))
    return {"kind": "batch", "meshes": _log(rng, 4, 64), "nmin": rng.randint(4, 12), "nmax": rng.randint(16, 48),
            "dom": rng.choice(["neg", "if", "neg+if"]), "mask": rng.choice([1, 2, 3])}


# ------------------------------------------------------------------ inputs
def _grid(*ns):
    return torch.meshgrid(*[torch.arange(n, device="cuda") for n in ns], indexing="ij")


def _mesh(D, nx, ny, nz=0):
    """(coords, el2v) of the structured simplex mesh: [-1.5,1.5]^2 with two triangles per cell, or the unit cube with
    six Kuhn tetrahedra per cell"""
    if D == 2:
        i, j = _grid(nx + 1, ny + 1)
        X = torch.stack([-1.5 + 3.0 * i.reshape(-1) / nx, -1.5 + 3.0 * j.reshape(-1) / ny], dim=1).double()
        ci, cj = (a.reshape(-1) for a in _grid(nx, ny))
        v = lambda a, b: (ci + a) * (ny + 1) + cj + b  # noqa: E731
        el = torch.stack([torch.stack([v(0, 0), v(1, 0), v(1, 1)], 1), torch.stack([v(0, 0), v(1, 1), v(0, 1)], 1)], 1)
        return X.contiguous(), el.reshape(-1, 3).int().contiguous()
    i, j, k = (a.reshape(-1).double() for a in _grid(nx + 1, ny + 1, nz + 1))
    X = torch.stack([i / nx, j / ny, k / nz], dim=1)
    ci, cj, ck = (a.reshape(-1) for a in _grid(nx, ny, nz))
    v = lambda o: ((ci + o[0]) * (ny + 1) + cj + o[1]) * (nz + 1) + ck + o[2]  # noqa: E731
    tets = []
    for perm in itertools.permutations(range(3)):
        o, vs = [0, 0, 0], [v((0, 0, 0))]
        for ax in perm:
            o[ax] += 1
            vs.append(v(o))
        tets.append(torch.stack(vs, 1))
    return X.contiguous(), torch.stack(tets, 1).reshape(-1, 4).int().contiguous()


def _cube_mesh(D, nx, ny, nz=0):
    """(coords, el2v) of the structured quadrilateral / hexahedral mesh"""
    v2 = [(0, 0), (1, 0), (1, 1), (0, 1)]
    if D == 2:
        i, j = _grid(nx + 1, ny + 1)
        X = torch.stack([-1.5 + 3.0 * i.reshape(-1) / nx, -1.5 + 3.0 * j.reshape(-1) / ny], dim=1).double()
        ci, cj = (a.reshape(-1) for a in _grid(nx, ny))
        el = torch.stack([(ci + a) * (ny + 1) + cj + b for a, b in v2], 1)
        return X.contiguous(), el.int().contiguous()
    i, j, k = (a.reshape(-1).double() for a in _grid(nx + 1, ny + 1, nz + 1))
    X = torch.stack([i / nx, j / ny, k / nz], dim=1)
    ci, cj, ck = (a.reshape(-1) for a in _grid(nx, ny, nz))
    el = torch.stack([((ci + a) * (ny + 1) + cj + b) * (nz + 1) + ck + c for c in (0, 1) for a, b in v2], 1)
    return X.contiguous(), el.int().contiguous()


def _ball(X, rng):
    """P1 values of a ball with a wavy surface (a circle in 2D), perturbed off zero as InterpolateToP1 does"""
    D = X.shape[1]
    if D == 2:
        c, r = rng.uniform(-0.2, 0.2, 2), rng.uniform(0.9, 1.1)
        phi = torch.sqrt((X[:, 0] - c[0]) ** 2 + (X[:, 1] - c[1]) ** 2) - r
    else:
        c, r = rng.uniform(0.47, 0.53, 3), rng.uniform(0.33, 0.37)
        s = sum((X[:, d] - c[d]) ** 2 for d in range(3))
        phi = torch.sqrt(s) - r + 0.01 * torch.sin(7 * X[:, 0]) * torch.sin(7 * X[:, 1]) * torch.sin(7 * X[:, 2])
    return torch.where(phi.abs() < 1e-14, torch.full_like(phi, 1e-14), phi)


def _is_cut(lset, el2v):
    v = lset[el2v.long()]
    return (v > 0).any(1) & (v < 0).any(1)


def _ids(mask):
    return torch.nonzero(mask).reshape(-1).int().contiguous()


def _p2_dofs(el2v, nv):
    """element dof table of the P2 space: vertices, then one dof per edge"""
    D = el2v.shape[1] - 1
    pairs = [(i, j) for i in range(D + 1) for j in range(i + 1, D + 1)]
    e = el2v.long()
    key = torch.stack([torch.minimum(e[:, i], e[:, j]) * nv + torch.maximum(e[:, i], e[:, j]) for i, j in pairs], 1)
    uniq, inv = torch.unique(key.reshape(-1), return_inverse=True)
    return torch.cat([e, nv + inv.reshape(key.shape)], 1).int().contiguous(), nv + uniq.numel()


def _ndof(D, p):
    return math.comb(p + D, D)


def _spheres_p2(nx, rng):
    """el2v, coords and the P2 nodal values (ne x 10) of the union of spheres on the nx^3 Kuhn mesh.  The vertices and
    edge midpoints are the points of the grid with half the mesh width."""
    X, el = _mesh(3, nx, nx, nx)
    C, R = rng.uniform(0.2, 0.8, (BALLS, 3)), rng.uniform(0.05, 0.15, BALLS)
    m = 2 * nx + 1
    t = torch.arange(m, device="cuda", dtype=torch.float64) / (2 * nx)
    val = torch.full((m, m, m), float("inf"), dtype=torch.float64, device="cuda")
    for c, r in zip(C, R):
        d = ((t - c[0]) ** 2)[:, None, None] + ((t - c[1]) ** 2)[None, :, None] + ((t - c[2]) ** 2)[None, None, :]
        val = torch.minimum(val, d.sqrt_().sub_(r))
    val = val.reshape(-1)
    n1 = nx + 1
    nod = torch.empty((el.shape[0], 10), dtype=torch.float64, device="cuda")
    e = el.long()
    ijk = [(e[:, k] // (n1 * n1), (e[:, k] // n1) % n1, e[:, k] % n1) for k in range(4)]
    for col, (a, b) in enumerate([(0, 0), (1, 1), (2, 2), (3, 3), (0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)]):
        i, j, k = (ijk[a][d] + ijk[b][d] for d in range(3))
        nod[:, col] = val[(i * m + j) * m + k]
    return X, el, nod


def _coefficient(gf):
    """(code, constants, grid functions) of c = 1 + x y / 2 + gf"""
    return [1, 0, 1, 1, 2, 0, 5, 2, 1, 5, 3, 19, 0, 3], [1.0, 0.5], [gf]


def _batch_shapes(case):
    """cells per direction and degree of every mesh: a property of the case, as is the plan that it needs"""
    rng = np.random.default_rng(case["meshes"])
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    return [(int(round(math.exp(rng.uniform(lo, hi)))), int(rng.integers(1, 4))) for _ in range(case["meshes"])]


def _batch_meshes(case, rng):
    X, el, ls, off, ps, nv = [], [], [], [0], [], 0
    for n, p in _batch_shapes(case):
        ax = rng.uniform(0.15, 0.45, 3)
        x, e = _mesh(3, n, n, n)
        phi = sum(((x[:, d] - 0.5) / ax[d]) ** 2 for d in range(3)) - 1.0
        X.append(x)
        el.append(e + nv)
        ls.append(torch.where(phi.abs() < 1e-14, torch.full_like(phi, 1e-14), phi))
        nv += x.shape[0]
        off.append(off[-1] + e.shape[0])
        ps.append(p)
    return torch.cat(X), torch.cat(el).contiguous(), torch.cat(ls), off, ps


def _room(case):
    """elements that the output buffers of a case have room for: more than any level set of the case cuts (cf, assemble:
    meets).  What is left over stays zero."""
    kind = case["kind"]
    if kind == "subdiv":
        return min(6 * case["nx"] ** 3, 40 * case["nx"] ** 2)
    D = case["D"]
    m = max(case["nx"], case["ny"], case["nz"])
    cells = case["nx"] * case["ny"] * max(case["nz"], 1)
    if kind == "hex":
        return min(cells, 4 * m + 16 if D == 2 else 4 * m * m + 64)
    ne = cells * (2 if D == 2 else 6)
    cut = min(ne, 8 * m + 32 if D == 2 else 16 * m * m + 64)
    if kind == "cf" and case["dom"] != "if":
        return min(ne, cut + int((0.5 if D == 2 else 0.3) * ne))
    return cut


def _batch_room(case):
    """floats for a batch's matrices: a ball of the largest semi-axis cuts 17.4 n^2 elements"""
    ndt = len(DTS[case["dom"]])
    return sum(min(6 * n ** 3, 20 * n * n + 64) * ndt * _ndof(3, p) ** 2 for n, p in _batch_shapes(case))


def _fits(n, case):
    if n > _room(case):
        raise ValueError("%d elements, and room for %d" % (n, _room(case)))
    return _room(case)


def _padded(t, n):
    """t (m, ...) flat, with zeros for the rows m .. n that a pass leaves as they are"""
    out = torch.zeros((n,) + tuple(t.shape[1:]), dtype=t.dtype, device="cuda")
    out[:t.shape[0]] = t
    return out.reshape(-1)


def _mark_buffers(ne):
    z = lambda n, t: torch.zeros(n, dtype=t, device="cuda")  # noqa: E731
    return {"dt": z(ne, torch.uint8), "cr": z(ne, torch.float64), "bits": z(8 * ((ne + 31) // 32), torch.int32),
            "cl": z(ne, torch.int32), "nc": z(1, torch.int32)}


def _fp(prec):
    return torch.float64 if prec == "fp64" else torch.float32


def _inputs(case, seed):
    """mesh, level set and element lists: what the library is given"""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = dict(case)
    if kind == "batch":
        s["X"], s["el"], s["ls"], s["off"], s["ps"] = _batch_meshes(case, rng)
        return s
    if kind == "subdiv":
        s["X"], s["el"], s["nod"] = _spheres_p2(case["nx"], rng)
        return s
    D = case["D"]
    s["X"], s["el"] = (_cube_mesh if kind == "hex" else _mesh)(D, case["nx"], case["ny"], case["nz"])
    s["ls"] = _ball(s["X"], rng)
    v = s["ls"][s["el"].long()]
    s["cut"] = _ids((v > 0).any(1) & (v < 0).any(1))
    if kind in ("cf", "assemble"):
        dt = DTS[case["dom"]][0]
        s["elems"] = s["cut"] if dt == IF else _ids((v < 0).any(1) if dt == NEG else (v > 0).any(1))
    if kind == "cf":
        s["gf"] = torch.sin(3 * s["X"][:, 0]) + 0.3 * s["X"][:, 1]
    if kind == "assemble":
        s["dofs"], s["n"] = (s["el"], s["X"].shape[0]) if case["p"] == 1 else _p2_dofs(s["el"], s["X"].shape[0])
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    ctx = s["ctx"] = _abi.Context(0)
    ne = s["el"].shape[0]
    cuda = {"device": "cuda"}
    if kind in ("step", "mark"):
        s.update(_mark_buffers(ne))
        if kind == "step":
            nd = _ndof(case["D"], case["p"])
            s["out"] = torch.zeros(_fits(s["cut"].numel(), case) * 2 * nd * nd, dtype=_fp(case["prec"]), **cuda)
    elif kind == "integrate":
        s["offsets"] = torch.zeros(ne + 1, dtype=torch.int32, **cuda)
        s["per_elem"] = torch.zeros(ne, dtype=torch.float64, **cuda)
        s["total"] = torch.zeros(1, dtype=torch.float64, **cuda)
    elif kind == "form":
        nd = _ndof(case["D"], case["p"])
        n = _fits(s["cut"].numel(), case) * len(DTS[case["dom"]]) * nd * nd
        s["out"] = torch.zeros(n, dtype=_fp(case["prec"]), **cuda)
    elif kind == "cf":
        nd, n = _ndof(case["D"], case["p"]), _fits(s["elems"].numel(), case)
        s["offsets"] = torch.zeros(n + 1, dtype=torch.int32, **cuda)
        s["mat"] = torch.zeros(n * nd * nd, dtype=_fp(case["prec"]), **cuda)
        s["vec"] = torch.zeros(n * nd, dtype=torch.float64, **cuda)
    elif kind == "subdiv":
        b = _mark_buffers(ne)
        ctx.mark_p2(s["nod"], case["L"], b["dt"], b["bits"], b["cl"], b["nc"])
        ctx.sync()
        s["cut"] = b["cl"][:int(b["nc"].item())].clone()
        nd = _ndof(3, case["p"])
        n = _fits(s["cut"].numel(), case) * len(DTS[case["dom"]]) * nd * nd
        s["out"] = torch.zeros(n, dtype=_fp(case["prec"]), **cuda)
    elif kind == "assemble":
        nd = s["dofs"].shape[1]
        s["edofs"] = s["dofs"][s["elems"].long()].contiguous()
        s["mat"] = torch.zeros(s["elems"].numel() * nd * nd, dtype=_fp(case["prec"]), **cuda)
        s["row_ptr"] = torch.zeros(s["n"] + 1, dtype=torch.int32, **cuda)
        s["col"] = torch.zeros(ne * nd * nd, dtype=torch.int32, **cuda)
        s["nnz"] = torch.zeros(1, dtype=torch.int32, **cuda)
    elif kind == "hex":
        n, k = _fits(s["cut"].numel(), case), s["el"].shape[1]
        s["offsets"] = torch.zeros(n + 1, dtype=torch.int32, **cuda)
        s["mat"] = torch.zeros(n * k * k, dtype=_fp(case["prec"]), **cuda)
    elif kind == "batch":
        torch.cuda.synchronize()
        b = s["batch"] = _abi.Batch(ctx, s["X"], s["el"], s["ls"], s["off"], s["ps"], dts=DTS[case["dom"]],
                                    mask=case["mask"])
        b.method(_abi.XG_METHOD_MOMENTS)
        b.plan()
        s["out"] = torch.zeros(_batch_room(case), dtype=torch.float32, **cuda)
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    return _RUN[s["kind"]](s, s["ctx"])


def _run_step(s, ctx):
    D, p = s["D"], s["p"]
    ctx.mark(D, s["el"], s["ls"], s["dt"], s["cr"], s["bits"], s["cl"], s["nc"])
    n = int(s["nc"].item())
    ctx.cut_pipeline(D, p, 2 * p, s["el"], s["X"], s["ls"], [NEG, IF], 3, PREC[s["prec"]] | _abi.XG_METHOD_MOMENTS,
                     s["out"], elems=s["cl"][:n])
    return s["dt"], s["cr"], s["bits"], s["cl"], s["out"]


def _run_mark(s, ctx):
    ctx.mark(s["D"], s["el"], s["ls"], s["dt"], s["cr"], s["bits"], s["cl"], s["nc"])
    return s["dt"], s["cr"], s["bits"], s["cl"], s["nc"]


def _run_integrate(s, ctx):
    D, dt, order = s["D"], DTS[s["dom"]][0], s["order"]
    ctx.cut_rule_count(D, s["el"], s["ls"], dt, order, s["offsets"])
    pts = torch.empty((int(s["offsets"][-1].item()), 4), dtype=torch.float64, device="cuda")
    ctx.cut_rule_fill(D, s["el"], s["X"], s["ls"], dt, order, s["offsets"], pts)
    ctx.integrate(D, s["el"], s["X"], s["offsets"], pts, TERMS, s["total"], s["per_elem"])
    return s["offsets"], s["per_elem"], s["total"]


def _run_form(s, ctx):
    prec = PREC[s["prec"]] | (_abi.XG_METHOD_MOMENTS if s["moments"] else 0)
    ctx.cut_pipeline(s["D"], s["p"], s["order"], s["el"], s["X"], s["ls"], DTS[s["dom"]], s["mask"], prec, s["out"],
                     elems=s["cut"])
    return s["out"]


def _run_cf(s, ctx):
    D, p, dt, order = s["D"], s["p"], DTS[s["dom"]][0], s["order"]
    ctx.cut_rule_count(D, s["el"], s["ls"], dt, order, s["offsets"], elems=s["elems"])
    pts = torch.empty((int(s["offsets"][s["elems"].numel()].item()), 4), dtype=torch.float64, device="cuda")
    ctx.cut_rule_fill(D, s["el"], s["X"], s["ls"], dt, order, s["offsets"], pts, elems=s["elems"])
    code, consts, gfs = _coefficient(s["gf"])
    ctx.rule_scale_cf(D, s["el"], s["X"], s["offsets"], pts, code, consts, gfs, elems=s["elems"])
    ctx.elmat(D, p, s["el"], s["X"], s["offsets"], pts, 3, PREC[s["prec"]], s["mat"], elems=s["elems"])
    ctx.elvec(D, p, s["el"], s["X"], s["offsets"], pts, s["vec"], elems=s["elems"])
    return s["offsets"], s["mat"], s["vec"]


def _run_subdiv(s, ctx):
    ctx.subdiv_pipeline(s["p"], s["L"], 2 * s["p"], s["cut"], s["el"], s["X"], s["nod"], DTS[s["dom"]], s["mask"],
                        PREC[s["prec"]], s["out"])
    return s["out"]


def _run_assemble(s, ctx):
    D, p, prec = s["D"], s["p"], PREC[s["prec"]]
    ctx.csr_pattern(s["dofs"], s["n"], s["row_ptr"], s["col"], s["nnz"])
    nnz = int(s["nnz"].item())
    values = torch.zeros(nnz, dtype=torch.float64, device="cuda")
    ctx.cut_pipeline(D, p, 2 * p, s["el"], s["X"], s["ls"], DTS[s["dom"]], 3, prec | _abi.XG_METHOD_MOMENTS, s["mat"],
                     elems=s["elems"])
    ctx.assemble_csr(s["edofs"], s["mat"], prec, s["row_ptr"], s["col"], values)
    return s["row_ptr"], s["col"][:nnz], values


def _run_hex(s, ctx):
    D, dt, order, pol = s["D"], DTS[s["dom"]][0], s["order"], s["policy"]
    ctx.quad_rule_count(D, s["el"], s["ls"], dt, order, pol, s["offsets"], elems=s["cut"])
    pts = torch.empty((int(s["offsets"][s["cut"].numel()].item()), 4), dtype=torch.float64, device="cuda")
    ctx.quad_rule_fill(D, s["el"], s["X"], s["ls"], dt, order, pol, s["offsets"], pts, elems=s["cut"])
    ctx.quad_elmat(D, s["el"], s["X"], s["offsets"], pts, 3, PREC[s["prec"]], s["mat"], elems=s["cut"])
    return s["offsets"], s["mat"]


def _run_batch(s, ctx):
    s["batch"].run(s["out"])
    return s["out"]


_RUN = {"step": _run_step, "mark": _run_mark, "integrate": _run_integrate, "form": _run_form, "cf": _run_cf,
        "subdiv": _run_subdiv, "assemble": _run_assemble, "hex": _run_hex, "batch": _run_batch}


# ------------------------------------------------------------------ what a pass cannot do without
def _counts(case):
    """(elements, vertices, cut elements, share of the elements inside) as the level sets of these cases have them"""
    D = case.get("D", 3)
    if case["kind"] == "batch":
        # sizes log-uniform in [nmin, nmax], ellipsoids with semi-axes around 0.3
        a, b = case["nmin"], case["nmax"]
        m = lambda k: case["meshes"] * (b ** k - a ** k) / (k * math.log(b / a))  # noqa: E731
        return 6 * m(3), m(3), 7.5 * m(2), 0.1
    if case["kind"] == "subdiv":
        n = case["nx"]
        return 6.0 * n ** 3, (n + 1.0) ** 3, 24.7 * n * n, 0.15
    if D == 2:
        n = math.sqrt(case["nx"] * case["ny"])
        ne, nv, cut, frac = 2.0 * n * n, (n + 1) ** 2, 4.5 * n, 0.35
    else:
        n = (case["nx"] * case["ny"] * case["nz"]) ** (1 / 3)
        ne, nv, cut, frac = 6.0 * n ** 3, (n + 1) ** 3, 10.5 * n * n, 0.18
    if case["kind"] == "hex":
        ne, cut = (n * n, 2.2 * n) if D == 2 else (n ** 3, 2.3 * n * n)
    return ne, nv, cut, frac


def _matrix_flops(D, p, points):
    """a matrix from a rule: every point's symmetric rank-one update of the degree-p products"""
    nd = _ndof(D, p)
    return points * nd * (nd + 1) * (1 + D)


def work(case):
    kind, D, p = case["kind"], case.get("D", 3), case.get("p", 2)
    ne, nv, cut, frac = _counts(case)
    tab, nd = 4 * (D + 1), _ndof(D, p)
    b = 8 if case.get("prec") == "fp64" else 4
    ndt = len(DTS[case.get("dom", "neg")])
    geo = tab + 4 + 8 * D + 8  # an element's row and id, and about one vertex's coordinates and value for each
    mark = {"bytes": ne * (tab + 9 + 1) + 8 * nv + 4 * cut, "flops": 4 * ne + 60 * cut}
    if kind == "mark":
        return mark
    if kind == "step":
        return {"bytes": mark["bytes"] + cut * (geo + 2 * nd * nd * b),
                "flops": mark["flops"] + cut * _matrix_flops(D, p, (p + 1) ** D)}
    if kind == "integrate":
        q = (case["order"] // 2 + 1) ** D
        pts = {"neg": frac * ne * q + 2 * cut * q, "pos": (1 - frac) * ne * q + 2 * cut * q,
               "if": 1.3 * cut * q ** ((D - 1) / D)}[case["dom"]]
        return {"bytes": ne * (tab + 4 + 8) + nv * 8 * (D + 1) + 32 * pts, "flops": pts * (4 * D * D + 20)}
    if kind == "form":
        return {"bytes": cut * (geo + ndt * nd * nd * b), "flops": cut * ndt * _matrix_flops(D, p, (p + 1) ** (D - 1))}
    if kind == "cf":
        n = cut if case["dom"] == "if" else frac * ne + cut / 2
        q = (case["order"] // 2 + 1) ** (D - (case["dom"] == "if"))
        return {"bytes": n * (geo + 4 + nd * nd * b + nd * 8), "flops": n * _matrix_flops(D, p, q)}
    if kind == "subdiv":
        leaves = 1.25 * 4 ** case["L"]  # leaves that the interface meets
        return {"bytes": cut * (geo + 80 + ndt * nd * nd * b),
                "flops": cut * ndt * leaves * 6 * 2 * math.comb(2 * p + 3, 3)}
    if kind == "assemble":
        n = {"neg": frac * ne + cut / 2, "pos": (1 - frac) * ne + cut / 2, "if": cut}[case["dom"]]
        rows, per_row = (nv, 15 if D == 3 else 7) if p == 1 else ((8 * nv, 29) if D == 3 else (4 * nv, 12))
        return {"bytes": ne * 4 * nd + n * (geo + 4 * nd) + rows * (4 + 12 * per_row),
                "flops": n * (nd * nd + _matrix_flops(D, p, 1))}
    if kind == "hex":
        k = 2 ** D
        q = (case["order"] // 2 + 1) ** (D - (case["dom"] == "if"))
        return {"bytes": cut * (4 * k + 8 + 8 * (D + 1) + 32 * 2 * q + k * k * b), "flops": cut * 2 * q * k * k * 4}
    per = sum(_ndof(3, k) ** 2 for k in (1, 2, 3)) / 3
    return {"bytes": ne * (16 + 9 + 1) + 8 * nv + cut * (geo + ndt * per * 4),
            "flops": 4 * ne + cut * ndt * sum(_matrix_flops(3, k, (k + 1) ** 2) for k in (1, 2, 3)) / 3}


def tolerance(case):
    """four times what the path differs by from its 64-bit value: FP64 arithmetic rounded once to FP32 shows 2.5e-8, FP32
    shape values and products with FP64 sums of groups of points 1e-7, FP64 results 1.3e-15 (a sum over all elements,
    in no fixed order, 6e-13; sums over the thousands of pieces of a subdivision rule more than one rule's)"""
    kind = case["kind"]
    if kind == "mark":
        return "exact"
    if kind == "integrate":
        return {"rel": 2e-12}
    if kind == "cf" and case["prec"] == "fp32" or kind == "form" and not case["moments"]:
        return {"rel": 5e-7}
    if kind == "batch" or case["prec"] == "fp32":
        return {"rel": 1e-7}
    return {"rel": 1e-13 if kind == "subdiv" else 2e-14}


# ------------------------------------------------------------------ the same numbers in 64 bits
def _gauss(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1), 0.5 * w


def _simplex_rule(dim, n):
    """barycentric points (q, dim + 1) and weights (sum 1) exact for degree 2 n - dim on the unit simplex"""
    x, w = _gauss(n)
    if dim == 1:
        B, W = [[1 - a, a] for a in x], list(w)
    elif dim == 2:
        B, W = [], []
        for (a, wa), (b, wb) in itertools.product(zip(x, w), repeat=2):
            B.append([1 - a, a * (1 - b), a * b])
            W.append(2 * wa * wb * a)
    else:
        B, W = [], []
        for (a, wa), (b, wb), (c, wc) in itertools.product(zip(x, w), repeat=3):
            B.append([1 - a, a * (1 - b), a * b * (1 - c), a * b * c])
            W.append(6 * wa * wb * wc * a * a * b)
    t = lambda v: torch.tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
    return t(B), t(W)


#: pieces of {phi < 0} in a simplex whose vertices are sorted by value, by (dimension, number of negative vertices): a
#: piece's corner is a vertex (i,) or the cut point of an edge (i, j)
_NEG_PIECES = {
    (2, 1): [[(0,), (0, 1), (0, 2)]], (2, 2): [[(0,), (1,), (1, 2)], [(0,), (1, 2), (0, 2)]],
    (2, 3): [[(0,), (1,), (2,)]],
    (3, 1): [[(0,), (0, 1), (0, 2), (0, 3)]],
    (3, 2): [[(0,), (0, 2), (0, 3), (1, 3)], [(0,), (0, 2), (1, 2), (1, 3)], [(0,), (1,), (1, 2), (1, 3)]],
    (3, 3): [[(0,), (1,), (2,), (2, 3)], [(0,), (1,), (1, 3), (2, 3)], [(0,), (0, 3), (1, 3), (2, 3)]],
    (3, 4): [[(0,), (1,), (2,), (3,)]]}
_IF_PIECES = {
    (2, 1): [[(0, 1), (0, 2)]], (2, 2): [[(0, 2), (1, 2)]],
    (3, 1): [[(0, 1), (0, 2), (0, 3)]], (3, 3): [[(0, 3), (1, 3), (2, 3)]],
    (3, 2): [[(0, 2), (0, 3), (1, 3)], [(0, 2), (1, 3), (1, 2)]]}


def _pieces(l, dt):
    """(element numbers, corners in barycentric coordinates (m, k, D + 1)) of the part dt of simplices with vertex
    values l (n, D + 1)"""
    D = l.shape[1] - 1
    v = -l if dt == POS else l
    srt, perm = torch.sort(v, dim=1)
    nneg = ((v <= 0) if dt == POS else (v < 0)).sum(1)
    unit = torch.eye(D + 1, dtype=torch.float64, device="cuda")[perm]  # sorted vertex -> barycentric
    who, corners = [], []
    for (dim, k), pieces in (_IF_PIECES if dt == IF else _NEG_PIECES).items():
        if dim != D:
            continue
        at = torch.nonzero(nneg == k).reshape(-1)
        for piece in pieces:
            cs = []
            for c in piece:
                if len(c) == 1:
                    cs.append(unit[at, c[0]])
                else:
                    a, b = srt[at, c[0]], srt[at, c[1]]
                    t = (a / (a - b))[:, None]
                    cs.append((1 - t) * unit[at, c[0]] + t * unit[at, c[1]])
            who.append(at)
            corners.append(torch.stack(cs, 1))
    return torch.cat(who), torch.cat(corners)


def _measure(V):
    """measure of the simplices with corners V (m, k, D)"""
    E = V[:, 1:] - V[:, :1]
    k = E.shape[1]
    return torch.linalg.det(E @ E.transpose(1, 2)).clamp_min(0).sqrt() / math.factorial(k) if k < E.shape[2] else \
        torch.linalg.det(E).abs() / math.factorial(k)


def _alphas(D, p):
    """multi-indices of the Lagrange nodes: by number of vertices, then vertices, then descending"""
    al = [a for a in itertools.product(range(p, -1, -1), repeat=D + 1) if sum(a) == p]
    sup = lambda a: tuple(i for i, v in enumerate(a) if v)  # noqa: E731
    return sorted(al, key=lambda a: (len(sup(a)), sup(a), tuple(-v for v in a)))


def _shapes(lam, p):
    """Lagrange shape functions and their derivatives by the barycentrics at lam (..., D + 1)"""
    D = lam.shape[-1] - 1
    one = torch.ones_like(lam[..., 0])
    L, dL = [], []
    for k in range(D + 1):
        v, d = [one], [0 * one]
        for m in range(p):
            f = (p * lam[..., k] - m) / (m + 1)
            d.append(d[-1] * f + v[-1] * (p / (m + 1)))
            v.append(v[-1] * f)
        L.append(v)
        dL.append(d)
    phi, dphi = [], []
    for a in _alphas(D, p):
        t = one
        for k in range(D + 1):
            t = t * L[k][a[k]]
        phi.append(t)
        g = []
        for k in range(D + 1):
            t = dL[k][a[k]]
            for j in range(D + 1):
                if j != k:
                    t = t * L[j][a[j]]
            g.append(t)
        dphi.append(torch.stack(g, -1))
    return torch.stack(phi, -1), torch.stack(dphi, -2)


def _bary_grads(V):
    """gradients of the barycentrics of simplices V (n, D + 1, D)"""
    G = torch.linalg.inv(V[:, :-1] - V[:, -1:]).transpose(1, 2)  # row c: gradient of lam_c
    return torch.cat([G, -G.sum(1, keepdim=True)], 1)


def _points(who, corners, V, n):
    """element numbers, barycentrics (m, q, D + 1) and physical weights (m, q) of the pieces"""
    B, W = _simplex_rule(corners.shape[1] - 1, n)
    lam = torch.einsum("qk,mkd->mqd", B, corners)
    return lam, _measure(corners @ V[who])[:, None] * W


def _add_forms(out, vec, who, lam, w, V, p, mask, c=None):
    """adds the mass / stiffness matrices (and vectors) of weighted points to out (n, nd, nd)"""
    phi, dphi = _shapes(lam, p)
    if c is not None:
        w = w * c
    rows = []
    if mask & 1:
        rows.append(phi)
    if mask & 2:
        g = dphi @ _bary_grads(V)[who][:, None]
        rows += [g[..., d] for d in range(g.shape[-1])]
    A = torch.cat(rows, 1)  # (m, comps * q, nd)
    ww = w.repeat(1, len(rows))
    out.index_add_(0, who, (A * ww[..., None]).transpose(1, 2).contiguous() @ A)
    if vec is not None:
        vec.index_add_(0, who, (phi * w[..., None]).sum(1))


def _matrices(l, V, dts, p, mask, extra=0, coef=None, want_vec=False, step=4096):
    """matrices (n, len(dts), nd, nd) and vectors of the parts of the simplices"""
    n, D = l.shape[0], l.shape[1] - 1
    nd = _ndof(D, p)
    out = torch.zeros((n, len(dts), nd, nd), dtype=torch.float64, device="cuda")
    vec = torch.zeros((n, nd), dtype=torch.float64, device="cuda") if want_vec else None
    for a in range(0, n, step):
        ll, VV = l[a:a + step], V[a:a + step]
        for t, dt in enumerate(dts):
            who, corners = _pieces(ll, dt)
            if not who.numel():
                continue
            lam, w = _points(who, corners, VV, p + 2 + extra)
            o = torch.zeros((ll.shape[0], nd, nd), dtype=torch.float64, device="cuda")
            v = vec[a:a + step] if want_vec else None
            c = coef(slice(a, a + step), who, lam, lam @ VV[who]) if coef else None
            _add_forms(o, v, who, lam, w, VV, p, mask, c)
            out[a:a + step, t] = o
    return (out, vec) if want_vec else out


def _fractions(l):
    """share of the part phi < 0 of simplices with vertex values l"""
    D = l.shape[1] - 1
    f = torch.zeros(l.shape[0], dtype=torch.float64, device="cuda")
    for a in range(0, l.shape[0], 1 << 20):
        ll = l[a:a + (1 << 20)]
        who, corners = _pieces(ll, NEG)
        # corners hold D + 1 barycentrics: their determinant is the share
        f[a:a + (1 << 20)].index_add_(0, who, torch.linalg.det(corners).abs())
    return f


def _exact_integrate(s):
    D, dt = s["D"], DTS[s["dom"]][0]
    per = torch.zeros(s["el"].shape[0], dtype=torch.float64, device="cuda")
    for a in range(0, per.numel(), 1 << 15):
        e = s["el"][a:a + (1 << 15)].long()
        l, V = s["ls"][e], s["X"][e]
        who, corners = _pieces(l, dt)
        if who.numel():
            lam, w = _points(who, corners, V, 3)
            x = lam @ V[who]
            f = sum(c * torch.stack([x[..., d] ** ex[d] for d in range(D)]).prod(0) for c, ex in TERMS)
            per[a:a + (1 << 15)].index_add_(0, who, (w * f).sum(1))
    return None, per, per.sum().reshape(1)


#: children of a tetrahedron in the subdivision rule (cutint/xintegration.cpp:872-914): each corner is the midpoint of
#: two of the parent's vertices, or one of them twice
_CHILDREN = [[(0, 3), (0, 0), (0, 1), (0, 2)], [(1, 3), (0, 1), (1, 1), (1, 2)], [(2, 3), (0, 2), (1, 2), (2, 2)],
             [(1, 3), (0, 1), (1, 2), (2, 3)], [(1, 3), (0, 1), (0, 3), (2, 3)], [(3, 3), (0, 3), (1, 3), (2, 3)],
             [(1, 2), (2, 3), (0, 3), (0, 2)], [(1, 2), (0, 1), (0, 3), (0, 2)]]


def _exact(s):
    kind = s["kind"]
    if kind in ("mark", "step"):
        e = s["el"].long()
        l = s["ls"][e]
        dom = torch.where((l < 0).any(1), torch.where((l > 0).any(1), IF, NEG), POS).to(torch.uint8)
        cr = _fractions(l)
        if kind == "mark":
            return dom, cr, None, None, None
        c = s["cut"].long()
        m = _matrices(l[c], s["X"][e[c]], [NEG, IF], s["p"], 3)
        return dom, cr, None, None, _padded(m, _room(s))
    if kind == "integrate":
        return _exact_integrate(s)
    if kind == "form":
        e = s["el"][s["cut"].long()].long()
        m = _matrices(s["ls"][e], s["X"][e], DTS[s["dom"]], s["p"], s["mask"])
        return _padded(m, _room(s))
    if kind == "cf":
        e = s["el"][s["elems"].long()].long()
        g = s["gf"][e]

        def coef(part, who, lam, x):
            return 1 + 0.5 * x[..., 0] * x[..., 1] + (lam * g[part][who][:, None]).sum(-1)
        m, v = _matrices(s["ls"][e], s["X"][e], DTS[s["dom"]], s["p"], 3, 1, coef, True)
        return None, _padded(m, _room(s)), _padded(v, _room(s))
    if kind == "assemble":
        e = s["el"][s["elems"].long()].long()
        m = _matrices(s["ls"][e], s["X"][e], DTS[s["dom"]], s["p"], 3)[:, 0]
        d, n, nd = s["dofs"].long(), s["n"], s["dofs"].shape[1]
        key = torch.unique((d[:, :, None] * n + d[:, None, :]).reshape(-1))
        d = d[s["elems"].long()]
        at = torch.searchsorted(key, (d[:, :, None] * n + d[:, None, :]).reshape(-1))
        return None, None, torch.zeros(key.numel(), dtype=torch.float64, device="cuda").index_add_(0, at, m.reshape(-1))
    if kind == "batch":
        out = []
        for m, p in enumerate(s["ps"]):
            e = s["el"][s["off"][m]:s["off"][m + 1]].long()
            e = e[_is_cut(s["ls"], e)]
            out.append(_matrices(s["ls"][e], s["X"][e], DTS[s["dom"]], p, s["mask"]).reshape(-1))
        return _padded(torch.cat(out), _batch_room(s))
    return None


def exact(case, seed):
    # the hexahedral rule is a construction of its own (slices of a trilinear level set), with no value beside it, and
    # the subdivision rule of a large mesh takes minutes this way
    if case["kind"] == "hex" or (case["kind"] == "subdiv" and not _small_subdiv(case)):
        return None
    with torch.no_grad():
        if case["kind"] == "subdiv":
            return _exact_subdiv(case, seed)
        return _exact(_inputs(case, seed))


def _small_subdiv(case):
    return 24.7 * case["nx"] ** 2 * 8 ** case["L"] < 1.5e7 * 16


def _leaves(L):
    """corners (8^L, 4, 4) in barycentric coordinates of the leaves of the level-L refinement"""
    t = torch.eye(4, dtype=torch.float64, device="cuda")[None]
    for _ in range(L):
        kids = [torch.stack([0.5 * (t[:, i] + t[:, j]) for i, j in c], 1) for c in _CHILDREN]
        t = torch.stack(kids, 1).reshape(-1, 4, 4)
    return t


def _exact_subdiv(case, seed):
    """the matrices of the level-L rule: the level set interpolated linearly on every leaf of the refinement"""
    p, dts = case["p"], DTS[case["dom"]]
    s = prepare(case, seed)  # the cut list is an input of the call
    e = s["el"][s["cut"].long()].long()
    V, nod = s["X"][e], s["nod"][s["cut"].long()]
    leaf = _leaves(case["L"])
    phi, _ = _shapes(leaf, 2)
    nd = _ndof(3, p)
    out = torch.zeros((e.shape[0], len(dts), nd, nd), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 16) // leaf.shape[0])
    for a in range(0, e.shape[0], step):
        VV = V[a:a + step]
        l = torch.einsum("lkn,en->elk", phi, nod[a:a + step]).reshape(-1, 4)
        for t, dt in enumerate(dts):
            who, corners = _pieces(l, dt)
            if not who.numel():
                continue
            corners = corners @ leaf[who % leaf.shape[0]]
            who = who // leaf.shape[0]
            o = torch.zeros((VV.shape[0], nd, nd), dtype=torch.float64, device="cuda")
            for b in range(0, who.numel(), 1 << 16):
                lam, w = _points(who[b:b + (1 << 16)], corners[b:b + (1 << 16)], VV, p + 2)
                _add_forms(o, None, who[b:b + (1 << 16)], lam, w, VV, p, case["mask"])
            out[a:a + step, t] = o
    return _padded(out, _room(case))
