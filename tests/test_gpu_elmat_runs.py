"""Element matrices of rules of any length and of lists of any length: the contraction takes 64 points at a time
and 4 per matrix instruction, and a wave takes 1, 2, 4 or 8 elements in a run (more as the list grows)."""
import numpy as np
import pytest

from ngsxfem_amd import _abi
from ngsxfem_amd import workloads as W
from ngsxfem_amd.meshes import Make1DMesh, MakeStructured2DMesh, MakeStructured3DMesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu
COUNTS = [0, 0, 1, 3, 4, 5, 63, 64, 65, 0, 127, 128, 129, 200]


def _mesh(D):
    return Make1DMesh(5) if D == 1 else (MakeStructured2DMesh(nx=3, ny=4) if D == 2 else MakeStructured3DMesh(nx=2))


@pytest.mark.parametrize("D", [1, 2, 3])
@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("mask", [1, 2, 3])
def test_rules_of_every_length(D, p, mask):
    import torch
    mesh = _mesh(D)
    rng = np.random.default_rng(100 * D + 10 * p + mask)
    elems = rng.integers(0, mesh.ne, len(COUNTS)).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(COUNTS)]).astype(np.int32)
    pts = np.zeros((off[-1], 4))
    pts[:, :D] = rng.dirichlet(np.ones(D + 1), off[-1])[:, :D]
    pts[:, 3] = rng.uniform(-0.3, 1.0, off[-1])  # rules with negative weights too
    ctx = _abi.Context(0)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    nd = O.h1_ndof(D, p)
    for prec, dtype, bar in ((_abi.XG_PREC_FP64, torch.float64, 1e-13), (_abi.XG_PREC_FP32, torch.float32, 1e-6)):
        out = torch.full((len(COUNTS), nd, nd), float("nan"), dtype=dtype, device="cuda")
        ctx.elmat(D, p, up(mesh.el2v), up(mesh.coords), up(off), up(pts), mask, prec, out, elems=up(elems))
        ctx.sync()
        g = out.cpu().numpy().astype(np.float64)
        for i, e in enumerate(elems):
            a, b = off[i], off[i + 1]
            V = mesh.coords[mesh.el2v[e]]
            ref = O.elmat(D, p, V, pts[a:b, :3], pts[a:b, 3], mask) if b > a else np.zeros((nd, nd))
            # scale: the matrix of the absolute weights (the sums may cancel)
            sc = np.abs(O.elmat(D, p, V, pts[a:b, :3], np.abs(pts[a:b, 3]), mask)).max() if b > a else 0.0
            assert np.abs(g[i] - ref).max() <= bar * sc, (i, COUNTS[i])
    ctx.close()


@pytest.mark.parametrize("n", [1, 2, 32767, 32768, 65537, 131073])
@pytest.mark.parametrize("p", [1, 2])
def test_lists_of_every_length(n, p):
    """a long list gives the matrices of a short one, bit for bit (the same operations per element)"""
    import torch
    mesh, lset = W.config2(6)
    rng = np.random.default_rng(n)
    pick = rng.integers(0, mesh.ne, n).astype(np.int32)
    ctx = _abi.Context(0)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    el, X, ls = up(mesh.el2v), up(mesh.coords), up(lset)
    nd = O.h1_ndof(3, p)

    def both(ids):
        m = ids.numel()
        out = torch.zeros((m, 2, nd, nd), dtype=torch.float32, device="cuda")
        ctx.cut_pipeline(3, p, 2 * p, el, X, ls, [0, 2], 3, _abi.XG_PREC_FP32, out, elems=ids)
        off = torch.zeros(m + 1, dtype=torch.int32, device="cuda")
        ctx.cut_rule_count(3, el, ls, 0, 2 * p, off, elems=ids)
        pts = torch.zeros((max(int(off[-1].item()), 1), 4), dtype=torch.float64, device="cuda")
        ctx.cut_rule_fill(3, el, X, ls, 0, 2 * p, off, pts, elems=ids)
        csr = torch.zeros((m, nd, nd), dtype=torch.float64, device="cuda")
        vec = torch.zeros((m, nd), dtype=torch.float64, device="cuda")
        ctx.elmat(3, p, el, X, off, pts, 3, _abi.XG_PREC_FP64, csr, elems=ids)
        ctx.elvec(3, p, el, X, off, pts, vec, elems=ids)
        ctx.sync()
        return out, csr, vec

    long = both(up(pick))
    short = both(up(np.arange(mesh.ne, dtype=np.int32)))
    at = up(pick).long()
    for a, b in zip(long, short):
        assert torch.equal(a, b[at])
    # the short list against the oracle
    ref = O.cut_pipeline(3, p, 2 * p, np.arange(mesh.ne, dtype=np.int32), mesh.el2v, mesh.coords, lset, [0, 2], 3)
    g = short[0].cpu().numpy().astype(np.float64).reshape(ref.shape)
    sc = np.abs(ref).max(axis=(-2, -1), keepdims=True)
    assert np.all(np.abs(g - ref) <= 2e-7 * sc)
    ctx.close()


VEC_COUNTS = [0, 1, 4, 15, 16, 17, 31, 32, 33, 64, 95, 96, 97, 129, 200, 513]


def _long_rules(D, seed, reps):
    """(elements, offsets, points) of a list with rules of VEC_COUNTS points, `reps` times over"""
    mesh = _mesh(D)
    rng = np.random.default_rng(seed)
    n = np.tile(VEC_COUNTS, reps)
    elems = rng.integers(0, mesh.ne, len(n)).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    pts = np.zeros((off[-1], 4))
    pts[:, :D] = rng.dirichlet(np.ones(D + 1), off[-1])[:, :D]
    pts[:, 3] = rng.uniform(-0.3, 1.0, off[-1])
    return mesh, elems, off, pts


@pytest.mark.parametrize("D", [1, 2, 3])
@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("reps", [1, 257])
def test_vectors_of_rules_of_every_length(D, p, reps):
    """an element has 16 lanes of a wave, or all of them for a long rule in a list of up to 4096 elements (16 and
    4112 here), against the oracle's shape functions.  Bar: a rounding per point
    of the sum and 30 of a shape function and the Jacobian"""
    import torch
    mesh, elems, off, pts = _long_rules(D, 10 * D + p, reps)
    ctx = _abi.Context(0)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    nd = O.h1_ndof(D, p)
    out = torch.full((len(elems), nd), float("nan"), dtype=torch.float64, device="cuda")
    ctx.elvec(D, p, up(mesh.el2v), up(mesh.coords), up(off), up(pts), out, elems=up(elems))
    ctx.sync()
    g = out.cpu().numpy()
    assert len(elems) == 16 if reps == 1 else len(elems) > 4096
    first = len(elems) - len(VEC_COUNTS)  # the last of the repetitions, and the first
    for i in list(range(len(VEC_COUNTS))) + list(range(first, len(elems))):
        x, w = pts[off[i]:off[i + 1], :D], pts[off[i]:off[i + 1], 3]
        V = mesh.coords[mesh.el2v[elems[i]]]
        det = abs(np.linalg.det((V[:D] - V[D]).T.reshape(D, D)))
        phi = np.array([O.h1_shape(D, p, q)[0] for q in x]).reshape(-1, nd)
        bar = 1.2e-16 * (len(w) + 30) * det * np.abs(w).sum() * max(1.0, np.abs(phi).max(initial=0.0))
        assert np.abs(g[i] - det * (phi * w[:, None]).sum(0)).max() <= bar, (i, len(w))
    ctx.close()


@pytest.mark.parametrize("D", [1, 2, 3])
@pytest.mark.parametrize("reps", [1, 257])
def test_integrals_of_rules_of_every_length(D, reps):
    """an element has 2, 4 or 8 lanes, or a wave in a list of up to 4096 elements, and a lane takes 4 points at once
    while one of the wave has more, against the oracle.  Bar: a rounding per point and 30 of a term"""
    import torch
    mesh, elems, off, pts = _long_rules(D, 100 + D, reps)
    ctx = _abi.Context(0)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    terms = [(1.0 / (k + 1), (k % 4, k % 3 if D > 1 else 0, k % 2 if D > 2 else 0)) for k in range(11)]
    per = torch.full((len(elems),), float("nan"), dtype=torch.float64, device="cuda")
    tot = torch.full((1,), 7.0, dtype=torch.float64, device="cuda")
    ctx.integrate(D, up(mesh.el2v), up(mesh.coords), up(off), up(pts), terms, tot, per, elems=up(elems))
    ctx.sync()
    g = per.cpu().numpy()
    first = len(elems) - len(VEC_COUNTS)
    cmax = sum(c for c, _ in terms) * max(1.0, np.abs(mesh.coords).max()) ** 6
    for i in list(range(len(VEC_COUNTS))) + list(range(first, len(elems))):
        x, w = pts[off[i]:off[i + 1], :3], pts[off[i]:off[i + 1], 3]
        V = mesh.coords[mesh.el2v[elems[i]]]
        ref = O.integrate_poly(D, V, x, w, terms) if len(w) else 0.0
        det = abs(np.linalg.det((V[:D] - V[D]).T.reshape(D, D)))
        assert abs(g[i] - ref) <= 1.2e-16 * (len(w) + 30) * det * np.abs(w).sum() * cmax, (i, len(w))
    assert abs(tot.item() - g.sum()) <= 1.2e-16 * len(elems) * np.abs(g).sum()
    ctx.close()
