"""The straight cut rule and its integral over lists of every length that changes how a wave shares them out: one
element per wave up to 16,384 elements, then 2, 4, .. 64, with remainders, against the oracle and against the same
call on short pieces of the list (bit for bit: the same arithmetic per point)."""
import numpy as np
import pytest

from ngsxfem_amd import _abi
from ngsxfem_amd import workloads as W
from ngsxfem_amd.meshes import MakeStructured2DMesh, MakeStructured3DMesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _rule(ctx, D, el, X, ls, dt, order, elems, torch):
    n = elems.numel()
    off = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    ctx.cut_rule_count(D, el, ls, dt, order, off, elems=elems)
    pts = torch.zeros((max(int(off[-1].item()), 1), 4), dtype=torch.float64, device="cuda")
    ctx.cut_rule_fill(D, el, X, ls, dt, order, off, pts, elems=elems)
    return off, pts


@pytest.mark.parametrize("D,n,order", [(2, 1, 4), (2, 16384, 3), (2, 16385, 4), (3, 7, 6), (3, 32769, 2),
                                       (3, 131073, 5), (3, 1048577, 2)])
@pytest.mark.parametrize("dt", [0, 1, 2])
def test_lists_of_every_length(D, n, order, dt):
    import torch
    mesh = MakeStructured2DMesh(nx=61, ny=47) if D == 2 else MakeStructured3DMesh(nx=11, ny=13, nz=10)
    X = mesh.coords
    r = np.sqrt(((X - 0.5) ** 2).sum(axis=1))
    lset = W.p1_perturb(r - 0.31)
    rng = np.random.default_rng(n + dt)
    pick = rng.integers(0, mesh.ne, n).astype(np.int32)  # repeats and any order
    ctx = _abi.Context(0)
    d = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (mesh.el2v, X, lset, pick)]
    off, pts = _rule(ctx, D, d[0], d[1], d[2], dt, order, d[3], torch)
    tot = torch.full((1,), 7.0, dtype=torch.float64, device="cuda")
    per = torch.zeros(n, dtype=torch.float64, device="cuda")
    terms = [(1.0, (0, 0, 0)), (0.5, (1, 1, 0))]
    ctx.integrate(D, d[0], d[1], off, pts, terms, tot, per, elems=d[3])
    ctx.sync()
    o, p = off.cpu().numpy(), pts.cpu().numpy()
    # one call per distinct element: a list so short that every element has a wave
    ids = np.arange(mesh.ne, dtype=np.int32)
    o1, p1 = [a.cpu().numpy() for a in _rule(ctx, D, d[0], d[1], d[2], dt, order, torch.from_numpy(ids).cuda(), torch)]
    cnt = np.diff(o1)[pick]
    assert np.array_equal(np.diff(o), cnt)
    src = np.repeat(o1[pick], cnt) + np.arange(int(cnt.sum())) - np.repeat(np.cumsum(cnt) - cnt, cnt)
    assert np.array_equal(p[:len(src)], p1[src])
    # the oracle on every element
    ref = O.integrate_mesh(mesh, lset, dt, order, terms, element_wise=True)
    scale = np.abs(ref).max()
    g = per.cpu().numpy()
    assert np.abs(g - ref[pick]).max() <= 2e-14 * scale  # up to a hundred terms, each rounded a few times
    # n sums of one rounding each, in some order
    assert abs(tot.item() - ref[pick].sum()) <= 1e-15 * n * scale + 1e-300
    ctx.close()
