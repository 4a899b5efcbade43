"""The fused CBIE system's neighbour pairs and row reduction (both operators of
a pair from one evaluation) against the FP64 oracle, for every rule and for
triangle counts around the 64-row blocks, alone and in a batch.  Bar: the
operators' 1e-5."""
import numpy as np
import pytest
import torch

import oracle
from neuralat_amd import mesh

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _dev():
    return torch.device("cuda:0")


def _surface(nu, nv, seed):
    """A closed latitude-longitude sphere of 2 nu (nv - 1) triangles."""
    rng = np.random.default_rng(seed)
    th = np.pi * np.arange(1, nv) / nv
    ph = 2 * np.pi * np.arange(nu) / nu
    ring = np.stack([np.outer(np.sin(th), np.cos(ph)), np.outer(np.sin(th), np.sin(ph)),
                     np.outer(np.cos(th), np.ones(nu))], -1).reshape(-1, 3)
    v = np.concatenate([ring, [[0, 0, 1], [0, 0, -1]]]) * (0.2 + 0.01 * rng.random(3))
    n, top, bot = nu * (nv - 1), nu * (nv - 1), nu * (nv - 1) + 1
    t = []
    for a in range(nu):
        b = (a + 1) % nu
        t.append((top, a, b))
        t.append((bot, n - nu + b, n - nu + a))
        for r in range(nv - 2):
            t += [(r * nu + a, (r + 1) * nu + a, (r + 1) * nu + b), (r * nu + a, (r + 1) * nu + b, r * nu + b)]
    return v.astype(np.float32), np.array(t, np.int32)


def _psi(n, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)


def _check(v, t, k, clamp, psi, lhs, rhs, quad):
    K = oracle.assemble(v, t, k, "double", "DP0", quad=quad, clamp=clamp)
    V = oracle.assemble(v, t, k, "single", "DP0", quad=quad, clamp=clamp)
    e = v[t].astype(np.float64)
    area = 0.5 * np.linalg.norm(np.cross(e[:, 1] - e[:, 0], e[:, 2] - e[:, 0]), axis=1)
    L, r = 0.5 * np.diag(area) - K, -(V @ psi.astype(np.complex128))
    assert np.linalg.norm(lhs - L) < TOL * np.linalg.norm(L)
    assert np.linalg.norm(rhs - r) < TOL * np.linalg.norm(r)


@pytest.mark.parametrize("quad", ["full", "approx", "approx1"])
@pytest.mark.parametrize("nu,nv", [(3, 2), (9, 4), (8, 5), (5, 8), (16, 5)])  # 6, 54, 64, 70, 128 triangles
def test_cbie_system_rules(quad, nu, nv):
    from neuralat_amd.bem import BEM_Solver

    v, t = _surface(nu, nv, nu)
    approx = {"full": False, "approx": True, "approx1": "approx_1"}[quad]
    psi = _psi(len(t), nv)
    for clamp in (True, False):
        print("cbie pairs", quad, len(t), clamp, flush=True)
        s = BEM_Solver(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()), basis="DP0", clamp=clamp)
        lhs, rhs = s.cbie_system(9.0, torch.tensor(psi, device=_dev()), approx=approx)
        _check(v, t, 9.0, clamp, psi, lhs.cpu().numpy(), rhs.cpu().numpy(), quad)


@pytest.mark.parametrize("row_tile", [16, 32, 64])
def test_batch_of_uneven_items(row_tile):
    from neuralat_amd.bem.batch import Mesh, batch_cbie

    shapes = [(5, 8), (3, 2), (16, 5), (9, 4), (8, 5)]
    meshes = [_surface(a, b, a + b) for a, b in shapes]
    ks = [3.0, 7.5, 11.0, 2.0, 9.0]
    psis = [_psi(len(t), q) for q, (v, t) in enumerate(meshes)]
    print("cbie batch", row_tile, flush=True)
    handles = [Mesh(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev())) for v, t in meshes]
    outs = batch_cbie(handles, ks, [torch.tensor(p, device=_dev()) for p in psis], row_tile=row_tile)
    for (v, t), k, p, (lhs, rhs) in zip(meshes, ks, psis, outs):
        _check(v, t, k, True, p, lhs.cpu().numpy(), rhs.cpu().numpy(), "full")


def test_batch_past_the_grid_limit():
    """A batch of more neighbour pairs than one launch can take at a wavefront
    each (2^26 pairs are 2^32 work-items): 65 items of a 1024-triangle fan, whose
    triangles are all neighbours.  Items at both ends of the split equal the
    same item alone, bit for bit."""
    from neuralat_amd.bem.batch import Mesh, allocate_systems, batch_cbie

    d, items = 1024, 65
    a = 2 * np.pi * np.arange(d) / d
    v = np.concatenate([[[0, 0, 0.05]], np.stack([0.1 * np.cos(a), 0.1 * np.sin(a), 0 * a], 1)]).astype(np.float32)
    t = np.stack([0 * np.arange(d), 1 + np.arange(d), 1 + (np.arange(d) + 1) % d], 1).astype(np.int32)
    m = Mesh(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()))
    assert m.n_neighbor_pairs * items > 2 ** 26
    ks = [2.0 + 0.25 * q for q in range(items)]
    psis = [torch.tensor(_psi(d, q), device=_dev()) for q in range(items)]
    outs = [(lhs.fill_(float("nan")), rhs.fill_(float("nan"))) for lhs, rhs in allocate_systems([m] * items, _dev())]
    print("cbie batch past the grid limit", m.n_neighbor_pairs * items, flush=True)
    batch_cbie([m] * items, ks, psis, outs=outs, row_tile=64)
    for q in (0, 31, 32, 63, 64):
        (lhs, rhs), = batch_cbie([m], [ks[q]], [psis[q]], row_tile=64)
        assert torch.equal(lhs, outs[q][0]) and torch.equal(rhs, outs[q][1]), q
