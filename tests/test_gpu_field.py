"""The fused exterior pressure (bem_field*: D phi - S psi contracted inside the
evaluation) against the FP64 oracle's potential operators, at the edges of its
point tiles, triangle splits and batches.  Bar: the operators' own 1e-5."""
import numpy as np
import pytest
import torch

import oracle
from neuralat_amd import mesh

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _dev():
    return torch.device("cuda:0")


def _case(level, basis, seed, rows=1):
    v, t = mesh.icosphere(level, 0.1)
    v = mesh.sh_perturb(v, 4, 0.05, seed=seed).astype(np.float32)
    n = len(t) if basis == "DP0" else len(v)
    rng = np.random.default_rng(seed)
    data = (rng.standard_normal((2, rows, n)) + 1j * rng.standard_normal((2, rows, n))).astype(np.complex64)
    return v, t, data[0], data[1]


def _exact(v, t, pts, k, basis, clamp, psi, phi):
    return (oracle.potential(v, t, pts, k, "double", basis, clamp=clamp) @ phi.astype(np.complex128)
            - oracle.potential(v, t, pts, k, "single", basis, clamp=clamp) @ psi.astype(np.complex128))


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("basis", ["P1", "DP0"])
@pytest.mark.parametrize("level,npts", [(0, 1), (0, 65), (1, 64), (2, 1), (2, 63), (3, 200)])
def test_field_against_oracle(basis, level, npts):
    from neuralat_amd.bem import BEM_Solver

    v, t, psi, phi = _case(level, basis, 3 + level)
    pts = mesh.random_exterior_points(npts, 0.13, 0.5, seed=npts).astype(np.float32)
    for clamp in (True, False):
        print("field", basis, level, npts, clamp, flush=True)
        s = BEM_Solver(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()), basis=basis, clamp=clamp)
        p = s.boundary2potential(18.3, torch.tensor(psi[0], device=_dev()), torch.tensor(phi[0], device=_dev()),
                                 torch.tensor(pts, device=_dev()))
        assert p.shape == (npts,)
        assert _rel(p.cpu().numpy(), _exact(v, t, pts, 18.3, basis, clamp, psi[0], phi[0])) < TOL
        none = s.boundary2potential(18.3, torch.tensor(psi[0], device=_dev()), torch.tensor(phi[0], device=_dev()),
                                    torch.zeros((0, 3), device=_dev()))
        assert none.shape == (0,)


def test_field_batches_and_samples():
    """More systems than one launch takes (64), rows wider than the basis, and
    the samples of a geometry set, each equal to the single call."""
    from neuralat_amd.bem import BEM_Solver, GeometrySet, boundary2potential_samples

    nk = 66
    v, t, psi, phi = _case(1, "P1", 5, nk)
    pts = mesh.random_exterior_points(33, 0.2, 0.5, seed=2).astype(np.float32)
    ks = np.linspace(-40.0, 60.0, nk).astype(np.float32)
    s = BEM_Solver(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()))
    dpts = torch.tensor(pts, device=_dev())
    wide = [torch.nn.functional.pad(torch.tensor(a, device=_dev()), (0, 3), value=float("nan")) for a in (psi, phi)]
    print("field batch", nk, flush=True)
    p = s.boundary2potential_batch(ks, wide[0], wide[1], dpts)
    for z in (0, 1, 63, 64, 65):
        assert _rel(p[z].cpu().numpy(), _exact(v, t, pts, float(ks[z]), "P1", True, psi[z], phi[z])) < TOL, z
    vs = np.stack([v, v * np.float32(1.3), v + np.float32(0.02)])
    own = np.stack([pts, pts * np.float32(1.5), pts + np.float32(0.05)])
    print("field samples", flush=True)
    gs = GeometrySet(s.mesh, vs)
    q = boundary2potential_samples(gs, ks[:3], torch.tensor(psi[:3], device=_dev()),
                                   torch.tensor(phi[:3], device=_dev()), own)
    for z in range(3):
        assert _rel(q[z].cpu().numpy(), _exact(vs[z], t, own[z], float(ks[z]), "P1", True, psi[z], phi[z])) < TOL, z
