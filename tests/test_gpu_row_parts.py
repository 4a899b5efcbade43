"""P1 tile sweeps of small grids, whose row tiles are shared by several
workgroups: a lone wavenumber (up to 16 parts per row tile) against the same
wavenumber inside a batch that fills the chip (whole row tiles), for each operator
and rule.  Only the order of the FP32 sums over row triangles differs: at most 48
terms per entry, 48 * 2^-24 < 3e-6."""
import numpy as np
import pytest
import torch

from neuralat_amd import mesh

pytestmark = pytest.mark.gpu
TOL = 3e-6
KS = [3.0 + 0.25 * z for z in range(32)]


def _solver(level, drop=0):
    from neuralat_amd.bem import BEM_Solver

    v, t = mesh.icosphere(level, 0.2)
    v = mesh.sh_perturb(v, 4, 0.05, seed=3).astype(np.float32)
    t = t[: len(t) - drop]
    used = np.unique(t)
    ids = np.zeros(len(v), dtype=t.dtype)
    ids[used] = np.arange(len(used), dtype=t.dtype)
    d = torch.device("cuda:0")
    return BEM_Solver(torch.tensor(v[used], device=d), torch.tensor(ids[t], device=d)), len(used)


@pytest.mark.parametrize("level,drop", [(0, 0), (1, 3), (2, 0), (2, 37), (3, 0)])
@pytest.mark.parametrize("quad", [False, True, "approx_1"])
def test_operators(level, drop, quad):
    s, n = _solver(level, drop)
    for op in ("single", "double", "adjointdouble", "hypersingular", "bm_lhs", "bm_rhs"):
        print("row parts", level, drop, quad, op, flush=True)
        many = s.assemble_boundary_matrix_batch(KS, op, approx=quad)
        one = s.assemble_boundary_matrix(KS[5], op, approx=quad)
        assert float((one - many[5]).norm() / many[5].norm()) < TOL, op


@pytest.mark.parametrize("level,drop", [(0, 0), (1, 3), (2, 37), (3, 0)])
def test_burton_miller(level, drop):
    s, n = _solver(level, drop)
    g = torch.randn(len(KS), n, dtype=torch.complex64, device="cuda:0", generator=torch.Generator("cuda:0").manual_seed(2))
    print("row parts system", level, drop, flush=True)
    L, R = s.burton_miller_systems(KS, g)
    l1, r1 = s.burton_miller_system(KS[5], g[5], approx=True)
    assert float((l1 - L[5]).norm() / L[5].norm()) < TOL
    assert float((r1 - R[5]).norm() / R[5].norm()) < TOL
