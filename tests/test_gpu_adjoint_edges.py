"""The DP0 adjoint kernels where their row tiles (32 triangles) and pair groups
(16 pairs a workgroup) are only partly filled: vertex gradients of 20, 77 and 80
triangles along random directions against central differences of the FP64 oracle
pipeline, at the bound of the same comparison on larger meshes (2e-3); the same
for the P1 Burton-Miller gradient (row tiles of 32 triangles)."""
import numpy as np
import pytest
import torch

import fp64_grad
import oracle
from neuralat_amd import mesh
from test_gpu_grad import _dev, _loss_gpu, _setup
from test_gpu_grad_bm import _fp64_ops, _gpu_geometry, _loss64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,drop", [(0, 0), (1, 0), (1, 3)])
def test_vertex_gradient(level, drop):
    v, t, pts, src = _setup(level, seed=5)
    t = t[: len(t) - drop]  # an open surface: the discrete problem stays well posed
    assert len(np.unique(t)) == len(v)
    k0 = 2.5
    vt = torch.tensor(v, device=_dev(), requires_grad=True)
    print("adjoint edges", len(t), flush=True)
    L = _loss_gpu(vt, torch.tensor(t, device=_dev()), torch.tensor(k0, device=_dev()), src, torch.tensor(pts, device=_dev()))
    L.backward()
    gv = vt.grad.detach().cpu().numpy().astype(np.float64)
    v64, h = v.astype(np.float64), 1e-6
    rng = np.random.default_rng(3)
    ad, fd = [], []
    for _ in range(6):
        d = rng.standard_normal(v.shape)
        d /= np.linalg.norm(d)
        fd.append((fp64_grad.loss(v64 + h * d, t, k0, src, pts) - fp64_grad.loss(v64 - h * d, t, k0, src, pts)) / (2 * h))
        ad.append(np.sum(gv * d))
    assert np.linalg.norm(np.array(ad) - fd) < 2e-3 * np.linalg.norm(fd)


@pytest.mark.parametrize("level,drop", [(0, 0), (1, 3)])
def test_gradient_without_clamp(level, drop):
    """The exact kernel (clamp=False), where a triangle's own points are at
    distance zero in the regular kernel's excluded pairs: vertex and wavenumber
    gradients against the FP64 pipeline without the clamp, same bound."""
    from neuralat_amd.bem.grad import exterior_pressure, monopole_neumann_dp0

    v, t, pts, src = _setup(level, seed=5)
    t = t[: len(t) - drop]
    k0 = 2.5
    vt = torch.tensor(v, device=_dev(), requires_grad=True)
    kt = torch.tensor(k0, device=_dev(), requires_grad=True)
    tt = torch.tensor(t, device=_dev())
    print("adjoint without clamp", len(t), flush=True)
    p = exterior_pressure(vt, tt, kt, monopole_neumann_dp0(vt, tt, src, kt), torch.tensor(pts, device=_dev()),
                          clamp=False, tol=1e-7, adjoint_tol=1e-6)
    (p.real ** 2 + p.imag ** 2).sum().backward()
    gv = vt.grad.detach().cpu().numpy().astype(np.float64)

    def loss64(x, k):
        val, dn = mesh.sources_field([src], None, k)
        psi = mesh.project_dp0(x, t, lambda y, n: dn(y, n))
        S, D = (oracle.assemble(x, t, k, op, "DP0", clamp=False) for op in ("single", "double"))
        phi = np.linalg.solve(0.5 * oracle.identity(x, t, "DP0") - D, -S @ psi)
        Sp, Dp = (oracle.potential(x, t, pts, k, op, "DP0", clamp=False) for op in ("single", "double"))
        return float(np.sum(np.abs(Dp @ phi - Sp @ psi) ** 2))

    v64, h = v.astype(np.float64), 1e-6
    rng = np.random.default_rng(3)
    ad, fd = [float(kt.grad)], [(loss64(v64, k0 + h) - loss64(v64, k0 - h)) / (2 * h)]
    for _ in range(6):
        d = rng.standard_normal(v.shape)
        d /= np.linalg.norm(d)
        fd.append((loss64(v64 + h * d, k0) - loss64(v64 - h * d, k0)) / (2 * h))
        ad.append(np.sum(gv * d))
    assert abs(ad[0] - fd[0]) < 2e-3 * abs(fd[0])
    assert np.linalg.norm(np.array(ad) - fd) < 2e-3 * np.linalg.norm(fd)


@pytest.mark.parametrize("level", [0, 1])
def test_p1_vertex_gradient(level):
    k = 7.0
    v, t = mesh.icosphere(level, 0.1)
    v = mesh.sh_perturb(v, 4, 0.05, seed=6).astype(np.float32)
    _, dn = mesh.sources_field(np.array([[0.01, -0.005, 0.002]]), None, k)
    psi = mesh.project_p1(v, t, lambda x, n: dn(x, n))
    pts = mesh.random_exterior_points(24, 0.2, 0.5, seed=2)
    print("P1 adjoint edges", len(t), flush=True)
    gv, _ = _gpu_geometry(v, t, k, psi, pts)
    v64, h = v.astype(np.float64), 1e-6
    rng = np.random.default_rng(11)
    ad, fd = [], []
    for _ in range(6):
        d = rng.standard_normal(v.shape)
        lp, lm = (_loss64(_fp64_ops(v64 + s * h * d, t, k, pts), psi) for s in (1, -1))
        fd.append((lp - lm) / (2 * h))
        ad.append(float(np.sum(gv * d)))
    assert np.linalg.norm(np.array(ad) - fd) < 2e-3 * np.linalg.norm(fd)


def test_tall_row_tiles():
    """From 16384 triangles on a row tile holds 64 triangles: the scratch is an
    eighth of a byte per pair, V^H lambda equals the product with the assembled
    operator (1e-5, the operators' bar), and the vertex gradients add up to zero
    (every pair term depends on differences of positions only: what a pair gives
    its row triangle it takes from its column triangle; FP32 per triangle, 1e-3
    allowed)."""
    import ctypes

    from neuralat_amd import _lib
    from neuralat_amd.bem import BEM_Solver
    from neuralat_amd.bem.solver import matvec

    v, t = mesh.icosphere(5, 0.1)
    v = mesh.sh_perturb(v, 4, 0.05, seed=6).astype(np.float32)
    n = len(t)
    s = BEM_Solver(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()), basis="DP0")
    lib = _lib.load()
    size = lib.bem_adjoint_work_size(s.mesh.handle)
    assert size <= n * n // 8
    g = torch.Generator(_dev()).manual_seed(4)
    lam, psi, phi = (torch.randn(n, dtype=torch.complex64, device=_dev(), generator=g) for _ in range(3))
    gvert = torch.zeros((len(v), 3), dtype=torch.float64, device=_dev())
    gk = torch.zeros(1, dtype=torch.float64, device=_dev())
    vhl = torch.zeros((n, 2), dtype=torch.float64, device=_dev())
    work = torch.empty(size, dtype=torch.uint8, device=_dev())
    print("adjoint tall tiles", n, flush=True)
    ptr = lambda x: ctypes.c_void_p(x.data_ptr())  # noqa: E731
    _lib.check(lib.bem_adjoint_cbie_dp0(s.mesh.handle, 9.0, 1, ptr(lam), ptr(psi), ptr(phi), ptr(gvert), ptr(gk),
                                        ptr(vhl), ptr(work), ctypes.c_void_p(0)))
    torch.cuda.synchronize()
    want = matvec(s.assemble_boundary_matrix(9.0, "single"), lam, trans=2)
    got = torch.complex(vhl[:, 0], vhl[:, 1])
    assert float((got - want).norm() / want.norm()) < 1e-5
    assert float(gvert.sum(0).norm()) < 1e-3 * float(gvert.norm(dim=1).sum())
