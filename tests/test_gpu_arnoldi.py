"""The fused Arnoldi step of the GMRES solvers (basis in LDS; chunked kernels;
separate kernels beyond both) at the edges of its forms: 64-lane, 512-element
chunk and LDS limits, step counts that cross from one form to the next, and
systems of unequal length in lockstep.  Solutions against FP64 residuals and
direct solves at the bars the solver tests use (1e-5)."""
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev():
    return torch.device("cuda:0")


def _system(n, radius, seed, nrhs=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.randn(n, n, 2, generator=g, device=_dev())
    A = torch.view_as_complex(A) * (radius / np.sqrt(2 * n))
    A.diagonal().add_(1.0)
    b = torch.view_as_complex(torch.randn(nrhs, n, 2, generator=g, device=_dev()))
    return A.contiguous(), b.contiguous()


def _err(A, x, b, adjoint=False):
    """Relative residual in FP64."""
    M = A.to(torch.complex128)
    M = M.conj().T if adjoint else M
    b = b.to(torch.complex128)
    return float(torch.linalg.vector_norm(b - M @ x.to(torch.complex128)) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("n,radius,restart", [(1, 0.0, 5), (2, 0.3, 5), (63, 0.5, 60), (512, 0.5, 60), (513, 0.7, 60),
                                              (1100, 0.7, 60), (4097, 0.6, 40)])
def test_single_system(n, radius, restart):
    from neuralat_amd.bem.grad import _adjoint_solve
    from neuralat_amd.bem.solver import gmres

    print("arnoldi single", n, restart, flush=True)
    A, b = _system(n, radius, n)
    x, info = gmres(A, b[0], tol=1e-6, restart=restart, maxiter=1000)
    assert info["converged"], info
    assert _err(A, x, b[0]) < 2e-6, info
    if n in (513, 4097):  # the adjoint product's scratch is shared with the step's
        y, info = _adjoint_solve(A, b[0], 1e-6, restart, 1000)
        assert info["converged"] and _err(A, y, b[0], adjoint=True) < 2e-6, info


def test_long_basis():
    """Steps past the chunked form's partial sums (18 chunks: 227 steps) take
    the separate kernels.  The target is 1e-5: such a slowly converging
    system's FP32 residual bottoms out near 1e-6."""
    from neuralat_amd.bem.solver import gmres

    print("arnoldi long basis", flush=True)
    A, b = _system(9000, 0.98, 9)
    x, info = gmres(A, b[0], tol=1e-5, restart=400, maxiter=1000)
    assert info["converged"] and 227 < info["iterations"] <= 400, info
    assert _err(A, x, b[0]) < 1.2e-5, info


def test_long_basis_in_lockstep():
    """The same hand-over to the separate kernels inside a cycle for several
    right-hand sides, for a batch (beside a short system) and for the one-pass
    steps of a batch's 16-bit inner solves.  Those get one outer step, so that
    one inner cycle takes over 227 steps; its solution is then off by the fp16
    rounding of A, 2^-11 |A| |x| / |b| < 1e-2."""
    from neuralat_amd.bem.batch import batch_gmres, batch_solve_mixed
    from neuralat_amd.bem.precision import gmres_multi

    A, B = _system(9000, 0.98, 9, 2)
    print("arnoldi long basis, right-hand sides", flush=True)
    X, infos = gmres_multi(A, B, tol=1e-5, restart=400, maxiter=1000)
    for q in range(2):
        assert infos[q]["converged"] and _err(A, X[q], B[q]) < 1.2e-5, infos[q]
    assert 227 < infos[0]["iterations"] <= 400, infos[0]
    C, c = _system(700, 0.6, 700)
    print("arnoldi long basis, batch", flush=True)
    xs, infos = batch_gmres([A, C], [B[0], c[0]], tol=1e-5, restart=400)
    assert 227 < infos[0]["iterations"], infos
    for M, b, x, i in zip((A, C), (B[0], c[0]), xs, infos):
        assert i["converged"] and _err(M, x, b) < 1.2e-5, i
    print("arnoldi long basis, inner solves", flush=True)
    xs, infos = batch_solve_mixed([A, C], [B[0], c[0]], dtype="fp16", tol=1e-6, inner_tol=1e-5, outer_restart=1,
                                  inner_restart=400, max_inner_cycles=1, max_outer_cycles=1)
    assert 227 < infos[0]["inner_iterations"] < 400, infos
    for M, b, x in zip((A, C), (B[0], c[0]), xs):
        assert _err(M, x, b) < 1e-2


@pytest.mark.parametrize("n,nrhs", [(65, 3), (700, 17), (5000, 2)])
def test_many_right_hand_sides(n, nrhs):
    from neuralat_amd.bem.precision import gmres_multi

    print("arnoldi multi", n, nrhs, flush=True)
    A, B = _system(n, 0.6, n, nrhs)
    X, infos = gmres_multi(A, B, tol=1e-6, restart=50)
    assert all(i["converged"] for i in infos)
    for q in range(nrhs):
        assert _err(A, X[q], B[q]) < 2e-6, q


@pytest.mark.parametrize("use_graph", [True, False])
def test_uneven_lockstep(use_graph):
    from neuralat_amd.bem.batch import batch_gmres, batch_solve_mixed

    sizes = (1, 40, 513, 700, 2100)
    print("arnoldi lockstep", use_graph, flush=True)
    systems = [_system(n, 0.6, n) for n in sizes]
    As, bs = [a for a, _ in systems], [b[0] for _, b in systems]
    xs, infos = batch_gmres(As, bs, tol=1e-6, restart=20, max_cycles=30, use_graph=use_graph)
    for n, A, b, x, i in zip(sizes, As, bs, xs, infos):
        assert i["converged"] and _err(A, x, b) < 2e-6, (n, i)
    xs, infos = batch_solve_mixed(As, bs, dtype="fp16", tol=1e-6, inner_tol=1e-3, inner_restart=30, max_inner_cycles=1,
                                  max_outer_cycles=6, use_graph=use_graph)
    for n, A, b, x, i in zip(sizes, As, bs, xs, infos):
        assert i["converged"] and _err(A, x, b) < 2e-6, (n, i)


def _best(f, n=9):
    f()
    torch.cuda.synchronize()
    out = []
    for _ in range(n):
        a = time.perf_counter()
        f()
        torch.cuda.synchronize()
        out.append(time.perf_counter() - a)
    return min(out)


@pytest.mark.parametrize("n", [6000, 12000, 13000])
def test_one_step_takes_one_product(n):
    """A solve that converges in its first step takes no products past it: as
    long as with maxiter=1, whose residual is read after that step whatever the
    read window (two more steps would make five products of three)."""
    from neuralat_amd.bem.precision import gmres_multi
    from neuralat_amd.bem.solver import gmres

    A, B = _system(n, 1e-8, n, 16)
    print("arnoldi one step", n, flush=True)
    for solve in (lambda **kw: gmres(A, B[0], tol=1e-5, restart=50, **kw)[1],
                  lambda **kw: gmres_multi(A, B, tol=1e-5, restart=50, **kw)[1][0]):
        info = solve()
        assert info["converged"] and info["iterations"] == 1, info
        free, held = _best(solve), _best(lambda: solve(maxiter=1))
        assert free < 1.25 * held, (n, free, held)


def test_fp16_scale_of_one_large_system():
    """The scale of one large system's 16-bit copy reads its matrix at the
    chip's rate: the fp16 solve takes one more read of 3.4 GB than the bf16 one
    (0.7 ms of 3.8 at 5 TB/s; 1.7 ms on half the CUs)."""
    from neuralat_amd.bem.batch import batch_solve_mixed

    A, b = _system(20480, 1e-8, 1)
    A[20479, 7] = 300.0  # the largest entry, in the last row: the scale must see it
    print("fp16 scale", flush=True)
    t = {}
    for dtype in ("bf16", "fp16"):
        solve = lambda: batch_solve_mixed([A], [b[0]], dtype=dtype, tol=1e-5, inner_tol=1e-2, inner_restart=10)  # noqa: E731
        x, infos = solve()
        assert infos[0]["converged"] and _err_rows(A, x[0], b[0]) < 2e-5, infos
        t[dtype] = _best(solve)
    assert t["fp16"] < 1.3 * t["bf16"], t


def _err_rows(A, x, b):
    """Relative residual, the product in FP64 row blocks."""
    r = torch.cat([b[q:q + 2048].to(torch.complex128) - A[q:q + 2048].to(torch.complex128) @ x.to(torch.complex128)
                   for q in range(0, len(b), 2048)])
    return float(torch.linalg.vector_norm(r) / torch.linalg.vector_norm(b.to(torch.complex128)))


def test_short_lockstep_solve_stops_near_its_end():
    """A batch that converges in its eighth step launches no whole segment (16
    more steps) past it: as long as with restart=12, whose cycle ends at step 12."""
    from neuralat_amd.bem.batch import batch_gmres

    A, b = _system(1000, 0.2, 3)
    print("arnoldi short lockstep", flush=True)
    _, infos = batch_gmres([A], [b[0]], tol=1e-5, restart=50)
    assert infos[0]["converged"] and 4 < infos[0]["iterations"] < 12, infos
    free, held = (_best(lambda: batch_gmres([A], [b[0]], tol=1e-5, restart=r), 25) for r in (50, 12))
    assert free < 1.1 * held, (free, held)
