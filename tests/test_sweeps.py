"""The streaming triangular solves and the residual of the refinement: block
edges (64 rows), remainders, one, some and several groups of right-hand sides,
against torch in double precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(torch, n, nrhs, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.complex(*[torch.randn(n, n, generator=g, device="cuda", dtype=torch.float64) for _ in range(2)])
    A += 2 * n**0.5 * torch.eye(n, device="cuda")
    B = torch.complex(*[torch.randn(nrhs, n, generator=g, device="cuda", dtype=torch.float64) for _ in range(2)])
    return A, B


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 200, 449, 1000])
@pytest.mark.parametrize("nrhs", [1, 2, 8, 9, 63])
def test_solve_complex128(bfa, torch_cuda, n, nrhs):
    torch = torch_cuda
    A, B = _system(torch, n, nrhs, 7 * n + nrhs)
    LU = A.T.contiguous()                      # column-major A
    piv = torch.empty(n, dtype=torch.int32, device="cuda")
    assert bfa.lu_factor(LU, n, piv) == 0
    X = B.clone()
    bfa.lu_solve(LU, n, piv, X, nrhs)
    torch.cuda.synchronize()
    # backward error of a pivoted LU with growth of order n^(2/3): a few n eps
    r = (B - X @ A.T).norm() / (A.norm() * X.norm())
    assert r < 8 * max(n, 4) * np.finfo(np.float64).eps


@pytest.mark.parametrize("n", [40, 64, 130, 513, 1024])
@pytest.mark.parametrize("nrhs", [1, 7, 8, 31, 33, 70])
def test_refined_solve(bfa, torch_cuda, n, nrhs):
    torch = torch_cuda
    A, B = _system(torch, n, nrhs, 11 * n + nrhs)
    M = A.T.contiguous()
    LU = M.to(torch.complex64)
    piv = torch.empty(n, dtype=torch.int32, device="cuda")
    assert bfa.lu_factor_c(LU, n, piv) == 0
    X = B.clone()
    it, res = bfa.solve_refine(M, LU, piv, n, X, nrhs, tol=1e-12)
    torch.cuda.synchronize()
    R = B - X @ A.T
    worst = (R.norm(dim=1) / B.norm(dim=1)).max().item()
    # the reported residual is the one of the result, summed in another order
    assert res <= 1e-12 and worst <= 1e-12 + 8 * n * np.finfo(np.float64).eps
