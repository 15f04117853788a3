"""The CG iteration's kernels at vector sizes around their 256 chunks, from solves of a
few iterations to ones beyond 50 (which replace the residual), against a dense solve.

The residual is reduced to 1e-12; the system's condition number is at most 1e4 (its
largest eigenvalue, at most M, over lambda M): 1e-8 relative at most, 1e-7 is asked for."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,level,M", [(1, 1, 50), (1, 8, 3000), (2, 6, 3000), (3, 5, 3000), (4, 4, 3000)])
@pytest.mark.parametrize("reuse", [False, True])
def test_cg(gpu, d, level, M, reuse):
    capi = gpu
    print("case", d, level, M, reuse, flush=True)
    rng = np.random.default_rng(level)
    X, y = rng.random((M, d)), rng.standard_normal(M)
    lv, ix = capi.Grid(0, d).regular(level).level_index()
    N, lam = len(lv), 1e-4
    B = np.stack([oracle.mult(0, X, lv, ix, row) for row in np.eye(N)], axis=1)
    exact = np.linalg.solve(B.T @ B + lam * M * np.eye(N), B.T @ y)
    op = capi.MultiEval(0, X, precision=capi.PREC_FP64).prepare(lv, ix)
    alpha, _ = op.solve(y, lam, mode=capi.SOLVE_FP64, max_iterations=2000, epsilon=1e-12,
                        alpha0=exact * 1.001 if reuse else None)
    assert np.linalg.norm(alpha - exact) <= 1e-7 * np.linalg.norm(exact)
