"""The subspace tree's walks against the oracle at their edges: dimensions around
the register variants (4, 8, 10, 16, 20, above), depths around the recursion
variants (4, 6, 12 refined dimensions), level vectors whose parents the grid lacks,
tables larger than a block's LDS, one point per lane or several, data on cell edges
and at the corners, and a grid whose points repeat (not walked).

Tolerances as for the other operators: 1e-12 in FP64, 1e-5 in FP32 with inputs
representable in FP32."""
import itertools

import numpy as np
import pytest

import oracle
from sgpp_amd import workloads

pytestmark = pytest.mark.gpu

TOL = {0: 1e-12, 1: 1e-5}


def rel(a, b):
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (nb if nb > 0 else 1.0)


def full(d, dims, top):
    """All points of levels 1..top in the first dims of d dimensions."""
    one = [(l, i) for l in range(1, top + 1) for i in range(1, 1 << l, 2)]
    pts = np.array(list(itertools.product(one, repeat=dims)), dtype=np.uint32)
    lv = np.ones((len(pts), d), np.uint32)
    ix = np.ones((len(pts), d), np.uint32)
    lv[:, :dims], ix[:, :dims] = pts[:, :, 0], pts[:, :, 1]
    return lv, ix


def loose(d, depth, n, seed):
    """n random points without their ancestors, each refined in up to depth dimensions."""
    rng = np.random.default_rng(seed)
    pts = set()
    while len(pts) < n:
        lv = np.ones(d, np.uint32)
        k = rng.integers(1, depth + 1)
        lv[rng.choice(d, k, replace=False)] = rng.integers(2, 4, k)
        if lv.sum() - d <= 16:
            pts.add(tuple(zip(lv.tolist(), (2 * rng.integers(0, 1 << (lv - 1)) + 1).tolist())))
    a = np.array(sorted(pts), dtype=np.uint32)
    return np.ascontiguousarray(a[:, :, 0]), np.ascontiguousarray(a[:, :, 1])


@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("d,top,M", [(3, 5, 1), (3, 5, 255), (6, 4, 1025), (10, 3, 257), (24, 2, 513)])
def test_equal_points_and_points_by_the_faces(gpu, basis, prec, d, top, M):
    """All data in one cell (every add meets in one position), then data whose
    level-1 factors are the smallest, zero or denormal."""
    capi = gpu
    print("case", basis, prec, d, top, M, flush=True)
    lv, ix = capi.Grid(basis, d).regular(top).level_index()
    rng = np.random.default_rng(M)
    alpha, y = rng.standard_normal(len(lv)), rng.standard_normal(M)
    X = np.full((M, d), 0.3125)
    faces = rng.choice([0.0, 1.0, 1e-310, 1e-40, 2.0 ** -24, 1.0 - 2.0 ** -24, 0.5, 0.3], (M, d))
    faces = np.where(rng.random((M, d)) < 0.3, faces, rng.random((M, d)))
    for X in (X, faces.astype(np.float32).astype(np.float64) if prec else faces):
        op = capi.MultiEval(basis, X, precision=prec).prepare(lv, ix)
        r, a = op.mult(alpha), op.mult_transpose(y)
        assert rel(r, oracle.mult(basis, X, lv, ix, alpha)) <= TOL[prec]
        assert rel(a, oracle.mult_transpose(basis, X, lv, ix, y)) <= TOL[prec]
        assert np.array_equal(a, op.mult_transpose(y))


def grid(capi, basis, kind, d, arg):
    if kind == "regular":
        return capi.Grid(basis, d).regular(arg).level_index()
    if kind == "full":
        return full(d, *arg)
    if kind == "loose":
        return loose(d, arg, 300, d)
    lv, ix = full(d, *arg)  # repeated
    return np.concatenate([lv, lv[:5]]), np.concatenate([ix, ix[:5]])


@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("algorithm", [0, 1])
@pytest.mark.parametrize("kind,d,arg,M", [
    ("regular", 4, 6, 33001), ("regular", 9, 4, 4099), ("regular", 11, 3, 1000),
    ("regular", 16, 2, 65), ("regular", 17, 2, 64), ("regular", 21, 3, 3001),
    ("regular", 40, 2, 257), ("full", 7, (7, 2), 20001), ("full", 9, (5, 2), 130000),
    ("full", 2, (1, 14), 5000), ("loose", 12, 12, 2000), ("loose", 20, 5, 2000),
    ("repeated", 3, (3, 3), 1500)])
def test_walks(gpu, algorithm, basis, prec, kind, d, arg, M):
    capi = gpu
    if algorithm == capi.ALGO_SUBSPACE and (prec == 1 or d > 20):
        pytest.skip("not a subspace operator")
    print("case", algorithm, basis, prec, kind, d, arg, M, flush=True)
    lv, ix = grid(capi, basis, kind, d, arg)
    rng = np.random.default_rng(d)
    X = rng.random((M, d))
    X[:40] = rng.integers(0, 9, (40, d)) / 8.0
    X[0], X[1], X[2] = 0.0, 1.0, 0.5
    X = X.astype(np.float32).astype(np.float64)
    alpha, y = rng.standard_normal(len(lv)), rng.standard_normal(M)
    op = capi.MultiEval(basis, X, precision=prec, algorithm=algorithm).prepare(lv, ix)
    if kind == "repeated" and algorithm == capi.ALGO_SUBSPACE:
        # (of repeated points a table holds the last one only)
        lv, ix, keep = lv[5:], ix[5:], slice(5, None)
    else:
        keep = slice(None)
    r, a = op.mult(alpha), op.mult_transpose(y)
    assert rel(r, oracle.mult(basis, X, lv, ix, alpha[keep])) <= TOL[prec]
    assert rel(a[keep], oracle.mult_transpose(basis, X, lv, ix, y)) <= TOL[prec]
    assert np.array_equal(r, op.mult(alpha))
