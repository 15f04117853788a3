"""Single basis values (unit weights, unit sources) against their value in extended precision:
no more roundings than the product of D factors has, D - 1 (ModLinear: and one for each
boundary factor 2 - 2^l x, which the type need not hold); from 11 dimensions on, where a walk
takes a Linear level-1 factor out of a product of all, one and three per refined dimension."""
import numpy as np
import pytest


def basis_value(basis, X, lv, ix):
    p = np.ones(len(X), np.longdouble)
    for d in range(X.shape[1]):
        x, l, i = X[:, d].astype(np.longdouble), int(lv[d]), int(ix[d])
        if basis and l == 1:
            continue
        if basis and i == 1:
            f = 2 - 2 ** l * x
        elif basis and i == 2 ** l - 1:
            f = 2 ** l * x - i + 1
        else:
            f = 1 - abs(2 ** l * x - i)
        p *= np.maximum(f, 0)
    return p


@pytest.mark.gpu
@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("d,level", [(1, 8), (2, 8), (3, 6), (4, 5), (5, 5), (8, 4), (10, 3), (11, 4), (20, 3), (30, 3)])
def test_roundings(gpu, basis, prec, d, level):
    capi = gpu
    print("case", basis, prec, d, level, flush=True)
    lv, ix = capi.Grid(basis, d).regular(level).level_index()
    rng = np.random.default_rng(d)
    M, u = 700, 2.0 ** (-24 if prec else -53)
    X = rng.random((M, d))
    X = X.astype(np.float32).astype(np.float64) if prec else X
    op = capi.MultiEval(basis, X, precision=prec).prepare(lv, ix)

    def check(got, exact, refined):
        n = d - 1 + refined if basis else (d - 1 if d <= 10 else min(d - 1, 1 + 3 * refined))
        bound = n * u / (1 - n * u)
        assert np.all(abs(got - exact) <= bound * exact), n

    for j in [0] + list(rng.choice(len(lv), 24)):
        e = np.zeros(len(lv))
        e[j] = 1.0
        check(op.mult(e).astype(np.longdouble), basis_value(basis, X, lv[j], ix[j]), (lv[j] > 1).sum())
    for m in rng.choice(M, 6):
        e = np.zeros(M)
        e[m] = 1.0
        got = op.mult_transpose(e).astype(np.longdouble)
        for j in rng.choice(len(lv), 40):
            check(got[j], basis_value(basis, X[m:m + 1], lv[j], ix[j])[0], (lv[j] > 1).sum())


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("d", [3, 11, 24])
def test_small_coordinates(gpu, prec, d):
    """A coordinate far below the finest cell: the values are small, not 0."""
    capi = gpu
    lv, ix = np.ones((2, d), np.uint32), np.ones((2, d), np.uint32)
    lv[1, 0] = 12
    x0 = 2.0 ** -np.array([30, 60, 90, 100, 101, 110, 114])
    X = np.full((len(x0), d), 0.375)
    X[:, 0] = x0
    op = capi.MultiEval(0, X, precision=prec).prepare(lv, ix)
    u, n = 2.0 ** (-24 if prec else -53), max(d - 1, 4)
    for j, l in ((0, 1), (1, 12)):
        exact = x0 * 2.0 ** l * 0.75 ** (d - 1)
        assert np.all(exact > 2.0 ** -126)
        e = np.zeros(2)
        e[j] = 1.0
        assert np.all(abs(op.mult(e) - exact) <= 2 * n * u * exact)
