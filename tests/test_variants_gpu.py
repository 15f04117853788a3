"""Every kernel variant at its edges, with the variant that runs known: the walks with several
points per lane, and the kernels that grids without a walk use (culled, generic, subspace). The
host tests show, without a GPU, that these grids and data sizes get these kernels.

Tolerances as for the other operators: 1e-12 in FP64, 1e-5 in FP32 with inputs representable in
FP32."""

import numpy as np
import pytest

import oracle
from host_hip import on_host  # noqa: F401

TOL = {0: 1e-12, 1: 1e-5}


def rel(a, b):
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (nb if nb > 0 else 1.0)


def make_grid(capi, basis, kind, d, level):
    lv, ix = capi.Grid(basis, d).regular(level).level_index()
    if kind == "fine":  # a subspace of 2^13 cells in the first dimension: its table is walked in parts
        l1 = np.ones((1 << 13, d), np.uint32)
        i1 = np.ones((1 << 13, d), np.uint32)
        l1[:, 0], i1[:, 0] = 14, 2 * np.arange(1 << 13) + 1
        lv, ix = np.concatenate([lv, l1]), np.concatenate([ix, i1])
    if kind == "repeated":  # no walk: a table holds a point once
        lv, ix = np.concatenate([lv, lv[:1]]), np.concatenate([ix, ix[:1]])
    if kind == "deep":  # no walk: more levels above 1 than a walk has register sets
        one = np.full((1, d), 2, np.uint32)
        lv, ix = np.concatenate([lv, one]), np.concatenate([ix, one - 1])
    return lv, ix


def make_data(basis, d, M):
    """uniform points; some on cell edges, at the corners, and a run of equal ones"""
    rng = np.random.default_rng(100 * d + basis)
    X = rng.random((M, d))
    n = M // 20 + 1
    X[:n] = rng.integers(0, 17, (n, d)) / 16.0
    X[n:3 * n] = X[-1]
    X[0], X[-2], X[M // 2] = 0.0, 1.0, 0.5
    X = X.astype(np.float32).astype(np.float64)
    return X, rng.standard_normal(M)


def clustered(basis, d, M):
    rng = np.random.default_rng(100 * d + basis)
    X = rng.uniform(0.1, 0.9, (4, d))[rng.integers(0, 4, M)] + 0.05 * rng.standard_normal((M, d))
    X[:7] = rng.integers(0, 9, (min(7, M), d)) / 8.0
    return np.clip(X, 0, 1).astype(np.float32).astype(np.float64), rng.standard_normal(M)


# ------------------------------------------------------------------ walks

# (d, regular level, kind, data points in FP32 and FP64): enough that the FP32 walks take four or two
# points per lane, the FP64 ones two up to 10 dimensions; none is a multiple of a batch
WIDE = [(3, 6, "fine", 165001, 83001), (4, 7, "plain", 45001, 22555), (7, 5, "plain", 27003, 14005),
        (8, 4, "plain", 55001, 28001), (10, 4, "plain", 31003, 16001), (13, 3, "plain", 43001, None),
        (16, 3, "plain", 29001, None), (20, 3, "plain", 19003, None), (24, 3, "plain", 14001, None)]


def wide_points(d, prec):
    return (4 if d <= 10 else 2) if prec else 2


def check(capi, op, basis, X, y, lv, ix, prec, columns=300, keep=slice(None)):
    rng = np.random.default_rng(3)
    alpha = rng.standard_normal(len(lv))
    r, a = op.mult(alpha), op.mult_transpose(y)
    rows = np.unique(np.concatenate([np.arange(0, len(X), max(1, len(X) // 3000)), np.arange(max(0, len(X) - 80), len(X))]))
    assert rel(r[rows], oracle.mult(basis, X[rows], lv[keep], ix[keep], alpha[keep])) <= TOL[prec]
    cols = np.unique(rng.integers(0, len(lv), columns))
    if keep != slice(None):
        cols = cols[cols >= keep.start]
    assert rel(a[cols], oracle.mult_transpose(basis, X, lv[cols], ix[cols], y)) <= TOL[prec]
    assert abs(r @ y - alpha[keep] @ a[keep]) <= 10 * TOL[prec] * np.linalg.norm(r) * np.linalg.norm(y)
    assert np.array_equal(r, op.mult(alpha))


@pytest.mark.gpu
@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("d,level,kind,M32,M64", WIDE)
def test_several_points_per_lane(gpu, d, level, kind, M32, M64, prec, basis):
    capi, M = gpu, M32 if prec else M64
    if M is None:
        pytest.skip("one point per lane")
    print("case", d, level, kind, M, prec, basis, flush=True)
    lv, ix = make_grid(capi, basis, kind, d, level)
    X, y = make_data(basis, d, M)
    op = capi.MultiEval(basis, X, precision=prec).prepare(lv, ix)
    check(capi, op, basis, X, y, lv, ix, prec)


def test_several_points_per_lane_run(on_host):
    on_host("""
        import re
        import test_variants_gpu as t
        for d, level, kind, M32, M64 in t.WIDE:
            for prec, M in ((1, M32), (0, M64)):
                for basis in (0, 1):
                    if M is None:
                        continue
                    lv, ix = t.make_grid(capi, basis, kind, d, level)
                    X, y = t.make_data(basis, d, M)
                    op = capi.MultiEval(basis, X, precision=prec).prepare(lv, ix)
                    launches()
                    op.mult(np.zeros(len(lv)))
                    op.mult_transpose(y)
                    found = {m[1]: int(m[2]) for name, _, _, _ in launches()
                             for m in [re.search("tree_mult(T?)_kernelI[fd]Li[0-9]+ELi([0-9]+)E", name)] if m}
                    assert found == {"": t.wide_points(d, prec), "T": t.wide_points(d, prec)}, (d, prec, basis, found)
    """)


# ------------------------------------------------------------------ kernels without a walk

# (algorithm, d, regular level, kind, data points)
OWN = [(0, d, level, "repeated", M) for d, level, M in
       ((1, 5, 1), (1, 7, 4097), (2, 6, 255), (3, 5, 2049), (4, 4, 1023), (5, 4, 3001), (6, 4, 64), (7, 3, 65),
        (8, 4, 6007), (9, 3, 1000), (10, 3, 5003), (11, 3, 2047), (13, 2, 513), (15, 3, 3000), (16, 2, 1), (17, 2, 257),
        (20, 2, 4099), (21, 2, 300), (24, 3, 1031), (40, 2, 129), (64, 2, 257))]
OWN += [(0, 13, 3, "deep", 1500), (0, 20, 2, "deep", 700), (0, 30, 2, "deep", 500)]
OWN += [(1, 1, 9, "repeated", 3000), (1, 2, 7, "repeated", 5001), (1, 3, 5, "repeated", 257), (1, 5, 4, "repeated", 20011),
        (1, 8, 3, "repeated", 2000), (1, 10, 3, "repeated", 1), (1, 13, 2, "repeated", 999), (1, 20, 2, "repeated", 4001),
        (1, 13, 2, "deep", 700)]


@pytest.mark.gpu
@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("data", [make_data, clustered])
@pytest.mark.parametrize("algorithm,d,level,kind,M", OWN)
def test_own_kernels(gpu, algorithm, d, level, kind, M, data, prec, basis):
    capi = gpu
    if algorithm and prec:
        pytest.skip("not a subspace operator")
    print("case", algorithm, d, level, kind, M, data.__name__, prec, basis, flush=True)
    lv, ix = make_grid(capi, basis, kind, d, level)
    X, y = data(basis, d, M) if M > 3 else (np.full((M, d), 0.3125), np.ones(M))
    op = capi.MultiEval(basis, X, precision=prec, algorithm=algorithm).prepare(lv, ix)
    # (of a repeated point a subspace table holds the last one only)
    check(capi, op, basis, X, y, lv, ix, prec, keep=slice(1, None) if algorithm and kind == "repeated" else slice(None))


@pytest.mark.gpu
@pytest.mark.parametrize("basis", [0, 1])
def test_large_subspaces_of_the_subspace_kernels(gpu, basis):
    """Tables beyond the kernel's 4,096 LDS entries: added to with global atomics."""
    capi = gpu
    lv, ix = capi.Grid(basis, 1).regular(14).level_index()
    lv, ix = np.concatenate([lv, lv[:1]]), np.concatenate([ix, ix[:1]])
    X, y = make_data(basis, 1, 7001)
    op = capi.MultiEval(basis, X, algorithm=capi.ALGO_SUBSPACE).prepare(lv, ix)
    rng = np.random.default_rng(4)
    alpha = rng.standard_normal(len(lv))
    assert rel(op.mult(alpha), oracle.mult(basis, X, lv[1:], ix[1:], alpha[1:])) <= 1e-12
    assert rel(op.mult_transpose(y)[1:], oracle.mult_transpose(basis, X, lv[1:], ix[1:], y)) <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("d", [6, 12, 24])
def test_launch_shapes_of_own_kernels(gpu, d, prec, basis):
    """Any chunks, segments and blocks, and the entry point without allocations, give the same."""
    import torch
    capi = gpu
    lv, ix = make_grid(capi, basis, "repeated", d, 4 if d == 6 else 3)
    X, y = clustered(basis, d, 20000)
    alpha = np.random.default_rng(5).standard_normal(len(lv))
    base = capi.MultiEval(basis, X, precision=prec).prepare(lv, ix)
    r0, a0 = base.mult(alpha), base.mult_transpose(y)
    tol = 1e-14 if prec == 0 else 1e-6
    for G, S, blocks in ((1, 1, 0), (2, 3, 0), (7, 16, 0), (0, 0, 50), (0, 0, 5000)):
        op = capi.MultiEval(basis, X, precision=prec, mult_grid_chunks=G, multT_data_segs=S,
                            target_blocks=blocks).prepare(lv, ix)
        assert rel(op.mult(alpha), r0) <= tol and rel(op.mult_transpose(y), a0) <= tol
    d_alpha = torch.tensor(alpha, device="cuda:0")
    out = torch.empty(len(X), dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    capi.check(capi.F["sgpp_hip_meval_mult_device_noalloc"](base.h, d_alpha.data_ptr(), out.data_ptr(), prec))
    base.synchronize()
    assert rel(out.cpu().numpy(), r0) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("basis", [0, 1])
def test_three_algorithms_agree(gpu, basis):
    """The subspace kernels, the culled kernels and the walks, on one grid and data set."""
    capi = gpu
    d, M = 6, 150001
    plain, own = make_grid(capi, basis, "plain", d, 5), make_grid(capi, basis, "repeated", d, 5)
    X, y = clustered(basis, d, M)
    n = len(plain[0])
    alpha = np.random.default_rng(6).standard_normal(n)
    walked = capi.MultiEval(basis, X).prepare(*plain)
    r, a = walked.mult(alpha), walked.mult_transpose(y)
    for algorithm, weights in ((0, np.append(alpha, 0.0)), (1, np.append(alpha, alpha[0]))):
        op = capi.MultiEval(basis, X, algorithm=algorithm).prepare(*own)
        assert rel(op.mult(weights), r) <= 1e-12
        assert rel(op.mult_transpose(y)[:n], a) <= 1e-12


def test_own_kernels_run(on_host):
    on_host("""
        import test_variants_gpu as t
        cases = [c + (p, b) for c in t.OWN for p in (0, 1) for b in (0, 1) if not (c[0] and p)]
        cases += [(0, d, 4 if d == 6 else 3, "repeated", 20000, p, 0) for d in (6, 12, 24) for p in (0, 1)]
        cases += [(a, 6, 5, "repeated", 150001, 0, 0) for a in (0, 1)]
        for algorithm, d, level, kind, M, prec, basis in cases:
            lv, ix = t.make_grid(capi, basis, kind, d, level)
            X, y = t.clustered(basis, d, M) if M > 3 else (np.full((M, d), 0.3125), np.ones(M))
            op = capi.MultiEval(basis, X, precision=prec, algorithm=algorithm).prepare(lv, ix)
            launches()
            op.mult(np.zeros(len(lv)))
            op.mult_transpose(y)
            names = " ".join(name for name, _, _, _ in launches())
            want = ["subspace_mult_kernel", "subspace_multT_kernel"] if algorithm else (
                ["mult_kernel_generic", "multT_kernel_generic"] if d > 20 else ["11mult_kernelI", "12multT_kernelI"])
            assert all(w in names for w in want) and "tree_mult" not in names, (algorithm, d, kind, names)
    """)
