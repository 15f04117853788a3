"""Which kernels a grid and a data set get, on host memory: the walks along the subspace tree or
the instance's own (culled, generic, subspace), per direction."""
import pytest

from host_hip import on_host  # noqa: F401

GRIDS = """
import itertools

def around(d, dims, top):
    "levels 1 to top in the first dims dimensions, the points around (0.3, 0.3, ...)"
    lv = np.ones((top ** dims, d), np.uint32)
    lv[:, :dims] = list(itertools.product(range(1, top + 1), repeat=dims))
    return lv, 2 * (0.3 * 2.0 ** (lv - 1.0)).astype(np.uint32) + 1

def loose(d, depth, n, top):
    "n random points without their ancestors, levels 2 to top in up to depth dimensions"
    rng, pts = np.random.default_rng(d), set()
    while len(pts) < n:
        lv = np.ones(d, np.uint32)
        k = rng.integers(1, depth + 1)
        lv[rng.choice(d, k, replace=False)] = rng.integers(2, top + 1, k)
        if lv.sum() - d <= 24:
            pts.add(tuple(zip(lv.tolist(), (2 * rng.integers(0, 1 << (lv - 1)) + 1).tolist())))
    a = np.array(sorted(pts), dtype=np.uint32)
    return np.ascontiguousarray(a[:, :, 0]), np.ascontiguousarray(a[:, :, 1])

def adaptive(d, n):
    g = workloads.adaptive_grid(0, d, 2, workloads.damped_cosine_product, min(200, n // 20), n)[0]
    return g.level_index()

def regular(d, level):
    return capi.Grid(0, d).regular(level).level_index()

def mixture(M, d):
    rng = np.random.default_rng(1)
    return np.clip(rng.uniform(0.2, 0.8, (5, d))[rng.integers(0, 5, M)] + 0.08 * rng.standard_normal((M, d)), 0, 1)

def uniform(M, d):
    return np.random.default_rng(1).random((M, d))

def route(X, grid, basis, precision, algorithm):
    op = capi.MultiEval(basis, X, precision=precision, algorithm=algorithm).prepare(*grid)
    names = []
    for call, n in ((op.mult, op.N), (op.mult_transpose, op.M)):
        launches()
        call(np.zeros(n))
        names.append(" ".join(name for name, _, _, _ in launches()))
    return names
"""


@pytest.mark.parametrize("data,grid,basis,prec,algorithm,walked", [
    ("uniform(10000, 5)", "regular(5, 5)", 0, 0, 0, "both"),
    ("uniform(20000, 30)", "regular(30, 3)", 0, 0, 0, "both"),
    ("uniform(1000, 2)", "regular(2, 5)", 0, 0, 1, "both"),
    ("uniform(300, 7)", "regular(7, 5)", 1, 0, 1, "both"),
    ("uniform(20000, 24)", "loose(24, 3, 1000, 4)", 0, 1, 0, "both"),
    # few points in large tables: a block would copy them all
    ("uniform(20000, 24)", "around(24, 2, 12)", 0, 1, 0, "none"),
    ("uniform(300, 24)", "around(24, 2, 12)", 1, 0, 0, "none"),
    ("uniform(200000, 24)", "around(24, 3, 8)", 0, 1, 0, "none"),
    ("uniform(20000, 3)", "around(3, 2, 12)", 0, 1, 0, "none"),
    ("uniform(400000, 10)", "loose(10, 3, 1000, 6)", 0, 0, 1, "none"),
    ("uniform(400000, 6)", "loose(6, 4, 2000, 5)", 0, 0, 1, "none"),
    # few hits: culling leaves less than a node's walk
    ("mixture(200000, 8)", "adaptive(8, 20000)", 0, 1, 0, "none"),
    ("mixture(200000, 13)", "adaptive(13, 20000)", 0, 0, 0, "none"),
])
def test_routes(on_host, data, grid, basis, prec, algorithm, walked):
    out = on_host(GRIDS + "\nfor n in route(%s, %s, %d, %d, %d): print(n)" % (data, grid, basis, prec, algorithm))
    assert ["tree_mult" in line for line in out.splitlines()] == [walked == "both"] * 2, out


def test_launch_knobs_of_walks(on_host):
    """target_blocks sets the workgroups of both directions; chunks and segments that a caller
    asks for stay within the partial sums' 2 GiB."""
    on_host(GRIDS + """
lv, ix = regular(6, 6)  # 462 subspaces
X = uniform(100000, 6)

def grids(**more):
    op = capi.MultiEval(0, X, **more).prepare(lv, ix)
    out = {}
    for call, n in ((op.mult, op.N), (op.mult_transpose, op.M)):
        launches()
        hip.host_hip_clear()
        call(np.zeros(n))
        out["allocated"] = out.get("allocated", 0) + hip.host_hip_allocated()
        for name, x, y, _ in launches():
            if "tree_mult_k" in name: out["mult"] = x * y
            if "tree_multT_k" in name: out["multT"] = x * y
    return out

few, many = grids(target_blocks=200), grids(target_blocks=4000)
assert 200 <= few["mult"] <= 400 and 100 <= few["multT"] <= 400, few
assert 4000 <= many["mult"] <= 4400 and 3000 <= many["multT"] <= 5000, many
X = uniform(1500000, 6)
for algorithm in (0, 1):
    most = grids(mult_grid_chunks=1000000, multT_data_segs=1000000, algorithm=algorithm)
    assert most["allocated"] <= 2 * (2048 << 20) + (64 << 20), most
""")


def test_kernels_and_work_of_walks(on_host):
    """The kernels' names, and a walk's executed work: every data row, the padding to whole blocks
    included, looks each subspace up once, one of 2^13 cells in its parts (of 5,119 entries in FP64;
    of 1,280 in multTranspose); factors are at least the subspaces' but the root's."""
    on_host(GRIDS + """
def names(op):
    out = []
    for call, n in ((op.mult, op.N), (op.mult_transpose, op.M)):
        launches()
        call(np.zeros(n))
        out.append(" ".join(name for name, _, _, _ in launches()))
    return out

fine = np.ones((1 << 13, 3), np.uint32), np.ones((1 << 13, 3), np.uint32)
fine[0][:, 0], fine[1][:, 0] = 14, 2 * np.arange(1 << 13) + 1
lv, ix = regular(3, 5)  # 35 subspaces
for grid, mult, multT in (((lv, ix), 35, 35),
                          ((np.concatenate([lv, fine[0]]), np.concatenate([ix, fine[1]])), 37, 42)):
    op = capi.MultiEval(0, uniform(5000, 3)).prepare(*grid)
    assert op.kernels() == ("tree_mult_kernel", "tree_multT_kernel")
    w, rows = op.count_work(0), 5120  # one point per lane
    assert w["mult_pairs"] == rows * mult and w["multT_pairs"] == rows * multT, w
    assert rows * 34 <= w["mult_hat_steps"] <= 3 * rows * mult, w

repeated = np.concatenate([lv, lv[:1]]), np.concatenate([ix, ix[:1]])
for algorithm in (0, 1):
    for grid in ((lv, ix), repeated):
        op = capi.MultiEval(0, uniform(5000, 3), algorithm=algorithm).prepare(*grid)
        assert all(k in n for k, n in zip(op.kernels(), names(op))), (op.kernels(), names(op))
lv, ix = regular(24, 2)
op = capi.MultiEval(0, uniform(50, 24)).prepare(np.concatenate([lv, lv[:1]]), np.concatenate([ix, ix[:1]]))
assert op.kernels() == ("mult_kernel_generic", "multT_kernel_generic") and "generic" in names(op)[1]
try:
    capi.MultiEval(0, uniform(50, 3)).kernels()
    raise AssertionError("named kernels without a grid")
except capi.SGppHIPError:
    pass
""")
