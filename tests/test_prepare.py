"""Preparing a grid, on host memory: what a failed call leaves, and what a grid's layout takes."""
import textwrap

import pytest

from host_hip import on_host  # noqa: F401
from test_routes import GRIDS


@pytest.mark.parametrize("algorithm", [0, 1])
@pytest.mark.parametrize("basis", [0, 1])
def test_failed_prepare_leaves_no_grid(on_host, algorithm, basis):
    """Whichever allocation fails, no product runs on what the call left behind, and the
    next prepare works."""
    out = on_host("""
        X = workloads.uniform_points(1, 500, 3)
        small = capi.Grid(%d, 3).regular(2).level_index()
        large = capi.Grid(%d, 3).regular(6).level_index()
        failed = 0
        for first, then in ((None, large), (small, large), (large, small)):
            for after in range(30):
                op = capi.MultiEval(%d, X, algorithm=%d)
                if first is not None:
                    op.prepare(*first)
                launches()
                hip.host_hip_fail_malloc(after, 1)
                try:
                    op.prepare(*then)
                    ok = True
                except capi.SGppHIPError:
                    ok = False
                hip.host_hip_fail_malloc(-1, 0)
                if ok:
                    continue
                failed += 1
                launches()
                op.N = capi.F["sgpp_hip_meval_num_grid"](op.h)
                for call, n in ((op.mult, op.N), (op.mult_transpose, len(X))):
                    try:
                        call(np.zeros(n))
                    except capi.SGppHIPError as e:
                        assert "grid not set" in str(e), e
                    else:
                        raise AssertionError("a product ran after a failed prepare")
                assert launches() == []
                op.prepare(*small).mult(np.zeros(len(small[0])))
                assert launches()
        print(failed)
    """ % (basis, basis, basis, algorithm))
    assert int(out) > 0


def test_refused_grid_leaves_the_old_one(on_host):
    on_host("""
        X = workloads.uniform_points(1, 500, 3)
        lv, ix = capi.Grid(0, 3).regular(3).level_index()
        for algorithm in (0, 1):
            op = capi.MultiEval(0, X, algorithm=algorithm).prepare(lv, ix)
            bad = ix.copy()
            bad[0] = 2
            try:
                op.prepare(lv[:5], bad[:5])
                raise AssertionError("accepted")
            except capi.SGppHIPError as e:
                assert e.status_name == "INVALID_ARGUMENT"
            assert capi.F["sgpp_hip_meval_num_grid"](op.h) == len(lv)
            op.mult(np.zeros(len(lv)))
    """)


@pytest.mark.parametrize("algorithm", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
def test_no_memory_for_the_walks(on_host, algorithm, precision):
    """A grid that its algorithm's own kernels can evaluate is not refused because one of
    the walks' buffers could not be allocated."""
    if algorithm == 1 and precision == 1:
        pytest.skip("not a subspace operator")
    out = on_host("""
        X = workloads.uniform_points(1, 500, 3)
        lv, ix = capi.Grid(0, 3).regular(5).level_index()
        own = 0
        for after in range(20):
            op = capi.MultiEval(0, X, precision=%d, algorithm=%d)
            hip.host_hip_fail_malloc(after, 0)
            op.prepare(lv, ix)
            hip.host_hip_fail_malloc(-1, 0)
            launches()
            op.mult(np.zeros(len(lv)))
            op.mult_transpose(np.zeros(len(X)))
            own += not any("tree" in name for name, _, _, _ in launches())
            op.prepare(lv, ix).mult(np.zeros(len(lv)))
            assert any("tree" in name for name, _, _, _ in launches())
        print(own)
    """ % (precision, algorithm))
    assert int(out) >= 5


def test_tables_only_for_walked_grids(on_host):
    """A deep grid around one point: 144 points in 16.8 million cells of their subspaces. No
    table of them is filled for a grid that keeps the culled kernels (67 MB), and no second one
    for one that keeps the subspace kernels."""
    out = on_host("""
        import resource
        l = np.arange(1, 13)
        lv = np.ones((144, 3), np.uint32)
        lv[:, 0], lv[:, 1] = np.repeat(l, 12), np.tile(l, 12)
        ix = 2 * (0.3 * 2.0 ** (lv - 1.0)).astype(np.uint32) + 1
        X = workloads.uniform_points(1, 500, 3)
        peak = [resource.getrusage(resource.RUSAGE_SELF).ru_maxrss]
        for algorithm in (0, 1):
            op = capi.MultiEval(1, X, algorithm=algorithm).prepare(lv, ix)
            peak.append(resource.getrusage(resource.RUSAGE_SELF).ru_maxrss)
            launches()
            op.mult(np.zeros(144))
            assert not any("tree" in name for name, _, _, _ in launches())
            op = None
        print(peak[1] - peak[0], peak[2] - peak[1])
    """)
    streaming, subspace = (int(v) / 1024 for v in out.split())  # MiB
    assert streaming < 32
    assert subspace < 64 + 64 + 32  # the table, and the copy that stands for the GPU's


@pytest.mark.parametrize("data,grid,culled", [
    ("mixture(200000, 8)", "adaptive(8, 20000)", {"", "T"}),
    ("uniform(200000, 1)", "regular(1, 10)", {"T"}),
    ("uniform(10000, 5)", "regular(5, 5)", set())])
def test_only_culled_directions_are_probed(on_host, data, grid, culled):
    """The block order's timing launches are for the kernels that will run."""
    on_host(GRIDS + textwrap.dedent("""
        import re
        X, (lv, ix) = %s, %s
        op = capi.MultiEval(0, X, precision=1)
        launches()
        op.prepare(lv, ix)
        probed = {m[1] for name, _, _, _ in launches() for m in [re.search("[0-9]mult(T?)_kernel", name)] if m}
        assert probed == %r, probed
        op.mult(np.zeros(op.N))
        op.mult_transpose(np.zeros(op.M))
        used = {m[1] for name, _, _, _ in launches() for m in [re.search("[0-9]mult(T?)_kernel", name)] if m}
        assert used == probed, used
    """) % (data, grid, culled))
