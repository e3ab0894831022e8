"""The factorisation as one dataflow launch (gprat_amd/csrc/k_flow.hip) against
the panel schedule at the sizes around its 64-wide tiles and its panels of
eight (the tiled right-looking Cholesky of core/src/cpu/gp_algorithms.cpp)."""
import os
import threading
from contextlib import contextmanager

import numpy as np
import pytest

from conftest import norm_rel
from gprat_amd import capi, datagen

pytestmark = pytest.mark.gpu

# two Cholesky factors of one matrix agree to about n eps cond; cond <= (n v + noise) / noise
# <= 4e4 here and n <= 2500: 2500 * 1.1e-16 * 4e4 = 1.1e-8 is the worst case, the errors
# of the factor's entries are random: sqrt(n) in place of n, hence
TOL = 2e-10


def tol(n):
    """The same bound for larger n: sqrt(n) eps n v / noise."""
    return TOL * (max(n, 2500) / 2500) ** 1.5


@contextmanager
def panel_schedule():
    saved = os.environ.get("GPRAT_FLOW_LIMIT")
    os.environ["GPRAT_FLOW_LIMIT"] = "0"
    try:
        yield
    finally:
        if saved is None:
            del os.environ["GPRAT_FLOW_LIMIT"]
        else:
            os.environ["GPRAT_FLOW_LIMIT"] = saved


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0, 1)
    yield c
    c.close()


SIZES = [1, 64, 65, 500, 513, 1024, 1030, 1100, 1537, 2049, 2500]
# up to where the rule of engine.cpp's one_launch ends: an FP64 fit, a mixed fit, a gradient
LARGE_FP64, LARGE_MIXED, LARGE_GRADIENT = [5003, 9000, 11900], [5003, 11000], [5003, 8300]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("m", [1, 70, 1000])
def test_one_call(ctx, n, m):
    x, y, z = datagen.gp_problem(n, m, 5)
    args = (x, y, z, (1.0, 1.0, 0.1), 1, n, 1, m, 5)
    mean, var = ctx.predict(*args, variance=True)
    with panel_schedule():
        pm, pv = ctx.predict(*args, variance=True)
    assert norm_rel(mean, pm) < TOL and norm_rel(var, pv) < TOL


@pytest.mark.parametrize("precision, n", [(capi.PRECISION_FP64, n) for n in SIZES + LARGE_FP64]
                         + [(capi.PRECISION_MIXED, n) for n in SIZES + LARGE_MIXED])
def test_resident(ctx, n, precision):
    x, y, z = datagen.gp_problem(n, 33, 8)
    theta = (1.0, 1.0, 0.1)

    def results(p):
        m = ctx.fit(x, y, n, 8, theta, p)
        out = (*m.predict(z, 33), m.loss(), m.gradient()[1])
        m.release()
        return out
    got = results(precision)
    with panel_schedule():
        want = results(capi.PRECISION_FP64)
    # the mixed model's variance is refined from FP32 solves: 1e-7 is its stated bar
    t = tol(n)
    for a, b, bar in zip(got, want, (t, t if precision == capi.PRECISION_FP64 else 1e-7, t, 10 * t)):
        assert norm_rel(np.atleast_1d(a), np.atleast_1d(b)) < bar


@pytest.mark.parametrize("n", SIZES)
def test_tiles(ctx, n):
    x, _, _ = datagen.gp_problem(n, 1, 8)
    a = ctx.cholesky(x, (1.0, 1.0, 0.1), 1, n, 8)
    with panel_schedule():
        b = ctx.cholesky(x, (1.0, 1.0, 0.1), 1, n, 8)
    assert norm_rel(a.ravel(), b.ravel()) < TOL


@pytest.mark.parametrize("n", SIZES + LARGE_GRADIENT)
def test_gradient(ctx, n):
    x, y, _ = datagen.gp_problem(n, 1, 8)
    theta = (1.0, 1.0, 0.1)
    loss, grad = ctx.loss_gradient(x, y, theta, 1, n, 8)
    with panel_schedule():
        ploss, pgrad = ctx.loss_gradient(x, y, theta, 1, n, 8)
    assert norm_rel(np.atleast_1d(loss), np.atleast_1d(ploss)) < tol(n) and norm_rel(grad, pgrad) < 10 * tol(n)


def test_repeats_are_bit_identical(ctx):
    x, y, z = datagen.gp_problem(1800, 300, 8)
    args = (x, y, z, (1.0, 1.0, 0.1), 1, 1800, 1, 300, 8)
    first = ctx.predict(*args, variance=True)
    for _ in range(5):
        again = ctx.predict(*args, variance=True)
        assert np.array_equal(first[0], again[0]) and np.array_equal(first[1], again[1])


@pytest.mark.parametrize("column", [70, 600, 1100, 1500])
def test_first_failing_pivot(ctx, column):
    n, r = 1600, 4
    u = np.arange(n + r - 1) * 10.0
    u[column:column + r] = u[:r]  # this window repeats the first one: its pivot is about 2 * noise < 0
    with pytest.raises(capi.GpratError, match=f"at column {column}\\)"):
        ctx.cholesky(u, (0.3, 1.0, -1e-3), 1, n, r)
    assert ctx.cholesky(u, (0.3, 1.0, 1e-3), 1, n, r).shape == (1, n, n)


@pytest.mark.parametrize("n", [300, 1600])
def test_a_failed_factorisation_leaves_the_outputs(ctx, n):
    """Not positive definite: host arrays, arrays larger than the staging (65536
    test points) and device buffers keep what they held."""
    r, theta = 4, (0.3, 1.0, -1e-3)
    u = np.arange(n + r - 1) * 10.0
    u[n - 50:n - 50 + r] = u[:r]  # as above: the pivot of column n - 50 is about 2 * noise < 0
    y, t = np.zeros(n), np.array(theta)
    L, D = capi.lib(), capi._dptr
    tiles = np.full(n * n, 7.5)
    assert L.gprat_cholesky(ctx.handle, D(u), u.size, D(t), 1, n, r, D(tiles)) == capi.ERR_NOT_SPD
    assert np.all(tiles == 7.5)
    for m in (65, 65600):
        z = np.linspace(0.0, 1.0, m + r - 1)
        mean, var = np.full(m, 7.5), np.full(m, 7.5)
        args = (ctx.handle, D(u), u.size, D(y), y.size, D(z), z.size, D(t), 1, n, 1, m, r)
        assert L.gprat_predict_with_uncertainty(*args, D(mean), D(var)) == capi.ERR_NOT_SPD
        assert np.all(mean == 7.5) and np.all(var == 7.5)
    out = ctx.device_array(np.full(65, 7.5)), ctx.device_array(np.full(65, 7.5))
    with pytest.raises(capi.GpratError):
        ctx.predict(u, y, np.linspace(0.0, 1.0, 65 + r - 1), theta, 1, n, 1, 65, r, variance=True, out=out)
    assert all(np.all(d.numpy() == 7.5) for d in out)


# the second list: sizes around the lines of engine.cpp's forward_solve (4 and 10 Mi elements of n x m)
@pytest.mark.parametrize("n, m", [(n, m) for n in (100, 769, 2049, 2500) for m in (1, 16, 17, 32, 33, 64, 65, 200, 1100)]
                         + [(5003, 777), (8200, 16), (8200, 500), (16400, 250), (16400, 600), (32768, 100)])
def test_forward_solves_agree(ctx, n, m):
    """Few-row kernels (0), one launch (1) and the blocked solve (2)."""
    x, y, z = datagen.gp_problem(n, m, 8)
    model = ctx.fit(x, y, n, 8, (1.0, 1.0, 0.1))
    out = {}
    try:
        for how in "012":
            os.environ["GPRAT_FORWARD_SOLVE"] = how
            mean, var = model.predict(z, m)
            out[how] = mean, var, model.predict_full_cov(z, m)[1]
    finally:
        del os.environ["GPRAT_FORWARD_SOLVE"]
        model.release()
    for how in "01":
        assert np.array_equal(out[how][0], out["2"][0])
        assert norm_rel(out[how][1], out["2"][1]) < tol(n)
        assert norm_rel(out[how][2].ravel(), out["2"][2].ravel()) < tol(n)
        assert np.array_equal(out[how][2], out[how][2].T)


@pytest.mark.parametrize("n", [200, 1100])
def test_device_memory_in_and_out(ctx, n):
    """Results through pinned staging (host arrays) and through device buffers are the same."""
    m, theta = 77, (1.0, 1.0, 0.1)
    x, y, z = datagen.gp_problem(n, m, 8)
    dx, dy, dz = (ctx.device_array(v) for v in (x, y, z))
    out = ctx.device_empty(m), ctx.device_empty(m)
    host = ctx.predict(x, y, z, theta, 1, n, 1, m, 8, variance=True)
    ctx.predict(dx, dy, dz, theta, 1, n, 1, m, 8, variance=True, out=out)
    assert all(np.array_equal(h, d.numpy()) for h, d in zip(host, out))
    a, b = ctx.fit(x, y, n, 8, theta), ctx.fit(dx, dy, n, 8, theta)
    b.predict(dz, m, out=out)
    assert a.loss() == b.loss()
    assert all(np.array_equal(h, d.numpy()) for h, d in zip(a.predict(z, m), out))
    a.release()
    b.release()


def first_difference(got, want):
    """None, or the first quantity that is not bit-identical (a factor: its first 64x64 tile)."""
    for name, w in want.items():
        g = got[name]
        if np.array_equal(g, w):
            continue
        at = np.argwhere(np.atleast_1d(g) != np.atleast_1d(w))
        if name == "factor":
            tiles = sorted({(int(c) // 64, int(r) // 64) for r, c in at})
            return f"factor: {len(at)} entries, first in block column {tiles[0][0]}, block row {tiles[0][1]}"
        return f"{name}: {len(at)} entries, first at {at[0].tolist()}"
    return None


def test_results_do_not_depend_on_other_launches():
    """Two contexts in two threads: while their dataflow launches share the
    device, each gives bit by bit what it gives alone."""
    sizes, theta, m, rounds = (5003, 9000), (1.0, 1.0, 0.1), 33, 30
    contexts = [capi.Context(0, 1) for _ in sizes]
    problems = [datagen.gp_problem(n, m, 8) for n in sizes]

    def results(k, factor):
        n, c, (x, y, z) = sizes[k], contexts[k], problems[k]
        out = {}
        if factor:
            out["factor"] = c.cholesky(x, theta, 1, n, 8)[0]
        model = c.fit(x, y, n, 8, theta)
        try:
            out["loss"] = model.loss()
            out["mean"], out["variance"] = model.predict(z, m)
        finally:
            model.release()
        if n < 9000:
            out["gradient"] = c.loss_gradient(x, y, theta, 1, n, 8)[1]
        return out

    differences = []

    def work(k, alone, start):
        try:
            start.wait()
            for i in range(rounds):
                got = results(k, factor=i % 10 == 0)
                d = first_difference(got, {q: alone[q] for q in got})
                if d:
                    differences.append(f"n = {sizes[k]}, pass {i}: {d}")
        except Exception as e:
            differences.append(f"n = {sizes[k]}: {e!r}")

    try:
        alone = [results(k, factor=True) for k in range(len(sizes))]
        start = threading.Barrier(len(sizes))
        threads = [threading.Thread(target=work, args=(k, alone[k], start)) for k in range(len(sizes))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        for c in contexts:
            c.close()
    assert not differences, differences
