"""The 64x64 block factor (gprat_amd/csrc/block64.hpp) through Context.cholesky
at the sizes around its 16-wide steps and 64-wide blocks: the reference's
POTRF of core/src/cpu/gp_algorithms.cpp on one tile."""
import numpy as np
import pytest

from gprat_amd import capi

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0, 1)
    yield c
    c.close()


def covariance(x, n, r, theta):
    w = np.stack([x[i:i + r] for i in range(n)])
    d = ((w[:, None, :] - w[None, :, :]) ** 2).sum(-1)
    return theta[1] * np.exp(-0.5 / theta[0] ** 2 * d) + theta[2] * np.eye(n)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 63, 64, 65, 127, 130])
@pytest.mark.parametrize("theta", [(1.0, 1.0, 0.1), (4.0, 2.0, 1e-4), (0.3, 1e-3, 1e-6)])
def test_one_tile_factor(ctx, n, theta):
    x = np.random.default_rng(n).uniform(-1, 1, n + 7)
    tile = ctx.cholesky(x, theta, 1, n, 8)[0]
    L, K = np.tril(tile), covariance(x, n, 8, theta)
    # backward error of a Cholesky factor, element by element: (n + 1) eps sqrt(a_ii a_jj),
    # plus the covariance entries' own rounding (the exponential, 8 squared differences of size up to 4)
    own = (4 + 40 / theta[0] ** 2) * EPS * K.max()
    assert np.abs(L @ L.T - K).max() <= 2 * (n + 1) * EPS * K.max() + own


@pytest.mark.parametrize("column", [1, 15, 16, 20, 47, 63, 64, 100])
def test_first_failing_pivot(ctx, column):
    n, r = 128, 4
    # the window of `column` repeats the first one, so that pivot is about 2 * noise < 0
    # and every pivot before it is positive (the other windows are far apart)
    u = np.arange(n + r - 1) * 10.0
    u[column:column + r] = u[:r] if column >= r else u[0]
    if column < r:
        u[:column + r] = u[0]
    theta = (0.3, 1.0, -1e-3)
    K = covariance(u, n, r, theta)
    first = next(j for j in range(n) if np.linalg.eigvalsh(K[:j + 1, :j + 1]).min() <= 0)
    with pytest.raises(capi.GpratError, match=f"at column {first}\\)"):
        ctx.cholesky(u, theta, 1, n, r)
