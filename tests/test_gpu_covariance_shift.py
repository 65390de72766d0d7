"""GPU: the covariance of chunks long enough to take their shift from a sample, against two-pass sums in extended
precision: ordinary rows, rows with a trend, invalid rows at every step, a shift that the sample gets wrong (one row
carries the weight) and constant columns. The sums of n terms in FP64 with a shift within an eighth of a deviation:
1e-12 of the column scales."""
import numpy as np
import pytest

import decontamination_amd as dam
from decontamination_amd import _lib
from decontamination_amd.runtime import DeviceArray, get_context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _setup():
    assert dam.gpu_available(), "no GPU visible: the GPU tests must run on an MI355X"


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("kind", ["plain", "trend", "invalid", "heavy", "constant"])
def test_covariance_shift(kind, dim, dtype):
    print(f"covariance {kind} D{dim} {np.dtype(dtype)}", flush=True)
    n = 262_144 + 4_099
    rng = np.random.default_rng(dim)
    x = rng.standard_normal((n, dim)) * (1.0 + np.arange(dim)) + 3.0
    rho = rng.random(n) + 0.1
    if kind == "trend":
        x += np.linspace(-50.0, 50.0, n)[:, None]
    if kind == "invalid":
        x[::37, 0] = np.nan
        x[5::41, -1] = np.inf
        rho[::29], rho[1::31], rho[2::43] = 0.0, -1.0, np.nan
    if kind == "heavy":
        rho[:] = 1e-9
        rho[200_003:200_013] = 1e6
        x[200_003:200_013] += 1e4
    if kind == "constant":
        x[:, 0] = 0.1
    x = x.astype(dtype)
    ctx = get_context(0)
    dx, dr = DeviceArray.from_host(ctx, x), DeviceArray.from_host(ctx, rho)
    out = np.empty(1 + dim + dim * dim)
    _lib.call("somhip_covariance_chunk", ctx.handle, _lib.vp(dx.ptr), int(dtype == np.float64), _lib.vp(dr.ptr), n, dim,
              _lib.vp(out))
    ok = np.isfinite(x).all(1) & np.isfinite(rho) & (rho > 0.0)
    xs, w = x[ok].astype(np.longdouble), rho[ok].astype(np.longdouble)
    W = w.sum()
    mean = (w[:, None] * xs).sum(0) / W
    d = xs - mean
    s = np.sqrt((w[:, None] * d * d).sum(0))
    rows = np.unique([0, dim // 2, dim - 1])
    M2 = np.stack([((w * d[:, a])[:, None] * d).sum(0) for a in rows])
    scale = np.abs(mean) + s / np.sqrt(W)
    assert abs(out[0] - W) <= 1e-12 * W
    assert np.all(np.abs(out[1:1 + dim] - mean) <= 1e-12 * scale)
    lim = 1e-12 * np.outer(s[rows], s) + 1e-25 * W * np.outer(scale[rows], scale)
    assert np.all(np.abs(out[1 + dim:].reshape(dim, dim)[rows] - M2) <= lim)
