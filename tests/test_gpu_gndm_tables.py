"""GPU: the number density maps at the edges of their LDS tables (maps of 1, 31, 33, 13,653 neurons, the most that fit, and
13,654), of the unrolled steps and the workgroups' ranges, with winners out of range and densities that are left out.
Whole counts are exact; densities are multiples of 1/8, so their sums are too."""
import numpy as np
import pytest

import decontamination_amd as dam
from decontamination_amd import _lib
from decontamination_amd.runtime import DeviceArray, get_context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2047, 2049, 8192, 8193, 300_001])
@pytest.mark.parametrize("mn", [1, 31, 33, 13_653, 13_654])
def test_gndm_tables(mn, N):
    assert dam.gpu_available(), "no GPU visible: the GPU tests must run on an MI355X"
    print(f"gndm {mn} neurons {N} rows", flush=True)
    rng = np.random.default_rng(mn + N)
    w = rng.integers(-1, mn + 1, N).astype(np.int32)
    rho = rng.integers(-2, 40, N) / 8.0
    rho[::17], rho[1::19], rho[2::23] = np.nan, np.inf, 0.0
    ctx = get_context(0)
    dw, dr = DeviceArray.from_host(ctx, w), DeviceArray.from_host(ctx, rho)
    maps, out = DeviceArray.empty(ctx, (3, mn), np.float32), DeviceArray.empty(ctx, (N,), np.float32)
    _lib.call("somhip_gndm", ctx.handle, _lib.vp(dw.ptr), _lib.vp(dr.ptr), N, mn, _lib.vp(maps.view_ptr(0)),
              _lib.vp(maps.view_ptr(mn)), _lib.vp(maps.view_ptr(2 * mn)), _lib.vp(out.ptr))
    cat, foot, gnd = maps.copy_to_host()
    inside = (w >= 0) & (w < mn)
    use = inside & np.isfinite(rho) & (rho > 0.0)
    want_cat = np.bincount(w[use], weights=rho[use], minlength=mn).astype(np.float32)
    want_foot = np.bincount(w[inside], minlength=mn).astype(np.float32)
    with np.errstate(divide="ignore", invalid="ignore"):
        want = np.where(want_foot > 0.0, want_cat / want_foot, np.float32(np.nan)).astype(np.float32)
    assert np.array_equal(cat, want_cat) and np.array_equal(foot, want_foot)
    assert np.array_equal(gnd, want, equal_nan=True)
    assert np.array_equal(out.copy_to_host(), np.where(inside, want[np.clip(w, 0, mn - 1)], np.float32(np.nan)), equal_nan=True)
