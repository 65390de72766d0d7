"""GPU: the 16-bit matrix search against the exact scan and the oracle, at the edges of its own dispatch: dims
either side of each slot and slice limit, rows either side of each tile size, the data's own dimensions and
rotated ones (searches long enough to rotate), and maps that ask for each kind of plan. Winners are equal; the
errors, which also carry the second winner and the distance, agree to the rounding of their sums (1e-12).
"""
import numpy as np
import pytest

import decontamination_amd as dam
from oracle import FP64, REF32, build as build_oracle
from oracle import som_ref as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _setup():
    build_oracle()
    assert dam.gpu_available(), "no GPU visible: the GPU tests must run on an MI355X"


def _case(kind, m, n, dim, N, dtype, seed):
    rng = np.random.default_rng(seed)
    if kind == "noise":
        W = rng.standard_normal((m * n, dim))
    elif kind == "sheet":  # a smooth surface, its modes falling by a decade every few dims
        a, b = np.divmod(np.arange(m * n), n)
        k = np.arange(dim)
        W = np.sin(np.outer(a / m, 1 + k % 3) + k) * np.cos(np.outer(b / n, 1 + k % 2) - k) * 10.0 ** (-k / 6.0)
        W = W @ np.linalg.qr(rng.standard_normal((dim, dim)))[0]
    elif kind == "flat":   # far from the origin, nearly one point
        W = 5.0 + 1e-5 * rng.standard_normal((m * n, dim))
    else:                  # columns of very different sizes
        W = rng.standard_normal((m * n, dim)) * 10.0 ** rng.integers(-6, 7, dim)
    W = W.astype(dtype)
    X = (W[rng.integers(0, m * n, N)] + W.std(0) * 0.3 * rng.standard_normal((N, dim))).astype(dtype)
    if m * n > 2:
        W[m * n // 2] = W[1]  # equal distances: the lower index wins
    X[0] = W[min(1, m * n - 1)]
    if N > 8:
        X[5, 0] = np.nan
        X[6, -1] = np.inf
        X[7] = 1e30
    return W, X


def _check(kind, m, n, dim, N, dtype, arithmetic, seed):
    W, X = _case(kind, m, n, dim, N, dtype, seed)
    som = dam.SOM_Batch(m, n, dim, dtype=dtype, topology="square", precision="exact" if dtype == np.float64 else
                        "bf16_rerank", arithmetic=arithmetic)
    som._weights[...] = W
    got = som.get_winners(X)
    rows = np.unique(np.concatenate([np.arange(min(N, 600)), np.arange(max(0, N - 600), N),
                                     np.arange(0, N, max(1, N // 600))]))
    if dtype == np.float64:
        want = R.find_bmus_f64(W, X[rows])
    else:
        want = R.find_bmus(W, X[rows], FP64 if arithmetic == "fp64" else REF32)
    assert np.array_equal(got[rows], want)
    if dtype == np.float32:
        ref = dam.SOM_Batch(m, n, dim, topology="square", precision="exact", arithmetic=arithmetic)
        ref._weights[...] = W
        assert np.array_equal(got, ref.get_winners(X))
        ok = X[np.all(np.abs(X) < 1e20, axis=1)]
        if len(ok):
            assert np.allclose(som.compute_errors(ok), ref.compute_errors(ok), rtol=1e-12, atol=0.0)


@pytest.mark.parametrize("arithmetic", ["ref32", "fp64"])
@pytest.mark.parametrize("dim", [1, 2, 15, 16, 17, 20, 31, 32, 33, 40, 46, 47, 62, 63, 64])
@pytest.mark.parametrize("kind", ["noise", "sheet", "flat", "scaled"])
def test_search_dims(kind, dim, arithmetic):
    print(f"search {kind} D{dim} {arithmetic}", flush=True)
    _check(kind, 9, 15, dim, 700, np.float32, arithmetic, dim)


@pytest.mark.parametrize("N", [1, 31, 32, 33, 127, 128, 129, 131072, 131073])
@pytest.mark.parametrize("dim", [16, 32, 64])
def test_search_rows(dim, N):
    print(f"search rows {N} D{dim}", flush=True)
    _check("sheet", 11, 12, dim, N, np.float32, "ref32", N % 97)


# (map, dim, rows): at least 2^31, 2^30 and 2^29 (row, neuron) pairs at up to 16, 32 and 64 dims
@pytest.mark.parametrize("shape", [(128, 128, 5, 131072), (100, 100, 16, 214750), (100, 100, 17, 107376),
                                   (64, 64, 32, 262145), (80, 60, 33, 131073), (64, 64, 46, 131100),
                                   (64, 64, 47, 131072), (50, 70, 64, 160001)])
@pytest.mark.parametrize("kind", ["noise", "sheet", "flat", "scaled"])
def test_search_rotated(kind, shape):
    m, n, dim, N = shape
    print(f"search rotated {kind} {m}x{n} D{dim} rows {N}", flush=True)
    _check(kind, m, n, dim, N, np.float32, "fp64", dim)


@pytest.mark.parametrize("shape", [(9, 15, 1, 700), (9, 15, 15, 131073), (9, 15, 17, 129), (9, 15, 40, 128),
                                   (9, 15, 64, 131073), (100, 100, 16, 214750), (64, 64, 30, 262145),
                                   (64, 64, 63, 131073)])
@pytest.mark.parametrize("kind", ["noise", "sheet", "flat", "scaled"])
def test_search_float64(kind, shape):
    m, n, dim, N = shape
    print(f"search float64 {kind} {m}x{n} D{dim} rows {N}", flush=True)
    _check(kind, m, n, dim, N, np.float64, "fp64", dim)


def test_search_after_fp32_search():
    """The FP32 search of a prepared map leaves the plan of the 16-bit search alone."""
    W, X = _case("sheet", 20, 20, 12, 900, np.float32, 3)
    som = dam.SOM_Batch(20, 20, 12, topology="square")
    som._weights[...] = W
    first = som.get_winners(X)
    som._precision = "fp32"
    som.get_winners(X)
    som._precision = "bf16_rerank"
    assert np.array_equal(som.get_winners(X), first)
    assert np.array_equal(first, R.find_bmus(W, X, REF32))
