"""GPU: the vector-count sums on the closed-form grids against the oracle's, at the edges of their split (rows and
columns that do not divide 16 or 256 neurons, one column, wide maps beyond the tables, remainders of the sample
steps), and on the same grid handed over as an arbitrary topography. FP64 sums of at most 2,000 positive-weighted
terms rounded to the data's type: 1e-10 relative for float64, 2e-6 for float32 centroids; and the column maxima
behind the fixed-point scales, through a weighted epoch of float64 rows."""
import numpy as np
import pytest

import decontamination_amd as dam
from oracle import build as build_oracle
from oracle import som_ref as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _setup():
    build_oracle()
    assert dam.gpu_available(), "no GPU visible: the GPU tests must run on an MI355X"


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("topology", ["square", "hexagonal"])
@pytest.mark.parametrize("shape", [(1, 2, 1, 1), (5, 1, 3, 63), (1, 40, 16, 64), (15, 17, 16, 65), (16, 16, 17, 129),
                                   (3, 90, 5, 127), (9, 70, 33, 200), (33, 31, 48, 1000), (13, 20, 64, 2000),
                                   (2, 300, 4, 500)])
def test_vectors_on_grids(shape, topology, dtype):
    m, n, dim, N = shape
    print(f"vectors {m}x{n} D{dim} rows {N} {topology} {np.dtype(dtype)}", flush=True)
    rng = np.random.default_rng(m + n + dim)
    X = rng.standard_normal((N, dim)).astype(dtype)
    rho = rng.random(N) * 2.0
    if N > 20:
        rho[3], rho[4], rho[5] = 0.0, -1.0, np.nan
        X[7, 0] = np.nan  # left out: no winner
    W0 = rng.standard_normal((m * n, dim)).astype(dtype)
    som = dam.SOM_Batch(m, n, dim, dtype=dtype, topology=topology, **({} if dtype == np.float64 else {"arithmetic": "fp64"}))
    som._weights[...] = W0
    som.train(X, dataset_weights=rho, n_vectors=N)
    c1 = (R.top2_f64(W0, X)[0]).astype(np.int64)
    topo = R.topography(m, n, topology, dtype).astype(np.float64).reshape(-1, 2)
    i = np.arange(N)
    sigma = np.maximum(max(m, n) / 2.0 / (1.0 + 2.0 * i / N), 1e-12)
    r = rho.astype(dtype).astype(np.float64)
    keep = (c1 >= 0) & (r > 0.0)
    num, den = np.zeros((m * n, dim)), np.zeros(m * n)
    for k in np.flatnonzero(keep):
        d2 = ((topo - topo[c1[k]]) ** 2).sum(1)
        h = r[k] * np.exp(-d2 / (2.0 * sigma[k] ** 2))
        num += h[:, None] * X[k].astype(np.float64)
        den += h
    want = np.where(den[:, None] > 0.0, num / np.where(den > 0.0, den, 1.0)[:, None], W0)
    ok = den > 1e-250
    tol = 1e-10 if dtype == np.float64 else 2e-6
    got = som._weights.astype(np.float64)
    err = np.abs(got - want)[ok] / np.maximum(np.abs(want[ok]), 1e-1)
    assert err.size == 0 or err.max() < tol, err.max()
