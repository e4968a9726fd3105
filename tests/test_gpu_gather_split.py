"""The gather's wide products on both sides of the line between workgroups of
256 and of 384 rows (192 columns: 8,192 padded patches), against FP64 on a
sample of rows.  Tolerances are those of the stored formats: BF16 products
within 2^-7 of sum |M||x| per element, refined ones within 1e-4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [7681, 8192, 8193])
def test_wide_products_either_side_of_one_round(rad, n):
    R = 192
    rng = np.random.default_rng(n)
    tri = rng.uniform(-1, 1, (n, 3, 3)).astype(np.float32)
    nrm = np.tile(np.float32([0, 0, 1]), (n, 1))
    up = np.tile(np.float32([0, 1, 0]), (n, 1))
    one = np.ones((n, 3), np.float32)
    sc = rad.Scene(tri, np.arange(n), np.concatenate([tri.mean(1), nrm, up], 1), 0.5 * one,
                   np.ones(n), one, 0 * one)
    M = rng.random((n, n), np.float32) / np.float32(n)
    x = rng.uniform(-1.0, 2.0, (R, n)).astype(np.float32)
    print(f"wide products: {n} patches", flush=True)
    s = rad.Solver(hemicube=16, hemicubes=1)
    s.upload(sc)
    s.dense_upload(M)
    # both ends, every workgroup's first and last row, and others
    idx = np.unique(np.concatenate([np.arange(0, n, 128), np.arange(127, n, 128),
                                    np.arange(n - 40, n), rng.integers(0, n, 100)]))
    Ms = M[idx].astype(np.float64)
    want = x.astype(np.float64) @ Ms.T
    mag = np.abs(x).astype(np.float64) @ np.abs(Ms).T
    y = s.dense_apply(x, split=False)[:, idx]
    assert np.max(np.abs(y - want) / mag) < 2.0 ** -7
    y2 = s.dense_apply(x, split=True)[:, idx]
    assert np.max(np.abs(y2 - want) / mag) < 1e-4
