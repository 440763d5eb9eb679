"""Imported sparse matrices: row blocks at their edges (empty rows, a block of exactly the
entries or rows that fit, one more, rows longer than a block) against scipy's product.

FP64: a row is one chain of fused multiply-adds, n eps relative to sum |v x| for rows of n
entries.  FP32: x is rounded to float and the products are summed in float, (n + 1) 2^-24."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _matrix(lens, m, seed):
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i, n in enumerate(lens):
        rows += [i] * n
        cols += list(np.sort(rng.choice(m, n, replace=False)))
    return sp.csc_matrix((rng.standard_normal(len(rows)), (rows, cols)), shape=(m, m))


SHAPES = {
    "one_by_one": [1],
    "empty": [0] * 5,
    "empty_rows": [0, 3, 0, 0, 7] + [0] * 300 + [2],
    "rows_256_and_257": [1] * 257,
    "entries_1024_exact": [512, 512, 1, 1023, 1],
    "entries_1025": [512, 513, 1024, 1],
    "long_rows": [3, 1025, 2, 2500, 4096, 5],
    "ragged": list(np.random.default_rng(3).integers(0, 120, 700)),
}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_csr_row_blocks(g, gpu, shape, prec):
    lens = SHAPES[shape]
    m = max(len(lens), max(lens), 1)
    lens = list(lens) + [0] * (m - len(lens))
    print(f"[gpu] csr {shape} {prec}", flush=True)
    A = _matrix(lens, m, 1)
    x = np.random.default_rng(2).standard_normal(m)
    op = g.csc_matrix(A, precision=prec)
    y = op @ x
    op.close()
    scale = abs(A) @ abs(x)
    eps = (np.array(lens) + 1) * (2.0 ** -52 if prec == "fp64" else 2.0 ** -23)
    assert np.all(np.abs(y - A @ x) <= eps * scale)
