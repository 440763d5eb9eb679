"""Imported sparse matrices of about one entry a row run a thread a row: the edges of that
rule (1.5 entries a row on average, 8 in the longest) against scipy's product.

Bounds as for the row blocks: n eps (FP64), (n + 1) 2^-24 (FP32) of sum |v x| for n entries."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

SHAPES = {
    "empty": [0] * 300,
    "diagonal_256": [1] * 256,
    "diagonal_257": [1] * 257,
    "mean_at_the_line": [1, 2] * 300,
    "mean_above": [1, 2] * 300 + [2],
    "longest_8": [8] + [0, 1] * 200,
    "longest_9": [9] + [0, 1] * 200,
}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_short_rows(g, gpu, shape, prec):
    lens = SHAPES[shape]
    m = len(lens)
    print(f"[gpu] csr short rows {shape} {prec}", flush=True)
    rng = np.random.default_rng(1)
    rows = np.repeat(np.arange(m), lens)
    cols = np.concatenate([np.sort(rng.choice(m, n, replace=False)) for n in lens]) if len(rows) else rows
    A = sp.csc_matrix((rng.standard_normal(len(rows)), (rows, cols)), shape=(m, m))
    x = rng.standard_normal(m)
    op = g.csc_matrix(A, precision=prec)
    y = op @ x
    op.close()
    eps = (np.array(lens) + 1) * (2.0 ** -52 if prec == "fp64" else 2.0 ** -23)
    assert np.all(np.abs(y - A @ x) <= eps * (abs(A) @ abs(x)))
