"""Transform sweeps at their edges against the assembled matrix (transform_csc, host): k^D a
power of two and not (the index arithmetic), k^D just below, at and above the 128 that still
gives a long-list cell a workgroup, lists of at most 8, just above and of many entries, a last
workgroup with few DoFs, and grids of less than one workgroup.

Tolerance: a sweep's row is a sum of at most n 2^n k products, each rounded; D sweeps of the
1-D matrices' conditioning (below 1e2 here) leave less than 1e-12 relative L2."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, 0), (1, 5, 7), (2, 2, 9), (2, 3, 7), (2, 5, 4), (3, 3, 5), (3, 5, 4), (4, 3, 4), (5, 2, 4), (5, 3, 3),
          (7, 2, 4), (8, 2, 1)]


@pytest.mark.parametrize("D,k,n", SHAPES)
def test_sweeps_match_the_assembled_matrix(g, gpu, D, k, n):
    x = np.random.default_rng([D, k, n]).standard_normal(g.get_size(D, k, n))
    for a, b in [("modal", "nodal"), ("nodal", "points"), ("points", "nodal"), ("nodal", "modal")]:
        print(f"[gpu] sweeps D={D} k={k} n={n} {a} -> {b}", flush=True)
        op = g.transform(D, k, n, a, b)
        assert rel(op @ x, g.transform_csc(D, k, n, a, b) @ x) < 1e-12, (a, b)
        op.close()
