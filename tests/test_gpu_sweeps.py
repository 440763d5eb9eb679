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


@pytest.mark.parametrize("Dx,k,n,prec", [(1, 2, 9, "fp32"), (1, 5, 5, "fp64"), (2, 2, 3, "fp32"), (2, 2, 9, "fp32"),
                                         (2, 2, 9, "fp64"), (2, 3, 5, "fp32"), (2, 3, 6, "fp64"), (2, 5, 2, "fp64"),
                                         (3, 2, 5, "fp32")])
def test_without_a_force_only_space_is_differentiated(g, gpu, Dx, k, n, prec):
    """The velocity derivatives are left out exactly where a zero force multiplies them."""
    print(f"[gpu] vlasov Dx={Dx} k={k} n={n} {prec}", flush=True)
    N = g.get_size(2 * Dx, k, n)
    x = np.random.default_rng([Dx, k, n]).standard_normal(N)
    free, zero = (g.vlasov_operator(Dx, k, n, F, precision=prec) for F in (None, [np.zeros(N)] * Dx))
    np.testing.assert_array_equal(free @ x, zero @ x)
