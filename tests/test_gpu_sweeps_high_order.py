"""Transform sweeps on cells of many values (k^D up to 390,625) against the 1-D transform
applied along each axis on the host.

n = 0: one cell, and a sparse grid that is the full tensor product.  Tolerance: D sweeps of
k-term rows whose 1-D matrices are conditioned below 1e2 leave less than 1e-12 relative L2."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,k", [(8, 5), (7, 5), (6, 5), (8, 3), (8, 2)])
def test_one_cell_matches_the_axes(g, gpu, D, k):
    x = np.random.default_rng([D, k]).standard_normal(k ** D)
    for a, b in [("modal", "nodal"), ("nodal", "points"), ("points", "nodal"), ("nodal", "modal")]:
        print(f"[gpu] sweeps of one cell D={D} k={k} {a} -> {b}", flush=True)
        T = g.transform_1D(k, 0, a, b).toarray()
        y = x.reshape((k,) * D)
        for d in range(D):
            y = np.moveaxis(np.tensordot(T, y, axes=(1, d)), 0, d)
        op = g.transform(D, k, 0, a, b)
        assert rel(op @ x, y.ravel()) < 1e-12, (a, b)
        op.close()
