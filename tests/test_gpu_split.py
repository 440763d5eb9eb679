"""Kernels with one wavefront per direction, and the launch order with long lists first.

A small launch of the segmented and direct kernels runs a wavefront per direction; a large
one a wavefront per cell group.  Both take entries in list order and directions in
direction order, so one solve alone (split) equals the same solve among enough copies for
the other form, bit for bit in FP32 and to the last bits in FP64 (1e-15 relative, the
rounding of one sum per direction)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(g, kind, D, k, n, prec, copies, steps=3):
    N = g.get_size(D, k, n) * (2 if kind == "wave" else 1)
    y0 = np.random.default_rng(D * 10 + k).standard_normal(N)
    b = g.Batch(prec)
    for _ in range(copies):
        b.add(kind, D, k, n, y0, 0.02 * 2.0 ** -n, steps, a=[0.3, -0.8, 0.5, 0.1][:D] if kind == "transport" else None)
    b.run()
    out = b.get(0), b.get(copies - 1)
    b.close()
    np.testing.assert_array_equal(out[0], out[1])
    return out[0]


# (D, k, n, copies for more wavefronts than the split form takes)
@pytest.mark.parametrize("D,k,n,copies", [(2, 2, 9, 50), (2, 3, 8, 110), (2, 4, 7, 240), (3, 2, 7, 80), (3, 3, 6, 50),
                                          (3, 4, 5, 125), (4, 2, 6, 45), (4, 3, 5, 31), (4, 4, 5, 8)])
@pytest.mark.parametrize("kind", ["transport", "wave"])
def test_split_equals_whole_fp32(g, gpu, D, k, n, copies, kind):
    print(f"[gpu] split {kind} D={D} k={k} n={n}", flush=True)
    np.testing.assert_array_equal(_solve(g, kind, D, k, n, "fp32", 1), _solve(g, kind, D, k, n, "fp32", copies))


@pytest.mark.parametrize("D,k,n,copies", [(3, 4, 5, 31), (4, 3, 5, 15), (4, 4, 5, 45)])
def test_split_equals_whole_fp64(g, gpu, D, k, n, copies):
    for kind in ("transport", "wave"):
        one, many = _solve(g, kind, D, k, n, "fp64", 1), _solve(g, kind, D, k, n, "fp64", copies)
        assert np.linalg.norm(one - many) <= 1e-15 * np.linalg.norm(many)
