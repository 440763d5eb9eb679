"""The plan kernel with one wavefront per direction (small launches): applications and RK4
against the oracle at the shapes it serves, partial last wavefronts and tiles among them, and
bit for bit against a launch of enough copies to run without the split."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,k,n", [(2, 1, 7), (2, 2, 8), (2, 4, 6), (2, 5, 6), (3, 2, 6), (3, 3, 5), (3, 5, 4), (4, 2, 5),
                                   (4, 5, 2), (5, 2, 4), (5, 3, 2), (6, 2, 3)])
def test_plan_split_oracle(g, O, gpu, D, k, n):
    print(f"[gpu] plan split D={D} k={k} n={n}", flush=True)
    a = [0.7, -0.3, 0.5, 0.2, 0.9, -0.4][:D]
    rng = np.random.default_rng(D + 10 * k)
    for kind in ("transport", "wave", "laplacian"):
        op = (g.transport_matrix(D, k, n, a) if kind == "transport" else g.wave_matrix(D, k, n) if kind == "wave" else
              g.laplacian_matrix(D, k, n))
        x = rng.standard_normal(op.len)
        ref = O.System("wave" if kind == "laplacian" else kind, D, k, n, a=a if kind == "transport" else None)
        if kind == "laplacian":
            yo = ref.rhs(np.concatenate([x, 0 * x]))[op.len:]
        else:
            yo = ref.rhs(x)
        y = op @ x
        assert np.linalg.norm(y - yo) < 1e-12 * np.linalg.norm(yo), kind
        if kind != "laplacian":
            dt = 0.02 * 2.0 ** -n
            yr, ro = op.rk4(x, dt, 3), ref.rk4(x, dt, 3)
            assert np.linalg.norm(yr - ro) < 1e-12 * np.linalg.norm(ro), kind
        op.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("D,k,n,copies", [(2, 5, 6, 90), (3, 5, 4, 45), (4, 5, 2, 60), (5, 2, 4, 60)])
def test_plan_split_equals_whole(g, gpu, D, k, n, copies, prec):
    print(f"[gpu] plan split / whole D={D} k={k} n={n} {prec}", flush=True)
    for kind in ("transport", "wave"):
        y0 = np.random.default_rng(k).standard_normal(g.get_size(D, k, n) * (2 if kind == "wave" else 1))
        out = []
        for m in (1, copies):
            b = g.Batch(prec)
            for _ in range(m):
                b.add(kind, D, k, n, y0, 0.02 * 2.0 ** -n, 3, a=[0.3, -0.8, 0.5, 0.1, 0.6][:D] if kind == "transport" else None)
            b.run()
            out.append(b.get(m - 1))
            b.close()
        np.testing.assert_array_equal(out[0], out[1])
