"""Which kernel runs: one that gsg_tune_set asks for runs in every launch, a tuned entry in the
launches that fill the chip, and the tuner times launches of the kernels it names."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

PLAN, TILE = 1, 2


def _run(g, D, k, n, prec, copies=1, steps=3):
    """The final state, and (variant, launches) of the class's statistics."""
    y0 = np.random.default_rng([D, k, n]).standard_normal(g.get_size(D, k, n))
    b = g.Batch(prec)
    for _ in range(copies):
        b.add("transport", D, k, n, y0, 0.02 * 2.0 ** -n, steps, a=[0.3, -0.8, 0.5, 0.1, 0.6, -0.2][:D])
    b.profile(True)
    b.run()
    stats = [(s["variant"], s["launches"]) for s in b.kernel_stats()]
    y = b.get(copies - 1)
    b.close()
    return y, stats


# FP64 grids of the LDS fiber kernel: small ones that would run resident, and ones past the
# rule's dimensions
@pytest.mark.parametrize("D,k,n", [(1, 5, 8), (2, 3, 5), (2, 3, 8), (2, 5, 6), (3, 3, 5), (3, 5, 3), (5, 2, 4)])
def test_a_kernel_asked_for_runs(g, O, gpu, D, k, n):
    from galerkinsparsegrids_jl_amd import tune
    print(f"[gpu] asked D={D} k={k} n={n}", flush=True)
    got = {}
    try:
        for v, code in (("plan", PLAN), ("tile", TILE)):
            tune.set_variant(D, k, n, "fp64", v)
            got[v], stats = _run(g, D, k, n, "fp64")
            assert stats == [(code, 4 * 3)], v  # a launch a stage
    finally:
        tune.set_variant(D, k, n, "fp64", "auto")
    ref = O.System("transport", D, k, n, a=[0.3, -0.8, 0.5, 0.1, 0.6, -0.2][:D])
    y0 = np.random.default_rng([D, k, n]).standard_normal(g.get_size(D, k, n))
    yo = ref.rk4(y0, 0.02 * 2.0 ** -n, 3)
    assert rel(got["plan"], yo) < 1e-12 and rel(got["tile"], yo) < 1e-12


def test_a_tuned_entry_goes_by_size(g, gpu):
    from galerkinsparsegrids_jl_amd import tune
    from galerkinsparsegrids_jl_amd._lib import check, lib
    D, k, n = 2, 5, 8  # 32 K coefficients: 500 wavefronts, past the rule's n
    try:
        for v, one, many in (("tile", PLAN, TILE), ("auto", PLAN, PLAN), ("plan", PLAN, PLAN)):
            print(f"[gpu] tuned {v}", flush=True)
            check(lib().gsg_tune_set(D, k, n, 0, tune.VARIANT[v] | tune.TUNED))
            assert _run(g, D, k, n, "fp64")[1] == [(one, 12)]
            assert _run(g, D, k, n, "fp64", copies=40)[1] == [(many, 12)]
    finally:
        tune.set_variant(D, k, n, "fp64", "auto")


def test_tuner_times_stage_launches(g, gpu, tmp_path):
    """A grid small enough to run resident: the tuner's times are of a stage launch of each
    kernel, and its choice leaves the grid's solves resident."""
    from galerkinsparsegrids_jl_amd import tune
    print("[gpu] tuner on a small grid", flush=True)
    D, k, n = 2, 3, 4
    try:
        rows = tune.autotune([(D, k, n)], ("fp64",), steps=3, min_dofs=500_000, path=tmp_path / "t.txt")
        assert set(rows[0]) >= {"plan_ms", "tile_ms"} and rows[0]["variant"] in ("plan", "tile")
        assert tune.read_table(tmp_path / "t.txt") == {(D, k, n, "fp64"): rows[0]["variant"]}
        assert [launches for _, launches in _run(g, D, k, n, "fp64")[1]] == [1]  # all steps in one
        assert tune.get_variant(D, k, n, "fp64") == rows[0]["variant"]
    finally:
        tune.set_variant(D, k, n, "fp64", "auto")
