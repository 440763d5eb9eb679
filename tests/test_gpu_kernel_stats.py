"""A batch's kernel statistics count the unfinished solves of a class, and resident solves in
an entry of their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(g, prec, solves):
    b = g.Batch(prec)
    for kind, D, k, n, steps in solves:
        y0 = np.random.default_rng(n).standard_normal(g.get_size(D, k, n) * (2 if kind == "wave" else 1))
        b.add(kind, D, k, n, y0, 0.02 * 2.0 ** -n, steps, a=[0.3, -0.8, 0.5][:D] if kind == "transport" else None)
    b.profile(True)
    b.run()
    st = {(s["D"], s["k"], s["sys"], s["variant"]): s for s in b.kernel_stats()}
    b.close()
    return st


def test_finished_solves_are_not_counted(g, gpu):
    print("[gpu] statistics of finished solves", flush=True)
    N5, N8 = g.get_size(3, 3, 5), g.get_size(3, 3, 8)
    # no rebuild: the solves that finish hold less than a quarter of the batch
    st = _batch(g, "fp32", [("transport", 3, 3, 8, 10), ("transport", 3, 3, 5, 4), ("transport", 3, 4, 5, 3)])
    # per entry and step: the float input, and the stage's reads and writes
    per = sum(4 + e for e in (8 + 8 + 4, 8 + 16 + 4, 8 + 16 + 4, 8 + 8 + 4))
    a, c = st[(3, 3, 0, 2)], st[(3, 4, 0, 2)]
    assert a["launches"] == 4 * 10 and a["dofs"] == N8
    assert a["algo_bytes"] == per * (10 * N8 + 4 * N5)
    assert c["launches"] == 4 * 3 and c["algo_bytes"] == per * 3 * g.get_size(3, 4, 5)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_resident_solves_have_their_own_entry(g, gpu, prec):
    print(f"[gpu] statistics of resident solves {prec}", flush=True)
    N5, N4 = g.get_size(2, 3, 5), g.get_size(2, 3, 4)
    st = _batch(g, prec, [("transport", 2, 3, 5, 300), ("wave", 2, 3, 4, 300), ("transport", 2, 3, 9, 300)])
    r, w = st[(2, 3, 0, 4)], st[(2, 3, 1, 4)]
    lo = 4 if prec == "fp32" else 0
    assert r["launches"] == 2 and r["dofs"] == N5 and r["algo_bytes"] == N5 * (80 * 300 + 2 * (8 + lo))
    assert w["launches"] == 2 and w["algo_bytes"] == N4 * (160 * 300 + 2 * (16 + 3 * lo))
    staged = [s for key, s in st.items() if key[3] != 4]
    assert len(staged) == 1 and staged[0]["launches"] == 4 * 300 and staged[0]["dofs"] == g.get_size(2, 3, 9)


@pytest.mark.parametrize("when", ["before", "after"])
def test_fused_batches_keep_small_solves_in_the_launch(g, gpu, when):
    """Beside others a small solve runs in the fused launch, resident only alone; a schedule
    set after the first steps counts from then on."""
    print(f"[gpu] fused batch, schedule set {when} the first steps", flush=True)
    for solves, resident in (([(2, 3, 5), (2, 3, 9)], False), ([(2, 3, 5), (2, 3, 4)], True)):
        b = g.Batch("fp32")
        if when == "before":
            b.schedule("fused")
        for D, k, n in solves:
            y0 = np.random.default_rng(n).standard_normal(g.get_size(D, k, n))
            b.add("transport", D, k, n, y0, 0.02 * 2.0 ** -n, 20, a=[0.3, -0.8])
        b.step(4)
        b.schedule("fused")
        b.profile(True)
        b.step(4)
        assert ([s["variant"] for s in b.kernel_stats()] == [4]) == resident
        assert all((s["variant"] == 4) == resident for s in b.kernel_stats())
        b.close()
