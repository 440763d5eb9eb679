"""Single applications run on the caller's stream: the handle's scratch is ordered over
streams, host calls follow device calls, and a call can be captured into a graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _late(torch, x):
    """x, written by a kernel that ends milliseconds after this call returns."""
    a = torch.randn(3000, 3000, device=x.device)
    for _ in range(20):
        a = a @ a * 1e-3
    return x + 0.0 * a[0, 0].double().nan_to_num()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_calls_on_two_streams_share_scratch(g, gpu, precision):
    import torch
    print(f"[gpu] two streams {precision}", flush=True)
    op = g.laplacian_matrix(3, 3, 5, precision=precision)
    xs = [np.random.default_rng(i).standard_normal(op.len) for i in range(4)]
    ref = [op @ x for x in xs]
    base = [torch.tensor(x, device=gpu) for x in xs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    out = []
    for i in range(4):  # the second stream's call is enqueued while the first's input is still being written
        with torch.cuda.stream(streams[i % 2]):
            out.append(op @ (_late(torch, base[i]) if i % 2 == 0 else base[i]))
    host = op @ xs[3]  # after the device calls, whose scratch it reuses
    torch.cuda.synchronize()
    for y, r in zip(out, ref):
        np.testing.assert_array_equal(y.cpu().numpy(), r)
    np.testing.assert_array_equal(host, ref[3])
    op.close()


@pytest.mark.parametrize("kind", ["transport", "laplacian"])
def test_apply_captured_into_a_graph(g, gpu, kind):
    import torch
    print(f"[gpu] captured {kind}", flush=True)
    op = g.transport_matrix(2, 3, 5, [1.0, 0.5], precision="fp32") if kind == "transport" else g.laplacian_matrix(3, 3, 4)
    x = torch.zeros(op.len, dtype=torch.float64, device=gpu)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        op @ x
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        y = op @ x
    for i in range(4):
        v = np.random.default_rng(i).standard_normal(op.len)
        eager = op @ torch.tensor(v, device=gpu)  # an uncaptured call between the replays
        x.copy_(torch.tensor(v, device=gpu))
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(y.cpu().numpy(), eager.cpu().numpy())
    op.close()
