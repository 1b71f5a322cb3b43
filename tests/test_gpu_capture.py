"""Passes captured into a graph: a first forward pass, which goes without
segment lists, and later ones, which keep them; every replay against the eager
pass, with eager work and synchronisation between the replays."""
import numpy as np
import pytest

from test_gpu_rows import CASES, CASES_R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("mode", ["R", "A"])
@pytest.mark.parametrize("name", ["faces", "wide"])
@pytest.mark.parametrize("warm", [False, True])
def test_forward_pass_in_a_graph(name, mode, warm):
    import kevernals_amd as K

    mode = {"R": K.MODE_R, "A": K.MODE_A}[mode]
    g = (CASES.get(name) or CASES_R[name])()
    rng = np.random.Generator(np.random.PCG64(43))
    vol = torch.from_numpy(rng.random(g.vol_shape, dtype=np.float32)).cuda()
    out = torch.zeros(g.proj_shape, device="cuda")
    ctx = K.Context(0, g)
    if warm:
        ctx.forward_project(vol, out, mode)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.forward_project(vol, out, mode)
    other = K.Context(0, g)
    for k in range(3):
        vol.add_(0.125)
        want = torch.empty_like(out)
        other.forward_project(vol, want, mode)
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), want.cpu().numpy(), err_msg=f"replay {k}")
    # the context's eager passes build the lists, the graph's go on as they are
    eager = torch.empty_like(out)
    ctx.forward_project(vol, eager, mode)
    out.fill_(float("nan"))
    graph.replay()
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), eager.cpu().numpy())
