"""Runs on registers of at most a tile inside a graph that the caller captures
(torch.cuda.graph): a kernel a gate.  Replayed several times with eager runs between,
whose programs use the same staging memory."""
import pytest

from quict_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 12])
@pytest.mark.parametrize("precision", ["double", "single"])
def test_small_runs_in_a_captured_graph(n, precision):
    print("[case] caller's graph", n, precision, flush=True)
    import torch
    from quict_amd.simulation import StateVectorSimulator
    c = workloads.random_mix_circuit(n, 40, 3)
    if precision == "single":
        c.convert_precision()
    other = workloads.random_mix_circuit(n, 90, 4)
    eager = StateVectorSimulator("GPU", precision=precision, fusion=False).run(c).tensor.clone()
    busy = StateVectorSimulator("GPU")
    sim = StateVectorSimulator("GPU", precision=precision, sync=False)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        sim.run(c)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = sim.run(c).tensor
    for _ in range(4):
        busy.run(other)
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
