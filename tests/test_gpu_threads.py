"""Simulators in several threads, each on a stream of its own, on one device: they
share the device's context and its program slots.  The same states as one after
another."""
import threading

import pytest

from quict_amd import workloads

pytestmark = pytest.mark.gpu


def test_runs_in_several_threads():
    print("[case] threads", flush=True)
    import torch
    from quict_amd.simulation import StateVectorSimulator
    sizes = [(5, 60), (8, 200), (11, 90), (14, 150)]
    circuits = [workloads.random_mix_circuit(n, g, n) for n, g in sizes]
    want = [StateVectorSimulator("GPU").run(c).tensor.clone() for c in circuits]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                sim = StateVectorSimulator("GPU", sync=False)
                for k in range(60):
                    out = sim.run(circuits[i]).tensor
                    torch.cuda.current_stream().synchronize()
                    if not torch.equal(out, want[i]):
                        wrong.append((i, k))
        except Exception as e:  # (reported by the assertion below)
            wrong.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
