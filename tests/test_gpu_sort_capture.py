"""Stand-alone sorts recorded into a graph: refused while the engine has no workspace (its clear would be
recorded, not run), and right at every replay once it has, with other sorts between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_sort_in_a_graph():
    import torch
    from torpedo_amd._capi import TpdError
    from torpedo_amd.engine import GaussianEngine, sort_pairs_device
    n, bits, side = 5_000, 43, torch.cuda.Stream()
    rng = np.random.default_rng(1)
    src = torch.zeros(n, dtype=torch.int64, device="cuda")
    vals = torch.arange(n, dtype=torch.int32, device="cuda")
    bufs = [torch.empty_like(src), torch.empty_like(vals), torch.empty_like(src), torch.empty_like(vals)]
    torch.cuda.synchronize()

    def sort():
        with torch.cuda.stream(side):
            bufs[0].copy_(src)
            bufs[1].copy_(vals)
            return sort_pairs_device(eng, *(t.data_ptr() for t in bufs), n, bits, side.cuda_stream)

    def check(run):
        keys = rng.integers(0, 2 ** bits, n, dtype=np.uint64)
        src.copy_(torch.from_numpy(keys.view(np.int64)))
        torch.cuda.synchronize()
        alt = run()
        torch.cuda.synchronize()
        order = np.argsort(keys, kind="stable")
        assert np.array_equal(bufs[2 if alt else 0].cpu().numpy().view(np.uint64), keys[order])
        assert np.array_equal(bufs[3 if alt else 1].cpu().numpy(), order)

    with GaussianEngine() as eng:
        with pytest.raises(TpdError, match="before a capture"):
            with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=side, capture_error_mode="relaxed"):
                sort()
        check(sort)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            recorded = sort()

        def replay():
            graph.replay()
            return recorded
        for _ in range(4):
            check(replay)
            check(sort)
