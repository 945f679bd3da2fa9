"""HIP graph capture of the batched solve at sizes that solve in passes, with folding off (unfolded passes) and on
(folded ones, the Neumann group's low modes in passes of their own), with and without the second stream: every
replay equals the eager solve to the bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    import duct_amd
    torch.cuda.set_device(0)
    duct_amd.init(0)
    yield duct_amd
    duct_amd.shutdown()


@pytest.mark.parametrize("m,M,bounds,kind,overlap", [
    (200, 10, "dddn", "plain", True), (200, 10, "dddn", "plain", False), (200, 10, "dddn", "fold", True),
    (200, 10, "dddn", "fold", False), (130, 12, "d", "fold", True)])
def test_passes_replay_in_a_graph(dev, m, M, bounds, kind, overlap):
    import torch
    from duct_amd import solver
    dev.setup(m)
    rng = np.random.default_rng(m + M)
    f = [torch.from_numpy(rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m))).cuda() for _ in bounds]
    alams = [1000.0 if b == "d" else 0.0 for b in bounds]

    def solve(sol):
        dev.helm3d_batch(f, sol, bounds, alams)

    print("graph capture m=%d M=%d %s %s overlap=%d" % (m, M, bounds, kind, overlap), flush=True)
    try:
        dev.set_fold(2 if kind == "fold" else 0)
        dev.set_overlap(overlap)
        eager = [torch.zeros_like(x) for x in f]
        with solver.KernelTimer() as t:
            solve(eager)
            torch.cuda.synchronize()
        assert t.count[{"plain": "proj_c2p", "fold": "fold_c2p"}[kind]] > 0 and t.count["plane"] == 0
        solve(eager)                                   # warmup: sizes the buffers, with the second stream's
        torch.cuda.synchronize()
        sol = [torch.zeros_like(x) for x in f]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            solve(sol)
        torch.cuda.synchronize()
        for rep in range(3):
            for x in sol:
                x.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            for a, b in zip(sol, eager):
                assert torch.equal(a, b), rep
            scratch = [torch.zeros_like(x) for x in f]  # eager work between the replays
            solve(scratch)
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(scratch, eager))
        del g
    finally:
        dev.set_fold(0)
        dev.set_overlap(True)
