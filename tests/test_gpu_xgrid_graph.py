"""GPU test of the x grids' tables (the roots of unity of k_xprod_fft, the dense DFT matrices): an advection
term captured into a graph on one grid replays to the eager result's bits after calls on other grids, between
which tensors of the tables' size are allocated; and calls that alternate between grids give what each gives alone.
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


# mgalx 48 ... 162: factors 2, 3 and 5; 112 = 16 * 7: the dense transforms
@pytest.mark.parametrize("mgalx", [48, 96, 112, 150])
def test_graph_of_one_grid_outlives_calls_on_others(dev, mgalx):
    import torch
    from duct_amd import step
    m, M = 17, 16
    dev.setup(m)
    rng = np.random.default_rng(mgalx)
    u = [torch.from_numpy(rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m))).cuda() for _ in range(3)]

    def adv(X, out):
        step.advection(*u, *out, mgalx=X, alp=0.9)

    new = lambda: [torch.full_like(u[0], float("nan")) for _ in range(3)]
    eager = new()
    adv(mgalx, eager)
    torch.cuda.synchronize()
    out = new()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        adv(mgalx, out)
    torch.cuda.synchronize()
    others = [X for X in (48, 96, 112, 150, 162) if X != mgalx]
    for rep in range(3):
        between = {X: new() for X in others}
        for X in others:
            adv(X, between[X])
        junk = [torch.full((2, X), float("nan"), dtype=torch.float64, device="cuda") for X in (mgalx,) * 8]
        for x in out:
            x.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        print("mgalx=%d replay %d" % (mgalx, rep), flush=True)
        assert all(torch.equal(a, b) for a, b in zip(out, eager))
        for X in others:           # 3 M <= X: every grid dealiases the same products
            for a, b in zip(between[X], eager):
                assert float((a - b).abs().max() / b.abs().max()) <= 1e-13
        del junk
    del g
