"""GPU test of right-hand sides that overlap each other: by other than whole planes, where zeroing the walls of the
one (helm3d.f90:48-60) touches the other's interior and the solves keep the passes, and by whole planes or wholly.

Reference: the same solves on right-hand sides that do not overlap, each alone.  Bar: the solve's, 1e-12.
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


@pytest.mark.parametrize("m", [18, 67, 129])
@pytest.mark.parametrize("shift", ["point", "line", "planes", "none"])
@pytest.mark.parametrize("swap", [False, True])
def test_overlapping_right_hand_sides(dev, m, shift, swap):
    import torch
    from duct_amd import solver
    M, n = 5, 5 * m * m
    off = {"point": 1, "line": 3 * m + 7, "planes": 2 * m * m, "none": 0}[shift]
    dev.setup(m)
    rng = np.random.default_rng(m + off)
    host = rng.standard_normal(n + off) + 1j * rng.standard_normal(n + off)
    buf = torch.from_numpy(host).cuda()
    rhs = [buf[k:k + n].view(M, m, m) for k in ((off, 0) if swap else (0, off))]
    alone = [r.clone() for r in rhs]
    sol, ref = ([torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in rhs] for _ in "ab")
    with solver.KernelTimer() as t:
        dev.helm3d_batch(rhs, sol, "dd", [700.0, 3.0], alp=0.9, ib=2)
        torch.cuda.synchronize()
    assert (t.count["plane"] > 0) == (shift in ("planes", "none"))
    for k in range(2):
        dev.helm3d_batch([alone[k]], [ref[k]], "d", [[700.0, 3.0][k]], alp=0.9, ib=2)
    torch.cuda.synchronize()
    for k in range(2):
        e = float((sol[k] - ref[k]).abs().max() / ref[k].abs().max())
        print("m=%d %s field %d rel.err %.2e" % (m, shift, k, e), flush=True)
        assert e <= 1e-12
