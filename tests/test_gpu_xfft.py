"""GPU tests of the advection products on x grids of factors 2, 3 and 5 (k_xprod_fft), against the
oracle's FFT route: every fused radix (4, 6, 10) with and without further passes of each radix
(2, 3, 4, 5, 8), few and many modes for the grid, one to three waves and more than 256 threads per
workgroup, and line counts that leave the last tile of 2, 4 or 8 lines ragged.

Bar: the transforms round at ~eps log2(X) <= 2.5e-15 and the derivative products at ~eps m, both
relative to random fields whose results do not cancel: 1e-13 of each component's maximum.
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


@pytest.mark.parametrize("m,M,mgalx", [
    (9, 1, 4), (9, 2, 6), (9, 3, 10), (9, 2, 8), (9, 4, 12), (9, 6, 18), (9, 6, 20), (17, 5, 16), (17, 8, 24),
    (17, 3, 32), (9, 16, 50), (9, 21, 64), (65, 10, 30), (17, 42, 128), (9, 40, 120), (9, 54, 162), (9, 80, 250),
    (9, 85, 256), (9, 64, 384), (6, 100, 300), (6, 170, 512), (9, 240, 720), (6, 256, 768), (6, 300, 900),
    (6, 333, 1000), (6, 512, 1536), (5, 600, 2048)])
def test_advection_on_smooth_x_grids(dev, m, M, mgalx):
    import torch
    from duct_amd import step
    from oracle import spectral
    dev.setup(m)
    rng = np.random.default_rng(1000 * m + mgalx)
    fields = [rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m)) for _ in range(3)]
    u = [torch.from_numpy(f).cuda() for f in fields]
    adv = [torch.zeros_like(u[0]) for _ in range(3)]
    step.advection(*u, *adv, mgalx=mgalx, alp=0.9)
    torch.cuda.synchronize()
    ref = spectral.advection3d(*fields, mgalx=mgalx, alp=0.9)
    for c in range(3):
        got = adv[c].cpu().numpy()
        e = float(np.max(np.abs(got - ref[c])) / np.max(np.abs(ref[c])))
        print("m=%d M=%d mgalx=%d adv%d rel.err %.2e" % (m, M, mgalx, c + 1, e), flush=True)
        assert e <= 1e-13
