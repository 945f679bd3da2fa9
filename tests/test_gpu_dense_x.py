"""GPU test of the advection products on the x grids that the dense x-transforms keep (16, 32 or 48 modes and
mgalx = 112 or 176, with a factor past 5) and on the smallest grids of 16 modes, which k_xprod_fft takes: against
the oracle's FFT route.

Bar: the dense sums of mgalx terms round at ~eps sqrt(mgalx), the derivative products at ~eps m, both relative to
random fields whose results do not cancel: 1e-13 of each component's maximum.
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


@pytest.mark.parametrize("m,M,mgalx", [(9, 16, 112), (17, 32, 112), (33, 16, 176), (40, 48, 176), (65, 32, 176),
                                       (9, 16, 48), (33, 16, 48), (97, 16, 48), (33, 16, 64)])
def test_advection_products(dev, m, M, mgalx):
    import torch
    from duct_amd import step
    from oracle import spectral
    dev.setup(m)
    rng = np.random.default_rng(1000 * m + mgalx)
    fields = [rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m)) for _ in range(3)]
    u = [torch.from_numpy(f).cuda() for f in fields]
    adv = [torch.full_like(u[0], float("nan")) for _ in range(3)]
    step.advection(*u, *adv, mgalx=mgalx, alp=0.9)
    torch.cuda.synchronize()
    ref = spectral.advection3d(*fields, mgalx=mgalx, alp=0.9)
    for c in range(3):
        e = float(np.max(np.abs(adv[c].cpu().numpy() - ref[c])) / np.max(np.abs(ref[c])))
        print("m=%d M=%d mgalx=%d adv%d rel.err %.2e" % (m, M, mgalx, c + 1, e), flush=True)
        assert e <= 1e-13
