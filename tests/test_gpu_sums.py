"""GPU tests of the derivative sums along both directions in one launch (k_sums) at the edges of its tiles
and of its range: planes of one to four tiles with remainders 0, 1 and 15, odd mode counts, the largest
batches that it takes and the first that it leaves to the y and z launches, aspect ratios other than 1.

References: the oracle's advection and substep.  Bars: those of the advection (1e-12: sums of m <= 64
terms round to a few eps of their magnitudes) and of the substep (1e-10, the pressure Poisson solve).
"""
import numpy as np
import pytest

from test_gpu_rk3 import initial_state, oracle_helm, relerr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    import duct_amd
    torch.cuda.set_device(0)
    duct_amd.init(0)
    yield duct_amd
    duct_amd.shutdown()


@pytest.mark.parametrize("m,M,aspect", [(4, 3, 1.0), (15, 5, 2.0), (16, 16, 1.0), (17, 9, 0.5), (31, 16, 1.0), (32, 7, 1.5),
                                        (33, 3, 1.0), (47, 16, 1.0), (48, 5, 0.8), (49, 8, 1.0), (63, 9, 1.0),
                                        (64, 56, 1.2), (64, 57, 1.0), (65, 8, 1.0)])
def test_advection_sums(dev, m, M, aspect):
    import torch
    from duct_amd import step
    from oracle import spectral
    dev.setup(m)
    rng = np.random.default_rng(100 * m + M)
    f = []
    for _ in range(3):
        x = (rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m))) * np.exp(-0.1 * np.arange(M))[:, None, None]
        x[0] = x[0].real
        f.append(x)
    adv = [torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in range(3)]
    step.advection(*[torch.from_numpy(x).cuda() for x in f], *adv, mgalx=4 * M, alp=0.7, aspect=aspect)
    torch.cuda.synchronize()
    ref = spectral.advection3d(*f, mgalx=4 * M, alp=0.7, aspect=aspect)
    errs = [relerr(a.cpu().numpy(), r) for a, r in zip(adv, ref)]
    print("m=%d M=%d aspect=%g rel.err %s" % (m, M, aspect, errs), flush=True)
    assert max(errs) <= 1e-12


@pytest.mark.parametrize("m,M,aspect", [(15, 3, 1.0), (16, 5, 1.5), (17, 16, 1.0), (32, 4, 1.0), (33, 16, 0.7), (48, 3, 1.0),
                                        (49, 7, 1.0), (64, 6, 1.3), (65, 4, 1.3)])
def test_substeps_with_sums(dev, oracle_mod, m, M, aspect):
    import torch
    from duct_amd import step
    from oracle import rk3 as R
    fnu, dt, alp, dpdx = 0.01, 0.02, 0.9, 0.3
    dev.setup(m)
    fields, adv = initial_state(m, M, m)
    helm3d = oracle_helm(oracle_mod, m, alp)
    F, A = ([torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in g] for g in (fields, adv))
    ref, a = list(fields), tuple(adv)
    for krk in (1, 2, 3):
        step.rk3_substep(*F, A, krk, fnu, dt, 3 * M + M % 2, alp=alp, aspect=aspect, dpdx=dpdx)
        torch.cuda.synchronize()
        *ref, a, _ = R.rk3_substep(*ref, a, krk, fnu, dt, 3 * M + M % 2, helm3d, alp, aspect=aspect, dpdx=dpdx)
        errs = [relerr(g.cpu().numpy(), r) for g, r in zip(F + A, list(ref) + list(a))]
        print("m=%d M=%d krk=%d rel.err %s" % (m, M, krk, " ".join("%.1e" % e for e in errs)), flush=True)
        assert max(errs) <= 1e-10
