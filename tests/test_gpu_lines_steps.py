"""GPU tests of whole substeps whose derivative sums are those of the y and z launches (k_lines) on odd grids,
whose centre row is summed over the waves of a workgroup: few and many folded rows, batches small enough for
jobs of their own and larger ones, every krk, and an update whose last output (u, no product of its own)
follows one with a centre row (w).

Reference: the oracle's substep.  Bar: the substep's, 1e-10 of each field's maximum, on the whole field and on
its centre lines alone; p's grows as m^4 past m = 129 with the condition of the pressure Poisson planes (the
oracle and the same substep with collocation matrices, both on the CPU in 64 bits, differ in p by 6.2e-12 at
129^2 x 12 and by 1.7e-10 at 257^2 x 3, in the other fields by at most 4e-12).
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


@pytest.mark.parametrize("m,M,aspect", [(49, 72, 1.0), (65, 16, 1.5), (65, 24, 1.0), (97, 5, 1.0), (97, 16, 1.0),
                                        (129, 12, 2.0), (257, 3, 1.0), (257, 6, 1.0)])
def test_substeps_on_odd_grids(dev, oracle_mod, m, M, aspect):
    import torch
    from duct_amd import step
    from oracle import rk3 as R
    fnu, dt, alp, dpdx, X = 0.01, 0.02, 0.9, 0.3, 3 * M + M % 2
    dev.setup(m)
    fields, adv = initial_state(m, M, m + M)
    oracle_mod.use_blas(True)
    try:
        helm3d = oracle_helm(oracle_mod, m, alp)
        F, A = ([torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in g] for g in (fields, adv))
        ref, a = list(fields), tuple(adv)
        for krk in (1, 2, 3):
            print("m=%d M=%d krk=%d" % (m, M, krk), flush=True)
            step.rk3_substep(*F, A, krk, fnu, dt, X, alp=alp, aspect=aspect, dpdx=dpdx)
            torch.cuda.synchronize()
            *ref, a, _ = R.rk3_substep(*ref, a, krk, fnu, dt, X, helm3d, alp, aspect=aspect, dpdx=dpdx)
            c = m // 2
            for name, g, r in zip(("u", "v", "w", "p", "adv1", "adv2", "adv3"), F + A, list(ref) + list(a)):
                g = g.cpu().numpy()
                top = np.max(np.abs(r))
                e = [relerr(g, r), np.max(np.abs(g - r)[:, c]) / top, np.max(np.abs(g - r)[:, :, c]) / top]
                print("  %s rel.err %.1e, on the centre lines along y %.1e, along z %.1e" % (name, *e), flush=True)
                assert max(e) <= (1e-10 * max(1.0, (m / 129.0) ** 4) if name == "p" else 1e-10)
    finally:
        oracle_mod.use_blas(False)


@pytest.mark.parametrize("m,M", [(65, 4), (65, 24)])
def test_substep_without_z_derivatives(dev, oracle_mod, m, M):
    """aspect = inf: 1 / aspect is zero, and so are the coefficients of the z products, some of which join sums that
    others have begun."""
    import torch
    from duct_amd import step
    from oracle import rk3 as R
    fnu, dt, alp, dpdx, X = 0.01, 0.02, 0.9, 0.3, 3 * M
    dev.setup(m)
    fields, adv = initial_state(m, M, m)
    F, A = ([torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in g] for g in (fields, adv))
    step.rk3_substep(*F, A, 2, fnu, dt, X, alp=alp, aspect=float("inf"), dpdx=dpdx)
    torch.cuda.synchronize()
    ref = R.rk3_substep(*fields, tuple(adv), 2, fnu, dt, X, oracle_helm(oracle_mod, m, alp), alp, aspect=float("inf"), dpdx=dpdx)
    errs = [relerr(g.cpu().numpy(), r) for g, r in zip(F + A, list(ref[:4]) + list(ref[4]))]
    print("m=%d M=%d aspect=inf rel.err %s" % (m, M, " ".join("%.1e" % e for e in errs)), flush=True)
    assert max(errs) <= 1e-10
