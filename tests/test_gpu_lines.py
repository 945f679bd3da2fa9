"""GPU tests of the derivative products at the edges of their tiles: single ones (k_line, through
duct_colloc_deriv_dev_) and the folded sums of them (k_lines, through the advection term): one to nine
row tiles of folded rows, rows and contractions with remainders, odd sizes with their centre row, slabs
of lines that span planes and end ragged, D and D^T, accumulation.

References: the collocation matrix in extended precision, rounded once, times the field in float64; the
oracle's advection.  Bars: a dot product of m terms rounds to at most ~m/2 eps of the sum of the terms'
magnitudes, in practice a few eps of it: 16 eps of max(|D| |u|); 1e-12 for the advection.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def dev():
    import torch
    import duct_amd
    torch.cuda.set_device(0)
    duct_amd.init(0)
    yield duct_amd
    duct_amd.shutdown()


def colloc(m):
    N = m - 1
    j = np.arange(m)
    pi = np.longdouble("3.14159265358979323846264338327950288")
    d = 2 * np.sin(pi * (j[:, None] + j[None, :]) / (2 * N)) * np.sin(pi * (j[:, None] - j[None, :]) / (2 * N))
    np.fill_diagonal(d, 1)
    c = np.ones(m, dtype=np.longdouble)
    c[0] = c[-1] = 2
    D = (c[:, None] / c[None, :]) * np.where((j[:, None] + j[None, :]) % 2, -1, 1) / d
    np.fill_diagonal(D, 0)
    np.fill_diagonal(D, -D.sum(axis=1))
    return D.astype(np.float64)


@pytest.mark.parametrize("m,M", [(4, 9), (5, 7), (16, 3), (17, 3), (32, 2), (33, 16), (34, 5), (35, 3), (64, 2), (65, 3),
                                 (97, 2), (129, 3), (130, 2), (161, 2), (257, 2), (258, 1), (287, 1), (288, 2)])
@pytest.mark.parametrize("trans,beta", [(False, 0.0), (True, -0.5)])
def test_colloc_deriv_tiles(dev, m, M, trans, beta):
    import torch
    from duct_amd import adjoint
    dev.setup(m)
    rng = np.random.default_rng(7 * m + M)
    u = rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m))
    o = rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m))
    D = colloc(m)
    A = 1.25 * (D.T if trans else D)
    for cdir in "yz":
        got = torch.from_numpy(o).cuda()
        adjoint.colloc_deriv(torch.from_numpy(u).cuda(), got, cdir, trans=trans, scal=1.25, beta=beta)
        torch.cuda.synchronize()
        ref = (u @ A.T if cdir == "y" else A @ u) + beta * o
        bar = 16 * EPS * max(np.max(np.abs(u.real) @ np.abs(A).T), np.max(np.abs(A) @ np.abs(u.imag)))
        e = float(np.max(np.abs(got.cpu().numpy() - ref)))
        print("m=%d M=%d %s trans=%d err %.2e bar %.2e" % (m, M, cdir, trans, e, bar), flush=True)
        assert e <= bar


@pytest.mark.parametrize("m,M,aspect", [(65, 5, 1.0), (66, 3, 1.4), (96, 5, 1.0), (97, 3, 1.0), (130, 3, 0.8), (161, 2, 1.0),
                                        (193, 2, 1.0), (226, 2, 1.0), (258, 1, 1.2), (287, 1, 1.0)])
def test_folded_sums_through_advection(dev, m, M, aspect):
    import torch
    from duct_amd import step
    from oracle import spectral
    dev.setup(m)
    rng = np.random.default_rng(100 * m + M)
    f = []
    for _ in range(3):
        x = rng.standard_normal((M, m, m)) + 1j * rng.standard_normal((M, m, m))
        x[0] = x[0].real
        f.append(x)
    adv = [torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in range(3)]
    step.advection(*[torch.from_numpy(x).cuda() for x in f], *adv, mgalx=4 * M, alp=0.7, aspect=aspect)
    torch.cuda.synchronize()
    ref = spectral.advection3d(*f, mgalx=4 * M, alp=0.7, aspect=aspect)
    errs = [float(np.max(np.abs(a.cpu().numpy() - r)) / np.max(np.abs(r))) for a, r in zip(adv, ref)]
    print("m=%d M=%d rel.err %s" % (m, M, errs), flush=True)
    assert max(errs) <= 1e-12
