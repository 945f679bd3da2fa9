"""GPU tests of the folded derivative products (k_lines, through duct_colloc_deriv_dev_) at the edges
of its tiles: one to nine row tiles, rows and contractions with remainders, odd sizes with their
centre row, slabs of lines that span planes and end ragged, D and D^T, accumulation.

Reference: the collocation matrix in extended precision, rounded once, times the field in float64.
Bar: a dot product of m terms rounds to at most ~m/2 eps of the sum of the terms' magnitudes, in
practice a few eps of it: 16 eps of max(|D| |u|).
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
