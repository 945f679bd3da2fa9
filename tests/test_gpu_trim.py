"""GPU tests of the projection passes that compute only the 16s in use of a plane padded to 256 or 512:
interiors of 9 to 32 tiles of 16 with remainders 0, 1 and 15 (so every share of row tiles over the waves, odd
and even stage counts), the transposed solve, and mixed walls on rectangular planes whose short side has fewer
tiles than a block has waves.

References: the CPU oracle, and the adjoint identity.  Bar: both sides round products of n <= 512 terms, ~n eps
each against solutions that do not cancel: 1e-12 of the maximum, the FP64 bar.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(scope="module")
def dev():
    import torch
    import duct_amd
    torch.cuda.set_device(0)
    duct_amd.init(0)
    yield duct_amd
    duct_amd.shutdown()


def field(M, m, seed, mz=None):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((M, mz or m, m)) + 1j * rng.standard_normal((M, mz or m, m))


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("m", [131, 145, 146, 147, 162, 178, 194, 195, 209, 226, 243, 258, 259, 290, 322, 371, 400, 449, 514])
def test_trimmed_solve_and_adjoint(dev, oracle_mod, m):
    import torch
    from duct_amd import adjoint
    dev.setup(m)
    ob = oracle_mod.OracleBasis(oracle_mod.pseudomat(m))
    # one Neumann basis on both sides: two eigensolves of the operator differ by more than the solves do
    dev.solver.upload_basis("n", m, ob.b.PN, ob.b.PNM1, ob.b.EN, ob.b.DC, ob.b.AM1, ob.b.iofzero, ob.b.wanted)
    M = 3
    for bound, alam in (("d", 700.0), ("n", 40.0)):
        f, g = field(M, m, 10 * m), field(M, m, 10 * m + 1)
        # alp k of 2 and more: no singular plane, whose gauge node depends on the order of the eigenvalues
        ref, _ = oracle_mod.helm3d(ob, f, bound, alam, alp=0.9, ib=3)
        print("m=%d bound %s" % (m, bound), flush=True)
        sol, adj = (torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in "ab")
        dev.helm3d_batch([torch.from_numpy(f.copy()).cuda()], [sol], bound, [alam], alp=0.9, ib=3)
        adjoint.helm3d_adjoint_batch([torch.from_numpy(g).cuda()], [adj], bound, [alam], alp=0.9, ib=3)
        torch.cuda.synchronize()
        s, t = sol.cpu().numpy(), adj.cpu().numpy()
        e = relerr(s, ref)
        scale = np.linalg.norm(s) * np.linalg.norm(g)
        d = float(np.real(np.vdot(s, g)) - np.real(np.vdot(f, t)))
        print("  rel.err %.2e, <Sf,g> - <f,S'g> = %.2e of %.2e" % (e, d, scale), flush=True)
        assert e <= TOL
        assert abs(d) <= TOL * scale


@pytest.mark.parametrize("my,mz,walls", [(131, 20, "dndd"), (18, 146, "ndnd"), (200, 40, "nnnd"), (258, 67, "dnnn"),
                                        (10, 300, "dddd"), (290, 35, "dnnd"), (161, 195, "ndnn")])
def test_trimmed_walls_match_oracle(dev, my, mz, walls):
    import torch
    from duct_amd import temperature
    from oracle import temp as T
    M, alp, alam = 3, 0.8, 5.0
    rhs = field(M, my, my + 7 * mz, mz=mz)
    rng = np.random.default_rng(my * mz)
    bcy, bcz = rng.standard_normal((M, 2, mz)), rng.standard_normal((M, 2, my))
    temperature.setup_temp(my, walls, 1.0, 1.5, mz=mz)
    sol = torch.full((M, mz, my), float("nan"), dtype=torch.complex128, device="cuda")
    temperature.helm3d_temp(*[torch.from_numpy(x).cuda() if x is not None else sol for x in (rhs, None, bcy, bcz)],
                            alam, alp=alp, ib=0)
    torch.cuda.synchronize()
    ref = T.helm3d_temp(T.TempBasis(my, walls, 1.0, 1.5, mz=mz), rhs, alam, bcy, bcz, alp=alp)
    e = relerr(sol.cpu().numpy(), ref)
    print("my=%d mz=%d %s rel.err %.2e" % (my, mz, walls, e), flush=True)
    assert e <= TOL
