"""GPU tests of the solves with the plane in LDS (k_plane) at the edges of their tiles: interiors of one
to eight tiles of 16 with remainders 0, 1 and 15, odd mode counts, a mode offset, in-place solves,
the transposed solve, and the mixed walls on rectangular planes.

References: the projection passes over planar intermediates, which a batch whose solutions overwrite
each other's right-hand sides still takes (every right-hand side is read before a solution is
written), and the oracle for the mixed walls.  Bar: both routes round the same products of n <= 128
terms, ~n eps each against solutions that do not cancel: 1e-12 of the maximum, the FP64 bar.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12
SIZES = [4, 17, 18, 19, 33, 34, 35, 50, 51, 66, 67, 82, 83, 98, 99, 114, 115, 129, 130]


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


@pytest.mark.parametrize("m", SIZES)
@pytest.mark.parametrize("ib", [0, 3])
def test_plane_solve_equals_passes(dev, m, ib):
    import torch
    dev.setup(m)
    M = 5
    for bound, alam in (("d", 700.0), ("n", 0.0)):
        f = [field(M, m, 10 * m + k) for k in range(2)]
        rhs = [torch.from_numpy(x).cuda() for x in f]
        sol = [torch.full_like(x, float("nan")) for x in rhs]
        print("m=%d ib=%d bound %s" % (m, ib, bound), flush=True)
        dev.helm3d_batch(rhs, sol, bound * 2, [alam, alam + 9.0], alp=0.9, ib=ib)
        torch.cuda.synchronize()
        got = [x.cpu().numpy() for x in sol]
        place = torch.from_numpy(f[0]).cuda()                  # in place, one field
        dev.helm3d_batch([place], [place], bound, [alam], alp=0.9, ib=ib)
        torch.cuda.synchronize()
        assert np.array_equal(place.cpu().numpy(), got[0])
        a, b = (torch.from_numpy(x).cuda() for x in f)          # each solution over the other's right-hand side
        dev.helm3d_batch([a, b], [b, a], bound * 2, [alam, alam + 9.0], alp=0.9, ib=ib)
        torch.cuda.synchronize()
        for k, ref in enumerate((b, a)):
            e = relerr(got[k], ref.cpu().numpy())
            print("  field %d rel.err %.2e" % (k, e), flush=True)
            assert e <= TOL
        if bound == "d":
            r = rhs[0].cpu().numpy()
            for edge in (r[:, 0], r[:, -1], r[:, :, 0], r[:, :, -1]):
                assert not edge.any()                            # helm3d.f90:48-60
            assert np.array_equal(r[:, 1:-1, 1:-1], f[0][:, 1:-1, 1:-1])


@pytest.mark.parametrize("m", [4, 18, 35, 66, 83, 99, 114, 130])
def test_plane_adjoint_identity(dev, m):
    import torch
    from duct_amd import adjoint
    dev.setup(m)
    M = 3
    bounds, alams = "dnn", [300.0, 0.0, 2.0]
    f, g = ([field(M, m, 100 * m + 10 * k + s) for k in range(3)] for s in (1, 2))
    sf, stg = ([torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in range(3)] for _ in "ab")
    dev.helm3d_batch([torch.from_numpy(x).cuda() for x in f], sf, bounds, alams)
    adjoint.helm3d_adjoint_batch([torch.from_numpy(x).cuda() for x in g], stg, bounds, alams)
    torch.cuda.synchronize()
    for k in range(3):
        s, t = sf[k].cpu().numpy(), stg[k].cpu().numpy()
        scale = np.linalg.norm(s) * np.linalg.norm(g[k])
        d = float(np.real(np.vdot(s, g[k])) - np.real(np.vdot(f[k], t)))
        print("m=%d field %d <Sf,g> - <f,S'g> = %.2e of %.2e" % (m, k, d, scale), flush=True)
        assert abs(d) <= TOL * scale
        assert not t[:, 0].any() and not t[:, :, -1].any() and not t[0].imag.any()


@pytest.mark.parametrize("my,mz,walls", [(4, 5, "dndd"), (18, 35, "ndnd"), (67, 20, "nnnd"), (83, 82, "dnnn"),
                                        (100, 130, "dddd"), (115, 98, "ndnn"), (130, 18, "dnnd")])
def test_plane_walls_match_oracle(dev, my, mz, walls):
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


def test_plane_many_planes_and_folding(dev):
    """More planes than the CUs hold at once, against the projection passes; and the folded solver where it
    leaves whole solves to LDS: the same bits with folding on as off."""
    import torch
    from duct_amd import solver
    m, M = 129, 165
    dev.setup(m)
    f = [field(M, m, k) for k in range(2)]
    for bounds in ("dd", "nn"):
        sol = [torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in f]
        dev.helm3d_batch([torch.from_numpy(x).cuda() for x in f], sol, bounds, [700.0, 3.0], alp=0.9, ib=2)
        a, b = (torch.from_numpy(x).cuda() for x in f)
        dev.helm3d_batch([a, b], [b, a], bounds, [700.0, 3.0], alp=0.9, ib=2)
        torch.cuda.synchronize()
        for s, r in zip(sol, (b, a)):
            e = relerr(s.cpu().numpy(), r.cpu().numpy())
            print("m=%d M=%d %s rel.err %.2e" % (m, M, bounds, e), flush=True)
            assert e <= TOL
    for m, M in ((67, 4), (114, 3), (129, 4)):
        dev.setup(m)
        f = [field(M, m, 7 * m + k) for k in range(2)]
        got = []
        for fold in (0, 2):
            solver.set_fold(fold)
            try:
                s = [torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in f]
                dev.helm3d_batch([torch.from_numpy(x).cuda() for x in f], s, "dn", [700.0, 0.0], alp=0.9)
                torch.cuda.synchronize()
                got.append([x.cpu().numpy() for x in s])
            finally:
                solver.set_fold(0)
        assert all(np.array_equal(x, y) for x, y in zip(*got))


@pytest.mark.parametrize("m,M,bounds", [(67, 3, "d"), (97, 2, "dn"), (98, 3, "ddn"), (130, 4, "dn"), (131, 2, "dn"), (146, 3, "d"),
                                        (147, 2, "d"), (162, 64, "d")])
def test_folded_schemes_left_to_unfolded_solves(dev, m, M, bounds):
    """Where the unfolded FP64 solve is the faster one, the folded solver gives its bits, and so does the refined
    one (the right-hand sides' Dirichlet walls zeroed alike); with residuals asked for it refines as before."""
    import torch
    from duct_amd import solver
    dev.setup(m)
    alam = [700.0, 2.0, 1.0][:len(bounds)]
    f = [field(M, m, 9 * m + k) for k in range(len(bounds))]
    out = []
    for kind in ("plain", "fold", "refine", "stats"):
        rhs = [torch.from_numpy(x).cuda() for x in f]
        s = [torch.full((M, m, m), float("nan"), dtype=torch.complex128, device="cuda") for _ in f]
        if kind in ("plain", "fold"):
            solver.set_fold(0 if kind == "plain" else 2)
            try:
                dev.helm3d_batch(rhs, s, bounds, alam, alp=0.9)
            finally:
                solver.set_fold(0)
        else:
            solver.helm3d_mixed_batch(rhs, s, bounds, alam, alp=0.9, scheme0="fold16q", scheme1="fold16q", niter=1,
                                      stats=kind == "stats")
        torch.cuda.synchronize()
        out.append([x.cpu().numpy() for x in s])
        after = [r.cpu().numpy() for r in rhs]
        if kind == "plain":
            want = after
        assert all(np.array_equal(a, b) for a, b in zip(after, want))
    folds = 131 <= m and not (m <= 146 or (m <= 162 and M >= 64))   # m = 147: three modes stay folded
    for k, x in enumerate(out[0]):
        assert folds or np.array_equal(out[1][k], x)
        assert folds or np.array_equal(out[2][k], x)
        e = [relerr(out[j][k], x) for j in (1, 2, 3)]
        print("m=%d field %d fold %.2e refine %.2e with stats %.2e" % (m, k, *e), flush=True)
        assert e[0] <= 1e-11 and e[1] <= 1e-9 and e[2] <= 1e-9
