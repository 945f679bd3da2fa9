"""GPU tests of the rule that takes solves with folding on to the unfolded FP64 solve or to the folded passes, on
both sides of each of its lines, and of the folded passes at the folded size 64 (113 to 128 interior points).

The route is read from the library's per-kernel-class counts, the results are compared with the unfolded solve
of the same fields and with the oracle.  Bars: each solve holds 1e-12 of the field's maximum against the oracle
at these sizes, so two of them agree to 2e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12
FOLD = ("fold_c2p", "fold_p2p_div", "fold_p2p", "fold_p2c", "fold_mid")


@pytest.fixture(scope="module")
def dev():
    import torch
    import duct_amd
    torch.cuda.set_device(0)
    duct_amd.init(0)
    yield duct_amd
    duct_amd.set_fold(0)
    duct_amd.shutdown()


_cur = {"m": None}


def ensure(dev, m):
    if _cur["m"] != m:
        dev.setup(m)
        _cur["m"] = m


def fields(nf, M, m, seed):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return [torch.view_as_complex(torch.randn((M, m, m, 2), generator=g, dtype=torch.float64, device="cuda"))
            for _ in range(nf)]


def solve(dev, f, bounds, fold, ib=0, out=None):
    """The solutions (into `out`, or new fields) and the counts of the kernel classes."""
    import torch
    from duct_amd import solver
    rhs = [x.clone() for x in f] if out is None else f
    sol = [torch.full_like(x, float("nan")) for x in f] if out is None else out
    alam = [700.0 if b == "d" else 0.0 for b in bounds]
    dev.set_fold(fold)
    try:
        with solver.KernelTimer() as t:
            dev.helm3d_batch(rhs, sol, bounds, alam, alp=1.0, ib=ib)
            torch.cuda.synchronize()
    finally:
        dev.set_fold(0)
    return sol, t.count


@pytest.mark.parametrize("m,M,bounds,fold,folds", [
    (113, 192, "d", 2, False), (114, 64, "ddd", 1, False),             # 111 and 112 points: always in LDS
    (115, 4, "d", 2, True), (130, 63, "d", 1, True),                   # Dirichlet alone: fewer than 128 planes,
    (115, 64, "d", 2, False), (130, 128, "d", 2, False), (130, 32, "dd", 1, False),   # 128 to 256,
    (130, 129, "d", 2, True), (115, 64, "ddd", 2, True),               # and more
    (115, 3, "n", 2, False), (130, 512, "n", 2, False), (130, 513, "n", 2, True),     # with Neumann fields: 1024
    (130, 256, "dn", 2, False), (115, 257, "dn", 1, True), (129, 129, "dddn", 2, True), (129, 513, "n", 1, False),
    (131, 4, "d", 2, False), (146, 2, "dn", 2, False), (147, 63, "d", 2, True), (162, 64, "d", 2, False),   # passes
    (162, 21, "ddd", 2, True), (162, 22, "ddd", 2, False), (163, 64, "d", 2, True)])
def test_routes_of_folded_solves(dev, m, M, bounds, fold, folds):
    ensure(dev, m)
    f = fields(len(bounds), M, m, 31 * m + M)
    got, count = solve(dev, f, bounds, fold)
    ref, plain = solve(dev, f, bounds, 0)
    took = sum(count[k] for k in FOLD)
    print("m=%d M=%d %s fold=%d: %s" % (m, M, bounds, fold, {k: v for k, v in count.items() if v}), flush=True)
    assert (took > 0) == folds and sum(plain[k] for k in FOLD) == 0
    for a, b in zip(got, ref):
        e = float((a - b).abs().max() / b.abs().max())
        print("  against the unfolded solve %.2e" % e, flush=True)
        assert e <= 2 * TOL
        assert folds or e == 0.0


@pytest.mark.parametrize("m", [115, 130])
def test_folded_neumann_passes_of_size_64_match_oracle(dev, oracle_mod, m):
    """Modes of a batch of 513 that stays folded: the low ones (unfolded) and those past xlambda = 64."""
    ensure(dev, m)
    f = fields(1, 513, m, m)
    got, count = solve(dev, f, "n", 2)
    assert count["fold_c2p"] > 0
    ob = oracle_mod.OracleBasis(oracle_mod.pseudomat(m))
    for k0 in (0, 1, 7, 8, 9, 100, 512):
        ref, _ = oracle_mod.helm3d(ob, f[0][k0:k0 + 1].cpu().numpy(), "n", 0.0, ib=k0)
        e = float(np.max(np.abs(got[0][k0:k0 + 1].cpu().numpy() - ref)) / np.max(np.abs(ref)))
        print("m=%d mode %d rel.err %.2e" % (m, k0, e), flush=True)
        assert e <= TOL


@pytest.mark.parametrize("m,bounds,ib", [(115, "dd", 0), (130, "nn", 0), (129, "nn", 8), (98, "nn", 3)])
def test_crosswise_fields_stay_folded(dev, m, bounds, ib):
    """Solutions that overwrite the other field's right-hand side: not in LDS, so with folding on the folded passes."""
    ensure(dev, m)
    f = fields(2, 12, m, m + ib)
    ref, _ = solve(dev, f, bounds, 0, ib=ib)
    a, b = (x.clone() for x in f)
    (b, a), count = solve(dev, [a, b], bounds, 2, ib=ib, out=[b, a])
    assert sum(count[k] for k in FOLD) > 0 and count["plane"] == 0
    for x, r in zip((b, a), ref):
        e = float((x - r).abs().max() / r.abs().max())
        print("m=%d %s ib=%d rel.err %.2e" % (m, bounds, ib, e), flush=True)
        assert e <= 2 * TOL
