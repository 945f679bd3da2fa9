"""GPU test of aliased fields that the derivative entries refuse: an output that is an input or another output."""
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


@pytest.mark.parametrize("m,M", [(33, 4), (65, 24)])   # both directions in one launch, y and z launches
def test_aliased_outputs_are_refused(dev, m, M):
    import torch
    from duct_amd import adjoint, step
    from duct_amd._lib import DuctError
    dev.setup(m)
    f = [torch.zeros((M, m, m), dtype=torch.complex128, device="cuda") for _ in range(6)]
    for out in ((3, 3, 5), (3, 4, 3), (3, 4, 4), (3, 4, 0), (1, 4, 5)):
        with pytest.raises(DuctError, match="alias"):
            step.advection(*f[:3], *[f[i] for i in out], mgalx=3 * M)
    with pytest.raises(DuctError, match="alias"):
        adjoint.colloc_deriv(f[0], f[0], "y")
    with pytest.raises(DuctError, match="alias"):
        step.transyz(f[0], f[0], "z", 1)
    step.advection(*f, mgalx=3 * M)
    torch.cuda.synchronize()
