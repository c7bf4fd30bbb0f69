"""Default variants that depend on the model: a single-precision Tungsten plan
steps on the first variant of every role, a role set by the caller stays as set
in either order, and operators of the PFC model bring the defaults back."""
import math

import pytest

pytestmark = pytest.mark.gpu

DX = math.pi / 4


@pytest.mark.parametrize("n", [(32, 32, 32), (256, 128, 128)])
def test_single_precision_tungsten_defaults(torch_gpu, n):
    import openpfc_amd as P
    f = P.HipFft(*n, precision=P.F32)
    before = {r: f.get_variant(r) for r in P.TungstenStepper.TUNE_ROLES + ["pfc_x"]}
    layout = f.get_variant("step_layout")
    P.TungstenStepper(f, (1.1,) * 3).initialize(1.0)
    assert all(f.get_variant(r) == 0 for r in P.TungstenStepper.TUNE_ROLES if f.variants(r))
    assert f.get_variant("step_layout") == layout
    P.PfcStepper(f, (DX,) * 3, -0.25).initialize(0.5)
    for r, v in before.items():
        if r != "t_z":  # set by the operators themselves
            assert f.get_variant(r) == v, r
    last = len(f.variants("x_c2r")) - 1
    f.set_variant("x_c2r", last)
    P.TungstenStepper(f, (1.1,) * 3).initialize(1.0)
    assert f.get_variant("x_c2r") == last and f.get_variant("x_r2c") == 0


def test_double_tungsten_keeps_the_defaults(torch_gpu):
    import openpfc_amd as P
    f = P.HipFft(32, 32, 32)
    before = {r: f.get_variant(r) for r in P.TungstenStepper.TUNE_ROLES}
    P.TungstenStepper(f, (1.1,) * 3).initialize(1.0)
    assert {r: f.get_variant(r) for r in before} == before
