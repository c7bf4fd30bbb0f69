"""Default variants of the transposed passes by footprint: plain lines for PFC plans
whose grids stay in the last-level cache, non-temporal ones beyond it, and the forms
of large grids for the other model, whichever operators were set before."""
import math

import pytest

pytestmark = pytest.mark.gpu

ROLES = ("t_x_fwd", "t_y_fwd", "t_z", "t_y_inv", "t_x_inv")


def names(f):
    return {r: f.variants(r)[f.get_variant(r)] for r in ROLES}


@pytest.mark.parametrize("n, prec, plain", [
    ((256, 256, 128), 0, ROLES),            # 68 MB a spectrum
    ((512, 128, 128), 0, ROLES),
    ((256, 256, 128), 1, ROLES),            # 34 MB
    ((512, 128, 128), 1, ROLES),
    ((256, 256, 256), 1, ROLES[1:]),        # 68 MB: only the x pass is past its line
    ((1024, 128, 128), 1, ROLES[1:]),
    ((256, 512, 128), 1, ROLES[1:]),
    ((256, 512, 128), 0, ()),               # 135 MB
    ((512, 512, 128), 1, ())])
def test_plain_lines_in_the_cache(torch_gpu, n, prec, plain):
    import openpfc_amd as P
    f = P.HipFft(*n, precision=P.F32 if prec else P.F64)
    P.PfcStepper(f, (math.pi / 4,) * 3, -0.25).initialize(0.5)
    got = names(f)
    for r in plain:
        assert not got[r].endswith(("/nt", "/mt", "/mtp")), (r, got)
    if plain != ROLES:
        assert got["t_x_fwd"].endswith("/nt"), got
    if not plain:
        assert got["t_z"].endswith(("/mt", "/mtp")), got


def test_the_model_sets_the_footprint(torch_gpu):
    import openpfc_amd as P
    f = P.HipFft(256, 256, 128)
    pfc = names(f)
    P.TungstenStepper(f, (1.1,) * 3).initialize(1.0)
    tungsten = names(f)
    assert tungsten["t_z"].endswith("/mt") and tungsten["t_y_fwd"].endswith("/nt")
    first = f.variants("t_y_fwd")[0]
    f.set_variant("t_y_fwd", 0)
    P.PfcStepper(f, (math.pi / 4,) * 3, -0.25).initialize(0.5)
    assert names(f) == {**pfc, "t_y_fwd": first}  # a role set by the caller stays
