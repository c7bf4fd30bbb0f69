"""Natural-layout z pass at the ends of its multiplier table: columns of one
point, of the longest tabulated length (256) and beyond it, with a partial last
tile of kx columns, for the plain step and both Tungsten z passes, against the
oracle (the tolerance of the step: 1e-12 over two steps in FP64)."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX, DT, EPS = math.pi / 4, 0.5, -0.25


@pytest.mark.parametrize("nz", [1, 2, 12, 96, 192, 256, 512, 1024])
def test_natural_z_lengths(torch_gpu, nz):
    import openpfc_amd as P
    from openpfc_amd import TungstenParams
    from test_gpu_tungsten import DX_G, GOLDEN_PARAMS
    torch = torch_gpu
    n = (48, 4, nz)
    psi0 = O.uniform_noise(n, 31, -0.01, 0.01, base=-0.2)
    f = P.HipFft(*n)
    st = P.PfcStepper(f, (DX, DX, DX), EPS)
    st.initialize(DT)
    psi = torch.from_numpy(psi0).cuda()
    st.step(psi, 2)
    opL, opN = O.pfc_operators(n, (DX, DX, DX), EPS, DT)
    ref = O.pfc_step(psi0, opL, opN, 2)
    assert np.abs(psi.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
    prm = TungstenParams(**GOLDEN_PARAMS)
    t = P.TungstenStepper(P.HipFft(*n), (DX_G,) * 3, prm)
    t.initialize(1.0)
    psi = torch.from_numpy(psi0).cuda()
    t.step(psi, 2)
    ops = O.tungsten_operators(n, (DX_G,) * 3, prm.operator_params(), 1.0)
    ref, _ = O.tungsten_step(psi0, *ops, prm.nonlinear_params(), 2)
    assert np.abs(psi.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
