"""Fused z pass of the adjoint step at every column length, with whole and
partial column tiles (W = nx/2 + 1 is never a multiple of 4 or 8 columns), the
plane kernels and the row kernels around it, mixed choices of the two, a single
plane and a single row per plane: against the oracle's adjoint
step within 1e-10 (the bound of the adjoint step's own test).  The field does not
depend on whether the derivative is asked for, bit for bit."""
import ctypes
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX, DT, EPS = math.pi / 4, 0.5, -0.3
NZ = [1, 2, 4, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 512, 1024]
CASES = [((16, 8, nz), c) for nz in NZ for c in ("plane", "rows")]
CASES += [((24, 4, 16), "mixed"), ((8, 1, 24), "rows"), ((2, 2, 8), "rows"),
          ((1024, 32, 8), "rows"), ((128, 128, 4), "plane")]


@pytest.mark.parametrize("n,choice", CASES)
def test_adjoint_z(torch_gpu, n, choice):
    import openpfc_amd as P
    torch = torch_gpu
    print(f"adjoint {n} {choice}", flush=True)
    f = P.HipFft(*n)
    for role in ("x_r2c", "x_c2r", "pfc_x"):
        names = f.variants(role)
        if choice == "plane" and names[-1] == "plane":
            f.set_variant(role, len(names) - 1)
        elif choice == "mixed" and names[-1] == "plane":
            f.set_variant(role, len(names) - 1 if role == "pfc_x" else 0)
        else:
            f.set_variant(role, 0)
    st = P.PfcStepper(f, (DX,) * 3, EPS)
    st.initialize(DT)
    rng = np.random.default_rng(11)
    shape = (n[2], n[1], n[0])
    psi, lam = (-0.2 + 0.1 * rng.uniform(-1, 1, shape) for _ in range(2))
    dpsi, dlam = torch.from_numpy(psi).cuda(), torch.from_numpy(lam).cuda()
    dr = ctypes.c_double(0.0)

    def step(out, r):
        P.check(f._lib.pfc_hip_pfc_adjoint_step(f.handle, ctypes.c_void_p(dpsi.data_ptr()),
                                                ctypes.c_void_p(out.data_ptr()), r, None))
    step(dlam, ctypes.byref(dr))
    opL, opN = O.pfc_operators(n, (DX,) * 3, EPS, DT)
    dL, dN = O.pfc_operator_derivs(n, (DX,) * 3, EPS, DT)
    ref, ref_dr = O.pfc_adjoint_step(psi, lam, opL, opN, dL, dN)
    assert np.abs(dlam.cpu().numpy() - ref).max() <= 1e-10 * np.abs(ref).max()
    assert abs(dr.value - ref_dr) <= 1e-10 * abs(ref_dr), (dr.value, ref_dr)
    dlam2 = torch.from_numpy(lam).cuda()
    step(dlam2, None)
    assert torch.equal(dlam2, dlam)
