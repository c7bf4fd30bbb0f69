"""Plane kernels (x and y passes of a whole plane in one block) at the ends of
what they take: every row and column length, partial wave groups (nx/2 + 1
lines), planes up to the LDS limit, one plane, and planes just beyond it.

* transforms against the oracle (1e-13 FP64, 2e-6 FP32: the bounds of the
  transform tests) and steps of both models (1e-12 FP64, 2e-5 FP32 over three
  steps: those of the variant tests), plane kernels and row kernels alike;
* a run of K steps gives the bits of K single steps;
* the combine of the adjoint step (1e-10, as its own test);
* extents whose plane does not fit have no "plane" variant.
"""
import ctypes
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX, DT, EPS = math.pi / 4, 0.5, -0.25
SHAPES = [(16, 8, 4), (24, 12, 2), (32, 16, 1), (48, 24, 12), (64, 32, 8), (96, 48, 4),
          (128, 64, 4), (192, 96, 2), (96, 96, 4), (64, 128, 2), (128, 128, 2), (256, 64, 2),
          (64, 192, 2), (16, 256, 2), (24, 512, 2), (512, 24, 2), (1024, 16, 2), (192, 192, 2)]


def _has(f, role):
    return f.variants(role)[-1] == "plane"


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", SHAPES)
def test_plane_kernels(torch_gpu, n, prec):
    import openpfc_amd as P
    from openpfc_amd import TungstenParams
    from test_gpu_tungsten import DX_G, GOLDEN_PARAMS
    torch = torch_gpu
    f64 = prec == "f64"
    rdt, cdt = (torch.float64, torch.complex128) if f64 else (torch.float32, torch.complex64)
    f = P.HipFft(*n, precision=P.F64 if f64 else P.F32)
    bytes_ = (n[0] // 2 + 1) * n[1] * (16 if f64 else 8)
    assert _has(f, "x_r2c") == _has(f, "pfc_x") == (bytes_ <= 160 * 1024)
    if bytes_ > 160 * 1024:
        return
    print(f"plane {n} {prec}", flush=True)
    for role in ("x_r2c", "x_c2r", "pfc_x", "x_tung"):
        f.set_variant(role, len(f.variants(role)) - 1)
    # transforms
    a = np.random.default_rng(7).standard_normal((n[2], n[1], n[0]))
    ref = O.r2c(a)
    X = torch.empty((n[2], n[1], n[0] // 2 + 1), dtype=cdt, device="cuda")
    f.forward(torch.from_numpy(a).to(rdt).cuda(), X)
    tol = 1e-13 if f64 else 2e-6
    assert np.abs(X.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
    y = torch.empty((n[2], n[1], n[0]), dtype=rdt, device="cuda")
    f.backward(torch.from_numpy(ref).to(cdt).cuda(), y)
    assert np.abs(y.double().cpu().numpy() - a).max() <= tol * np.abs(a).max()
    # PFC steps: a run against the oracle and against single steps
    psi0 = O.uniform_noise(n, 99, -0.01, 0.01, base=-0.2)
    st = P.PfcStepper(f, (DX,) * 3, EPS)
    st.initialize(DT)
    psi = torch.from_numpy(psi0).to(rdt).cuda()
    one = psi.clone()
    st.step(psi, 3)
    for _ in range(3):
        st.step(one, 1)
    assert torch.equal(psi, one)
    opL, opN = O.pfc_operators(n, (DX,) * 3, EPS, DT)
    ref = O.pfc_step(psi0, opL, opN, 3)
    tol = 1e-12 if f64 else 2e-5
    assert np.abs(psi.double().cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
    # adjoint combine
    if f64:
        lam = np.random.default_rng(3).standard_normal(psi0.shape)
        dl = torch.from_numpy(lam).cuda()
        dp = torch.from_numpy(psi0).cuda()
        dr = ctypes.c_double(0.0)
        P.check(f._lib.pfc_hip_pfc_adjoint_step(f.handle, ctypes.c_void_p(dp.data_ptr()),
                                                ctypes.c_void_p(dl.data_ptr()),
                                                ctypes.byref(dr), None))
        dL, dN = O.pfc_operator_derivs(n, (DX,) * 3, EPS, DT)
        want, want_dr = O.pfc_adjoint_step(psi0, lam, opL, opN, dL, dN)
        assert np.abs(dl.cpu().numpy() - want).max() <= 1e-10 * np.abs(want).max()
        assert abs(dr.value - want_dr) <= 1e-10 * max(abs(want_dr), 1e-3 * np.abs(lam).sum())
    # Tungsten
    prm = TungstenParams(**GOLDEN_PARAMS)
    t = P.TungstenStepper(f, (DX_G,) * 3, prm)
    t.initialize(1.0)
    psi0 = O.uniform_noise(n, 77, -0.05, 0.05, base=-0.1)
    psi = torch.from_numpy(psi0).to(rdt).cuda()
    mf = torch.empty_like(psi)
    t.step(psi, 2, psi_mf=mf)
    ops = O.tungsten_operators(n, (DX_G,) * 3, prm.operator_params(), 1.0)
    ref, ref_mf = O.tungsten_step(psi0, *ops, prm.nonlinear_params(), 2)
    assert np.abs(psi.double().cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
    assert np.abs(mf.double().cpu().numpy() - ref_mf).max() <= tol * np.abs(ref_mf).max()


@pytest.mark.parametrize("split", [False, True])
def test_plane_mixed_with_row_kernels(torch_gpu, split):
    """One direction on the plane kernels, the other on the row kernels."""
    import openpfc_amd as P
    torch = torch_gpu
    n = (96, 48, 24)
    psi0 = O.uniform_noise(n, 5, -0.01, 0.01, base=-0.2)
    base = float(psi0.mean())  # the mean-split step conserves the field's mean
    opL, opN = O.pfc_operators(n, (DX,) * 3, EPS, DT)
    ref = O.pfc_step(psi0, opL, opN, 2)
    for fwd in (0, 1):
        for inv in (0, 1):
            f = P.HipFft(*n)
            f.set_variant("pfc_x", len(f.variants("pfc_x")) - 1 if fwd else 0)
            f.set_variant("x_c2r", len(f.variants("x_c2r")) - 1 if inv else 0)
            st = P.PfcStepper(f, (DX,) * 3, EPS)
            st.initialize(DT)
            if split:
                st.set_mean(base)
            psi = torch.from_numpy(psi0 - (base if split else 0.0)).cuda()
            st.step(psi, 2)
            got = psi.cpu().numpy() + (base if split else 0.0)
            assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max(), (fwd, inv)
