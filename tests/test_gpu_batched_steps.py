"""Batched plans in the transposed layout field by field against single plans, bit
for bit: multi-step calls as single steps (role step_fuse 0), and calls that keep
the spectrum over fields whose spectra are remade at different steps."""
import ctypes
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX = math.pi / 4
DT = 0.5
N = (256, 128, 128)


@pytest.mark.parametrize("prec,split,fuse,eps,steps", [
    ("f64", False, 0, [-0.20, -0.31], 4),
    ("f32", True, 0, [-0.20, -0.31], 4),
    ("f64", False, 1, [-0.25, -0.8], 20),  # remade after 60 and after 17 steps
    ("f32", True, 1, [-0.8, -0.25], 20)])
def test_batched_runs_equal_single_plans(torch_gpu, prec, split, fuse, eps, steps):
    import openpfc_amd as P
    torch = torch_gpu
    lib = P.load()
    mean = [-0.18, -0.22]
    pr = P.F64 if prec == "f64" else P.F32
    rdt = torch.float64 if prec == "f64" else torch.float32
    fields = [O.uniform_noise(N, 29 + b, -0.01, 0.01, base=0.0 if split else mean[b])
              for b in range(2)]
    h = ctypes.c_void_p()
    P.check(lib.pfc_hip_plan_create_batched(*N, 2, pr, 0, ctypes.byref(h)))
    try:
        op = (ctypes.c_double * 4)(DX, DX, DX, eps[0])
        P.check(lib.pfc_hip_pfc_set_operators(h, 0, op, 4, DT))
        P.check(lib.pfc_hip_pfc_set_members(h, (ctypes.c_double * 2)(*eps),
                                            (ctypes.c_double * 2)(*mean), int(split)))
        P.check(lib.pfc_hip_variant_set(h, P.HipFft.ROLES["step_layout"], 0))
        P.check(lib.pfc_hip_variant_set(h, P.HipFft.ROLES["step_fuse"], fuse))
        stacked = torch.from_numpy(np.stack(fields)).to(rdt).cuda().contiguous()
        s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        P.check(lib.pfc_hip_pfc_step(h, ctypes.c_void_p(stacked.data_ptr()), steps, s))
        for b in range(2):
            f = P.HipFft(*N, precision=pr)
            st = P.PfcStepper(f, (DX,) * 3, eps[b])
            st.initialize(DT)
            if split:
                st.set_mean(mean[b])
            f.set_variant("step_layout", 0)
            f.set_variant("step_fuse", fuse)
            one = torch.from_numpy(fields[b]).to(rdt).cuda()
            for n in ([1] * steps if fuse == 0 else [steps]):
                st.step(one, n)
            assert bool(torch.isfinite(one).all())
            assert torch.equal(one, stacked[b]), f"field {b} differs"
    finally:
        lib.pfc_hip_plan_destroy(h)
