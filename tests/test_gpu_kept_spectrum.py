"""Multi-step runs that keep psi's spectrum between steps (transposed layout,
role step_fuse = 1): a run of every length round the first steps, runs that
cross the point where the spectrum is made anew, and strongly unstable
operators, against single steps.

Tolerances: two runs differ by roundings (a few units of 1e-16 a step) that the
unstable modes amplify by at most exp(g n) over n steps, g the largest growth
exponent of a mode; 1e-14 * exp(g n) (FP64) and 1e-5 * exp(g n) (FP32), well
above that, is required."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX = math.pi / 4
N = (256, 128, 128)


def _growth(eps, dt):
    k2 = np.linspace(0, 3, 3001)
    return max(0.0, float((-k2 * (eps + (1 - k2) ** 2) * dt).max()))


def _pair(torch, prec, eps, dt, steps, split=False, chunks=None):
    import openpfc_amd as P
    psi0 = O.uniform_noise(N, 61, -0.01, 0.01, base=-0.2)
    mean = float(psi0.mean())
    rdt = torch.float64 if prec == "f64" else torch.float32
    out = []
    for fuse in (1, 0):
        f = P.HipFft(*N, precision=P.F64 if prec == "f64" else P.F32)
        assert f.variants("step_fuse") == ["per_step", "fused"]
        assert f.get_variant("step_fuse") == 1  # the default
        f.set_variant("step_fuse", fuse)
        st = P.PfcStepper(f, (DX,) * 3, eps)
        st.initialize(dt)
        if split:
            st.set_mean(mean)
        psi = torch.from_numpy(psi0 - mean if split else psi0).to(rdt).cuda()
        for n in chunks or [steps]:
            st.step(psi, n)
        out.append(psi.double())
    err = float(((out[0] - out[1]).abs().max() / out[1].abs().max()).item())
    bound = (1e-14 if prec == "f64" else 1e-5) * math.exp(_growth(eps, dt) * steps)
    print(f"{prec} eps={eps} dt={dt} steps={steps}: {err:.2e} (bound {bound:.1e})", flush=True)
    assert bool(torch.isfinite(out[0]).all())
    assert err <= bound
    return out


@pytest.mark.parametrize("steps", [1, 2, 3, 5])
@pytest.mark.parametrize("prec,split", [("f64", False), ("f64", True), ("f32", True)])
def test_short_runs(torch_gpu, prec, split, steps):
    a, b = _pair(torch_gpu, prec, -0.25, 0.5, steps, split)
    if steps == 1:
        assert torch_gpu.equal(a, b)


def test_run_past_the_refresh(torch_gpu):
    _pair(torch_gpu, "f64", -0.25, 0.5, 70)


def test_unstable_operator(torch_gpu):
    # largest growth exponent 1.19 a step: the spectrum is made anew every 6 steps
    _pair(torch_gpu, "f64", -1.0, 1.0, 9)


def test_stable_operator(torch_gpu):
    a, _ = _pair(torch_gpu, "f64", 0.1, 0.5, 130)
    assert abs(float(a.mean()) + 0.2) < 1e-3


def test_per_step_run_is_its_single_steps(torch_gpu):
    import openpfc_amd as P
    torch = torch_gpu
    f = P.HipFft(*N)
    f.set_variant("step_fuse", 0)
    st = P.PfcStepper(f, (DX,) * 3, -0.25)
    st.initialize(0.5)
    a = torch.from_numpy(O.uniform_noise(N, 3, -0.01, 0.01, base=-0.2)).cuda()
    b = a.clone()
    st.step(a, 4)
    st.step(b, 1)
    st.step(b, 3)
    assert torch.equal(a, b)
