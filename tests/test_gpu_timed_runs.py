"""Timed kept-spectrum runs (step_timed_fused) and long runs on both sides of the
points where the spectrum is made anew.

step_timed_fused is step() with events round its launches, so it has to leave
the bits of step() at every length.

Tolerances of the long runs, fixed and not growing with the length: the
pattern saturates after some 50 steps, from where on no mode grows.  Until then
roundings grow as the field itself does (its noise starts at 0.01 and ends at
0.3 of the pattern's amplitude), so that they stay relative ones of some units
of 1e-16 (FP64) and 6e-8 (FP32) times the root of the step count and a pattern
selection factor below 1e3: 1e-10 and 1e-3.  A kept spectrum that is never
made anew multiplies its own roundings by exp(0.13 n): of order 1 at 300 steps
in FP32 and at 600 in FP64."""
import math

import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX = math.pi / 4
N = (256, 128, 128)


def _stepper(P, prec, eps, dt, mean=None):
    f = P.HipFft(*N, precision=P.F64 if prec == "f64" else P.F32)
    st = P.PfcStepper(f, (DX,) * 3, eps)
    st.initialize(dt)
    if mean is not None:
        st.set_mean(mean)
    return f, st


def _field(torch, prec, split, seed):
    psi0 = O.uniform_noise(N, seed, -0.01, 0.01, base=-0.2)
    mean = float(psi0.mean()) if split else None
    psi = torch.from_numpy(psi0 - mean if split else psi0)
    return psi.to(torch.float64 if prec == "f64" else torch.float32).cuda(), mean


# the spectrum is made anew every 6 (eps = -1, dt = 1), 17 (eps = -0.8) and 60 steps; eps = -5,
# dt = 2 grows by more than exp(8) a step, where every step is a run
@pytest.mark.parametrize("prec,eps,dt,steps", [
    ("f64", -1.0, 1.0, 6), ("f64", -1.0, 1.0, 7), ("f64", -1.0, 1.0, 13),
    ("f32", -0.8, 0.5, 35), ("f64", -0.25, 0.5, 61), ("f64", -5.0, 2.0, 2)])
def test_timed_run_leaves_the_bits_of_step(torch_gpu, prec, eps, dt, steps):
    import openpfc_amd as P
    a, _ = _field(torch_gpu, prec, False, 5)
    b = a.clone()
    _, st = _stepper(P, prec, eps, dt)
    st.step(a, steps)
    t = st.step_timed_fused(b, steps)
    assert bool(torch_gpu.isfinite(a).all())
    assert torch_gpu.equal(a, b)
    assert all(v > 0 for v in t[:5]), t
    assert (t[5] > 0) == (eps != -5.0), t


@pytest.mark.parametrize("prec,steps,tol", [("f64", 600, 1e-10), ("f32", 300, 1e-3)])
def test_long_run_against_single_steps(torch_gpu, prec, steps, tol):
    import openpfc_amd as P
    psi0, mean = _field(torch_gpu, prec, True, 61)
    out = []
    for call, fuse in (("step", 1), ("step_timed_fused", 1), ("step", 0)):
        f, st = _stepper(P, prec, -0.25, 0.5, mean)
        f.set_variant("step_fuse", fuse)
        psi = psi0.clone()
        getattr(st, call)(psi, steps)
        assert bool(torch_gpu.isfinite(psi).all())
        out.append(psi.double())
    assert torch_gpu.equal(out[0], out[1])
    err = float(((out[0] - out[2]).abs().max() / out[2].abs().max()).item())
    print(f"{prec} {steps} steps: {err:.2e}", flush=True)
    assert err <= tol
