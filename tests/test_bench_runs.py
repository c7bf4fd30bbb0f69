"""bench.py on multi-step runs that keep psi's spectrum: the kernel names of
their passes as openpfc_amd.profile_summary shortens what rocprofv3 prints, and
the bytes a call moves, counted pass by pass."""
import math
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402
from openpfc_amd.profile_summary import short_name  # noqa: E402

PLAN16 = "pfc_amd::FftPlan<1024, 16, pfc_amd::RadixList<16, 16, 4>, false>"
HALF8 = "pfc_amd::FftPlan<512, 8, pfc_amd::RadixList<8, 8, 8>, false>"
HALF16 = "pfc_amd::FftPlan<512, 16, pfc_amd::RadixList<16, 16, 2>, false>"


@pytest.mark.parametrize("kernel,prec,variant,mode,name,t,plan,rest", [
    ("k_tx_bnd", "f32", "r16x16x2/E16/G16/nt", 0, "k_tx_bnd", "float", HALF16, "16, 1, true"),
    ("k_tx_bnd", "f64", "r8x8x8/E8/G8", 0, "k_tx_bnd", "double", HALF8, "8, 1, false"),
    ("k_tx_bnd", "f64", "r8x8x8/E8/G8/w4/nt", 0, "k_tx_bnd", "double", HALF8, "8, 4, true"),
    ("k_tx_bnd", "f64", "r8x8x8/E8/G8/cols/w4", 0, "k_tx_cols", "double", HALF8, "8, 4, false"),
    ("k_tx_bnd", "f64", "r8x8x8/E8/G8/cols/w2/nt", 0, "k_tx_cols", "double", HALF8,
     "8, 2, true"),
    ("k_tz", "f64", "r16x16x4/E16/G1/split/mt", 3, "k_tz_mt", "double", PLAN16,
     "1, true, 3, false"),
    ("k_tz", "f32", "r16x16x4/E16/G2/split/mtp", 4, "k_tz_mt", "float", PLAN16,
     "2, true, 4, true"),
    ("k_tz", "f64", "r16x16x4/E16/G1/split/pre", 3, "k_tz", "double", PLAN16,
     "1, true, 3, true, false"),
])
def test_kernel_names_of_kept_spectrum_passes(kernel, prec, variant, mode, name, t, plan, rest):
    full = f"void pfc_amd::{name}<{t}, {plan}, {rest}>(pfc_amd::TStepArgs<{t}>)"
    assert bench.variant_key(kernel, prec, 1024, variant, mode=mode) == short_name(full)


@pytest.mark.parametrize("steps,span", [(1, 1), (1, 60), (2, 60), (20, 60), (60, 60), (61, 60),
                                        (130, 60), (7, 1)])
def test_bytes_of_a_call(steps, span):
    n, esize = 64, 8
    R, C = esize * n ** 3, 2 * esize * (n // 2 + 1) * n * n
    total, done = 0, 0
    while done < steps:
        k = min(span, steps - done)
        for i in range(k):
            last = i == k - 1
            total += R + 2 * C if i == 0 else 2 * C  # forward x of psi and N | boundary
            total += 4 * C if i == 0 else 2 * C      # forward y
            total += 3 * C if last else 4 * C        # z: A and N in, inverse out, kept unless last
            total += 2 * C                           # inverse y
        total += C + R                               # inverse x
        done += k
    assert bench.run_step_bytes(n, esize, steps, span) * steps == pytest.approx(total, rel=1e-12)


def test_length_of_a_run():
    # growth exponents of the bench's operators (0.132), a strong one (1.19) and none
    assert bench.kept_run_steps(-0.25, 0.5) == 60
    assert bench.kept_run_steps(-1.0, 1.0) == 6
    assert bench.kept_run_steps(0.1, 0.5) == 64
    assert bench.kept_run_steps(-0.25, 0.0) == 1
    assert math.isfinite(bench.run_step_bytes(1024, 8, 20, 60))
