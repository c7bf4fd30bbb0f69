"""PFC runs of the settings-file App on extents whose multi-step calls keep psi's
spectrum (256x128x128, FP64):

* a restart from a save point continues with the bits of the uninterrupted run,
  since every call starts from psi itself at a save point;
* with model.params.keep_spectrum false the result does not depend on the save
  interval, bit for bit; by default two intervals agree to rounding (1e-12: ten
  steps of a few 1e-16 each, amplified by at most exp(0.132 * 10) = 3.7);
* anything but true or false is refused."""
import json
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
APP = os.path.join(ROOT, "openpfc_amd", "host", "openpfc_amd_app")
DX = 0.7853981633974483


def _settings(out, saveat, t1=5.0, **params):
    return {"model": {"name": "pfc", "params": {"epsilon": -0.25, **params}},
            "domain": {"Lx": 256, "Ly": 128, "Lz": 128, "dx": DX, "dy": DX, "dz": DX,
                       "origin": "center"},
            "timestepping": {"t0": 0.0, "t1": t1, "dt": 0.5, "saveat": saveat},
            "fields": [{"name": "density", "data": str(out / "psi_%d.bin")}],
            "initial_conditions": [{"target": "density", "type": "constant", "n0": -0.2},
                                   {"target": "density", "type": "uniform_noise", "seed": 7,
                                    "low": -0.01, "high": 0.01}],
            "boundary_conditions": []}


def _run(tmp_path, name, s, ok=True):
    cfg = tmp_path / f"{name}.json"
    cfg.write_text(json.dumps(s))
    env = dict(os.environ, OPENPFC_GPU_AUTOTUNE_DISABLE="1")
    r = subprocess.run([APP, str(cfg)], capture_output=True, text=True, timeout=100, env=env)
    print(r.stdout, r.stderr, flush=True)
    assert (r.returncode == 0) == ok
    return r


def _last(d, k):
    return np.fromfile(d / f"psi_{k}.bin", dtype="<f8")


def test_restart_from_a_save_point(torch_gpu, tmp_path):
    a, b = tmp_path / "a", tmp_path / "b"
    _run(tmp_path, "a", _settings(a, 2.0, t1=6.0))   # saves after 4, 8 and 12 steps
    s = _settings(b, 2.0, t1=6.0)
    s["initial_conditions"] = [{"target": "density", "type": "from_file",
                                "filename": str(a / "psi_1.bin")}]
    s["simulator"] = {"result_counter": 1, "increment": 4}
    _run(tmp_path, "b", s)
    for k in (2, 3):
        assert (a / f"psi_{k}.bin").read_bytes() == (b / f"psi_{k}.bin").read_bytes(), k


@pytest.mark.parametrize("keep", [False, None])
def test_save_interval(torch_gpu, tmp_path, keep):
    p = {} if keep is None else {"keep_spectrum": keep}
    a, b = tmp_path / "a", tmp_path / "b"
    _run(tmp_path, "a", _settings(a, 5.0, **p))   # ten steps, saved at the end
    _run(tmp_path, "b", _settings(b, 1.0, **p))   # saved every two steps
    x, y = _last(a, 1), _last(b, 5)
    if keep is False:
        assert np.array_equal(x, y)
    assert np.abs(x - y).max() <= 1e-12 * np.abs(y).max()


def test_keep_spectrum_is_a_truth_value(torch_gpu, tmp_path):
    r = _run(tmp_path, "c", _settings(tmp_path / "c", 5.0, keep_spectrum=0), ok=False)
    assert "keep_spectrum" in r.stderr
