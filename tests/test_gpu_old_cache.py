"""Autotune caches of earlier builds (openpfc_amd_app, FP64 256x128x128): entries
that name variants since removed still run under OPENPFC_GPU_AUTOTUNE_MODE=
cache_only, which refuses names no build offered."""
import json
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
APP = os.path.join(ROOT, "openpfc_amd", "host", "openpfc_amd_app")
DX = 0.7853981633974483


def test_cache_only_takes_entries_with_removed_variants(torch_gpu, tmp_path):
    cfg = tmp_path / "run.json"
    cfg.write_text(json.dumps({
        "model": {"name": "pfc", "params": {"epsilon": -0.25}},
        "domain": {"Lx": 256, "Ly": 128, "Lz": 128, "dx": DX, "dy": DX, "dz": DX,
                   "origin": "center"},
        "timestepping": {"t0": 0.0, "t1": 2.0, "dt": 0.5, "saveat": 0.0},
        "initial_conditions": [{"target": "density", "type": "constant", "n0": -0.2}],
        "boundary_conditions": []}))

    def run(mode):
        env = dict(os.environ, OPENPFC_GPU_AUTOTUNE_DISABLE="0", OPENPFC_GPU_AUTOTUNE_MODE=mode,
                   OPENPFC_GPU_AUTOTUNE_CACHE_DIR=str(tmp_path))
        r = subprocess.run([APP, str(cfg)], capture_output=True, text=True, timeout=110, env=env)
        print(mode, r.stdout, r.stderr, flush=True)
        return r

    import openpfc_amd as P
    f = P.HipFft(256, 128, 128)
    P.PfcStepper(f, (DX,) * 3, -0.25).initialize(0.5)
    key = P.step_key("pfc", P.F64, (256, 128, 128))
    path = P.store_cache_entry(f, key, cache_dir=str(tmp_path))
    assert run("cache_only").returncode == 0
    with open(path) as fh:
        cache = json.load(fh)
    entry = cache["entries"][key]
    assert "15" in entry and "9" in entry

    def store(**names):
        cache["entries"][key] = dict(entry, **names)
        with open(path, "w") as fh:
            json.dump(cache, fh)

    store(**{"15": "r16x8/E16+r16x16/E16/G4/split/w4"})
    assert run("cache_only").returncode == 0
    store(**{"15": "r8x4x4/E8+r8x8x4/E8/G8/full", "9": "r8x4x4/E8/G1/split/pre/nt"})
    assert run("cache_only").returncode == 0
    store(**{"15": "no-such-variant"})
    r = run("cache_only")
    assert r.returncode != 0 and "No cached configuration" in r.stderr
