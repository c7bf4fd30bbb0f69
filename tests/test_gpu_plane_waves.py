"""Plane kernels with 8 waves a block (single precision, more blocks than CUs)
against the same planes with 16: the bits do not depend on the waves.  One plane
with zeros beyond it along z has, at every kz, the spectrum of the plane alone;
runs compare a boundary pass with an inverse and a forward pass; a batched
plan crosses the line where its fields alone do not.  Transforms also against
the oracle (2e-6, the bound of the transform tests)."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX = math.pi / 4


def _on_plane(f):
    for role in ("x_r2c", "x_c2r", "pfc_x"):
        names = f.variants(role)
        assert names[-1] == "plane"
        f.set_variant(role, len(names) - 1)


@pytest.mark.parametrize("nx,ny", [(128, 128), (64, 256), (256, 64), (96, 192), (192, 96)])
def test_forward_bits_and_error(torch_gpu, nx, ny):
    import openpfc_amd as P
    torch = torch_gpu
    nz = 512
    print(f"waves {nx}x{ny}", flush=True)
    big, one = P.HipFft(nx, ny, nz, precision=P.F32), P.HipFft(nx, ny, 1, precision=P.F32)
    _on_plane(big)
    _on_plane(one)
    plane = torch.from_numpy(np.random.default_rng(3).standard_normal((1, ny, nx))).float().cuda()
    a = torch.zeros((nz, ny, nx), device="cuda")
    a[0] = plane[0]  # its transform along z is the plane's spectrum at every kz
    X = torch.empty((nz, ny, nx // 2 + 1), dtype=torch.complex64, device="cuda")
    Y = torch.empty((1, ny, nx // 2 + 1), dtype=torch.complex64, device="cuda")
    big.forward(a, X)
    one.forward(plane, Y)
    assert torch.equal(X, Y.expand_as(X))
    ref = O.r2c(plane.double().cpu().numpy())
    assert np.abs(Y.cpu().numpy() - ref).max() <= 2e-6 * np.abs(ref).max()


@pytest.mark.parametrize("n", [(128, 128, 256), (96, 192, 192), (96, 192, 128), (128, 128, 128)])
def test_run_equals_single_steps(torch_gpu, n):
    """A boundary (two fields: 8 waves from 129 planes on) has the bits of an
    inverse pass (16 waves) and a forward pass."""
    import openpfc_amd as P
    torch = torch_gpu
    psi0 = O.uniform_noise(n, 5, -0.01, 0.01)
    out = []
    for runs in ([3], [1, 1, 1]):
        f = P.HipFft(*n, precision=P.F32)
        f.set_variant("step_layout", f.variants("step_layout").index("natural"))
        _on_plane(f)
        st = P.PfcStepper(f, (DX,) * 3, -0.25)
        st.initialize(0.5)
        st.set_mean(-0.2)
        psi = torch.from_numpy(psi0).float().cuda()
        for k in runs:
            st.step(psi, k)
        out.append(psi)
    assert torch.equal(out[0], out[1])


def test_batched_bits(torch_gpu):
    """Three 128^3 fields in one batched plan (768 blocks) and alone (256)."""
    import openpfc_amd as P
    from openpfc_amd.ensemble import Ensemble, Run
    torch = torch_gpu
    runs = [Run.cubic(128, DX, -0.25 + 0.01 * i, 0.5, -0.2) for i in range(3)]
    both = []
    for group in ([runs], [[r] for r in runs]):
        res = []
        for rs in group:
            e = Ensemble(rs, precision=P.F32, mean_split=True)
            for i, r in enumerate(rs):
                psi = O.uniform_noise((128,) * 3, 40 + runs.index(r), -0.01, 0.01)
                e.field(i).copy_(torch.from_numpy(psi).float().reshape(e.field(i).shape))
            e.step(2)
            torch.cuda.synchronize()
            res += [e.field(i).clone() for i in range(len(rs))]
        both.append(res)
    for a, b in zip(*both):
        assert bool(torch.isfinite(a).all())
        assert torch.equal(a, b)
