"""Every launch variant of the fused step boundary (role t_x_fuse), the staged
ones and those with threads across the tile, at each row length they take, for
plain and mean-split fields: runs of 4 steps against single steps.  Both round a
few units of 1e-16 (FP64) or 6e-8 (FP32) a step: 1e-13 and 1e-5 are required."""
import math

import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DX = math.pi / 4


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nx", [256, 512, 1024])
def test_boundary_variants(torch_gpu, nx, prec, split):
    import openpfc_amd as P
    torch = torch_gpu
    n = (nx, 128, 128)
    f64 = prec == "f64"
    psi0 = O.uniform_noise(n, 17, -0.01, 0.01, base=-0.2)
    mean = float(psi0.mean())
    rdt = torch.float64 if f64 else torch.float32
    start = torch.from_numpy(psi0 - mean if split else psi0).to(rdt).cuda()
    f = P.HipFft(*n, precision=P.F64 if f64 else P.F32)
    st = P.PfcStepper(f, (DX,) * 3, -0.25)
    st.initialize(0.5)
    if split:
        st.set_mean(mean)
    f.set_variant("step_fuse", 0)
    ref = start.clone()
    st.step(ref, 4)
    scale = float(ref.double().abs().max())
    f.set_variant("step_fuse", 1)
    names = f.variants("t_x_fuse")
    assert any("cols" in v for v in names) == f64
    for i, name in enumerate(names):
        f.set_variant("t_x_fuse", i)
        psi = start.clone()
        st.step(psi, 4)
        err = float((psi - ref).double().abs().max()) / scale
        print(f"{n} {prec} split={split} {name}: {err:.2e}", flush=True)
        assert err <= (1e-13 if f64 else 1e-5), name
