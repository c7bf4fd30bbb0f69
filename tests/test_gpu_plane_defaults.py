"""Which extents start on the plane kernels (x and y passes of a whole plane in one
block): not where a call is slower with them than with the row and column
kernels.  Measured, us, plane | rows: FP32 64x512x128 one step 110 | 70,
512x32x48 34.0 | 29.8, 128x256x64 53 | 44, 128x192x192 75 | 69; FP64 24x512x256 101 |
92, 128x128x32 37 | 34."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec,plane", [
    ((32, 32, 32), "f64", True), ((128, 128, 64), "f64", True), ((128, 128, 32), "f64", False),
    ((24, 512, 256), "f64", False), ((96, 96, 24), "f64", False),
    ((96, 96, 96), "f32", True), ((64, 64, 12), "f32", True), ((128, 128, 96), "f32", True),
    ((128, 256, 256), "f32", True), ((64, 512, 128), "f32", False), ((48, 512, 256), "f32", False),
    ((512, 32, 48), "f32", False), ((128, 256, 64), "f32", False), ((128, 192, 192), "f32", False)])
def test_plane_default(torch_gpu, n, prec, plane):
    import openpfc_amd as P
    f = P.HipFft(*n, precision=P.F64 if prec == "f64" else P.F32)
    for role in ("x_r2c", "x_c2r", "pfc_x", "x_tung"):
        names = f.variants(role)
        assert names[-1] == "plane"
        assert (names[f.get_variant(role)] == "plane") == plane, (role, names)
