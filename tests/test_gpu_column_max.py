"""Column maxima at the edges of the two-stage reduction: fewer columns than
a block's 64, a partial last block, fewer rows than the 256 partial rows and
than the 16 slices of the second stage.  A maximum is exact, so the result
equals numpy's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(2, 1, 1), (24, 1, 2), (64, 3 * 4, 1), (96, 4, 4), (192, 16, 16),
                               (1024, 24, 12), (2048, 2, 2)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_column_max_edges(torch_gpu, n, prec):
    import openpfc_amd as P
    torch = torch_gpu
    dt = np.float64 if prec == "f64" else np.float32
    a = np.random.default_rng(5).standard_normal((n[2], n[1], n[0])).astype(dt)
    a[:, :, 0] = -np.inf  # the reduction starts at the lowest finite value
    f = P.HipFft(*n, precision=P.F64 if prec == "f64" else P.F32)
    got = P.column_max(f, torch.from_numpy(a).cuda())
    want = np.maximum(a.max(axis=(0, 1)).astype(np.float64), -np.finfo(np.float64).max)
    assert np.array_equal(got, want)
