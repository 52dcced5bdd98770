"""The Q8_0 GEMM's scale products on the f16 matrix cores against the first-generation tile's f32 products."""
import numpy as np
import pytest
import torch

from inference_amd import GgmlDType, QMatMul, QTensor
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


# f16 scales that are normal, denormal (down to one unit) and infinite (an activation row's block by its values,
# a weight's block by its scale's bytes); sizes around the 128-row and 128-column tiles, one K step and several
@pytest.mark.parametrize("n,k,m", [(130, 512, 9), (257, 1024, 129), (128, 256, 128)])
@pytest.mark.parametrize("ws,xs", [(0.02, 1.0), (2e-5, 1.0), (0.02, 3e-6), (1e-6, 1e-5), (1.0, 1e9), ("inf", 1.0)])
def test_scale_products_keep_the_f32_bits(monkeypatch, n, k, m, ws, xs):
    rng = np.random.default_rng(n + m)
    inf = ws == "inf"
    w = (rng.standard_normal((n, k)) * (0.02 if inf else ws)).astype(np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    if xs > 1e6:
        x[0, :32] *= xs  # one block of one row past f16's range: its scale is infinite
    else:
        x *= xs
    raw = np.frombuffer(bytes(orc.quantize(orc.Q8_0, w)), np.uint8).copy()
    if inf:
        raw[34 * (k // 32) + 34:][:2] = (0x00, 0x7C)  # the second block of the second row
    qt = QTensor.from_ggml(raw, GgmlDType.Q8_0, (n, k), device=torch.device("cuda", 0))
    xd = torch.from_numpy(x).cuda()
    monkeypatch.setenv("QMM_SPLITK", "1")
    y = QMatMul.from_qtensor(qt).forward(xd)
    monkeypatch.setenv("QMM_MMQ8", "1")
    ref = QMatMul.from_qtensor(qt).forward(xd)
    np.testing.assert_array_equal(y.cpu().numpy(), ref.cpu().numpy())
    ok = torch.isfinite(y)
    if inf:  # only the second row's column
        assert not ok[:, 1].any()
        ok[:, 1] = True
    assert ok[1:].all() and (xs < 1e6 or not torch.isfinite(y[0]).any()) and (y != 0).any()
