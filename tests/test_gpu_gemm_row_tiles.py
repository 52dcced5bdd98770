"""GEMM tiles that are filled in part: row tiles past the last row are skipped, the others keep their bits."""
import pytest
import torch

from inference_amd import GgmlDType, QMatMul, QTensor

pytestmark = pytest.mark.gpu


# either side of 32, 64, 96 and 128 rows (a wave's row tiles and the workgroup tile), and past one whole tile
@pytest.mark.parametrize("dt", [GgmlDType.Q4K, GgmlDType.Q6K, GgmlDType.Q8_0])
@pytest.mark.parametrize("splits", ["1", "2"])
def test_rows_do_not_depend_on_the_row_count(monkeypatch, dt, splits):
    monkeypatch.setenv("QMM_SPLITK", splits)
    g = torch.Generator(device="cuda").manual_seed(6)
    n, k = 200, 1024
    mm = QMatMul.from_qtensor(QTensor.quantize(torch.randn((n, k), generator=g, device="cuda") * 0.02, dt))
    x = torch.randn((256, k), generator=g, device="cuda")
    whole = mm.forward(x)  # whole tiles only
    assert torch.isfinite(whole).all() and (whole != 0).all()
    for m in (9, 31, 32, 33, 64, 65, 96, 97, 127, 129, 160, 161, 193, 255):
        assert torch.equal(mm.forward(x[:m]), whole[:m]), m
