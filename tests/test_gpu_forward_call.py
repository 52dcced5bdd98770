"""QMatMul.forward's own work around the kernel launch: the rows it hands over as they are, the calls
without a workspace (one and two rows) and the stream it launches on."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from inference_amd import qmm


@pytest.fixture(scope="module")
def layer():
    w = torch.randn((96, 512), generator=torch.Generator().manual_seed(5))
    qt = qmm.QTensor.quantize(w.cuda(), qmm.GgmlDType.Q4K)
    return qmm.QMatMul.from_qtensor(qt)


@pytest.mark.parametrize("m", [0, 1, 2, 3, 9])
def test_every_form_of_the_rows_gives_the_same_bits(layer, m):
    x = torch.randn((m, 512), generator=torch.Generator().manual_seed(m)).cuda()
    want = layer.forward(x)
    assert want.shape == (m, 96)
    wide = torch.zeros((m, 640), device="cuda")
    wide[:, :512] = x
    forms = [x.reshape(1, m, 512), wide[:, :512], x.t().contiguous().t()]
    if m == 1:
        forms.append(x[0])
    for f in forms:
        got = layer.forward(f)
        assert got.shape == (*f.shape[:-1], 96)
        assert np.array_equal(got.reshape(m, 96).cpu().numpy(), want.cpu().numpy())


@pytest.mark.parametrize("m", [1, 2, 3])
def test_runs_on_the_current_stream_and_under_capture(layer, m):
    x = torch.randn((m, 512), generator=torch.Generator().manual_seed(m)).cuda()
    want = layer.forward(x).cpu()
    buf = torch.zeros_like(x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        buf.copy_(x)
        got = layer.forward(buf)
    side.synchronize()
    assert torch.equal(got.cpu(), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer.forward(buf)
    for scale in (1.0, 2.0, 4.0):  # a power of two scales the block scales and nothing else
        buf.copy_(x * scale)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), want * scale)
