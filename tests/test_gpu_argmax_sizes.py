"""Greedy argmax at the edges of its slices (128 workgroups, four logits a thread in flight): the lowest
index of the largest logit, a NaN above every number, and an index of the logits where all are -inf."""
import ctypes

import pytest
import torch

from inference_amd import qmm

pytestmark = pytest.mark.gpu


def _oracle(x):
    nan = torch.isnan(x)
    return int((nan if nan.any() else x == x.max()).nonzero()[0])


@pytest.mark.parametrize("n", [1, 2, 63, 127, 128, 129, 32767, 32768, 32769, 131071, 131072, 131073, 200001])
def test_argmax_of_every_slice_edge(n):
    L = qmm.lib()
    g = torch.Generator().manual_seed(n)
    ws = torch.zeros(int(L.qmm_greedy_workspace_size(n)), dtype=torch.uint8, device="cuda")
    toks = torch.zeros(4, dtype=torch.int32, device="cuda")
    pos = torch.zeros(1, dtype=torch.int32, device="cuda")
    per = -(-n // 128)
    at = sorted({0, min(per, n) - 1, min(per, n - 1), n // 2, n - 1})
    cases = [torch.full((n,), -float("inf")), torch.full((n,), 3.0)]
    for i in at:
        x = torch.randn(n, generator=g)
        x[i] = 9.0
        cases.append(x)
        x = x.clone()
        x[i] = float("nan")
        cases.append(x)
    x = torch.randn(n, generator=g)
    x[torch.tensor(at)] = float("inf")
    cases.append(x)
    for x in cases:
        pos.zero_()
        xd = x.cuda()
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert L.qmm_greedy_advance(xd.data_ptr(), n, toks.data_ptr(), 4, pos.data_ptr(), 1, ws.data_ptr(),
                                    ws.numel(), stream) == 0
        assert (toks[1].item(), pos.item()) == (_oracle(x), 1)
    assert not ws[:256].any()
