"""Decode attention around the count of positions that one workgroup per kv head takes whole (16)."""
import ctypes
import math

import pytest
import torch

from inference_amd import qmm

pytestmark = pytest.mark.gpu
DEV = "cuda"
U = 2.0 ** -24


# the first position, either side of 16, one and two positions a chunk; four- and eight-wave kernels
@pytest.mark.parametrize("heads,kv_heads,hd", [(32, 8, 128), (8, 1, 128), (6, 2, 64), (16, 16, 128), (16, 2, 256)])
@pytest.mark.parametrize("p", [0, 1, 14, 15, 16, 17, 31, 32, 40])
def test_short_caches(heads, kv_heads, hd, p):
    """Against f64 attention: a score has hd roundings of its absolute sum, which moves a weight by twice that
    relatively; the sums add up to p and the exponentials and the division a few. The cache past p, and for the
    rotating entry p itself, is NaN before the call."""
    L = qmm.lib()
    g = torch.Generator(device=DEV).manual_seed(100 * p + heads)
    span = 64
    q, kn, vn = (torch.randn((x, hd), generator=g, device=DEV) for x in (heads, kv_heads, kv_heads))
    kc, vc = (torch.randn((kv_heads, span, hd), generator=g, device=DEV) for _ in range(2))
    kc[:, p:] = math.nan
    vc[:, p:] = math.nan
    ones, zeros = torch.ones((span, hd), device=DEV), torch.zeros((span, hd), device=DEV)  # no rotation
    pos = torch.tensor([p], dtype=torch.int32, device=DEV)
    out = torch.full((heads, hd), 7.0, device=DEV)
    ws = torch.zeros(int(L.qmm_decode_attention_workspace_size(heads, kv_heads, hd, span)), dtype=torch.uint8,
                     device=DEV)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    scale = ctypes.c_float(hd ** -0.5)
    k64, v64 = torch.cat([kc[:, :p], kn[:, None]], 1).double(), torch.cat([vc[:, :p], vn[:, None]], 1).double()
    s = torch.einsum("hd,hjd->hj", q.double().cpu(), k64.cpu().repeat_interleave(heads // kv_heads, 0)) * hd ** -0.5
    vv = v64.cpu().repeat_interleave(heads // kv_heads, 0)
    want = (torch.softmax(s, -1)[:, :, None] * vv).sum(1).to(DEV)
    mag = torch.einsum("hd,hjd->hj", q.double().abs().cpu(),
                       k64.abs().cpu().repeat_interleave(heads // kv_heads, 0)).amax() * hd ** -0.5
    bound = U * (2 * (hd + 2) * mag.item() + p + 16) * vv.abs().amax().item()
    for _ in range(2):  # the second call finds the workspace as the first one left it
        qmm._check(L.qmm_decode_rope_attention(q.data_ptr(), kn.data_ptr(), vn.data_ptr(), ones.data_ptr(),
                                               zeros.data_ptr(), pos.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                                               out.data_ptr(), heads, kv_heads, hd, span, scale, ws.data_ptr(),
                                               ws.numel(), stream))
        assert (out.double() - want).abs().max().item() <= bound
        assert torch.equal(kc[:, p], kn) and torch.equal(vc[:, p], vn)
    out.fill_(7.0)
    qmm._check(L.qmm_decode_attention(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), pos.data_ptr(), out.data_ptr(),
                                      heads, kv_heads, hd, span, scale, ws.data_ptr(), ws.numel(), stream))
    assert (out.double() - want).abs().max().item() <= bound
