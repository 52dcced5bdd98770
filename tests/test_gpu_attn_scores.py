"""Attention scores up to the largest finite f32: decode (one workgroup, chunks) and prompts (rows, tiles)."""
import ctypes
import math

import pytest
import torch

from inference_amd import qmm

pytestmark = pytest.mark.gpu
DEV = "cuda"
Q0 = 2.0 ** 63  # the only element of q that is not zero: a score is Q0 * k[0], exactly


def scores(kind, n, seed):
    """f32 scores of n positions (the first one always a small one under "low_normal", so that every row sees
    one): beyond 2.36e38 in magnitude score * log2(e) is infinite, and from about 1e9 ("large") the rounding of
    that product is large enough for 2^x to over- or underflow."""
    g = torch.Generator().manual_seed(seed)
    u = torch.rand(n, generator=g)
    big = (2.4 + 0.9 * u) * 1e38
    if kind == "large":
        s = (1 + u) * 1e12
    elif kind == "high":
        s = big
    elif kind == "low":
        s = -big
    elif kind == "mixed":
        s = torch.where(torch.rand(n, generator=g) < 0.5, big, -big)
    else:
        s = torch.where(torch.rand(n, generator=g) < 0.5, 4 * u - 2, -big)
        s[0] = 0.5
    return s.float()


def setup(kind, n, kv_heads, hd):
    """Caches of n positions, their scores, and f64 outputs [n, kv_heads, hd] of queries at each position."""
    g = torch.Generator().manual_seed(n + hd)
    s = scores(kind, n, n)
    kc, vc = (torch.randn((kv_heads, n, hd), generator=g) for _ in range(2))
    kc[:, :, 0] = s / Q0
    assert torch.equal(kc[0, :, 0] * Q0, s) and torch.isfinite(s).all()
    hide = torch.arange(n)[None, :] > torch.arange(n)[:, None]
    w = torch.softmax(s.double()[None, :].expand(n, n).masked_fill(hide, -math.inf), -1)
    want = torch.einsum("pj,gjd->pgd", w, vc.double())
    return kc.to(DEV), vc.to(DEV), want.to(DEV)


def query(rows, heads, hd):
    q = torch.zeros((rows, heads, hd), device=DEV)
    q[:, :, 0] = Q0
    return q


# The scores are exact and the large ones equal or too far apart for a second weight, so what remains is the
# roundings of the small ones' exponentials and of the sums (n of them at most), relative to |v| < 6.
def close(got, want, n):
    assert ((got.double() - want).abs() <= 2.0 ** -24 * (n + 32) * 6).all()


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


KINDS = ["large", "high", "low", "mixed", "low_normal"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("heads,kv_heads,hd", [(8, 2, 128), (4, 4, 64), (8, 1, 256)])
@pytest.mark.parametrize("p", [11, 16, 40, 299])
def test_decode(kind, heads, kv_heads, hd, p):
    L = qmm.lib()
    kc, vc, want = setup(kind, p + 1, kv_heads, hd)
    q, out = query(1, heads, hd), torch.empty((heads, hd), device=DEV)
    pos = torch.tensor([p], dtype=torch.int32, device=DEV)
    ws = torch.zeros(int(L.qmm_decode_attention_workspace_size(heads, kv_heads, hd, p + 1)), dtype=torch.uint8,
                     device=DEV)
    qmm._check(L.qmm_decode_attention(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), pos.data_ptr(), out.data_ptr(),
                                      heads, kv_heads, hd, p + 1, ctypes.c_float(1.0), ws.data_ptr(), ws.numel(),
                                      stream()))
    close(out, want[p].repeat_interleave(heads // kv_heads, 0), p + 1)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("path", ["rows", "tiles"])
@pytest.mark.parametrize("heads,kv_heads,hd", [(8, 2, 128), (4, 4, 64)])
def test_prompt(monkeypatch, kind, path, heads, kv_heads, hd):
    monkeypatch.setenv("QMM_PREFILL_ATTN", path)
    n = 300
    kc, vc, want = setup(kind, n, kv_heads, hd)
    q, out = query(n, heads, hd), torch.empty((n, heads, hd), device=DEV)
    qmm._check(qmm.lib().qmm_prefill_attention(q.data_ptr(), heads * hd, kc.data_ptr(), vc.data_ptr(), 0, n,
                                               out.data_ptr(), heads * hd, heads, kv_heads, hd, n,
                                               ctypes.c_float(1.0), stream()))
    close(out, want.repeat_interleave(heads // kv_heads, 1), n)
