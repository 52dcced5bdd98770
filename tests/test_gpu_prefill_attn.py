"""Causal prompt attention on MFMA tiles (qmm_prefill_attn_tile_*) and by rows against f64 softmax attention."""
import ctypes
import math

import pytest
import torch

from inference_amd import GgmlDType, QTensor, qmm

pytestmark = pytest.mark.gpu
DEV = "cuda"
U = 2.0 ** -24


def L():
    return qmm.lib()


def S():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def inputs(first, count, heads, kv_heads, hd, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    span = first + count + 5
    q = torch.randn((count, heads * hd + 4), generator=g, device=DEV)  # a row stride of its own
    kc = torch.randn((kv_heads, span, hd), generator=g, device=DEV)
    vc = torch.randn((kv_heads, span, hd), generator=g, device=DEV)
    kc[:, first + count:] = math.nan  # unwritten rows
    vc[:, first + count:] = math.nan
    return q, kc, vc


def call(q, kc, vc, first, heads, hd):
    count, kv_heads, span = q.shape[0], kc.shape[0], kc.shape[1]
    out = torch.full((count, heads * hd + 8), 7.0, device=DEV)
    qmm._check(L().qmm_prefill_attention(q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), first, count,
                                         out.data_ptr(), out.stride(0), heads, kv_heads, hd, span,
                                         ctypes.c_float(hd ** -0.5), S()))
    assert (out[:, heads * hd:] == 7.0).all()
    return out[:, : heads * hd]


def reference(q, kc, vc, first, heads, hd):
    """f64 output, and the worst-case f32 error of each head: a score's dot has hd roundings of its absolute
    sum, which moves a weight by twice that relatively; the weighted sum adds n roundings and the
    exponential and division a few."""
    count, kv_heads = q.shape[0], kc.shape[0]
    last = first + count
    out = torch.empty((count, heads, hd), dtype=torch.float64, device=DEV)
    bound = torch.empty((count, heads, 1), dtype=torch.float64, device=DEV)
    hide = torch.arange(last, device=DEV)[None, :] > torch.arange(first, last, device=DEV)[:, None]
    for h in range(heads):
        g = h // (heads // kv_heads)
        qh, k, v = q[:, h * hd:(h + 1) * hd].double(), kc[g, :last].double(), vc[g, :last].double()
        s = (qh @ k.t() * hd ** -0.5).masked_fill(hide, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v
        mag = (qh.abs() @ k.abs().t() * hd ** -0.5).amax()
        bound[:, h] = U * (2 * (hd + 2) * mag + last + 16) * v[torch.isfinite(v)].abs().max()
    return out.view(count, -1), bound.expand(-1, -1, hd).reshape(count, -1)


# one row, a tile's last / first row either side, several tiles, group sizes that do not divide 32, and
# first / last positions on both sides of a 32-key tile and of the four waves' 128
CASES = [(0, 1, 32, 8, 128), (0, 9, 32, 8, 128), (31, 8, 32, 8, 128), (24, 8, 32, 8, 128), (3, 127, 32, 8, 128),
         (0, 129, 16, 4, 64), (100, 33, 16, 16, 128), (5, 33, 24, 8, 128), (0, 64, 7, 1, 64), (0, 40, 15, 3, 128),
         (127, 2, 8, 1, 64), (600, 70, 10, 2, 128)]


@pytest.mark.parametrize("path", ["rows", "tiles", None])
@pytest.mark.parametrize("first,count,heads,kv_heads,hd", CASES + [(2, 300, 16, 2, 256), (0, 600, 32, 8, 128)])
def test_prefill_attention(monkeypatch, first, count, heads, kv_heads, hd, path):
    if path:
        monkeypatch.setenv("QMM_PREFILL_ATTN", path)
    q, kc, vc = inputs(first, count, heads, kv_heads, hd, 900 + count)
    got = call(q, kc, vc, first, heads, hd)
    want, bound = reference(q, kc, vc, first, heads, hd)
    assert ((got.double() - want).abs() <= bound).all()


# Sizes where one form is faster by 13% or more (microseconds, rows / tiles).
FASTER = [("rows", 0, 64, 32, 8, 128),    # 7.3 / 10.7
          ("rows", 0, 160, 16, 16, 128),  # 12.7 / 16.3
          ("rows", 30, 128, 16, 16, 128),  # 11.9 / 16.2
          ("rows", 0, 64, 32, 16, 128),   # 6.7 / 10.6
          ("rows", 0, 8, 64, 8, 128),     # 7.1 / 10.4
          ("rows", 500, 64, 32, 8, 128),  # 27.0 / 32.1
          ("tiles", 0, 127, 32, 8, 128),  # 12.8 / 11.3
          ("tiles", 500, 128, 32, 8, 128),  # 47.8 / 32.3
          ("tiles", 0, 256, 32, 8, 128),  # 30.5 / 16.8
          ("tiles", 0, 384, 8, 1, 64)]    # 18.2 / 14.0


@pytest.mark.parametrize("form,first,count,heads,kv_heads,hd", FASTER)
def test_the_faster_form_is_taken(monkeypatch, form, first, count, heads, kv_heads, hd):
    """The two forms sum in different orders, so the bits tell which one ran."""
    q, kc, vc = inputs(first, count, heads, kv_heads, hd, 79)
    got = {None: call(q, kc, vc, first, heads, hd)}
    for path in ("rows", "tiles"):
        monkeypatch.setenv("QMM_PREFILL_ATTN", path)
        got[path] = call(q, kc, vc, first, heads, hd)
    assert not torch.equal(got["rows"], got["tiles"])
    assert torch.equal(got[None], got[form])


@pytest.mark.parametrize("which", ["k", "v"])
def test_caches_off_the_16_byte_grid(monkeypatch, which):
    """A cache that starts 4 bytes past the grid runs by rows, also where tiles are asked for, with their bits."""
    first, count, heads, kv_heads, hd = 3, 300, 8, 2, 128
    q, kc, vc = inputs(first, count, heads, kv_heads, hd, 80)
    monkeypatch.setenv("QMM_PREFILL_ATTN", "rows")
    want = call(q, kc, vc, first, heads, hd)
    monkeypatch.setenv("QMM_PREFILL_ATTN", "tiles")
    assert not torch.equal(call(q, kc, vc, first, heads, hd), want)
    moved = torch.empty(kc.numel() + 1, device=DEV)[1:].view(kc.shape).copy_(kc if which == "k" else vc)
    assert moved.data_ptr() % 16 == 4
    kc, vc = (moved, vc) if which == "k" else (kc, moved)
    assert torch.equal(call(q, kc, vc, first, heads, hd), want)


@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("what", ["q", "k", "v"])
def test_non_finite_values_reach_only_the_rows_that_see_them(monkeypatch, what, value):
    """One non-finite element of q, of a key row or of a value row: the tile path's outputs are finite, NaN and
    infinite exactly where the row path's are, and elsewhere within the f32 bound of the f64 result."""
    first, count, heads, kv_heads, hd = 2, 61, 16, 4, 128
    q, kc, vc = inputs(first, count, heads, kv_heads, hd, 77)
    if what == "q":
        q[20, 5] = value
    else:
        (kc if what == "k" else vc)[1, 30, 9] = value
    got = {}
    for path in ("rows", "tiles"):
        monkeypatch.setenv("QMM_PREFILL_ATTN", path)
        got[path] = call(q, kc, vc, first, heads, hd)
    rows, tiles = got["rows"], got["tiles"]
    assert torch.equal(torch.isnan(rows), torch.isnan(tiles)) and torch.equal(torch.isinf(rows), torch.isinf(tiles))
    ok = torch.isfinite(rows)
    assert not ok.all() and ok.any()
    clean = inputs(first, count, heads, kv_heads, hd, 77)
    want, bound = reference(*clean, first, heads, hd)
    # rows that do not see the element keep the clean result (-inf scores only drop a weight)
    same = torch.ones(count, dtype=torch.bool, device=DEV)
    if what == "q":
        same[20] = False
    else:
        same[30 - first:] = False
    assert ((tiles.double() - want).abs() <= bound)[same].all()


@pytest.mark.parametrize("key", [32, 64, 96])
def test_nan_key_that_is_all_a_wave_sees(monkeypatch, key):
    """A NaN key row at the first position of the second, third or fourth key tile is the only one that the
    tile's wave sees for that position's query: every row that sees it is NaN, on both paths, and no other."""
    first, count, heads, kv_heads, hd = 1, 110, 8, 2, 128
    q, kc, vc = inputs(first, count, heads, kv_heads, hd, 78)
    want, bound = reference(q, kc, vc, first, heads, hd)
    kc[:, key, 17] = math.nan
    for path in ("tiles", "rows"):
        monkeypatch.setenv("QMM_PREFILL_ATTN", path)
        got = call(q, kc, vc, first, heads, hd)
        assert ((got.double() - want).abs() <= bound)[: key - first].all(), path
        assert torch.isnan(got[key - first:]).all(), path


@pytest.mark.parametrize("m,heads,kv_heads,hd", [(127, 32, 8, 128), (9, 32, 8, 128), (33, 16, 4, 64), (24, 24, 12, 128)])
def test_tiles_write_the_o_gemms_planes(monkeypatch, m, heads, kv_heads, hd):
    """qmm_prefill_attention_o on the tile path (which writes the o GEMM's Q8_K planes) == the two calls."""
    monkeypatch.setenv("QMM_PREFILL_ATTN", "tiles")
    H, first = heads * hd, 3
    g = torch.Generator(device=DEV).manual_seed(3)
    wo = QTensor.quantize(torch.randn((512, H), generator=g, device=DEV) * 0.02, GgmlDType.Q4K)
    q, kc, vc = inputs(first, m, heads, kv_heads, hd, 40 + m)
    x0 = torch.randn((m, 512), generator=g, device=DEV)
    got, want = x0.clone(), x0.clone()
    wsb = int(L().qmm_prefill_attention_o_workspace_size(wo.handle, m))
    ws = torch.empty(wsb, dtype=torch.uint8, device=DEV)
    qmm._check(L().qmm_prefill_attention_o(q.data_ptr(), q.stride(0), kc.data_ptr(), vc.data_ptr(), first, m,
                                           heads, kv_heads, hd, kc.shape[1], ctypes.c_float(hd ** -0.5),
                                           wo.handle, got.data_ptr(), 512, ws.data_ptr(), wsb, S()))
    att = call(q, kc, vc, first, heads, hd).contiguous()
    wsb = int(L().qmm_matmul_ex_workspace_size(wo.handle, m, 0))
    ws = torch.empty(wsb, dtype=torch.uint8, device=DEV)
    qmm._check(L().qmm_matmul_ex((ctypes.c_void_p * 1)(wo.handle.value), 1, att.data_ptr(), m, H, None,
                                 ctypes.c_float(0), 1, (ctypes.c_void_p * 1)(want.data_ptr()),
                                 (ctypes.c_int64 * 1)(512), ws.data_ptr(), wsb, S()))
    assert torch.equal(got, want)
