"""Weight quantizers (one lane per sub-block, 64 sub-blocks a wave) against the oracle's bytes."""
import numpy as np
import pytest
import torch

from inference_amd import GgmlDType, QTensor
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def values(kind, n, k):
    rng = np.random.default_rng(31 * n + k)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    if kind == "ties":  # many values half way between codes
        w = (np.round(w * 100) * 0.5 + 0.5).astype(np.float32)
    elif kind == "scales":  # sub-blocks of very different sizes, some all zero or constant
        w = (w.reshape(n, k // 16, 16) * np.exp(rng.standard_normal((n, k // 16, 1)) * 5)).astype(np.float32)
        w[:, ::5] = 0.0
        w[:, 1::7] = 0.25
        w = w.reshape(n, k)
    return np.ascontiguousarray(w)


# one block (a wave's last lanes repeat it), counts that leave part of a wave, of a workgroup, and whole ones
@pytest.mark.parametrize("n,k", [(1, 256), (3, 256), (7, 512), (33, 768), (32, 2048)])
@pytest.mark.parametrize("kind", ["normal", "ties", "scales"])
@pytest.mark.parametrize("dt,odt", [(GgmlDType.Q4K, orc.Q4K), (GgmlDType.Q6K, orc.Q6K), (GgmlDType.Q8_0, orc.Q8_0)])
def test_bytes_equal_the_oracles(dt, odt, kind, n, k):
    w = values(kind, n, k)
    got = QTensor.quantize(torch.from_numpy(w).cuda(), dt).to_ggml()
    np.testing.assert_array_equal(got, np.asarray(orc.quantize(odt, w)).reshape(-1))
