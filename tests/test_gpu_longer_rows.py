"""Rows at the ends of the classes by which a launch takes them: the row quantiser's (csrc/quant.hip), against the CPU oracle."""
import numpy as np
import pytest
import torch

from khaosz_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16, F32 = torch.bfloat16, torch.float32


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _rows(M, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g) * (0.2 + 3 * torch.rand(M, 1, generator=g))


# 1024 and 2048 vectors of 16 bytes, and one on either side
@pytest.mark.parametrize("M", [1, 70])
@pytest.mark.parametrize("dtype,K", [(F32, 4096), (F32, 4112), (F32, 8176), (F32, 8192), (F32, 8208), (BF16, 8192), (BF16, 8208), (BF16, 16384),
                                     (BF16, 16400)])
def test_long_rows_are_quantised_like_the_oracle(oracle, dtype, K, M):
    x = _rows(M, K, K + M).to(dtype)
    x[0, K - 1] = 1e4  # the maximum in the row's last vector
    q, s = ops.quant_rowwise_i8(x.to(DEV))
    bf = dtype == BF16
    qo, so = oracle.c_quant_rowwise_i8(_bits(x) if bf else x.numpy(), bf16_bits=bf)
    assert np.array_equal(q.cpu().numpy(), qo) and np.array_equal(s.cpu().numpy(), so)
