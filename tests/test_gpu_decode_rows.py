"""The decode GEMV that quantises rows of any length (csrc/gemv_rows.hip), where its tiles can go wrong: rows that are not
whole 128-byte lines, the ends of its row length classes, batches on both sides of 8, matrices that end inside a
workgroup of each height, 16-bit and 32-bit rows, int8 and FP8 -- against the CPU oracle."""
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


# N against workgroups of 8, 16, 32 and 64 rows on 256 compute units; K at line and class edges
CASES = [(5, 1, 16), (8, 9, 112), (9, 33, 128), (16, 7, 144), (1, 2049, 1024), (4, 2047, 1040), (16, 2056, 2032), (11, 4097, 2048),
         (7, 8201, 2064), (16, 8193, 528), (9, 1537, 4096), (16, 520, 4112), (3, 9000, 4128), (12, 100, 8176), (16, 16, 8192),
         (2, 8208, 8192), (6, 16385, 272),
         # few rows of a matrix of two rounds and more, short rows and long ones (which count their rounds differently)
         (3, 500, 8192), (5, 2500, 4608), (2, 4600, 2400), (3, 9001, 1040), (4, 8300, 2064), (1, 4353, 6864),
         (2, 9000, 4016), (1, 10248, 3200), (3, 16400, 1040), (12, 16400, 2048), (2, 32784, 528), (1, 6200, 1488),
         # up to 4 rows, where the dot-product kernel takes over and where it does not
         (2, 3000, 6000), (1, 1500, 3168), (4, 6000, 3200), (2, 4097, 1040), (1, 16392, 2112), (2, 16380, 3072)]


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("M,N,K", CASES)
def test_int8_rows_bit_exact(oracle, M, N, K, dtype):
    x = _rows(M, K, M + K).to(dtype)
    wq = torch.randint(-127, 128, (N, K), generator=torch.Generator().manual_seed(N), dtype=torch.int8)
    sw = torch.rand(N, generator=torch.Generator().manual_seed(N + 1)) * 1e-3
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2)) * 0.1
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(3)).to(dtype)
    args = x.to(DEV), wq.to(DEV), sw.to(DEV), bias.to(DEV)
    y = ops.gemv_w8a8_decode(*args)
    bf = dtype == BF16
    want = oracle.c_linear_w8a8(_bits(x) if bf else x.numpy(), wq.numpy(), sw.numpy(), bias.numpy(), x_bf16_bits=bf, bf16_out=bf)
    got = _bits(y) if bf else y.cpu().numpy()
    assert np.array_equal(got.view(np.uint16 if bf else np.uint32), want.view(np.uint16 if bf else np.uint32))
    assert torch.equal(ops.gemv_w8a8_decode(*args, residual=res.to(DEV)), y + res.to(DEV))


@pytest.mark.parametrize("M,N,K", [c for c in CASES if c[2] <= 2048])
def test_norm_in_front_bit_exact(oracle, M, N, K):
    x = _rows(M, K, M + K).to(BF16)
    gam = (1 + 0.2 * torch.randn(K, generator=torch.Generator().manual_seed(4))).to(BF16)
    wq = torch.randint(-127, 128, (N, K), generator=torch.Generator().manual_seed(N), dtype=torch.int8)
    sw = torch.rand(N, generator=torch.Generator().manual_seed(N + 1)) * 1e-3
    y = ops.gemv_w8a8_decode(x.to(DEV), wq.to(DEV), sw.to(DEV), norm=(gam.to(DEV), 1e-5))
    qx, sx = oracle.c_rmsnorm_quant_i8(_bits(x), _bits(gam), 1e-5, bf16_bits=True)
    want = oracle.c_dequant_epilogue(oracle.c_gemm_i8_i32(qx, wq.numpy()), sx, sw.numpy(), None, bf16_out=True)
    assert np.array_equal(_bits(y), want)


@pytest.mark.parametrize("M,N,K", CASES)
def test_fp8_rows_within_tolerance(oracle, M, N, K):
    """Codes that differ by one, a lost line, or NaN codes read behind a row's end would be far outside 1e-3 of the rms."""
    x = _rows(M, K, M + K).to(BF16)
    w = _rows(N, K, N) * 0.02
    xq, sx = oracle.c_quant_tensor_fp8(_bits(x), bf16_bits=True)
    wq, sw = oracle.c_quant_tensor_fp8(w.numpy())
    y = ops.gemv_fp8_decode(x.to(DEV), torch.from_numpy(wq).to(DEV), torch.tensor([sw], device=DEV), out_dtype=F32).cpu().numpy()
    exact = oracle.np_linear_fp8(xq, sx, wq, sw)
    assert np.max(np.abs(y - exact)) <= 1e-3 * np.sqrt(np.mean(exact.astype(np.float64) ** 2))


# rows that are cast without a branch per vector and rows that are not, one and two to a wavefront, every length class
@pytest.mark.parametrize("scale", [3e-26, 1e-22, 1.0, 7e21, 2e28])
@pytest.mark.parametrize("M,K", [(1, 512), (8, 2048), (5, 4080), (8, 8192), (9, 1040), (16, 2048), (11, 4096), (7, 2560), (6, 2576), (8, 5120),
                                 (3, 5136)])
def test_fp8_rows_are_cast_like_the_oracle(oracle, M, K, scale):
    """The codes that the GEMV's own cast makes, read back through a weight of ones on the diagonal: scales on both sides of
    [2^-64, 2^64], outside of which the cast takes the full divide, values on and next to the midpoints of e4m3."""
    tab = oracle.np_e4m3fn_table().astype(np.float32)
    steps = np.sort(np.unique(np.concatenate([tab[:127], (tab[:126] + tab[1:127]) / 2])))
    g = torch.Generator().manual_seed(M * K)
    x = torch.from_numpy(steps)[torch.randint(0, len(steps), (M, K), generator=g)] * (1 - 2 * torch.randint(0, 2, (M, K), generator=g))
    x[:, ::3] = (torch.rand(M, (K + 2) // 3, generator=g) * 2 - 1) * 448
    x[M - 1, K - 1] = -448.0  # the largest: the scale is the one asked for, but for its rounding to bf16
    x = (x.double() * scale).to(BF16)
    xq, sx = oracle.c_quant_tensor_fp8(_bits(x), bf16_bits=True)
    w = torch.zeros(K, K, dtype=torch.uint8, device=DEV)
    w.diagonal().fill_(0x38)
    y = ops.gemv_fp8_decode(x.to(DEV), w, torch.ones(1, device=DEV), out_dtype=F32).cpu().numpy()
    assert np.array_equal(y, tab[xq] * np.float32(sx))


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("M,F,K", [(1, 16, 512), (8, 48, 1024), (9, 4112, 512), (16, 6912, 1536), (5, 5632, 2048), (13, 8272, 1536)])
def test_up_gate_swiglu_is_the_separate_launches(M, F, K, norm):
    g = torch.Generator(device=DEV).manual_seed(M + F)
    x = torch.randn(M, K, generator=g, device=DEV).to(BF16)
    wq = torch.randint(-127, 128, (2 * F, K), generator=g, device=DEV, dtype=torch.int8)
    sw = torch.rand(2 * F, generator=g, device=DEV) * 1e-3
    nm = ((1 + 0.2 * torch.randn(K, generator=g, device=DEV)).to(BF16), 1e-5) if norm else None
    h = ops.gemv_w8a8_decode_swiglu(x, wq, sw, norm=nm)
    ug = ops.gemv_w8a8_decode(x, wq, sw, norm=nm).float()
    u, gate = ug[:, :F], ug[:, F:]
    want = u * (gate / (1 + torch.exp(-gate)))
    assert torch.allclose(h.float(), want, rtol=8e-3, atol=1e-6)


@pytest.mark.parametrize("M,K", [(8, 6912), (9, 4112), (11, 6912), (16, 8192), (16, 2048)])
def test_rows_with_nan_and_infinities_equal_single_rows(M, K):
    """The row maximum by bits (more rows than keep their floats in registers) and by floats: NaN is left out of both, infinities and
    denormals count.  A batch gives each row what the row gives alone."""
    x = _rows(M, K, M * K).to(BF16)
    x[0, K - 1] = float("nan")
    x[1, 5], x[1, K // 2] = float("nan"), 1e4
    x[2, 77] = float("-inf")
    x[3] = float("nan")
    x[4], x[5] = 0.0, -0.0
    x[6] *= 1e-38
    x[7, 0], x[7, 1] = float("-nan"), float("inf")
    x[M - 1, 3] = -3e38
    wq = torch.randint(-127, 128, (300, K), generator=torch.Generator().manual_seed(K), dtype=torch.int8).to(DEV)
    sw = (torch.rand(300, generator=torch.Generator().manual_seed(5)) * 1e-3).to(DEV)
    x = x.to(DEV)
    got = ops.gemv_w8a8_decode(x, wq, sw).float()
    want = torch.cat([ops.gemv_w8a8_decode(x[m:m + 1], wq, sw) for m in range(M)]).float()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    assert bool(got[:2].isfinite().all()) and bool((got[4:6] == 0).all())
