"""The tiles whose K is cut among the wavefronts of a workgroup, in steps of 16 rows and outputs: each of them against the oracle, and the
rule that takes a call to them against one of them."""
import numpy as np
import pytest
import torch

from khaosz_amd import _abi, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def bf16_bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def to_np(t):
    return t.detach().cpu().numpy()


# 48 x 32, 32 x 48, 32 x 64, 48 x 48, 16 x 16, 16 x 32, 32 x 16, 16 x 64: fewer K steps than wavefronts, K that ends in a step and at one's end, ragged rows and outputs, odd N
@pytest.mark.parametrize("kind", [36, 37, 38, 39, 40, 41, 42, 43])
@pytest.mark.parametrize("M,N,K", [(1, 40, 16), (17, 33, 16), (33, 97, 400), (97, 130, 1040), (65, 1001, 2064), (49, 64, 2048), (200, 512, 1936)])
def test_tiles_of_sixteens(oracle, M, N, K, kind):
    rng = np.random.default_rng(M + N + K)
    xq, wq = (rng.integers(-128, 128, (n, K), dtype=np.int8) for n in (M, N))
    sx, sw = (rng.random(n, dtype=np.float32) * 0.01 + 1e-4 for n in (M, N))
    b = rng.standard_normal(N).astype(np.float32)
    acc = oracle.c_gemm_i8_i32(xq, wq)
    d = [torch.from_numpy(t).to(DEV) for t in (xq, sx, wq, sw, b)]
    with _abi.lab_library() as lab:
        assert lab.aq_lab_set_gemm_tile(kind) == 0
        for out in (torch.bfloat16, torch.float32):
            bias = d[4].to(torch.bfloat16) if out is torch.bfloat16 else d[4]
            y = ops.linear_w8a8(d[0], d[1], d[2], d[3], bias, out_dtype=out)
            want = oracle.c_dequant_epilogue(acc, sx, sw, bias.float().cpu().numpy(), bf16_out=out is torch.bfloat16)
            assert np.array_equal(bf16_bits(y) if out is torch.bfloat16 else to_np(y), want)
            res = torch.randn(M, N, device=DEV, dtype=out)
            assert torch.equal(ops.linear_w8a8(d[0], d[1], d[2], d[3], bias, out_dtype=out, residual=res), y + res)
        x8, w8 = (torch.from_numpy(rng.standard_normal((n, K)).astype(np.float32)).to(DEV).to(torch.float8_e4m3fn) for n in (M, N))
        y = ops.linear_fp8(x8.view(torch.uint8), d[1][:1], w8.view(torch.uint8), d[3][:1], None, out_dtype=torch.float32)
    a, c = x8.float().cpu().double(), w8.float().cpu().double()
    # the matrix products of e4m3 values line a step's products up to the largest of them and cut off what is below: up to 5.4e-5 of the sum
    # of the magnitudes at K 16 (alike in 16 x 16 and in 32 x 32 products), less in longer sums; then K roundings of fp32
    bound = (6e-5 + (K + 2) * 2.0 ** -24) * (a.abs() @ c.abs().T) * float(sx[0]) * float(sw[0])
    assert ((y.cpu().double() - (a @ c.T) * float(sx[0]) * float(sw[0])).abs() <= bound).all()


# Both sides of the rule's lines on 256 compute units: 256 tiles of a shape and a few more, K 512 and 3072, 64 rows
@pytest.mark.parametrize("M,N,K,tile", [(64, 4096, 528, 34), (96, 4096, 528, 36), (97, 2752, 528, 37), (64, 4097, 528, 37), (64, 8192, 528, 33),
                                        (65, 4100, 512, 38), (65, 4100, 496, 65), (32, 12288, 272, 37), (333, 1536, 3072, 39),
                                        (333, 1536, 3056, 65), (336, 1728, 3088, 39), (336, 1729, 3088, 65), (64, 6145, 3088, 35), (16, 4096, 528, 40),
                                        (16, 4097, 528, 41), (33, 1360, 528, 40), (33, 1361, 528, 41), (9, 8193, 528, 43), (3, 16385, 272, 41),
                                        (32, 2048, 1040, 40), (32, 2049, 1040, 41), (17, 4097, 1040, 34), (2100, 48, 528, 42)])
def test_the_rule_for_tiles_of_sixteens(M, N, K, tile):
    """Whichever tile the rule takes, int8 sums are the bits of the 64 x 64 tile; FP8 sums differ by their order alone: fp32 sums of K
    products by at most 2 K 2^-24 of the sum of their magnitudes, bf16 results by a rounding more."""
    assert _abi.load_lab().aq_lab_choose_gemm_tile(M, N, K, 0, _abi.AQ_BF16, 0, 256) == tile
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    xq, wq = (torch.randint(-128, 128, (n, K), generator=g, device=DEV, dtype=torch.int8) for n in (M, N))
    sx, sw = (torch.rand(n, generator=g, device=DEV) * 0.01 + 1e-4 for n in (M, N))
    x8, w8 = (torch.randn(n, K, generator=g, device=DEV).to(torch.float8_e4m3fn) for n in (M, N))
    run = lambda: (ops.linear_w8a8(xq, sx, wq, sw, None, out_dtype=torch.bfloat16),
                   ops.linear_fp8(x8.view(torch.uint8), sx[:1], w8.view(torch.uint8), sw[:1], None, out_dtype=torch.bfloat16))
    got = run()
    with _abi.lab_library() as lab:
        assert lab.aq_lab_set_gemm_tile(65) == 0
        want = run()
    assert torch.equal(got[0], want[0])
    sums = (x8.float().abs() @ w8.float().abs().T) * (sx[0] * sw[0])
    diff = (got[1].float() - want[1].float()).abs()
    assert (diff <= 2.0 ** -7 * want[1].float().abs() + 2 * K * 2.0 ** -24 * sums).all()


@pytest.mark.parametrize("M,N,K", [(1, 300, 256), (9, 4100, 512), (12, 816, 6416), (16, 8200, 4352), (5, 16400, 272), (9, 130, 8448), (12, 8200, 11008), (16, 200, 10240)])
def test_up_to_sixteen_rows_of_codes(M, N, K):
    """FP8 rows that are cast by a launch of their own (K in whole 256-byte steps and not): against fp64 sums, with a bias and a residual."""
    g = torch.Generator().manual_seed(M + N + K)
    x8, w8 = (torch.randn(n, K, generator=g).to(torch.float8_e4m3fn) for n in (M, N))
    bias, res = torch.randn(N, generator=g), torch.randn(M, N, generator=g)
    one = torch.ones(1, device=DEV)
    y = ops.gemv_fp8_codes(x8.view(torch.uint8).to(DEV), one, w8.view(torch.uint8).to(DEV), one, bias.to(DEV), out_dtype=torch.float32, residual=res.to(DEV))
    a, c = x8.double(), w8.double()
    want = a @ c.T + bias.double() + res.double()
    bound = (6e-5 + (K + 4) * 2.0 ** -24) * (a.abs() @ c.abs().T) + 2.0 ** -22 * (want.abs() + bias.abs() + res.abs())  # as above, and two additions
    assert ((y.cpu().double() - want).abs() <= bound).all()
