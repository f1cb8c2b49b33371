"""Rows at the ends of the classes by which a launch takes them, against the CPU oracle: the row quantiser's (csrc/quant.hip), and the
tiles of up to 16 rows of a launch that quantises more than 16 itself (csrc/gemv_rows.hip)."""
import ctypes

import numpy as np
import pytest
import torch

from khaosz_amd import QuantLinear, _abi, ops

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


def _few_rows(x, wq, sw, bias=None, residual=None, gamma=None, fp8=False):
    """aq_linear_few_rows on a shape that it takes"""
    lib, (M, K), N = _abi.load(), x.shape, wq.shape[0]
    code = _abi.AQ_BF16 if x.dtype == BF16 else _abi.AQ_F32
    p = lambda t: None if t is None else t.data_ptr()
    assert lib.aq_linear_few_rows_ok(code, int(gamma is not None), int(fp8), M, N, K) == 1
    y = torch.full((M, N), float("nan"), device=DEV, dtype=x.dtype)
    rc = lib.aq_linear_few_rows(p(x), code, p(gamma), 1e-5, p(wq), int(fp8), p(sw), p(bias), _abi.AQ_F32, p(residual), p(y), code, M, N, K,
                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return y


# tiles of up to 8 and of 9..16 rows, whole and with a last one of fewer; N inside workgroups of each height; K at line and class edges
TILED = [(17, 513, 528), (18, 1537, 1024), (24, 2048, 512), (25, 100, 1040), (31, 1500, 2048), (32, 2048, 2048), (33, 700, 1024), (48, 1600, 1008),
         (63, 37, 1024), (64, 2048, 512), (65, 513, 272), (97, 300, 1024)]


LONG = [(17, 520, 2064, BF16), (18, 300, 3072, BF16), (17, 1030, 4096, BF16), (20, 1000, 8192, F32)]  # and of the longer classes of rows


@pytest.mark.parametrize("M,N,K,dtype", [(*c, d) for c in TILED for d in (BF16, F32)] + LONG)
def test_tiles_of_rows_bit_exact(oracle, M, N, K, dtype):
    x = _rows(M, K, M + K).to(dtype)
    g = torch.Generator().manual_seed(N)
    wq = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    sw, bias = torch.rand(N, generator=g) * 1e-3, torch.randn(N, generator=g) * 0.1
    res = torch.randn(M, N, generator=g).to(dtype).to(DEV)
    args = x.to(DEV), wq.to(DEV), sw.to(DEV), bias.to(DEV)
    y = _few_rows(*args)
    bf = dtype == BF16
    want = oracle.c_linear_w8a8(_bits(x) if bf else x.numpy(), wq.numpy(), sw.numpy(), bias.numpy(), x_bf16_bits=bf, bf16_out=bf)
    assert np.array_equal(_bits(y) if bf else y.cpu().numpy().view(np.uint32), want if bf else want.view(np.uint32))
    assert torch.equal(_few_rows(*args, residual=res), y + res)


@pytest.mark.parametrize("M,N,K", [c for c in TILED if c[2] <= 2048])
def test_tiles_of_rows_with_the_norm_bit_exact(oracle, M, N, K):
    x = _rows(M, K, M + K).to(BF16)
    g = torch.Generator().manual_seed(N)
    gam = (1 + 0.2 * torch.randn(K, generator=g)).to(BF16)
    wq, sw = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8), torch.rand(N, generator=g) * 1e-3
    y = _few_rows(x.to(DEV), wq.to(DEV), sw.to(DEV), gamma=gam.to(DEV))
    qx, sx = oracle.c_rmsnorm_quant_i8(_bits(x), _bits(gam), 1e-5, bf16_bits=True)
    want = oracle.c_dequant_epilogue(oracle.c_gemm_i8_i32(qx, wq.numpy()), sx, sw.numpy(), None, bf16_out=True)
    assert np.array_equal(_bits(y), want)


@pytest.mark.parametrize("largest_in", [0, -1])  # the row whose value sets the tensor's scale: of the first tile, of the last
@pytest.mark.parametrize("M,N,K", [c for c in TILED if c[2] < 2048 and c[0] != 48] + [(17, 2000, 2048), (32, 1024, 2048), (48, 512, 2048)])
def test_tiles_of_fp8_rows_within_tolerance(oracle, M, N, K, largest_in):
    """bf16 outputs: a quarter of a per cent each way from rounding, and the sums as in the decode tests (1e-3 of the rms)."""
    x = _rows(M, K, M + K).to(BF16)
    x[largest_in, K - 1] = 60.0
    w = _rows(N, K, N) * 0.02
    xq, sx = oracle.c_quant_tensor_fp8(_bits(x), bf16_bits=True)
    wq, sw = oracle.c_quant_tensor_fp8(w.numpy())
    y = _few_rows(x.to(DEV), torch.from_numpy(wq).to(DEV), torch.tensor([sw], device=DEV), fp8=True).float().cpu().numpy()
    exact = oracle.np_linear_fp8(xq, sx, wq, sw)
    assert np.all(np.abs(y - exact) <= 2.0 ** -8 * np.abs(exact) + 1e-3 * np.sqrt(np.mean(exact.astype(np.float64) ** 2)))


@pytest.mark.parametrize("M", [17, 32, 60])
def test_a_layer_gives_the_bits_of_its_two_launches(M):
    g = torch.Generator().manual_seed(M)
    layer = QuantLinear(1024, 1536).to(DEV)
    layer.load_float_weight(torch.randn(1536, 1024, generator=g).to(DEV) * 0.02)
    x, res = torch.randn(M, 1024, generator=g).to(BF16).to(DEV), torch.randn(M, 1536, generator=g).to(BF16).to(DEV)
    with torch.inference_mode():
        got = layer(x, residual=res)
        want = ops.linear_w8a8(*ops.quant_rowwise_i8(x), layer.qweight, layer.w_scale, None, out_dtype=BF16, residual=res)
    assert torch.equal(got, want)


def test_shapes_that_take_two_launches_are_refused():
    lib = _abi.load()
    x = torch.zeros(64, 2048, device=DEV, dtype=BF16)
    for M, N, K, fp8, norm in ((16, 512, 512, 0, 0), (64, 8192, 2048, 0, 0), (64, 512, 504, 0, 0), (17, 512, 512, 1, 1), (17, 300, 4112, 0, 1)):
        assert lib.aq_linear_few_rows_ok(_abi.AQ_BF16, norm, fp8, M, N, K) == 0
    p = x.data_ptr()
    assert lib.aq_linear_few_rows(p, _abi.AQ_BF16, None, 0.0, p, 0, p, None, 0, None, p, _abi.AQ_BF16, 64, 8192, 2048, None) == -6  # AQ_E_RANGE
    assert lib.aq_linear_few_rows(p, _abi.AQ_BF16, p, -1.0, p, 0, p, None, 0, None, p, _abi.AQ_BF16, 32, 512, 512, None) == -2  # AQ_E_SHAPE


def _kernel_launches(graph):
    hip = ctypes.CDLL(next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l))
    n = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("M,N,K,dtype,norm,launches", [(64, 2048, 2048, F32, False, 2), (125, 1824, 1216, BF16, False, 2), (93, 1184, 1072, BF16, True, 2),
                                                       (64, 2048, 512, F32, False, 1), (32, 2048, 2048, BF16, False, 1), (32, 1024, 1024, BF16, True, 1)])
def test_a_captured_layer_takes_the_launches_that_are_faster_in_a_graph(M, N, K, dtype, norm, launches):
    """Where one launch only saves the host's time for a second (the first three), a graph has the two; the same bits on every replay."""
    layer = QuantLinear.from_linear(torch.nn.Linear(K, N).to(DEV).to(dtype))
    kw = {"norm": (torch.ones(K, device=DEV, dtype=dtype), 1e-5)} if norm else {}
    x = _rows(M, K, M).to(dtype).to(DEV)
    with torch.inference_mode():
        for _ in range(2):
            layer(x, **kw)
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            y = layer(x, **kw)
        assert _kernel_launches(graph) == launches
        for i in range(3):
            x.copy_(_rows(M, K, 100 + i).to(dtype))
            want = layer(x, **kw)
            graph.replay()
            assert torch.equal(y, want)


# vectors of 16 bytes around the sizes that one launch covers with 1, 4, 8 and 12 (fp32: 16) per thread, and beyond
@pytest.mark.parametrize("dtype,vectors", [(BF16, v) for v in (2, 1024, 1026, 4096, 4098, 8192, 8194, 12288, 12290)] +
                         [(F32, v) for v in (4, 1024, 1028, 4096, 4100, 8192, 8196, 16384, 16388)])
def test_small_tensors_are_cast_in_one_launch(oracle, dtype, vectors):
    n = vectors * (8 if dtype == BF16 else 4)
    x = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 3).to(dtype)
    x[0], x[n // 2] = -0.0, 0.0
    for last, scale in ((99.0, 1.0), (-77.0, 1e-3), (5.0, 2.0 ** -60)):  # the maximum in the last vector
        y = x * scale
        y[n - 1] = last * scale
        q, s = ops.quant_tensor_fp8(y.to(DEV))
        qo, so = oracle.c_quant_tensor_fp8(_bits(y) if dtype == BF16 else y.numpy(), bf16_bits=dtype == BF16)
        assert np.array_equal(q.cpu().numpy().reshape(-1), qo.reshape(-1)) and s.item() == float(so)
    state = ops.fp8_onepass_state(torch.device(DEV))
    for special in (float("inf"), float("nan"), 0.0):  # as the form for large tensors has them
        y = x * 0 if special == 0.0 else x.clone()
        y[n - 3] = special
        q, s = ops.quant_tensor_fp8(y.to(DEV))
        want, ws = ops.quant_tensor_fp8(y.to(DEV), state=state, onepass=True)
        assert torch.equal(q, want) and torch.equal(s.view(torch.int32), ws.view(torch.int32))
