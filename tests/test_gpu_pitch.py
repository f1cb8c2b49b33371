"""Codes whose rows begin further apart than they are long (on 128-byte lines): the quantisers that write them and every kernel that
multiplies them, against the same calls on rows without a gap -- which the parity tests hold to the oracle."""
import pytest
import torch

from khaosz_amd import Fp8Linear, QuantLinear, _abi, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16, F32 = torch.bfloat16, torch.float32


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _codes(rows, K, fp8, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, K, generator=g)
    return x.to(torch.float8_e4m3fn).view(torch.uint8).to(DEV) if fp8 else (x * 30).clamp(-127, 127).to(torch.int8).to(DEV)


# tile by tile (lab numbering) as the library picks them on 256 compute units: K of no whole number of 128-byte lines, ragged M and N
TILES = [(40, 40, 130, 1040), (41, 60, 1800, 1040), (42, 2100, 48, 1040), (43, 9, 12000, 1040), (34, 100, 2000, 1040), (39, 330, 1600, 3088), (36, 200, 1500, 1616), (37, 60, 6000, 272), (38, 70, 5000, 1040), (35, 200, 2048, 1616), (33, 200, 2048, 272), (65, 330, 1536, 1040), (64, 700, 1600, 2064),
         (128, 1500, 1537, 336), (258, 2000, 2050, 1040), (192, 4000, 3070, 528), (256, 4097, 2049, 624), (258, 6000, 8186, 1008)]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("out", [BF16, F32])
@pytest.mark.parametrize("tile,M,N,K", TILES)
def test_a_gap_between_rows_changes_no_bit(tile, M, N, K, out, fp8):
    lib, code = _abi.load(), _abi.AQ_BF16 if out == BF16 else _abi.AQ_F32
    if out == BF16:
        assert _abi.load_lab().aq_lab_choose_gemm_tile(M, N, K, int(fp8), code, 0, 256) == tile
    a, w = _codes(M, K, fp8, 1), _codes(N, K, fp8, 2)
    sx, sw = torch.rand(1 if fp8 else M, device=DEV) * 1e-2, torch.rand(1 if fp8 else N, device=DEV) * 1e-2
    bias, res = torch.randn(N, device=DEV), torch.randn(M, N, device=DEV).to(out)
    fn = lib.aq_linear_fp8_strided if fp8 else lib.aq_linear_w8a8_strided
    got = []
    for ld in (K, (K + 127) // 128 * 128, K + 16):
        rows = torch.full((M, ld), 0x7F, dtype=a.dtype, device=DEV)  # the gap holds large values (e4m3: NaN), which no sum may meet
        rows[:, :K] = a
        y = torch.full((M, N), float("nan"), device=DEV, dtype=out)
        rc = fn(rows.data_ptr(), ld, sx.data_ptr(), w.data_ptr(), sw.data_ptr(), bias.data_ptr(), _abi.AQ_F32, res.data_ptr(), y.data_ptr(), code,
                M, N, K, _stream())
        assert rc == 0
        got.append(y)
    assert torch.isfinite(got[0]).all()
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("K", [1392, 1424, 1520, 1648, 2032])
@pytest.mark.parametrize("tile,M,N", [(65, 330, 1536), (65, 321, 1535), (64, 700, 1600), (64, 700, 1603), (128, 1500, 2050), (256, 6700, 1345)])
def test_weights_that_begin_anywhere_in_a_line(tile, M, N, K, fp8):
    """Around the length from which the tiles load the weights by lines: the same steps as on rows filled with zeros to whole lines, hence the
    same bits; a row of large values (e4m3: NaN) shows in its own column only."""
    lib = _abi.load()
    assert _abi.load_lab().aq_lab_choose_gemm_tile(M, N, K, int(fp8), _abi.AQ_BF16, 0, 256) == tile
    ld = (K + 127) // 128 * 128
    a, w = _codes(M, K, fp8, 3), _codes(N, K, fp8, 4)
    w[N // 2] = 0x7F
    rows, full = torch.zeros(M, ld, dtype=a.dtype, device=DEV), torch.zeros(N, ld, dtype=a.dtype, device=DEV)
    rows[:, :K], full[:, :K] = a, w
    sx, sw = torch.rand(1 if fp8 else M, device=DEV) * 1e-2, torch.rand(1 if fp8 else N, device=DEV) * 1e-2
    fn = lib.aq_linear_fp8_strided if fp8 else lib.aq_linear_w8a8_strided
    for out in (BF16, F32):
        code = _abi.AQ_BF16 if out == BF16 else _abi.AQ_F32
        want = torch.empty(M, N, device=DEV, dtype=out)
        assert fn(rows.data_ptr(), ld, sx.data_ptr(), full.data_ptr(), sw.data_ptr(), None, 0, None, want.data_ptr(), code, M, N, ld, _stream()) == 0
        assert torch.isfinite(want).sum().item() == M * (N - 1 if fp8 else N)
        for start in (0, 16, 80):
            base = torch.empty(N * K + 128, dtype=w.dtype, device=DEV)
            b = base[start:start + N * K].view(N, K)
            b.copy_(w)
            y = torch.zeros(M, N, device=DEV, dtype=out)
            assert fn(rows.data_ptr(), ld, sx.data_ptr(), b.data_ptr(), sw.data_ptr(), None, 0, None, y.data_ptr(), code, M, N, K, _stream()) == 0
            assert torch.equal(torch.nan_to_num(y, 7.0), torch.nan_to_num(want, 7.0))


@pytest.mark.parametrize("K", [6016, 6144, 6272, 6400, 6528, 6656, 6784])
@pytest.mark.parametrize("tile", [128, 64, 65, 33])
def test_long_rows_in_whole_turns_of_the_stages(tile, K):
    """Around the length from which a turn of the loop is as many steps as there are stages, with every remainder of 3, 4 and 6: the bits of
    the tile that goes step by step (sums run in the same order)."""
    M, N = 150, 200
    a, w, a8, w8 = _codes(M, K, False, 5), _codes(N, K, False, 6), _codes(M, K, True, 7), _codes(N, K, True, 8)
    sx, sw, r = torch.rand(M, device=DEV) * 1e-2, torch.rand(N, device=DEV) * 1e-2, torch.randn(M, N, device=DEV).to(BF16)
    run = lambda: (ops.linear_w8a8(a, sx, w, sw, None, out_dtype=F32), ops.linear_w8a8(a, sx, w, sw, None, out_dtype=BF16, residual=r),
                   ops.linear_fp8(a8, sx[:1], w8, sw[:1], None, out_dtype=F32))
    with _abi.lab_library() as lab:
        assert lab.aq_lab_set_gemm_tile(tile) == 0
        got = run()
        assert lab.aq_lab_set_gemm_tile(256) == 0
        for y, want in zip(got, run()):
            assert torch.isfinite(y).all() and torch.equal(y, want)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("M,K", [(1, 48), (70, 1040), (70, 2064), (300, 4112), (5000, 272), (300, 9008), (20, 16400)])
def test_quantisers_write_rows_with_a_gap(M, K, dtype):
    lib, code = _abi.load(), _abi.AQ_BF16 if dtype == BF16 else _abi.AQ_F32
    x = (torch.randn(M, K, device=DEV) * 3).to(dtype)
    ld = (K + 127) // 128 * 128
    q, s = torch.full((M, ld), 77, dtype=torch.int8, device=DEV), torch.empty(M, device=DEV)
    assert lib.aq_quant_rowwise_i8_strided(x.data_ptr(), code, M, K, K, q.data_ptr(), ld, s.data_ptr(), _stream()) == 0
    want, ws = ops.quant_rowwise_i8(x)
    assert torch.equal(q[:, :K], want) and torch.equal(s, ws) and bool((q[:, K:] == 77).all())
    want, ws = ops.quant_tensor_fp8(x)
    for state in (None, ops.fp8_onepass_state(x.device)):
        q, s = ops.quant_tensor_fp8(x, state=state, onepass=state is not None, pitch=ld)
        assert q.stride() == (ld, 1) and torch.equal(q, want) and torch.equal(s, ws)


def test_distances_that_are_refused():
    lib = _abi.load()
    x, q, s = torch.zeros(32, 64, device=DEV, dtype=BF16), torch.zeros(64 * 64, device=DEV, dtype=torch.int8), torch.ones(64, device=DEV)
    p, qp, sp = x.data_ptr(), q.data_ptr(), s.data_ptr()
    for ld, rc in ((48, -2), (72, -4)):  # AQ_E_SHAPE, AQ_E_ALIGN
        assert lib.aq_quant_rowwise_i8_strided(p, _abi.AQ_BF16, 32, 64, 64, qp, ld, sp, _stream()) == rc
        assert lib.aq_quant_tensor_fp8_strided(p, _abi.AQ_BF16, 32, 64, qp, ld, sp, qp, 1024, _stream()) == rc
        assert lib.aq_linear_w8a8_strided(qp, ld, sp, qp, sp, None, 0, None, p, _abi.AQ_BF16, 32, 32, 64, _stream()) == rc
    with pytest.raises(ValueError):
        ops.quant_tensor_fp8(x.view(-1), pitch=128)


@pytest.mark.parametrize("M,N,K,step", [(3, 48, 64, 1 << 23), (3, 48, 64, (1 << 22) + 16), (3, 48, 64, 1 << 22), (40, 300, 1040, 4176), (40, 300, 1040, 1048)])
def test_codes_whose_rows_lie_anywhere(M, N, K, step):
    """Rows up to and beyond the distance that the entry point takes, and rows that are no multiple of 16 bytes apart: codes that the kernels
    cannot read in place are copied, as they always were."""
    a, w = _codes(M, K, True, 9), _codes(N, K, True, 10)
    rows = torch.empty((M - 1) * step + K, dtype=torch.uint8, device=DEV).as_strided((M, K), (step, 1))
    rows.copy_(a)
    one = torch.full((1,), 0.01, device=DEV)
    for out in (BF16, F32):
        assert torch.equal(ops.linear_fp8(rows, one, w, one, None, out_dtype=out), ops.linear_fp8(a, one, w, one, None, out_dtype=out))


@pytest.mark.parametrize("M,N,K", [(40, 6000, 1040), (300, 1601, 2064), (2100, 1040, 4016), (1500, 2048, 1024)])
def test_layers_give_the_bits_of_their_operators(M, N, K):
    """(2100 x 4016 bf16 values: the FP8 quantiser's one-launch form)"""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).to(BF16).to(DEV)
    res = torch.randn(M, N, generator=g).to(BF16).to(DEV)
    base = torch.nn.Linear(K, N, bias=True).to(DEV).to(BF16)
    q, f = QuantLinear.from_linear(base), Fp8Linear.from_linear(base)
    with torch.inference_mode():
        for _ in range(2):
            xq, sx = ops.quant_rowwise_i8(x)
            assert torch.equal(q(x, residual=res), ops.linear_w8a8(xq, sx, q.qweight, q.w_scale, q.bias, residual=res))
            xq, sx = ops.quant_tensor_fp8(x)
            assert torch.equal(f(x, residual=res), ops.linear_fp8(xq, sx, f.qweight, f.w_scale, f.bias, residual=res))
