"""CPU-side checks: the C-ABI library loads, exports every symbol the header
declares, rejects bad arguments before touching a GPU, and the host module keeps
the reference's Linear surface (astrai/model/components/linear.py:7-21) and swap
invariants (tests/module/test_lora.py in the reference)."""
import ctypes
import os
import re
import subprocess

import pytest
import torch
import torch.nn as nn

import khaosz_amd
from khaosz_amd import _abi, ops
from khaosz_amd.linear import Fp8Linear, Linear, QuantLinear, quantize_model

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "astrai_q.h")).read()
    declared = set(re.findall(r"\b(aq_[a-z0-9_]+)\s*\(", header))
    assert declared == set(_abi.SYMBOLS), declared ^ set(_abi.SYMBOLS)
    lib = _abi.load()
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.aq_version() == 100


def _kernel_notes(path, tmp_path):
    """{kernel: {.vgpr_spill_count, .private_segment_fixed_size, ..}} of the gfx950 code in a library built here."""
    llvm = "/opt/rocm/llvm/bin/"
    fat = tmp_path / "fat"
    subprocess.run([llvm + "llvm-objcopy", "-O", "binary", "--only-section=.hip_fatbin", path, str(fat)], check=True)
    blob, magic, notes = fat.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__", {}
    start = blob.find(magic)
    while start >= 0:  # a bundle per source file: magic, count, then (offset, size, length of the target's name, name) each
        at = start + len(magic) + 8
        for _ in range(int.from_bytes(blob[at - 8:at], "little")):
            offset, size, length = (int.from_bytes(blob[at + 8 * i:at + 8 * i + 8], "little") for i in range(3))
            if b"gfx950" in blob[at + 24:at + 24 + length]:
                obj = tmp_path / "obj"
                obj.write_bytes(blob[start + offset:start + offset + size])
                text = subprocess.run([llvm + "llvm-readelf", "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
                for kernel in text.split("- .agpr_count")[1:]:
                    fields = dict(re.findall(r"^ +(\.[a-z_]+): +(\S+)$", kernel, re.M))
                    notes[fields[".symbol"]] = fields
            at += 24 + length
        start = blob.find(magic, start + 1)
    return notes


def test_kernels_of_walked_tiles_keep_everything_in_registers(tmp_path):
    """A spilled value comes back through memory in front of the epilogue that needs it (12 of them: 7 % of the launch)."""
    walk = {k: v for k, v in _kernel_notes(_abi.LIB_PATH, tmp_path).items() if "gemm_walk_kernel" in k}
    assert len(walk) == 12
    assert {k: v for k, v in walk.items() if v[".vgpr_spill_count"] != "0" or v[".private_segment_fixed_size"] != "0"} == {}


def test_lab_library_holds_the_product_and_the_lab_symbols():
    """The probes and the tile-forcing hook live in a second library built from the same objects:
    the product library exports none of them."""
    lab_header = open(os.path.join(ROOT, "khaosz_amd", "csrc", "aq_lab.h")).read()
    declared = set(re.findall(r"\b(aq_lab_[a-z0-9_]+)\s*\(", lab_header))
    assert declared == set(_abi.LAB_SYMBOLS), declared ^ set(_abi.LAB_SYMBOLS)
    lab, lib = _abi.load_lab(), _abi.load()
    for name in declared:
        assert hasattr(lab, name), name
        assert not hasattr(lib, name), f"{name} leaked into the product library"
    for name in _abi.SYMBOLS:
        assert hasattr(lab, name), name
    assert lab.aq_lab_set_gemm_tile(3) == -2 and lab.aq_lab_set_gemm_tile(0) == 0


@pytest.mark.parametrize("ptr,nbytes,code", [(1 << 20, -128, -2), (0, 128, -1), ((1 << 20) + 2, 128, -4)])
def test_ranges_to_read_ahead_are_checked(ptr, nbytes, code):
    lib, P = _abi.load(), 1 << 20  # a fake pointer; refused before any launch
    good = [1 << 20, 1 << 10]
    spans = (ctypes.c_int64 * 4)(*good, ptr, nbytes)
    assert lib.aq_prefill_attn_causal_ahead(P, 64, P, 64, P, 64, P, 0.1, 1, 1, 1, 1, 64, ctypes.addressof(spans), 2, None) == code
    assert lib.aq_prefill_attn_paged_ahead(P, 64, P, P, P, 1, 0, 16, 1, P, 0.1, 1, 1, 1, 1, 64, ctypes.addressof(spans), 2, None) == code


def test_argument_validation_happens_before_any_launch():
    lib = _abi.load()
    P = 1 << 20  # a 16-byte aligned fake pointer; never dereferenced on these paths
    assert lib.aq_quant_rowwise_i8(P, 0, 4, 17, 17, P, P, None) == -2      # K % 16
    assert lib.aq_quant_rowwise_i8(P, 7, 4, 16, 16, P, P, None) == -3      # dtype
    assert lib.aq_quant_rowwise_i8(None, 0, 4, 16, 16, P, P, None) == -1   # null
    assert lib.aq_quant_rowwise_i8(P + 4, 0, 4, 16, 16, P, P, None) == -4  # alignment
    assert lib.aq_quant_rowwise_i8(P, 0, 4, 32, 16, P, P, None) == -2      # ldx < K
    assert lib.aq_quant_rowwise_i8(P, 0, 0, 16, 16, P, P, None) == 0       # empty is fine
    assert lib.aq_gemm_i8_i32(P, P, P, 4, 4, 24, None) == -2
    assert lib.aq_gemm_i8_i32(P, P, P, 0, 4, 32, None) == 0
    assert lib.aq_gemm_i8_i32(P, None, P, 4, 4, 32, None) == -1
    assert lib.aq_linear_w8a8(P, P, P, P, None, 0, P, 5, 4, 4, 32, None) == -3
    assert lib.aq_linear_w8a8(P, None, P, P, None, 0, P, 1, 4, 4, 32, None) == -1
    assert lib.aq_linear_fp8(P, P, P, P, P, 9, 4, 4, 32, None) == -3
    assert lib.aq_linear_fp8_residual(P, P, P, P, P, 7, None, P, 1, 4, 4, 32, None) == -3       # bias dtype
    assert lib.aq_linear_fp8_residual(P, P, P, P, None, 0, P + 2, P, 1, 4, 4, 32, None) == -4   # residual alignment
    assert lib.aq_gemv_w8a8_decode(P, 1, P, P, None, 0, P, 1, 17, 8, 32, P, 1 << 20, None) == -2  # M > 16
    assert lib.aq_gemv_w8a8_decode(P, 1, P, P, None, 0, P, 1, 4, 8, 32, P, 8, None) == -5         # workspace
    assert lib.aq_gemv_w8a8_decode(P, 1, P, P, None, 0, P + 2, 1, 4, 8, 32, P, 1 << 20, None) == -4  # y alignment
    assert lib.aq_gemv_w8a8_codes(P, P, P, P + 1, None, 0, P, 1, 4, 8, 32, None) == -4            # scale alignment
    assert lib.aq_linear_w8a8(P, P, P, P, None, 0, P, 1, 4, 1 << 21, 32, None) == -6              # N beyond the epilogue's offsets
    assert lib.aq_gemv_w8a8_workspace_bytes(16, 2048) >= 16 * 2048 + 64
    assert b"multiple of 16" in lib.aq_error_string(-2)
    with pytest.raises(ValueError):
        _abi.check(-2, "x")
    with pytest.raises(RuntimeError):
        _abi.check(-1, "x")


def test_ops_refuse_cpu_tensors_loudly():
    x = torch.randn(4, 32)
    with pytest.raises(RuntimeError, match="GPU only"):
        ops.quant_rowwise_i8(x)
    with pytest.raises(RuntimeError, match="GPU only"):
        ops.gemm_i8_i32(torch.zeros(4, 32, dtype=torch.int8), torch.zeros(4, 32, dtype=torch.int8))
    ql = QuantLinear(32, 16)
    with pytest.raises(RuntimeError, match="GPU only"):
        ql(x)
    lin = Linear(32, 16)
    lin.reset_parameters()
    with pytest.raises(RuntimeError, match="GPU"):
        QuantLinear.from_linear(lin)


def test_linear_keeps_the_reference_surface():
    torch.manual_seed(0)
    lin = Linear(24, 8)
    assert lin.bias is None and tuple(lin.weight.shape) == (8, 24)
    lin.reset_parameters()
    assert lin.weight.abs().max() <= 1 / 24 ** 0.5 + 1e-6
    x = torch.randn(2, 5, 24)
    assert torch.equal(lin(x), torch.nn.functional.linear(x, lin.weight))
    lb = Linear(24, 8, bias=True)
    lb.reset_parameters()
    assert set(lb.state_dict()) == {"weight", "bias"}
    assert torch.allclose(lb(x), x @ lb.weight.T + lb.bias, atol=1e-6)


def test_quant_linear_is_a_linear_with_quantized_state():
    q = QuantLinear(32, 16, bias=True)
    assert isinstance(q, Linear) and isinstance(q, nn.Module)
    assert set(q.state_dict()) == {"qweight", "w_scale", "bias"}
    assert q.qweight.dtype == torch.int8 and q.w_scale.dtype == torch.float32
    q.qweight.fill_(3)
    q.w_scale.fill_(0.5)
    assert torch.equal(q.weight, torch.full((16, 32), 1.5))
    assert q.in_dim == 32 and q.out_dim == 16
    f = Fp8Linear(32, 16)
    assert isinstance(f, Linear) and set(f.state_dict()) == {"qweight", "w_scale"}
    fb = Fp8Linear(32, 16, bias=True)
    assert set(fb.state_dict()) == {"qweight", "w_scale", "bias"} and tuple(fb.bias.shape) == (16,)
    with pytest.raises(RuntimeError):
        q.reset_parameters()


class _Block(nn.Module):
    def __init__(self):
        super().__init__()
        self.q_proj = Linear(32, 32)
        self.up = Linear(32, 64)
        self.lm_head = Linear(32, 100)
        self.other = nn.Linear(32, 32)


def test_quantize_model_walks_like_inject_lora_and_skips_untargeted(monkeypatch):
    # from_linear needs a GPU; stand in a recorder so the walk itself is tested on CPU
    made = []

    def fake(cls, base):
        made.append(base)
        return QuantLinear(base.weight.shape[1], base.weight.shape[0], bias=base.bias is not None)

    monkeypatch.setattr(QuantLinear, "from_linear", classmethod(fake))
    m = nn.Sequential(_Block(), _Block())
    n = quantize_model(m)
    assert n == 4 and len(made) == 4
    assert isinstance(m[0].q_proj, QuantLinear) and isinstance(m[1].up, QuantLinear)
    assert type(m[0].lm_head) is Linear and type(m[0].other) is nn.Linear
    keys = set(m.state_dict())
    assert "0.q_proj.qweight" in keys and "0.q_proj.w_scale" in keys and "0.lm_head.weight" in keys
    assert quantize_model(m) == 0  # idempotent: quantized layers are not float Linears
    with pytest.raises(ValueError):
        quantize_model(m, mode="int4")


def _reference_linear_class():
    """A class that looks, to code that never imports the reference, exactly like the reference's
    own Linear (astrai/model/components/linear.py:7-21): same name, same module path, same attributes
    and forward -- and no relation to this package's Linear."""

    class RefLinear(nn.Module):
        def __init__(self, in_dim, out_dim, bias=False):
            super().__init__()
            self.weight = nn.Parameter(torch.randn(out_dim, in_dim) * 0.05)
            self.bias = nn.Parameter(torch.zeros(out_dim)) if bias else None

        def forward(self, x):
            return nn.functional.linear(x, self.weight, self.bias)

    RefLinear.__name__ = RefLinear.__qualname__ = "Linear"
    RefLinear.__module__ = "astrai.model.components.linear"
    return RefLinear


def test_the_reference_class_is_recognised_by_name_without_importing_it(monkeypatch):
    from khaosz_amd.linear import _is_float_linear

    Ref = _reference_linear_class()
    assert not issubclass(Ref, Linear)
    assert _is_float_linear(Ref(16, 8), ())
    # the same class under another module path, or another name, is somebody else's layer
    Other = _reference_linear_class()
    Other.__module__ = "somewhere.else"
    assert not _is_float_linear(Other(16, 8), ())
    assert _is_float_linear(Other(16, 8), (Other,))  # unless the caller names its type
    Renamed = _reference_linear_class()
    Renamed.__name__ = "Dense"
    assert not _is_float_linear(Renamed(16, 8), ())
    assert not _is_float_linear(nn.Linear(16, 8), ())

    made = []

    def fake(cls, base):
        made.append(base)
        return QuantLinear(base.weight.shape[1], base.weight.shape[0], bias=base.bias is not None)

    monkeypatch.setattr(QuantLinear, "from_linear", classmethod(fake))

    class MLABlock(nn.Module):  # child names of the reference's MLA and DeepSeekMoE (attention.py:140-156, mlp.py:48-55)
        def __init__(self):
            super().__init__()
            self.q_proj, self.kv_a_proj, self.kv_b_proj, self.o_proj = Ref(32, 48), Ref(32, 16), Ref(16, 96), Ref(32, 32)
            self.router = Ref(32, 8)
            self.routed_experts = nn.ModuleList([_RefMLP(Ref) for _ in range(2)])

    class _Holder(nn.Module):
        def __init__(self):
            super().__init__()
            self.attn = MLABlock()
            self.up = Ref(8, 32)   # the reference's dim-8 test models: in_dim not a multiple of 16

    m = _Holder()
    n = quantize_model(m)
    # q/kv_a/kv_b/o + 2 experts x (up, gate, down); router stays float by default, `up` with in_dim 8 is skipped
    assert n == 4 + 6 and len(made) == n
    assert type(m.attn.router) is Ref and type(m.up) is Ref
    assert isinstance(m.attn.kv_a_proj, QuantLinear) and isinstance(m.attn.routed_experts[1].down, QuantLinear)
    assert quantize_model(m, target_modules={"router"}) == 1 and isinstance(m.attn.router, QuantLinear)


class _RefMLP(nn.Module):
    def __init__(self, L):
        super().__init__()
        self.up, self.gate, self.down = L(32, 64), L(32, 64), L(64, 32)


def test_package_exports():
    assert {"Linear", "QuantLinear", "Fp8Linear", "quantize_model"} <= set(dir(khaosz_amd))


def test_gemm_tile_choice_for_the_benchmark_shapes_and_a_few_hundred_rows():
    """The tile of a launch by tiles alone (int32 sums: no kernel that walks tiles or cuts K) is picked on the host from M, N and the
    number of compute units.  Pinned here for 256 compute units: the benchmark configurations keep the wide tiles (one round of
    256 tiles of 256 x 128 for the prefill configuration, 256 tiles of 128 x 128 for the FP8 one), a few hundred rows get the small
    tiles that still give every compute unit at most one tile, and a launch of many rounds never takes a small tile."""
    lab = _abi.load_lab()
    pick = lambda M, N: lab.aq_lab_choose_gemm_tile(M, N, 2048, 0, -1, 0, 256)
    assert pick(4096, 2048) == 256          # configuration 3: 256 tiles of 256 x 128, one round
    assert pick(2048, 2048) == 128          # configuration 4: 256 tiles of 128 x 128
    assert pick(8192, 8192) == 256
    assert pick(4096, 3072) == 256 and pick(4096, 11264) == 256   # block prefill: q/k/v, up/gate
    assert pick(2048, 13824) == 256         # model prefill, up/gate
    assert pick(64, 8192) == 33 and pick(48, 2048) == 33          # 64 x 32: 256 and 64 tiles
    assert pick(128, 8192) == 65            # 64 x 64: 256 tiles (64 x 32 would need two rounds)
    assert pick(256, 8192) == 64            # 128 x 64
    assert pick(128, 11264) == 64 and pick(64, 11264) == 65
    assert pick(384, 8192) == 128 and pick(512, 8192) == 128
    assert pick(768, 8192) == 256 and pick(1024, 8192) == 256
    assert pick(512, 2048) == 65 and pick(1024, 2048) == 64 and pick(256, 2048) == 33
    for M, N in ((8192, 8192), (100000, 4096), (1 << 20, 1 << 20)):
        assert pick(M, N) in (128, 256)
    for bad in ((0, 8, 64, 0, -1, 0, 256), (8, 8, 64, 0, -1, 0, 0), (8, 8, 24, 0, 1, 0, 256)):
        assert lab.aq_lab_choose_gemm_tile(*bad) == -2
    for bad in ((8, 8, 64, 1, -1, 0, 256), (8, 8, 64, 0, -1, 1, 256), (8, 8, 64, 0, 2, 0, 256)):  # FP8 sums, a residual on sums, no type
        assert lab.aq_lab_choose_gemm_tile(*bad) == -3


def test_gemm_tile_choice_where_tiles_are_walked_or_k_is_cut():
    """What a Linear's launch takes on 256 compute units: walked tiles of 256 x 128 (258) or 256 x 192 (192) with K from 512 and an even
    N, tiles with K cut among the wavefronts (34 to 43) for few rows, 256 x 256 (512) for some FP8 launches, else the tile above."""
    lab = _abi.load_lab()
    f32, bf16 = _abi.AQ_F32, _abi.AQ_BF16
    pick = lambda M, N, K, fp8=0, out=bf16, res=0: lab.aq_lab_choose_gemm_tile(M, N, K, fp8, out, res, 256)
    # block of 2048, 8 x 512 tokens: q/k/v, o, down; up/gate, whose last round is halved (5.55 rounds of 15 against 3.84 of 21.75; whole
    # it would be 5.75); the 24-layer model's up/gate on 4 x 512, halved too
    assert pick(4096, 3072, 2048) == 192 and pick(4096, 2048, 2048, res=1) == 258 and pick(4096, 2048, 5632, res=1) == 258
    assert pick(4096, 11264, 2048) == 258 and pick(2048, 13824, 1536) == 258
    # the residual's cost
    assert pick(3668, 4864, 512, fp8=1) == 192 and pick(3668, 4864, 512, fp8=1, res=1) == 258
    # what is not walked: short K, an odd N, a residual under fp32 outputs
    assert pick(4096, 3072, 496) == 256 and pick(4096, 3071, 2048) == 256
    assert pick(4096, 3072, 2048, out=f32) == 192 and pick(4096, 3072, 2048, out=f32, res=1) == 256
    # FP8: an odd number of 64-byte steps above 3072, a last round more than half full, whole rows of tiles, no residual
    assert pick(4864, 8640, 3264, fp8=1) == 512 and pick(4864, 8640, 3264) != 512
    for M, N, K, res in ((4864, 8640, 3328, 0), (4864, 8640, 3008, 0), (4863, 8640, 3264, 0), (4864, 8640, 3264, 1), (4096, 9216, 3264, 0),
                         (8192, 8192, 8192, 0)):
        assert pick(M, N, K, fp8=1, res=res) in (192, 258)
    # K cut among the wavefronts; a tile too many for that
    assert pick(64, 2048, 2048, out=f32) == 41 and pick(200, 2048, 6912) == 35 and pick(200, 2048, 1520) == 33
    assert pick(333, 1536, 6912, res=1) == 39
    # the smallest of which 256 are enough: 16 x 16, 16 x 32, 16 x 64 (up to 16 rows; then 16 x 32 in rounds), 32 x 16, 32 x 32
    for M, N, tile in ((16, 4096, 40), (16, 4097, 41), (16, 8192, 41), (16, 8193, 43), (16, 16384, 43), (16, 16385, 41), (17, 2048, 40), (17, 2049, 41),
                       (16, 1 << 20, 41), (32, 4096, 41), (32, 4097, 34), (2100, 48, 42), (33, 1360, 40), (33, 1361, 41), (64, 4096, 34), (64, 4097, 37)):
        assert pick(M, N, 1040) == pick(M, N, 1040, fp8=1, out=f32, res=1) == tile
    # 17 to 32 rows in whole lines of more outputs than those: weights streamed (31); no fewer rows, however long
    for M, N, K, tile in ((32, 12288, 1024, 37), (32, 12289, 1024, 31), (17, 12289, 11008, 31), (32, 12289, 1040, 65), (16, 12289, 11008, 43),
                          (9, 8193, 10240, 43), (8, 40000, 20480, 41), (33, 16384, 1024, 65)):
        assert pick(M, N, K) == pick(M, N, K, fp8=1, out=f32, res=1) == tile


def test_the_distance_between_rows_of_codes_is_one_that_their_quantiser_writes():
    """Rows on 128-byte lines where the quantisers write them (fewer than 2^31 vectors of four fp32 values) and the kernels take them as
    well as rows without a gap (31-bit offsets of the walked tiles); the 256 x 256 FP8 tile, which no residual takes, reads them as they are."""
    pitch = lambda M, N, K, fp8=1, res=0: _abi.load().aq_linear_codes_pitch(fp8, res, M, N, K)
    assert pitch(300, 1500, 1040) == 1152 and pitch(300, 1500, 1040, fp8=0) == 1152
    assert pitch(300, 1500, 1024) == 1024 and pitch(16, 1500, 1040) == 1040 and pitch(20, 1500, 0) == 0
    most = (1 << 33) // 8176  # rows of 8176 with fewer than 2^31 vectors of fp32
    for fp8 in (0, 1):
        assert pitch(most, 2048, 8176, fp8) == 8192 and pitch(most + 1, 2048, 8176, fp8) == 8176 and pitch(1100000, 2048, 8176, fp8) == 8176
    reach = 0x7ffffff0
    for M, want in ((reach // 7168, 7168), (reach // 7168 + 1, 7152), (reach // 7152, 7152), (reach // 7152 + 1, 7168)):
        assert pitch(M, 2048, 7152) == want and pitch(M, 2048, 7152, fp8=0) == want
    assert pitch(4864, 8640, 3264) == 3264 and pitch(4864, 8640, 3264, res=1) == 3328 and pitch(4864, 8640, 3264, fp8=0) == 3328
    for M in (0, -1, 1 << 31):
        assert pitch(M, 2048, 1040) == 1040
    # walked tiles (258, 192) read short rows as they are; the other tiles do not
    for M, N, K in ((6181, 1096, 720), (6020, 4400, 880), (7182, 4192, 1088), (8000, 8186, 1200), (4097, 2048, 2032)):
        assert _abi.load_lab().aq_lab_choose_gemm_tile(M, N, K, 0, _abi.AQ_BF16, 0, 256) in (258, 192)
        for fp8 in (0, 1):
            assert pitch(M, N, K, fp8) == pitch(M, N, K, fp8, res=1) == K
    for fp8 in (0, 1):
        assert pitch(4097, 2048, 2064, fp8) == 2176 and pitch(6181, 1095, 720, fp8) == 768 and pitch(700, 1600, 1040, fp8) == 1152


def test_one_launch_for_few_rows_where_the_host_pays_for_launches_and_in_a_graph():
    """Taken for less in a call on its own (int8 rows), where a launch saved is the host's time; FP8, whose bits depend on it, for the same."""
    lib = _abi.load()
    f32, bf16 = _abi.AQ_F32, _abi.AQ_BF16
    both = lambda dt, norm, fp8, M, N, K: (lib.aq_linear_few_rows_ok(dt, norm, fp8, M, N, K), lib.aq_linear_few_rows_queued_ok(dt, norm, fp8, M, N, K))
    assert both(f32, 0, 0, 64, 2048, 2048) == both(bf16, 0, 0, 125, 1824, 1216) == both(bf16, 1, 0, 93, 1184, 1072) == (1, 0)
    assert both(f32, 0, 0, 64, 2048, 512) == both(bf16, 0, 0, 32, 2048, 2048) == both(bf16, 1, 0, 32, 1024, 1024) == (1, 1)
    assert both(f32, 0, 0, 64, 2048, 4096) == both(bf16, 0, 0, 16, 512, 512) == both(bf16, 0, 0, 64, 8192, 2048) == (0, 0)
    for M in range(17, 200, 7):
        for N in (300, 1100, 2048, 5000):
            for K in range(16, 2064, 80):
                ok, queued = both(bf16, 0, 1, M, N, K)
                assert ok == queued
                for case in ((f32, 0, 0, M, N, K), (bf16, 0, 0, M, N, K), (bf16, 1, 0, M, N, K)):
                    ok, queued = both(*case)
                    assert ok >= queued


def test_quant_tensor_fp8_refuses_a_workspace_smaller_than_its_slots():
    """aq_quant_tensor_fp8 writes AQ_FP8_AMAX_WS_BYTES of partial maxima: a smaller workspace is refused before
    anything is launched (argument checks only: runs without a GPU)."""
    lib = _abi.load()
    dummy = 4096  # never dereferenced: the size check comes first
    assert lib.aq_quant_tensor_fp8(dummy, 1, 64, dummy, dummy, dummy, 4, None) == -5
    assert lib.aq_quant_tensor_fp8(dummy, 1, 64, dummy, dummy, dummy, _abi.AQ_FP8_AMAX_WS_BYTES - 1, None) == -5
    assert b"workspace" in lib.aq_error_string(-5).lower()
