"""The native host path (csrc/host.cpp): a fused block queued in one call gives the bits of the step-by-step path, keeps out of
the way of hooks and replaced operators, and operators fed with what the native functions do not take still answer."""
import ctypes
import pathlib
import subprocess
import sys
import threading

import pytest
import torch

from khaosz_amd import Fp8Linear, QuantLinear, _abi, fuse_shared_inputs, ops, quantize_model
from khaosz_amd.block import GQA, MLP, DecoderBlock, PagedKV, rotary_table

pytestmark = pytest.mark.gpu
DEV, DT = "cuda:0", torch.bfloat16


def _block(hidden=512, heads=8, kv=2, ffn=1408, **kw):
    torch.manual_seed(3)
    b = DecoderBlock(hidden, heads, ffn, kv, **kw)
    b.reset_parameters()
    b = b.to(DEV).to(DT)
    quantize_model(b)
    fuse_shared_inputs(b, norms=True, decode_attention=True, residuals=True)
    return b


def _case(b, B, S, cached, kv=2, d=64, page=32, unmapped=False):
    P = (cached + S + page - 1) // page
    table = torch.randperm(B * P, device=DEV).view(B, P)
    if unmapped:
        table[0, 0] = -1
    cache = PagedKV(B * P, page, kv, d, DEV, DT)
    cache.k_layers.normal_()
    cache.v_layers.normal_()
    fr = rotary_table(d, 4096, device=DEV)[cached:cached + S].unsqueeze(0).expand(B, -1, -1)
    return torch.randn(B, S, kv * 4 * d, device=DEV).to(DT), fr, cache, table


@pytest.mark.parametrize("qk_norm", [False, True])
@pytest.mark.parametrize("B,S,cached,unmapped", [
    (1, 1, 0, False), (4, 1, 299, False), (8, 1, 1100, False), (16, 1, 40, False), (17, 1, 70, False),  # decode rows
    (1, 2, 0, False), (3, 5, 0, False), (2, 45, 0, False), (2, 33, 51, False), (1, 3, 9, False), (2, 20, 0, True)])
def test_block_in_one_call_is_the_step_by_step_path(monkeypatch, qk_norm, B, S, cached, unmapped):
    b = _block(use_qk_norm=qk_norm)
    x, fr, cache, table = _case(b, B, S, cached, unmapped=unmapped)
    k0, v0 = cache.k_layers.clone(), cache.v_layers.clone()
    cache.bind(table, cached + S)
    lens = (cached + 1 - torch.arange(B, device=DEV).clamp(max=cached)) if S == 1 else None
    got = []
    with torch.inference_mode():
        for stepwise in (False, True):
            cache.k_layers.copy_(k0)
            cache.v_layers.copy_(v0)
            cache.seq_lens = lens
            if stepwise:  # a replaced operator: every call goes through it
                calls = []
                real = ops.rmsnorm_quant_rowwise_i8, ops.gemv_w8a8_decode
                monkeypatch.setattr(ops, "rmsnorm_quant_rowwise_i8", lambda *a: (calls.append(1), real[0](*a))[1])
                monkeypatch.setattr(ops, "gemv_w8a8_decode", lambda *a, **k: (calls.append(1), real[1](*a, **k))[1])
            y = b(x, fr, None, cache)
            got.append((y, cache.k_layers.clone(), cache.v_layers.clone()))
        assert calls
    for a, c in zip(*got):
        assert torch.equal(a, c)


@pytest.mark.parametrize("hidden,qk_norm,B,S,cached", [
    (512, False, 4, 1023, 0), (512, False, 4, 1025, 0), (512, False, 5, 900, 37), (512, True, 8, 1023, 0), (512, True, 8, 1025, 0),
    (512, True, 9, 950, 70), (1024, False, 3, 683, 0), (1024, False, 4, 600, 51), (1024, True, 5, 820, 0), (1024, True, 6, 700, 100)])
def test_block_that_rotates_queries_in_attention_is_the_step_by_step_path(monkeypatch, hidden, qk_norm, B, S, cached):
    """Prompts on both sides of the sizes from which the block has the attention rotate (and normalise) its queries."""
    d = hidden // 8
    b = _block(hidden=hidden, use_qk_norm=qk_norm)
    if qk_norm:
        with torch.no_grad():
            for norm in (b.attention.q_norm, b.attention.k_norm):
                norm.weight.copy_(torch.rand(d, device=DEV) + 0.5)
    x, fr, cache, table = _case(b, B, S, cached, d=d, page=64)
    cache.bind(table, cached + S)
    k0, v0 = cache.k_layers.clone(), cache.v_layers.clone()
    with torch.inference_mode():
        got = b(x, fr, None, cache), cache.k_layers.clone(), cache.v_layers.clone()
        cache.k_layers.copy_(k0)
        cache.v_layers.copy_(v0)
        calls = _counted(monkeypatch, ops, "rope_kv_write")  # a replaced operator: the step-by-step path serves
        want = b(x, fr, None, cache), cache.k_layers, cache.v_layers
    assert len(calls) == 1
    for a, c in zip(got, want):
        assert torch.equal(a, c)


def test_hooks_on_a_fused_blocks_children_still_run():
    b = _block()
    x, fr, cache, table = _case(b, 2, 1, 30)
    cache.bind(table, 31)
    seen = []
    with torch.inference_mode():
        want = b(x, fr, None, cache)
        h = b.mlp.down.register_forward_hook(lambda m, a, y: seen.append(tuple(y.shape)))
        assert torch.equal(b(x, fr, None, cache), want) and len(seen) == 1
        h.remove()
        assert torch.equal(b(x, fr, None, cache), want) and len(seen) == 1


def _counted(monkeypatch, owner, name):
    """Replaces owner.name by a function that does the same; the list it returns grows by one a call."""
    calls, real = [], getattr(owner, name)
    monkeypatch.setattr(owner, name, lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    return calls


@pytest.mark.parametrize("owner,name", [(QuantLinear, "forward"), (Fp8Linear, "forward"), (QuantLinear, "__call__"),
                                        (torch.nn.Module, "__call__"), (torch.nn.Module, "_call_impl"), (QuantLinear, "_call_impl")])
def test_a_method_replaced_on_a_layers_class_is_called(monkeypatch, owner, name):
    base = torch.nn.Linear(256, 128).to(DEV).to(DT)
    layer = (Fp8Linear if owner is Fp8Linear else QuantLinear).from_linear(base)
    x = torch.randn(5, 256, device=DEV).to(DT)
    with torch.inference_mode():
        want = layer(x)
        with monkeypatch.context() as m:
            calls = _counted(m, owner, name)
            assert torch.equal(layer(x), want) and len(calls) == 1
        assert torch.equal(layer(x), want) and len(calls) == 1


@pytest.mark.parametrize("S,owner,name", [(S, o, n) for S in (1, 40) for o, n in (
    (GQA, "forward"), (MLP, "forward"), (QuantLinear, "forward"), (torch.nn.Module, "__call__"), (GQA, "_project_qkv"))] + [
    (40, QuantLinear, "forward_codes"), (1, QuantLinear, "forward_attn"), (1, PagedKV, "attn_workspace"), (40, "down", "forward_codes"),
    (1, "o_proj", "forward_attn"), (1, "attention", "forward")])
def test_a_method_replaced_inside_a_fused_block_is_called(monkeypatch, S, owner, name):
    """On a class, or (a text) on one of the block's own modules."""
    b = _block()
    x, fr, cache, table = _case(b, 2, S, 0 if S > 1 else 299)
    cache.bind(table, S if S > 1 else 300)
    if isinstance(owner, str):
        owner = {"down": b.mlp.down, "o_proj": b.attention.o_proj, "attention": b.attention}[owner]
    with torch.inference_mode():
        want = b(x, fr, None, cache)
        with monkeypatch.context() as m:
            calls = _counted(m, owner, name)
            assert torch.equal(b(x, fr, None, cache), want) and calls
        n = len(calls)
        assert torch.equal(b(x, fr, None, cache), want)
        assert len(calls) == n


def _frames(f):
    """f() and the names of the Python functions that it ran (the native path runs none)."""
    seen = []
    sys.setprofile(lambda frame, event, arg: seen.append(frame.f_code.co_name) if event == "call" else None)
    try:
        y = f()
    finally:
        sys.setprofile(None)
    return y, seen


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("own", [False, True], ids=["of the class", "of the layer"])
def test_a_changed_row_limit_decides(monkeypatch, fp8, own):
    cls, gemm = (Fp8Linear, "linear_fp8") if fp8 else (QuantLinear, "linear_w8a8")
    layer = cls.from_linear(torch.nn.Linear(256, 128).to(DEV).to(DT))
    x = torch.randn(5, 256, device=DEV).to(DT)
    with torch.inference_mode():
        layer(x)
        assert gemm not in _frames(lambda: layer(x))[1]
        monkeypatch.setattr(layer if own else cls, "DECODE_MAX_ROWS", 4)
        y, seen = _frames(lambda: layer(x))
        assert gemm in seen and torch.equal(y, layer.forward(x))


def test_a_changed_size_for_the_one_launch_quantiser_decides(monkeypatch):
    layer = Fp8Linear.from_linear(torch.nn.Linear(256, 128).to(DEV).to(DT))
    x = torch.randn(40, 256, device=DEV).to(DT)
    with torch.inference_mode():
        want = layer(x)
        assert len(layer._quant_states) == 0
        monkeypatch.setattr(ops, "FP8_ONEPASS_MIN_BYTES", 0)
        assert torch.equal(layer(x), want) and len(layer._quant_states) == 1


@pytest.mark.parametrize("S,limit,value,function", [
    (40, "RMSNORM_QUANT_MAX_K", 256, "rmsnorm_quant_rowwise_i8"), (40, "SWIGLU_QUANT_MAX_F", 1024, "swiglu_quant_rowwise_i8"),
    (1, "GEMV_ATTN_MAX_ROWS", 1, "forward_attn"), (1, "GEMV_ATTN_MAX_K", 256, "forward_attn"),
    (1, "GEMV_ATTN_MAX_SLICES", 1, "forward_attn"), (1, "GEMV_ATTN_MAX_WORK", 100, "forward_attn")])
def test_a_changed_limit_of_an_operator_decides_in_a_fused_block(monkeypatch, S, limit, value, function):
    b = _block()
    x, fr, cache, table = _case(b, 2, S, 0 if S > 1 else 299)
    cache.bind(table, S if S > 1 else 300)
    step = lambda: b(x, fr, None, cache)
    monkeypatch.setattr(ops, "quant_tensor_fp8", None)  # no block uses it; layers by themselves go through their forward now
    with torch.inference_mode():
        step()
        assert "_project_qkv" not in _frames(step)[1]
        with monkeypatch.context() as m:
            m.setattr(ops, "gemv_swiglu_ok", lambda x, f: False)  # a replaced operator: the step-by-step path
            assert function in _frames(step)[1]
        if isinstance(getattr(ops, limit), dict):
            monkeypatch.setitem(getattr(ops, limit), DT, value)
        else:
            monkeypatch.setattr(ops, limit, value)
        seen = _frames(step)[1]
        assert "_project_qkv" in seen and function not in seen


@pytest.mark.parametrize("rows", [3, 40])
def test_what_the_native_functions_do_not_take_goes_the_general_way(rows):
    torch.manual_seed(1)
    q = QuantLinear(256, 96, bias=True, device=DEV)
    q.load_float_weight(torch.randn(96, 256, device=DEV) * 0.02)
    wide = torch.randn(rows, 512, device=DEV).to(DT)
    res = torch.randn(96, rows, device=DEV).to(DT)
    with torch.inference_mode():
        want = q(wide[:, :256].contiguous(), residual=res.t().contiguous())
        assert torch.equal(q(wide[:, :256], residual=res.t()), want)               # strided rows and residual
        assert torch.equal(q(wide[:, :256].reshape(1, rows, 256), residual=res.t()), want.view(1, rows, 96))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y = q(wide[:, :256].contiguous(), residual=res.t().contiguous())
        side.synchronize()
        assert torch.equal(y, want)
        with pytest.raises(ValueError):
            q(wide)
        with pytest.raises(ValueError):
            q(wide[:, :256].double())
        with pytest.raises(RuntimeError, match="GPU only"):
            q(wide[:, :256].cpu())


@pytest.mark.parametrize("M,N,K", [(17, 513, 528), (40, 1024, 1024), (64, 2048, 512), (100, 300, 1040), (300, 1601, 2064)])
def test_an_fp8_layer_gives_the_same_bits_however_it_is_called(monkeypatch, M, N, K):
    """Rows that one launch casts and multiplies, in an order of sums of its own, and rows that take two: called natively, by its forward,
    with a hook, compiled, with rows that are not contiguous.  Two large products cancel, so that another order shows in the result."""
    g = torch.Generator().manual_seed(M)
    base = torch.nn.Linear(K, N)
    x, res = torch.randn(M, K, generator=g).to(DT).to(DEV), torch.randn(M, N, generator=g).to(DT).to(DEV)
    with torch.no_grad():
        base.weight[:, 0], base.weight[:, K - 1], x[:, 0], x[:, K - 1] = 2.0, -2.0, 100.0, 100.0
    layer = Fp8Linear.from_linear(base.to(DEV).to(DT))
    wide = torch.zeros(M, K + 16, device=DEV, dtype=DT)
    wide[:, :K] = x
    with torch.inference_mode():
        for kw in ({}, {"residual": res}):
            layer(x, **kw)
            y, seen = _frames(lambda: layer(x, **kw))
            assert "forward" not in seen
            assert torch.equal(layer.forward(x, **kw), y) and torch.equal(layer(wide[:, :K], **kw), y)
            handle = layer.register_forward_hook(lambda m, a, y: None)
            assert torch.equal(layer(x, **kw), y)
            handle.remove()
            torch._dynamo.reset()
            assert torch.equal(torch.compile(lambda x: layer(x, **kw), backend="eager")(x), y)


@pytest.mark.parametrize("M,N,K", [(40, 1024, 1024), (300, 160, 2064), (2100, 160, 4016)])
def test_replaced_fp8_operators_are_called_as_ever(monkeypatch, M, N, K):
    """With dense codes and without a keyword that they do not know."""
    layer = Fp8Linear.from_linear(torch.nn.Linear(K, N).to(DEV).to(DT))
    x, real, seen = torch.randn(M, K, device=DEV).to(DT), (ops.quant_tensor_fp8, ops.linear_fp8), []

    def quant(x, state=None, onepass=None):
        return real[0](x, state=state, onepass=onepass)

    def linear(xq, sx, wq, sw, bias=None, out_dtype=DT, residual=None):
        seen.append(xq.is_contiguous())
        return real[1](xq, sx, wq, sw, bias, out_dtype=out_dtype, residual=residual)

    with torch.inference_mode():
        want = real[1](*real[0](x), layer.qweight, layer.w_scale, layer.bias)
        monkeypatch.setattr(ops, "linear_fp8", linear)
        assert torch.equal(layer(x), want)
        monkeypatch.setattr(ops, "quant_tensor_fp8", quant)
        assert torch.equal(layer(x), want)
        monkeypatch.setattr(ops, "linear_fp8", real[1])
        assert torch.equal(layer(x), want)
    assert seen == [True, True]


class _Sub(QuantLinear):
    pass


@pytest.mark.parametrize("rows", [1, 16, 17])
def test_forms_of_a_layer_call(rows):
    """The native method answers or hands over to nn.Module's call, whatever way the arguments come."""
    torch.manual_seed(5)
    base = torch.nn.Linear(256, 128).to(DEV).to(DT)
    layer, sub = QuantLinear.from_linear(base), _Sub.from_linear(base)
    x, r = torch.randn(2, rows, 256, device=DEV).to(DT)[0], torch.randn(rows, 128, device=DEV).to(DT)
    norm = torch.rand(256, device=DEV).to(DT), 1e-5
    with torch.inference_mode():
        for args, kw in (((), {}), ((), {"residual": None}), ((), {"residual": r}), ((r,), {}), ((), {"norm": norm}),
                         ((), {"residual": r, "norm": norm}), ((), {"norm": None})):
            want = layer.forward(x, *args, **kw)
            assert torch.equal(layer(x, *args, **kw), want) and torch.equal(sub(x, *args, **kw), want)
        assert torch.equal(layer(x=x), layer.forward(x))
        with pytest.raises(TypeError):
            layer(x, other=r)
        with pytest.raises(TypeError):
            layer()
        with pytest.raises(ValueError):
            layer(x[:, :128])
        seen = []
        handle = layer.register_forward_hook(lambda m, a, y: seen.append(y))
        y = layer(x)
        handle.remove()
        assert len(seen) == 1 and torch.equal(seen[0], y) and torch.equal(y, layer(x)) and len(seen) == 1


class _Full:
    """Inside it torch's allocator has 24 MiB left, and no piece of 28 MiB or more."""

    def __enter__(self):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (24 << 20)) / torch.cuda.mem_get_info()[1])
        self.held = []
        try:
            while True:  # what is free between the blocks in use
                self.held.append(torch.empty(28 << 20, dtype=torch.uint8, device=DEV))
        except torch.OutOfMemoryError:
            pass

    def __exit__(self, *exc):
        self.held = None
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_out_of_memory_in_a_block_is_an_error_and_the_program_goes_on():
    """The block's scratch memory, 31.5 MiB for these tokens, does not fit; its output, 4 MiB, does."""
    b = _block()
    x, fr, cache, table = _case(b, 1, 4096, 0)
    cache.bind(table, 4096)
    with torch.inference_mode():
        want = b(x, fr, None, cache)
        with _Full():
            torch.empty_like(x)
            with pytest.raises(torch.OutOfMemoryError):
                b(x, fr, None, cache)
        assert torch.equal(b(x, fr, None, cache), want)


def test_out_of_memory_in_a_layer_is_an_error_and_the_program_goes_on():
    q = QuantLinear(256, 8192, device=DEV)
    x = torch.randn(4096, 256, device=DEV).to(DT)
    with torch.inference_mode():
        want = q(x)
        with _Full(), pytest.raises(torch.OutOfMemoryError):
            q(x)
        assert torch.equal(q(x), want)


def test_out_of_memory_in_an_operator_has_torchs_type():
    x = torch.randn(8192, 4096, device=DEV, dtype=DT)
    wq, sw = torch.zeros(8192, 4096, dtype=torch.int8, device=DEV), torch.ones(8192, device=DEV)
    xq, sx = ops.quant_rowwise_i8(x)
    with _Full():
        for call in (lambda: ops.quant_rowwise_i8(x), lambda: ops.rmsnorm_quant_rowwise_i8(x, x[0], 1e-5),
                     lambda: ops.quant_tensor_fp8(x), lambda: ops.linear_w8a8(xq, sx, wq, sw)):
            with pytest.raises(torch.OutOfMemoryError):
                call()
    assert torch.equal(ops.quant_rowwise_i8(x)[0], xq)


_INTERRUPTED = """
#include <dlfcn.h>
#include "astrai_q.h"
void (*aq_test_between)(void);
int aq_linear_w8a8_residual(const int8_t* xq, const float* sx, const int8_t* wq, const float* sw, const void* b, int bt,
                            const void* r, void* y, int yt, int64_t M, int64_t N, int64_t K, void* st) {
  static int (*real)(const int8_t*, const float*, const int8_t*, const float*, const void*, int, const void*, void*, int,
                     int64_t, int64_t, int64_t, void*);
  if (!real) *(void**)&real = dlsym(RTLD_NEXT, "aq_linear_w8a8_residual");
  aq_test_between();
  return real(xq, sx, wq, sw, b, bt, r, y, yt, M, N, K, st);
}
"""


@pytest.fixture
def between(tmp_path):
    """Binds the native path to a library whose GEMM entry calls a Python function before it queues its launch -- what
    another thread may do while the interpreter lock is released."""
    src, so = tmp_path / "between.c", tmp_path / "between.so"
    src.write_text(_INTERRUPTED)
    product = _abi.LIB_PATH
    subprocess.run(["gcc", "-D_GNU_SOURCE", "-shared", "-fPIC", "-I", str(pathlib.Path(__file__).parent.parent / "include"), str(src),
                    "-o", str(so), "-Wl,--no-as-needed", product, f"-Wl,-rpath,{pathlib.Path(product).parent}"], check=True)
    lib, done = ctypes.CDLL(str(so)), []

    def bind(f):
        done.append(ctypes.CFUNCTYPE(None)(f))
        ctypes.c_void_p.in_dll(lib, "aq_test_between").value = ctypes.cast(done[-1], ctypes.c_void_p).value
        _abi.host().bind(lib._handle)

    yield bind
    _abi.host().bind(_abi.load()._handle)


def test_a_layer_holds_its_weight_for_the_length_of_a_call(between):
    """Another thread gives the module new buffers after the call has let go of the interpreter lock and before its GEMM
    is queued: the old ones stay until it is."""
    torch.manual_seed(2)
    base = torch.nn.Linear(512, 8192).to(DEV).to(DT)
    q, x = QuantLinear.from_linear(base), torch.randn(64, 512, device=DEV).to(DT)
    with torch.inference_mode():
        want = q(x)
        old = []

        def swap():
            old.append(torch.cuda.memory_allocated())
            q._buffers["qweight"], q._buffers["w_scale"] = torch.ones_like(q.qweight), torch.ones_like(q.w_scale)
            old.append(torch.cuda.memory_allocated())

        def another_thread():
            t = threading.Thread(target=swap)
            t.start()
            t.join()

        between(another_thread)
        y = q(x)
    assert torch.equal(y, want)
    assert old[1] - old[0] >= 8192 * 512 + 4 * 8192  # the new ones beside the old ones


def test_a_compiled_layer_and_block_give_the_same_bits():
    b = _block()
    x, fr, cache, table = _case(b, 2, 1, 30)
    cache.bind(table, 31)
    q = b.mlp.down
    h = torch.randn(5, 1408, device=DEV).to(DT)
    with torch.inference_mode():
        want, block_want = q(h), b(x, fr, None, cache)
        torch._dynamo.reset()
        assert torch.equal(torch.compile(lambda h: q(h) * 2, backend="eager")(h), want * 2)
        assert torch.equal(torch.compile(b, backend="eager")(x, fr, None, cache), block_want)


def test_threads_on_streams_of_their_own_share_a_layer_and_a_block():
    b = _block()
    x, fr, cache, table = _case(b, 3, 40, 0)
    cache.bind(table, 40)
    h = torch.randn(9, 1408, device=DEV).to(DT)
    with torch.inference_mode():
        want = b(x, fr, None, cache), b.mlp.down(h)
    torch.cuda.synchronize()
    wrong = []

    def work():
        with torch.cuda.stream(torch.cuda.Stream()), torch.inference_mode():
            for _ in range(50):
                got = b(x, fr, None, cache), b.mlp.down(h)  # every thread writes the same keys and values
                if not (torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])):
                    wrong.append(1)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
