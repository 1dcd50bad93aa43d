"""The direct calls (csrc/host/fast_calls.cpp) against the registered ops: the same bits where they answer, and no answer
where something sits between the call and the device implementation."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _w4(device, k, n, group, dtype, bias):
    from vllm_amd.layers.linear import LinearBase
    from vllm_amd.layers.quantization import get_quantization_config
    g = torch.Generator(device=device).manual_seed(k + n)
    config = get_quantization_config("gptq_marlin").from_config(dict(bits=4, group_size=group, desc_act=False, sym=True))
    layer = LinearBase(k, n, bias=bias, quant_config=config, params_dtype=dtype, return_bias=False).to(device)
    layer.qweight.data.copy_(torch.randint(-2 ** 31, 2 ** 31 - 1, layer.qweight.shape, dtype=torch.int32, device=device, generator=g))
    layer.scales.data.copy_(torch.rand(layer.scales.shape, device=device, generator=g) * 0.01 + 1e-3)
    layer.g_idx.data.copy_(torch.arange(k, device=device) // (group if group > 0 else k))
    layer.process_weights_after_loading()
    return layer


def _registered(layer, x):
    import vllm_amd._custom_ops as ops  # noqa: F401
    from vllm_amd.scalar_type import scalar_types
    kern, rows = layer.quant_method.kernel, x.reshape(-1, x.shape[-1])
    size_k, size_n = kern.config.partition_weight_shape
    out = torch.ops.vllm_amd.gptq_marlin_gemm(rows, None, layer.qweight, layer.bias, layer.scales, None, layer.qzeros, layer.g_idx,
                                              layer.g_idx_sort_indices, kern.workspace, scalar_types.uint4b8.id, rows.shape[0],
                                              size_n, size_k)
    return out.reshape(x.shape[:-1] + (size_n,))


@pytest.mark.parametrize("shape", [(1, 512), (65, 512), (2, 3, 512), (512,)])
@pytest.mark.parametrize("group,dtype,bias", [(128, torch.bfloat16, False), (32, torch.float16, True), (-1, torch.bfloat16, True)])
def test_w4_layer_equals_the_registered_op(device, shape, group, dtype, bias):
    from vllm_amd import _custom_ops as ops
    layer = _w4(device, 512, 192, group, dtype, bias)
    x = torch.randn(shape, device=device).to(dtype)
    got = layer(x)
    assert got.shape == shape[:-1] + (192,) and got.is_contiguous()
    assert torch.equal(got, _registered(layer, x))
    strided = torch.randn(7, 1024, device=device).to(dtype)[:, :512]
    assert torch.equal(layer(strided), _registered(layer, strided))
    direct = ops._fast.w4_linear(x, layer.qweight, layer.bias, layer.scales, layer.qzeros, layer.g_idx, layer.g_idx_sort_indices,
                                 layer.quant_method.kernel.workspace, layer.quant_method.quant_config.quant_type.id, 192, 512, True)
    assert direct is not None, "a plain call went through the dispatcher"


def test_w4_scratch_is_that_of_the_layers_own_format(device):
    """Two formats of one shape in turn that need different scratch for their K split: neither takes the other's size from the caches
    of either route, and a call allocates its output and the scratch of its own format, not that of any."""
    import ctypes
    import gc
    from vllm_amd import _lib
    lib = _lib.load()
    gc.collect()      # a layer and its parameters' loaders refer to each other: one of an earlier test may be freed within a call below
    layers = {g: _w4(device, 2048, 512, g, torch.bfloat16, False) for g in (128, 32)}
    smaller = 0
    for m in (33, 40, 48, 70, 100, 150):
        x = torch.randn(m, 2048, device=device).to(torch.bfloat16)
        sizes = [ctypes.c_size_t() for _ in range(3)]
        _lib.check(lib.vaq_w4a16_gemm_workspace(m, 512, 2048, 0, 0, *map(ctypes.byref, sizes)))
        every = sizes[0].value
        for _ in range(2):
            for layer in layers.values():
                assert torch.equal(layer(x), _registered(layer, x))
        for group, layer in layers.items():
            _lib.check(lib.vaq_w4a16_gemm_workspace_of_format(m, 512, 2048, group, _lib.VAQ_WTYPE_U4B8, 0, 0, *map(ctypes.byref, sizes)))
            own = sizes[0].value
            smaller += own < every
            for call in (lambda: layer(x), lambda: _registered(layer, x)):
                torch.cuda.reset_peak_memory_stats(device)
                before = torch.cuda.memory_allocated(device)
                out = call()
                assert torch.cuda.max_memory_allocated(device) - before == sum((n + 511) // 512 * 512 for n in (out.numel() * 2, own))
                del out
    assert smaller > 3


@pytest.mark.parametrize("shape", [(1, 256), (67, 256), (2, 5, 256)])
@pytest.mark.parametrize("static", [False, True])
@pytest.mark.parametrize("bias", [False, True])
def test_fp8_layer_equals_its_two_steps(device, shape, static, bias):
    from vllm_amd import _custom_ops as ops
    w = (torch.randn(320, 256, device=device) * 0.05).to(torch.bfloat16)
    wq, ws = ops.scaled_fp8_quant(w, use_per_token_if_dynamic=True)
    b = torch.randn(320, device=device).to(torch.bfloat16) if bias else None
    x = torch.randn(shape, device=device).to(torch.bfloat16)
    scale = torch.full((1,), 0.01, device=device) if static else None
    got = ops.fp8_linear(x, wq.t(), ws, scale, None, torch.bfloat16, b)
    rows = x.reshape(-1, 256)
    q = torch.empty(rows.shape, dtype=torch.float8_e4m3fn, device=device)
    s = scale if static else torch.empty(rows.shape[0], 1, device=device)
    if static:
        torch.ops.vllm_amd.static_scaled_fp8_quant(q, rows, s)
    else:
        torch.ops.vllm_amd.dynamic_per_token_scaled_fp8_quant(q, rows, s, None)
    ref = torch.empty(rows.shape[0], 320, dtype=torch.bfloat16, device=device)
    torch.ops.vllm_amd.cutlass_scaled_mm(ref, q, wq.t(), s, ws, b)
    assert got is not None and torch.equal(got, ref.reshape(shape[:-1] + (320,)))
    q2, s2 = ops._fast.fp8_quant(rows, scale, None, not static, None)
    assert torch.equal(q2.view(torch.uint8), q.view(torch.uint8)) and torch.equal(s2, s)
    assert torch.equal(ops._fast.scaled_mm(q2, wq.t(), s2, ws, torch.bfloat16, b), ref)


@pytest.mark.parametrize("k,n", [(16, 16), (144, 320), (1040, 256), (2064, 4128), (4096, 528), (4112, 64), (8176, 80), (8192, 48), (16384, 32)])
@pytest.mark.parametrize("static", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fp8_rows_quantised_by_the_gemm(device, k, n, static, dtype):
    """One launch for the quantisation and the product of a few rows: the bits of the two launches, special values too."""
    from vllm_amd import _custom_ops as ops, _lib
    lib, taken = _lib.load(), 0
    g = torch.Generator(device=device).manual_seed(k + n)
    wq, ws = ops.scaled_fp8_quant(torch.randn(n, k, device=device, generator=g).to(dtype), use_per_token_if_dynamic=True)
    for m in range(1, 10):
        x = torch.randn(m, k + 16, device=device, generator=g).to(dtype)[:, :k]
        if m >= 3:
            x[1] = 0
        if m >= 6:
            x[0, 3], x[2, 7], x[4, k - 1], x[5] = float("inf"), float("nan"), -float("inf"), x[5] * 1e-6
        if m >= 8:
            x[6], x[7] = float("nan"), -0.0
        scale = torch.full((1,), 0.011, device=device) if static else None
        bias = torch.randn(n, device=device, generator=g).to(dtype) if m % 2 else None
        taken += lib.vaq_fp8_quant_scaled_mm_takes(m, n, k, not static)
        got = ops.fp8_linear(x, wq.t(), ws if m % 3 else ws[:1].contiguous(), scale, None, dtype, bias)
        q, s = ops.scaled_fp8_quant(x.contiguous(), scale, use_per_token_if_dynamic=True)
        ref = ops.cutlass_scaled_mm(q, wq.t(), s, ws if m % 3 else ws[:1].contiguous(), dtype, bias)
        assert torch.equal(got.view(torch.int16), ref.view(torch.int16)), m
    assert taken >= (4 if k > 4096 else 8)


def test_no_answer_where_something_is_in_between(device):
    from torch.utils._python_dispatch import TorchDispatchMode
    from vllm_amd import _custom_ops as ops, _tuning

    class Seen(TorchDispatchMode):
        calls = ()

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.calls += (str(func),)
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    x = torch.randn(4, 64, device=device).to(torch.bfloat16)
    one = torch.ones(1, device=device)
    plain = ops._fast.fp8_quant(x, one, None, False, None)
    assert plain is not None
    with Seen() as seen:
        got = ops.scaled_fp8_quant(x, one)
    assert any("static_scaled_fp8_quant" in c for c in seen.calls)
    assert torch.equal(got[0].view(torch.uint8), plain[0].view(torch.uint8))
    assert ops._fast.fp8_quant(x.as_subclass(Sub), one, None, False, None) is None
    assert ops._fast.fp8_quant(x.cpu(), one, None, False, None) is None
    assert ops._fast.fp8_quant(x.t(), one, None, False, None) is None
    grad = x.float().requires_grad_()
    assert ops._fast.fp8_quant(grad, one, None, False, None) is None
    with torch.no_grad():
        assert ops._fast.fp8_quant(grad, one, None, False, None) is not None
    with torch.inference_mode():
        assert ops._fast.fp8_quant(x, one, None, False, None) is not None
    with _tuning.override(quant_wg_per_row=1):
        assert ops._fast.fp8_quant(x, one, None, False, None) is None
    assert ops._fast.fp8_quant(x, one, None, False, None) is not None


def _fp8_codes(n, k, device, seed):
    """Finite e4m3 codes, made in place (the weights below are 2 GiB)."""
    g = torch.Generator(device=device).manual_seed(seed)
    q = torch.empty(n, k, dtype=torch.uint8, device=device)
    q.random_(0, 0x60, generator=g)
    return q.view(torch.float8_e4m3fn)


@pytest.mark.parametrize("m", [1, 4, 9])
@pytest.mark.parametrize("static", [False, True])
def test_fp8_layer_with_weights_that_end_past_2_gib(device, m, static):
    """Contiguous and strided: few rows leave the kernel that quantises and multiplies, whose offsets are 32-bit."""
    from vllm_amd import _custom_ops as ops
    scale = torch.full((1,), 0.01, device=device) if static else None
    n, k = 270336, 8192
    big = _fp8_codes(n, k, device, 1)
    strided = torch.as_strided(big.view(-1), (32, 1024), (2 ** 26 + 2 ** 22, 1))      # the last row ends beyond 2 GiB
    assert 31 * strided.stride(0) + 1024 > 2 ** 31
    for w in (big, strided):
        x = torch.randn(m, w.shape[1], device=device).to(torch.bfloat16)
        ws = torch.rand(w.shape[0], 1, device=device) * 1e-2 + 1e-3
        got = ops.fp8_linear(x, w.t(), ws, scale, None, torch.bfloat16, None)
        assert got is not None and got.shape == (m, w.shape[0])
        q, s = ops.scaled_fp8_quant(x, scale, use_per_token_if_dynamic=True)
        cols = torch.cat([torch.arange(min(16, w.shape[0])), torch.arange(w.shape[0] - 16, w.shape[0])]).to(device)
        ref = (q.float() @ w[cols].float().t()) * s.reshape(-1, 1) * ws[cols].t()
        # one rounding to bf16 (2^-9) beside fp32 sums of products of like sign at most
        assert torch.allclose(got[:, cols].float(), ref, rtol=2 ** -8, atol=float(ref.abs().mean()) * 2e-3)


def test_other_threads_run_while_a_call_allocates(device):
    """The interpreter's lock is given up around allocation and launch.  Nothing else gives it up here: the interpreter itself
    would only after 1000 s."""
    import sys
    import threading
    from vllm_amd import _custom_ops as ops
    x = torch.randn(8192, 4096, device=device, dtype=torch.bfloat16)
    one = torch.ones(1, device=device)
    assert ops._fast.fp8_quant(x, one, None, False, None) is not None
    torch.cuda.empty_cache()      # (every output below is an allocation of its own from the driver)
    go, ran = threading.Event(), []
    other = threading.Thread(target=lambda: (go.wait(), ran.append(True)))
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1000)
    try:
        other.start()
        go.set()
        kept = [ops._fast.fp8_quant(x, one, None, False, None) for _ in range(32)]
        seen = bool(ran)
    finally:
        sys.setswitchinterval(interval)
        other.join()
    assert seen, "32 calls, and the other thread had no turn"
    assert all(torch.equal(q.view(torch.uint8), kept[0][0].view(torch.uint8)) for q, _ in kept)


def test_layers_called_from_two_threads(device):
    """Two threads on streams of their own, a W4A16 layer each and one FP8 layer between them, over sizes of every path
    (single launch, stream and tile kernels, split K with its counters per stream): the results of one thread alone."""
    import threading
    from vllm_amd import _custom_ops as ops
    from vllm_amd.layers.quantization.input_quant_fp8 import GroupShape
    from vllm_amd.layers.quantization.utils.w8a8_utils import Fp8LinearOp
    fp8 = Fp8LinearOp(act_quant_static=False, act_quant_group_shape=GroupShape.PER_TOKEN)
    layers = [_w4(device, 1024, 512, 128, torch.bfloat16, False), _w4(device, 2048, 256, 32, torch.bfloat16, True)]
    wq, ws = ops.scaled_fp8_quant((torch.randn(512, 8192, device=device) * 0.05).to(torch.bfloat16), use_per_token_if_dynamic=True)
    sizes = (1, 5, 16, 33, 100, 300)

    def step(layer, x4, x8):
        return layer(x4), fp8.apply(x8, wq.t(), ws, torch.bfloat16)

    inputs = [[(torch.randn(m, l.input_size, device=device).to(torch.bfloat16), torch.randn(m, 8192, device=device).to(torch.bfloat16))
               for m in sizes] for l in layers]
    expect = [[step(l, *i) for i in per] for l, per in zip(layers, inputs)]
    torch.cuda.synchronize()
    errors, start = [], threading.Barrier(2)

    def work(t):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait(30)
                got = [[step(layers[t], *i) for i in inputs[t]] for _ in range(60)]
                torch.cuda.current_stream().synchronize()
                for round_ in got:
                    for (a, b), (ra, rb) in zip(round_, expect[t]):
                        assert torch.equal(a, ra) and torch.equal(b, rb)
        except BaseException as e:      # noqa: BLE001 (reported by the test below)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_an_override_on_one_thread_leaves_the_others_their_direct_calls(device):
    import threading
    from vllm_amd import _custom_ops as ops, _tuning
    x, one = torch.randn(4, 64, device=device).to(torch.bfloat16), torch.ones(1, device=device)
    answers = []
    with _tuning.override(quant_wg_per_row=1):
        t = threading.Thread(target=lambda: answers.append(ops._fast.fp8_quant(x, one, None, False, None)))
        t.start()
        t.join()
        assert ops._fast.fp8_quant(x, one, None, False, None) is None
    assert answers[0] is not None
