"""The module calls as Python C functions (csrc/py_calls.cpp): bit for bit the
torch.ops route's results, and None -- the caller's sign to take the general
route -- for every call that is not the ordinary one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(K, N, bits, bias=True, gs=64, dtype=torch.bfloat16):
    import mflux_amd

    torch.manual_seed(N + bits)
    lin = mflux_amd.nn.Linear(K, N, bias=bias, device="cuda", dtype=dtype)
    return lin.to_quantized(gs, bits)


@pytest.mark.parametrize("bits,dtype,shape", [(8, torch.bfloat16, (1, 256)), (4, torch.float16, (2, 3, 256)),
                                              (6, torch.bfloat16, (40, 256)), (4, torch.bfloat16, (1, 300, 256)), (4, torch.bfloat16, (256,))])
def test_same_bits_as_the_operator(bits, dtype, shape):
    from mflux_amd import _lib

    layer = _layer(256, 192, bits, bias=bits != 4, dtype=dtype)
    x = torch.randn(shape, device="cuda", dtype=dtype)
    x2 = x.reshape(-1, 256)
    w = layer._operands()
    y = _lib.native().linear(x, *w, 64, bits)
    ref, ok = _lib.ops().qmm_t(x2, *w, 64, bits, dtype, None, None)
    assert ok and y.shape == (*shape[:-1], 192) and torch.equal(y, ref.reshape(y.shape))
    assert torch.equal(y, layer(x))
    if bits != 6 and x2.shape[0] <= 4:
        ref, ok = _lib.ops().qmv_silu(x2, *w, 64, bits)
        assert ok and torch.equal(_lib.native().silu_linear(x, *w, 64, bits), ref.reshape(y.shape))
    if x2.shape[0] > 16:
        gate, res = torch.randn(192, device="cuda", dtype=dtype), torch.randn_like(y)
        got = _lib.native().epilogue_linear(x, *w, 64, bits, _lib.EPILOGUE_GATE_RESIDUAL, gate, res, 0)
        ref, ok = _lib.ops().qmm_t_epilogue(x2, *w, 64, bits, _lib.EPILOGUE_GATE_RESIDUAL, gate, res.reshape(-1, 192), 0)
        assert ok and torch.equal(got, ref.reshape(y.shape))


def test_everything_else_is_left_to_the_general_route():
    from torch.utils._python_dispatch import TorchDispatchMode

    from mflux_amd import _lib

    layer = _layer(256, 192, 8)
    n, (w, s, b, bias) = _lib.native(), layer._operands()
    x = torch.randn(2, 256, device="cuda", dtype=torch.bfloat16)
    assert n.linear(x, w, s, b, bias, 64, 8) is not None

    class Sub(torch.Tensor):
        pass

    for bad in (x.cpu(), x.float(), x.half(), x[:, :192], x.t(), x[:0], torch.randn(256, 2, device="cuda", dtype=x.dtype).t(),
                x.clone().requires_grad_(True), x.as_subclass(Sub), torch._neg_view(x), x.tolist(), None):
        assert n.linear(bad, w, s, b, bias, 64, 8) is None
    for args in ((x, w.view(torch.int32), s, b, bias, 64, 8), (x, w, s, b, bias, 64, 4), (x, w, s, b, bias, 48, 8),
                 (x, w, s, b.float(), bias, 64, 8), (x, w, s, b, bias[:64], 64, 8), (x, w[:64], s, b, bias, 64, 8),
                 (x, w, s, b, bias, 64.0, 8), (x, w, s, b, bias, 64), (x, w, s, b, bias, 64, 1 << 80)):
        assert n.linear(*args) is None
    with torch.no_grad():
        assert n.linear(x.clone().requires_grad_(True), w, s, b, bias, 64, 8) is not None

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert n.linear(x, w, s, b, bias, 64, 8) is None
    answers = []

    def traced(t):
        answers.append(n.linear(t, w, s, b, bias, 64, 8))
        return t + 1

    torch.jit.trace(traced, x, check_trace=False)
    assert answers == [None]
    with pytest.raises(ValueError, match="does not match"):
        layer(x[:, :192])
    # autograd still sees the call
    xg = x.clone().requires_grad_(True)
    layer(xg).sum().backward()
    assert xg.grad is not None


def test_inputs_are_only_read():
    """A lazily cloned (copy-on-write) input stays one: only the output is written."""
    from mflux_amd import _lib

    layer = _layer(256, 192, 8)
    w = layer._operands()
    n = _lib.native()
    for M in (1, 6, 40):
        x = torch.randn(M, 256, device="cuda", dtype=torch.bfloat16)
        lazy = torch._lazy_clone(x)
        res, gate = torch.randn(M, 192, device="cuda", dtype=x.dtype), torch.randn(192, device="cuda", dtype=x.dtype)
        lazy_res = torch._lazy_clone(res)
        assert torch.equal(n.linear(lazy, *w, 64, 8), n.linear(x, *w, 64, 8))
        if M <= 16:
            n.silu_linear(lazy, *w, 64, 8)
        else:
            n.epilogue_linear(lazy, *w, 64, 8, _lib.EPILOGUE_GATE_RESIDUAL, gate, lazy_res, 0)
        assert torch._C._is_cow_tensor(lazy) and torch._C._is_cow_tensor(lazy_res)


def test_profiler_lists_the_calls():
    """A torch profile of module calls names the operators, as when they go through the dispatcher."""
    from torch.profiler import ProfilerActivity, profile

    import mflux_amd
    from mflux_amd import nn

    layer = _layer(256, 192, 8)
    x = torch.randn(40, 256, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad(), profile(activities=[ProfilerActivity.CPU]) as prof:
        layer(x)
        nn.silu_linear(layer, x[:1])
        nn.gelu_linear(layer, x)
    names = {e.name for e in prof.events()}
    assert {"mfq::qmm_t", "mfq::qmv_silu", "mfq::qmm_t_epilogue"} <= names


@pytest.mark.parametrize("epilogue,act_from", [("gelu", 0), ("gelu", 72), ("swiglu", 0)])
@pytest.mark.parametrize("bits", [4, 6, 8])
def test_epilogues_same_bits_as_the_operator(epilogue, act_from, bits):
    from mflux_amd import _lib, core

    layer = _layer(256, 192, bits)
    x = torch.randn(2, 20, 256, device="cuda", dtype=torch.bfloat16)
    w = layer._operands()
    got = _lib.native().epilogue_linear(x, *w, 64, bits, core.EPILOGUES[epilogue], None, None, act_from)
    ref, ok = _lib.ops().qmm_t_epilogue(x.reshape(-1, 256), *w, 64, bits, core.EPILOGUES[epilogue], None, None, act_from)
    assert ok and got.shape == (2, 20, ref.shape[-1]) and torch.equal(got, ref.reshape(got.shape))


@pytest.mark.parametrize("bits,dtype,shape", [(8, torch.bfloat16, (1, 256)), (4, torch.float16, (2, 3, 256)), (6, torch.bfloat16, (40, 256)),
                                              (4, torch.bfloat16, (1, 300, 256)), (4, torch.bfloat16, (256,)), (5, torch.float16, (7, 256)),
                                              (4, torch.bfloat16, (2304, 256))])
def test_float32_activations_are_the_operator_on_rounded_ones(bits, dtype, shape):
    from mflux_amd import _lib

    layer = _layer(256, 192, bits, bias=bits != 4, dtype=dtype)
    x = torch.randn(shape, device="cuda") * 3
    x.view(-1)[:4] = torch.tensor([1 + 2 ** -8, 1 + 3 * 2 ** -8, -1e-40, 3e38 if dtype == torch.bfloat16 else 65519.0])  # ties, tiny, large
    w = layer._operands()
    y = _lib.native().linear_float32(x, *w, 64, bits)
    ref, ok = _lib.ops().qmm_t(x.reshape(-1, 256).to(dtype), *w, 64, bits, torch.float32, None, None)
    assert ok and y.dtype == torch.float32 and y.shape == (*shape[:-1], 192) and torch.equal(y, ref.reshape(y.shape))
    assert torch.equal(y, layer(x))
    shifted = torch.empty(x.numel() + 1, device="cuda")[1:].view(shape).copy_(x)  # at an address of its own
    assert torch.equal(_lib.native().linear_float32(shifted, *w, 64, bits), y)
    for other in (x.to(dtype), x.double(), x.clone().requires_grad_(True), x.cpu()):
        assert _lib.native().linear_float32(other, *w, 64, bits) is None
