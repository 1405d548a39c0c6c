"""LoRA adapters on (quantized) linear layers.

Mirrors mflux's wrappers, same names and attributes:
``LoRALinear`` (src/mflux/models/common/lora/layer/linear_lora_layer.py:8-53:
``from_linear(linear, r, scale)``, ``linear``, ``scale``, ``lora_A [K, r]``,
``lora_B [r, N]``, ``base + scale * (x @ A) @ B``) and ``FusedLoRALinear``
(src/mflux/models/common/lora/layer/fused_linear_lora_layer.py:7-20:
``base_linear``, ``loras``, the sum over the adapters).

Around a ``QuantizedLinear`` base on the GPU, at inference, the whole layer is
one call of the quantized matmul: the adapters' down-projections are
concatenated into one ``[K, R]`` matrix (one small library GEMM gives ``t = x @ A``),
the scaled up-projections into one ``[N, R]`` matrix, and the kernel treats
them as ``R`` more ``k`` of the same product.  With gradients one adapter on a
quantized base keeps that form (``_LoRALinearFunction``); anything else, and a
base that is not quantized, is the reference's composition of separate matmuls.
"""
from __future__ import annotations

import math

import torch

from . import _lib, core
from .nn import Linear, QuantizedLinear

_RANK_STEP = 16  # the kernels take the low rank in steps of 16


class LoRALinear(torch.nn.Module):
    @staticmethod
    def from_linear(linear: torch.nn.Module, r: int = 16, scale: float = 1.0) -> "LoRALinear":
        output_dims, input_dims = linear.weight.shape
        if isinstance(linear, QuantizedLinear):
            # packed words -> elements (the reference multiplies by 32 // bits, which is only right for 4 and 8 bits)
            input_dims = input_dims * 32 // linear.bits
        ref = linear.scales if isinstance(linear, QuantizedLinear) else linear.weight
        lora_lin = LoRALinear(input_dims=input_dims, output_dims=output_dims, r=r, scale=scale, device=ref.device,
                              dtype=ref.dtype, _make_linear=False)
        lora_lin.linear = linear
        return lora_lin

    def __init__(self, input_dims: int, output_dims: int, r: int = 8, scale: float = 1.0, bias: bool = False, *,
                 device=None, dtype: torch.dtype = torch.bfloat16, _make_linear: bool = True):
        super().__init__()
        if _make_linear:
            self.linear = Linear(input_dims, output_dims, bias=bias, device=device, dtype=dtype)
        self.scale = scale
        bound = 1 / math.sqrt(input_dims)
        make = lambda *shape: torch.nn.Parameter(
            torch.empty(shape, device=device, dtype=torch.float32).uniform_(-bound, bound).to(dtype))
        self.lora_A = make(input_dims, r)
        self.lora_B = make(r, output_dims)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return _forward(self, self.linear, [self], x)


class FusedLoRALinear(torch.nn.Module):
    def __init__(self, base_linear: torch.nn.Module, loras: list[LoRALinear]):
        super().__init__()
        self.base_linear = base_linear
        self.loras = torch.nn.ModuleList(loras)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return _forward(self, self.base_linear, list(self.loras), x)


def _composed(base: torch.nn.Module, loras: list[LoRALinear], x: torch.Tensor) -> torch.Tensor:
    """The reference's arithmetic: separate matmuls, every intermediate rounded."""
    out = base(x)
    if len(loras) == 1:
        lora = loras[0]
        return out + lora.scale * torch.matmul(torch.matmul(x.to(lora.lora_A.dtype), lora.lora_A), lora.lora_B)
    lora_out = torch.zeros_like(out)
    for lora in loras:
        lora_out = lora_out + lora.scale * torch.matmul(torch.matmul(x.to(lora.lora_A.dtype), lora.lora_A),
                                                        lora.lora_B)
    return out + lora_out


def pack_adapters(loras: list[LoRALinear], dtype: torch.dtype) -> tuple[torch.Tensor, torch.Tensor]:
    """``(a_cat [K, R], bs [N, R])`` for ``quantized_matmul(..., low_rank=(x @ a_cat, bs))``:
    the down-projections side by side and the up-projections, scaled in float32
    and transposed, side by side, ``R`` = the sum of the ranks rounded up to a
    multiple of 16 with zero columns."""
    a_cat = torch.cat([lora.lora_A.detach().to(dtype) for lora in loras], dim=1)
    bs = torch.cat([(float(lora.scale) * lora.lora_B.detach().float()).t() for lora in loras], dim=1).to(dtype)
    pad = -a_cat.shape[1] % _RANK_STEP
    if pad:
        a_cat = torch.nn.functional.pad(a_cat, (0, pad))
        bs = torch.nn.functional.pad(bs, (0, pad))
    return a_cat.contiguous(), bs.contiguous()


_DOWN_KERNEL_MAX_K = 4096


def down_fragments(a_cat: torch.Tensor) -> torch.Tensor:
    """``a_cat [K, R]`` (``K % 32 == 0``, ``R % 16 == 0``) in the order the
    down-projection kernel's matrix instruction consumes it:
    ``[R/16, K/32, 4, 16, 8]`` with ``af[f, s, q, c, e] = a_cat[32 s + 8 q + e, 16 f + c]``."""
    K, R = a_cat.shape
    if K % 32 or R % 16:
        raise ValueError(f"[down_fragments] a_cat must be [K, R] with K % 32 == 0 and R % 16 == 0, got {tuple(a_cat.shape)}")
    return a_cat.reshape(K // 32, 4, 8, R // 16, 16).permute(3, 0, 1, 4, 2).contiguous()


def _packed_for(owner: torch.nn.Module, loras: list[LoRALinear], dtype: torch.dtype):
    # rebuilt when an adapter's tensors are replaced or written in place, or a scale changes
    key = (dtype,) + tuple((id(lora), lora.lora_A.data_ptr(), lora.lora_A._version, lora.lora_B.data_ptr(),
                            lora.lora_B._version, float(lora.scale)) for lora in loras)
    cache = owner.__dict__.get("_packed_adapters")
    if cache is None or cache[0] != key:
        a_cat, bs = pack_adapters(loras, dtype)
        cache = (key, (a_cat, down_fragments(a_cat) if a_cat.shape[0] <= _DOWN_KERNEL_MAX_K else None, bs))
        owner.__dict__["_packed_adapters"] = cache
    return cache[1]


class _LoRALinearFunction(torch.autograd.Function):
    """``base(x) + scale * (x @ A) @ B`` for training: the update rides in the base
    GEMM (``low_rank``), where the composition writes and reads the ``[M, N]``
    product three times more (a rank-16 matmul, the scaling, the add: 65 us of a
    step of 410 at 1536 rows, 3072 -> 12288), and backward in bfloat16 scales the
    ``[M, R]`` product of the gradient instead of the gradient.  One rounding where
    the composition has four.  The products with the factors are this package's
    kernels (``own``): the factors packed once per step, then one read of ``x`` and,
    backward, of ``x`` and of the gradient (304 -> 287 us of that step)."""

    @staticmethod
    def forward(ctx, x, lora_a, lora_b, w, scales, biases, bias, scale, group_size, bits):
        ctx.meta = (scale, group_size, bits)
        ctx.own = lora_a.shape[1] <= _TRAINING_MAX_RANK and lora_b.shape[1] % 32 == 0
        if ctx.own:
            ops = _lib.ops()
            af, bf, bs, ap = ops.low_rank_pack(lora_a.contiguous(), lora_b.contiguous(), scale)
            t, tf = ops.low_rank_forward(_rows(x), af, lora_a.shape[1])
            ctx.save_for_backward(x, lora_a, lora_b, w, scales, biases, tf, bf, ap)
        else:
            t = torch.matmul(x.reshape(-1, x.shape[-1]), lora_a)
            ctx.save_for_backward(x, lora_a, lora_b, w, scales, biases, t)
            bs = _operand((lora_b if scale == 1.0 else (scale * lora_b.float()).to(lora_b.dtype)).t())
            t = _operand(t)
        return core.quantized_matmul(x, w, scales, biases, True, group_size, bits, bias=bias,
                                     low_rank=(t.reshape(*x.shape[:-1], -1), bs))

    @staticmethod
    def backward(ctx, grad_y):
        x, lora_a, lora_b, w, scales, biases, *rest = ctx.saved_tensors
        scale, group_size, bits = ctx.meta
        x2, g = x.reshape(-1, x.shape[-1]), grad_y.reshape(-1, grad_y.shape[-1])
        twice = torch.is_grad_enabled()  # create_graph: everything below in operations that differentiate again
        # float16: the gradient is scaled before anything is summed over it, as the composition does.  A product of the
        # unscaled one leaves the type's range at 65504 |scale| of the true gradient, and a scaled-down lora_B of a
        # young adapter its normal numbers; bfloat16 has float32's range, and the [M, R] products are scaled instead.
        if scale != 1.0 and g.dtype == torch.float16:
            g, scale = scale * g, 1.0
        need_x, need_a, need_b = ctx.needs_input_grad[:3]
        grad_x = grad_a = grad_b = gt = None
        if ctx.own and not twice:
            tf, bf, ap = rest
            ops, rank = _lib.ops(), lora_a.shape[1]
            rows = _rows(grad_y)
            gt, gtf, grad_b = ops.low_rank_gradient(rows if scale == ctx.meta[0] else _rows(g), bf, tf, rank, scale,
                                                    need_x or need_a, need_b)
            grad_a = ops.low_rank_up(_rows(x), gtf, rank) if need_a else None
            if need_x:
                grad_x = core._matmul_untransposed(rows, w, scales, biases, group_size, bits, (gt, ap)).reshape(x.shape)
            return grad_x, grad_a, grad_b if need_b else None, None, None, None, None, None, None, None
        if need_x or need_a:
            gt = torch.matmul(g, lora_b.t())
            if scale != 1.0:
                gt = scale * gt
        if need_a:
            grad_a = torch.matmul(x2.t(), gt)
        if need_b:
            grad_b = torch.matmul((torch.matmul(x2, lora_a) if twice else rest[0]).t(), g)
            if scale != 1.0:
                grad_b = scale * grad_b
        if need_x:
            update = None if twice else (_operand(gt), _operand(lora_a))
            grad_x = core._matmul_untransposed(grad_y, w, scales, biases, group_size, bits, update)
            if twice:
                grad_x = grad_x + torch.matmul(gt, lora_a.t()).reshape(grad_x.shape)
        return grad_x, grad_a, grad_b, None, None, None, None, None, None, None


# of the kernels in csrc/lora.hip; above, and where N % 32, the products are torch's (rank 64, 1024 rows of 12288: 33 us for
# the first of them against the BLAS library's 13)
_TRAINING_MAX_RANK = 32


def _rows(t: torch.Tensor) -> torch.Tensor:
    """``t`` as a contiguous matrix of its last dimension's rows at a 16-byte address."""
    t = t.reshape(-1, t.shape[-1]).contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _operand(t: torch.Tensor) -> torch.Tensor:
    """A factor as the kernels take it: zero columns up to a multiple of the step
    they take the rank in, contiguous, 16-byte aligned (a parameter may be a view
    of a flat buffer at any offset)."""
    pad = -t.shape[1] % _RANK_STEP
    t = (torch.nn.functional.pad(t, (0, pad)) if pad else t).contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")
_GLOBAL_HOOKS = ("_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks",
                 "_global_backward_pre_hooks")


def _trains_in_one(base: torch.nn.Module, lora: LoRALinear, x: torch.Tensor) -> bool:
    """Whether a call with gradients is what ``_LoRALinearFunction`` computes: plain
    16-bit HIP tensors of one type against a plain ``QuantizedLinear`` whose own
    call nobody watches (hooks) or replaces, with more than 16 rows (below them the
    update is a launch of its own anyway), and none of the transforms that need
    the composition's own operations (tracing, functorch, forward mode, autocast)."""
    if type(base) is not QuantizedLinear or base.mode != "affine" or base.__dict__.get("_prepared") is not None:
        return False
    if not all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda and t.device == x.device and t.dtype == x.dtype
               for t in (x, lora.lora_A, lora.lora_B, base.scales, base.biases)):
        return False
    if x.dtype not in (torch.bfloat16, torch.float16) or type(lora.scale) not in (int, float):
        return False
    K, N, rank = base.input_dims, base.output_dims, lora.lora_A.shape[-1]
    if (x.shape[-1:] != (K,) or x.numel() <= 16 * K or lora.lora_A.shape != (K, rank) or lora.lora_B.shape != (rank, N)
            or not 1 <= rank <= 1024 or base.weight.ndim != 2 or base.weight.device != x.device):
        return False
    if base.bias is not None and (base.bias.requires_grad or base.bias.dtype != x.dtype or base.bias.device != x.device):
        return False
    if base.scales.requires_grad or base.biases.requires_grad:
        return False
    if "forward" in base.__dict__ or any(getattr(base, h) for h in _HOOKS):
        return False
    if any(getattr(torch.nn.modules.module, h, None) for h in _GLOBAL_HOOKS):
        return False
    return not (torch.jit.is_tracing() or torch.compiler.is_compiling() or torch.is_autocast_enabled("cuda")
                or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0)


def _forward(owner: torch.nn.Module, base: torch.nn.Module, loras: list[LoRALinear], x: torch.Tensor) -> torch.Tensor:
    if not loras:
        return base(x)
    needs_grad = torch.is_grad_enabled() and (
        x.requires_grad or any(lora.lora_A.requires_grad or lora.lora_B.requires_grad for lora in loras))
    rank = sum(lora.lora_A.shape[1] for lora in loras)
    fused = (isinstance(base, QuantizedLinear) and x.is_cuda and not needs_grad and rank <= 1024
             and base.scales.dtype in (torch.bfloat16, torch.float16) and x.numel() > 0)
    if not fused:
        if needs_grad and len(loras) == 1 and _trains_in_one(base, loras[0], x):
            lora = loras[0]
            return _LoRALinearFunction.apply(x, lora.lora_A, lora.lora_B, base.weight, base.scales, base.biases, base.bias,
                                             float(lora.scale), base.group_size, base.bits)
        return _composed(base, loras, x)
    compute = base.scales.dtype
    a_cat, af, bs = _packed_for(owner, loras, compute)
    # t = x @ [lora_A_1 | lora_A_2 | ...], float32 sums rounded once.  Rows of up to 4096 elements (the hidden
    # sizes of the transformer blocks): one read of x in csrc/lora.hip, on a par with or ahead of the BLAS
    # library.  Longer rows (the MLP down-projections, K = 10240 .. 15360): the library's skinny split-K GEMM,
    # which is 1.2-1.6x faster there (the kernel streams such rows from memory at 3.5 TB/s only).
    K = x.shape[-1]
    if K <= _DOWN_KERNEL_MAX_K:
        t = _lib.ops().low_rank_down(x.to(compute).reshape(-1, K).contiguous(), af).reshape(*x.shape[:-1], bs.shape[1])
    else:
        t = torch.matmul(x.to(compute), a_cat)
    return core.quantized_matmul(x, base.weight, base.scales, base.biases, transpose=True, group_size=base.group_size,
                                 bits=base.bits, mode=base.mode, bias=base.bias, low_rank=(t, bs))


# ---- baking adapters into the base weights (for saving) -------------------------
def _delta(lora: LoRALinear) -> torch.Tensor:
    """``scale * (lora_A @ lora_B).T``, ``[out, in]``, in float32."""
    return float(lora.scale) * torch.matmul(lora.lora_A.detach().float(), lora.lora_B.detach().float()).t()


def _bake(base: torch.nn.Module, loras: list[LoRALinear], requantize: bool) -> None:
    if not hasattr(base, "weight") or not loras:
        return
    quantized = isinstance(base, QuantizedLinear)
    shape = (base.output_dims, base.input_dims) if quantized and requantize else tuple(base.weight.shape)
    deltas = []
    for lora in loras:
        delta = _delta(lora)
        if tuple(delta.shape) != shape:
            print(f"⚠️  Skipping LoRA bake due to shape mismatch: weight {shape} vs delta {tuple(delta.shape)}")
            continue
        deltas.append(delta)
    if not deltas:
        return
    if quantized:
        # all adapters at once, so that the weight is requantized a single time
        full = core.dequantize(base.weight, base.scales, base.biases, base.group_size, base.bits)
        baked = (full.float() + sum(deltas).to(full.device)).to(full.dtype)
        # written into the layer's own tensors: they may be views of a stack (nn.concat_quantized)
        for old, new in zip((base.weight, base.scales, base.biases),
                            core.quantize(baked, base.group_size, base.bits, base.mode)):
            old.copy_(new)
        return
    with torch.no_grad():
        for delta in deltas:   # one rounded add per adapter, as the reference does
            base.weight.add_(delta.to(device=base.weight.device, dtype=base.weight.dtype))


def bake_and_strip_lora(module: torch.nn.Module, requantize: bool = False) -> torch.nn.Module:
    """Replaces every ``LoRALinear`` / ``FusedLoRALinear`` below ``module`` by its
    base layer with the adapters added into the weight, as
    ``LoRASaver.bake_and_strip_lora``
    (src/mflux/models/common/lora/mapping/lora_saver.py:9-82) does before a
    model is saved: ``weight += (scale * lora_A @ lora_B).T`` in the weight's
    dtype.  Around a quantized base the reference's shapes do not match and it
    strips the wrapper without baking (``:75-77``), and so does this function
    by default; ``requantize=True`` instead dequantizes the base, adds the
    adapters in float32, rounds to the 16-bit type and quantizes again with the
    layer's group size and bits (lossy by one requantization).  Returns
    ``module`` (the base layer when ``module`` itself is a wrapper)."""
    def strip(obj: torch.nn.Module) -> torch.nn.Module:
        if isinstance(obj, FusedLoRALinear):
            _bake(obj.base_linear, [lora for lora in obj.loras if isinstance(lora, LoRALinear)], requantize)
            return obj.base_linear
        if isinstance(obj, LoRALinear):
            _bake(obj.linear, [obj], requantize)
            return obj.linear
        return obj

    module = strip(module)
    for name, child in list(module.named_children()):
        module._modules[name] = bake_and_strip_lora(child, requantize)
    return module
