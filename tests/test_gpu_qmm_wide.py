"""GPU parity: the GEMM whose wavefronts dequantise into registers (csrc/qmm_wide.hip) at the edges of its 128 x 256 tiles,
with one quad of steps to a range and several, K whole and cut into ranges, and against the kernels that take the same call
when scales and biases lie at odd addresses (forms for those, K whole).  The shapes are ones that its rule takes on 256
compute units, where a test does not say otherwise; the tests ask the library.

Reference: float64 on the dequantised weights rounded once to the 16-bit type, which is what the kernels multiply.  What
is left is the rounding of the result (at most 2^-8 of it in bfloat16 and 2^-11 in float16; the bias add rounds once more)
and the float32 sums (K 2^-24 of the sum of magnitudes, below 2^-12 of a row's largest output on these operands).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _operands(M, K, N, bits, gs, dtype):
    import mflux_amd

    gen = torch.Generator(device="cuda").manual_seed(83)
    w = (torch.randn(N, K, generator=gen, device="cuda") * 0.02).to(dtype)
    x = torch.randn(M, K, generator=gen, device="cuda").to(dtype)
    bias = (torch.randn(N, generator=gen, device="cuda") * 0.02).to(dtype)
    packed = mflux_amd.quantize(w, gs, bits)
    w_hat = mflux_amd.dequantize(*packed, gs, bits, dtype=torch.float32).to(dtype).double()
    return x, packed, bias, x.double() @ w_hat.t()


def _close(y, ref, dtype, roundings):
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    bound = (unit * roundings + 2.0 ** -12) * ref.abs().amax(dim=1)
    err = (y.double() - ref).abs().amax(dim=1)
    assert bool((err <= bound).all()), float((err / bound).max())


def _at_odd_address(t):
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:].copy_(t.reshape(-1))
    return buf[1:].view(t.shape)


# rows: part of a tile, a tile, one more, several; columns: ragged (no epilogue), a tile's part, whole tiles
# K: one quad (256) and two, whole over many quads, an even and an uneven cut into ranges, long
WHOLE = {4: [(100, 2304, 38016), (257, 256, 20480), (385, 256, 32770), (600, 256, 24584), (257, 2816, 16392)],
         8: [(600, 256, 24584), (257, 2816, 32776)]}
CUT = {4: [(384, 4096, 4100), (513, 12288, 1032), (1000, 12288, 1032)], 8: [(513, 12288, 1032), (1000, 12288, 1032)]}
NOT_TAKEN = [(40, 512, 32770), (128, 512, 32770), (128, 6144, 24584)]  # (wide calls of few rows, which are left)
FORMS = {4: [(64, "bf16"), (32, "f16"), (128, "bf16")], 8: [(64, "f16"), (64, "bf16"), (128, "bf16")]}


@pytest.mark.parametrize("M,K,N,bits,gs,dtype", [
    (*shape, bits, *form) for bits in (4, 8) for shape in WHOLE[bits] + CUT[bits] + NOT_TAKEN for form in FORMS[bits]])
def test_tiles_ranges_and_the_other_kernels(M, K, N, bits, gs, dtype):
    import mflux_amd
    from gpu_util import kernel_of
    from mflux_amd import _lib

    kernel, ranges = kernel_of(M, K, N, bits, gs)
    assert (kernel == _lib.KERNEL_WIDE) == ((M, K, N) not in NOT_TAKEN)
    assert kernel != _lib.KERNEL_WIDE or (ranges > 1) == ((M, K, N) in CUT[bits])
    dtype = DT[dtype]
    x, (wq, s, b), bias, ref = _operands(M, K, N, bits, gs, dtype)
    y = mflux_amd.quantized_matmul(x, wq, s, b, group_size=gs, bits=bits, bias=bias)
    _close(y, ref + bias.double(), dtype, 2)
    other = mflux_amd.quantized_matmul(x, wq, _at_odd_address(s), _at_odd_address(b), group_size=gs, bits=bits, bias=bias)
    _close(other, ref + bias.double(), dtype, 2)
    y32 = mflux_amd.quantized_matmul(x.float(), wq, s, b, group_size=gs, bits=bits)  # float32 out: no rounding of the result
    assert y32.dtype == torch.float32
    _close(y32, ref, dtype, 0)


@pytest.mark.parametrize("M,K,N,bits", [(257, 256, 20480, 4), (640, 12288, 1032, 4), (257, 2816, 32776, 8)])
@pytest.mark.parametrize("rank", [16, 48])
def test_low_rank_update(M, K, N, bits, rank):
    import mflux_amd
    from gpu_util import kernel_of
    from mflux_amd import _lib

    assert kernel_of(M, K, N, bits, 64)[0] == _lib.KERNEL_WIDE
    x, packed, bias, ref = _operands(M, K, N, bits, 64, torch.bfloat16)
    t, bs = torch.randn(M, rank, device="cuda").bfloat16(), (torch.randn(N, rank, device="cuda") * 0.02).bfloat16()
    y = mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=bits, bias=bias, low_rank=(t, bs))
    _close(y, ref + bias.double() + t.double() @ bs.double().t(), torch.bfloat16, 2)


# K whole over one quad of steps and over eleven, and cut
@pytest.mark.parametrize("M,K,N,bits", [(257, 256, 20480, 4), (257, 2816, 16448, 4), (640, 12288, 1088, 4), (257, 2816, 32832, 8),
                                        (640, 12288, 1088, 8)])
def test_epilogues_are_the_separate_operations(M, K, N, bits):
    """Gate and residual, and SwiGLU, on the linear layer's own values; GELU rounds once where torch's does."""
    import mflux_amd
    from gpu_util import kernel_of
    from mflux_amd import _lib, core

    assert kernel_of(M, K, N, bits, 64)[0] == _lib.KERNEL_WIDE
    x, packed, bias, _ = _operands(M, K, N, bits, 64, torch.bfloat16)
    lin = mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=bits, bias=bias)
    gate, res = torch.randn(N, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="gate_residual", group_size=64, bits=bits, bias=bias, gate=gate, residual=res)
    assert torch.equal(y, res + gate * lin)
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="gelu", group_size=64, bits=bits, bias=bias, act_from=N // 2)
    assert torch.equal(y[:, : N // 2], lin[:, : N // 2])
    want = torch.nn.functional.gelu(lin[:, N // 2:].double(), approximate="tanh")
    assert bool(((y[:, N // 2:].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all())
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="swiglu", group_size=64, bits=bits, bias=bias)
    want = core.swiglu_unstack(lin).double()
    assert bool(((y.double() - want).abs() <= 2.0 ** -6 * want.abs() + 1e-6).all())  # the sigmoid's last place, twice rounded


# the last tile of a column with 44, 64 (half, the loop of its own) and 65 rows (the whole tile's loop); K whole and cut
@pytest.mark.parametrize("M", [300, 320, 321])
@pytest.mark.parametrize("K,N,bits,gs,dtype", [(2816, 16448, 4, 64, "bf16"), (2816, 16448, 4, 32, "f16"), (18944, 3592, 4, 128, "bf16"),
                                               (2816, 32832, 8, 64, "bf16")])
def test_a_last_tile_of_half_its_rows(M, K, N, bits, gs, dtype):
    import mflux_amd
    from gpu_util import kernel_of
    from mflux_amd import _lib

    assert kernel_of(M, K, N, bits, gs)[0] == _lib.KERNEL_WIDE
    x, packed, bias, ref = _operands(M, K, N, bits, gs, DT[dtype])
    y = mflux_amd.quantized_matmul(x, *packed, group_size=gs, bits=bits, bias=bias)
    _close(y, ref + bias.double(), DT[dtype], 2)
    rows = mflux_amd.quantized_matmul(x[:256], *packed, group_size=gs, bits=bits, bias=bias)  # (whole tiles only)
    if kernel_of(M, K, N, bits, gs) == kernel_of(256, K, N, bits, gs):
        assert torch.equal(y[:256], rows)
