"""GPU parity: the GEMM with K sliced over the wavefronts of a workgroup (csrc/qmm_slice.hip), at the edges of its tiles
(32 and 64 rows; 32, 48, 64, 80 and 96 columns), rings, chunks and windows, and the kernels that take the same call when scales
and biases lie at odd addresses (the 128-column tiles in their form for those, K whole).

Reference: float64 on the dequantised weights rounded once to the 16-bit type, which is what the kernels multiply.  What
is left is the rounding of the result (half a unit in the last of 8 or 11 significant bits, at most 2^-8 of it in bfloat16
and 2^-11 in float16; the bias add rounds once more) and the float32 sums (K 2^-24 of the sum of magnitudes, below 2^-12
of a row's largest output on these operands).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _operands(M, K, N, bits, gs, dtype, seed=81):
    import mflux_amd

    gen = torch.Generator(device="cuda").manual_seed(seed)
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


# rows: one, a tile's less one, a tile, one more, several; columns: a single piece, ragged, whole tiles
# K: wavefronts without a sub-step (128, 192), fewer than the ring holds, ends inside a chunk and a window, long
@pytest.mark.parametrize("M,K,N", [
    (17, 128, 40), (33, 256, 8), (32, 640, 96), (31, 768, 3064), (64, 1280, 264), (65, 768, 3072), (129, 1152, 1000),
    (300, 3072, 1032), (256, 3072, 3072), (200, 2560, 4096), (512, 3072, 3072), (1000, 512, 264)])
@pytest.mark.parametrize("bits,gs,dtype", [(4, 64, "bf16"), (4, 32, "f16"), (4, 128, "bf16"), (8, 64, "bf16"), (8, 32, "bf16"),
                                           (3, 64, "bf16"), (5, 32, "f16"), (6, 64, "bf16"), (6, 128, "f16")])
def test_tiles_rings_and_the_other_kernel(M, K, N, bits, gs, dtype):
    import mflux_amd

    dtype = DT[dtype]
    if K % (2 * gs):
        K += 2 * gs - K % (2 * gs)
    x, (wq, s, b), bias, ref = _operands(M, K, N, bits, gs, dtype)
    y = mflux_amd.quantized_matmul(x, wq, s, b, group_size=gs, bits=bits, bias=bias)
    _close(y, ref + bias.double(), dtype, 2)
    other = mflux_amd.quantized_matmul(x, wq, _at_odd_address(s), _at_odd_address(b), group_size=gs, bits=bits, bias=bias)
    _close(other, ref + bias.double(), dtype, 2)
    y32 = mflux_amd.quantized_matmul(x.float(), wq, s, b, group_size=gs, bits=bits)  # float32 out: no rounding of the result
    assert y32.dtype == torch.float32
    _close(y32, ref, dtype, 0)


# few tiles and a long K: cut over workgroups into float32 planes
@pytest.mark.parametrize("M,K,N,bits,gs", [(100, 18944, 520, 4, 64), (50, 12288, 2560, 4, 64), (20, 9728, 64, 8, 32),
                                           (90, 6144, 512, 3, 128), (400, 15360, 128, 6, 64)])
def test_k_cut_over_workgroups(M, K, N, bits, gs):
    import mflux_amd

    x, packed, bias, ref = _operands(M, K, N, bits, gs, torch.bfloat16)
    y = mflux_amd.quantized_matmul(x, *packed, group_size=gs, bits=bits, bias=bias)
    _close(y, ref + bias.double(), torch.bfloat16, 2)


@pytest.mark.parametrize("rank", [16, 48, 160])
@pytest.mark.parametrize("M,K,N", [(40, 768, 320), (256, 3072, 3072), (70, 9728, 64)])
def test_low_rank_update(M, K, N, rank):
    import mflux_amd

    x, packed, bias, ref = _operands(M, K, N, 4, 64, torch.bfloat16)
    t, bs = torch.randn(M, rank, device="cuda").bfloat16(), (torch.randn(N, rank, device="cuda") * 0.02).bfloat16()
    y = mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=4, bias=bias, low_rank=(t, bs))
    _close(y, ref + bias.double() + t.double() @ bs.double().t(), torch.bfloat16, 2)


@pytest.mark.parametrize("M,K,N", [(40, 768, 320), (256, 3072, 3072), (100, 2560, 4096), (512, 3072, 3072), (70, 9728, 64)])
def test_epilogues_are_the_separate_operations(M, K, N):
    """Gate and residual, and SwiGLU (whose tiles take other weight rows), on the linear layer's own values bit for bit;
    GELU rounds once where torch's does."""
    import mflux_amd
    from mflux_amd import core

    x, packed, bias, _ = _operands(M, K, N, 4, 64, torch.bfloat16)
    lin = mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=4, bias=bias)
    gate, res = torch.randn(N, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="gate_residual", group_size=64, bits=4, bias=bias, gate=gate, residual=res)
    assert torch.equal(y, res + gate * lin)
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="gelu", group_size=64, bits=4, bias=bias, act_from=N // 2)
    assert torch.equal(y[:, : N // 2], lin[:, : N // 2])
    want = torch.nn.functional.gelu(lin[:, N // 2:].double(), approximate="tanh")
    assert bool(((y[:, N // 2:].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all())
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="swiglu", group_size=64, bits=4, bias=bias)
    want = core.swiglu_unstack(lin).double()
    assert bool(((y.double() - want).abs() <= 2.0 ** -6 * want.abs() + 1e-6).all())  # the sigmoid's last place, twice rounded


def test_update_and_swiglu_together():
    """The update's rows are the tile's own weight rows, half of them the gate's and half the up projection's.  The C interface
    offers no call with both, so the launcher is called itself."""
    import ctypes

    import mflux_amd
    from mflux_amd import _lib, core

    class LowRank(ctypes.Structure):
        _fields_ = [("t", ctypes.c_void_p), ("bs", ctypes.c_void_p), ("R", ctypes.c_int)]

    class Epilogue(ctypes.Structure):
        _fields_ = [("kind", ctypes.c_int), ("gate", ctypes.c_void_p), ("residual", ctypes.c_void_p), ("act_from", ctypes.c_int)]

    M, K, N, rank = 70, 3072, 1024, 48
    ptr, i64, i32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    launch = getattr(_lib.load(), "_ZN3mfq16launch_qmm_sliceEPKvillPKjS1_S1_S1_liiPviS4_mP12ihipStream_tNS_7LowRankENS_8EpilogueE")
    launch.restype = i32
    launch.argtypes = [ptr, i32, i64, i64, ptr, ptr, ptr, ptr, i64, i32, i32, ptr, i32, ptr, ctypes.c_size_t, ptr, LowRank, Epilogue]
    x, (wq, s, b), bias, _ = _operands(M, K, N, 4, 64, torch.bfloat16)
    t, bs = torch.randn(M, rank, device="cuda").bfloat16(), (torch.randn(N, rank, device="cuda") * 0.3).bfloat16()
    y = torch.empty(M, N // 2, device="cuda", dtype=torch.bfloat16)
    rc = launch(x.data_ptr(), _lib.BF16, M, K, wq.data_ptr(), s.data_ptr(), b.data_ptr(), bias.data_ptr(), N, 64, 4, y.data_ptr(),
                _lib.BF16, None, 0, torch.cuda.current_stream().cuda_stream, LowRank(t.data_ptr(), bs.data_ptr(), rank),
                Epilogue(_lib.EPILOGUE_SWIGLU, None, None, 0))
    assert rc == 0
    lin = mflux_amd.quantized_matmul(x, wq, s, b, group_size=64, bits=4, bias=bias, low_rank=(t, bs))
    want = core.swiglu_unstack(lin).double()
    assert bool(((y.double() - want).abs() <= 2.0 ** -6 * want.abs() + 1e-6).all())


# whole and ragged last tiles of columns and rows; K: a wavefront's sub-steps fewer than the ring holds, and more
@pytest.mark.parametrize("M,K,N,bits,gs,dtype", [
    (449, 1280, 2552, 4, 64, "bf16"), (449, 1280, 2552, 8, 64, "f16"), (449, 1280, 2552, 6, 32, "bf16"), (449, 1280, 2560, 5, 64, "f16"),
    (300, 1024, 4072, 3, 64, "bf16"), (33, 2560, 19448, 4, 32, "f16"), (64, 2560, 19456, 8, 64, "bf16"),
    (449, 1280, 2560, 4, 64, "bf16"), (449, 1280, 2552, 4, 128, "f16"), (33, 2560, 19456, 8, 128, "bf16")])
def test_tiles_of_80_columns(M, K, N, bits, gs, dtype):
    import mflux_amd
    from gpu_util import tile_of
    from mflux_amd import _lib, core

    for epilogue in (0, _lib.EPILOGUE_SWIGLU) if N % 64 == 0 else (0,):
        assert tile_of(M, K, N, bits, gs, epilogue) == (_lib.KERNEL_SLICED, 64, 80)
    dtype = DT[dtype]
    x, packed, bias, ref = _operands(M, K, N, bits, gs, dtype)
    y = mflux_amd.quantized_matmul(x, *packed, group_size=gs, bits=bits, bias=bias)
    _close(y, ref + bias.double(), dtype, 2)
    _close(mflux_amd.quantized_matmul(x.float(), *packed, group_size=gs, bits=bits), ref, dtype, 0)
    t, bs = torch.randn(M, 48, device="cuda").to(dtype), (torch.randn(N, 48, device="cuda") * 0.02).to(dtype)
    y_lr = mflux_amd.quantized_matmul(x, *packed, group_size=gs, bits=bits, bias=bias, low_rank=(t, bs))
    _close(y_lr, ref + bias.double() + t.double() @ bs.double().t(), dtype, 2)
    if N % 64 == 0:  # half of a tile's columns the gate's, half the up projection's
        z = core.quantized_matmul_epilogue(x, *packed, epilogue="swiglu", group_size=gs, bits=bits, bias=bias)
        want = core.swiglu_unstack(y).double()
        assert bool(((z.double() - want).abs() <= 2.0 ** -6 * want.abs() + 1e-6).all())
