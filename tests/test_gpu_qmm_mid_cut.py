"""GPU parity: the 128-column-tile GEMM (csrc/qmm_mid.hip) where its plan cuts K
into ranges of unequal length and picks 128- or 256-row tiles, against float64
on the dequantised weights.

Tolerance: 1e-2 of a row's largest output (one rounding of the weights and one
of the result to bfloat16, 2^-9 each, as for the other GEMM kernels).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(M, K, N, bits, gs, seed):
    import mflux_amd

    gen = torch.Generator(device="cuda").manual_seed(seed)
    w = (torch.randn(N, K, generator=gen, device="cuda") * 0.02).bfloat16()
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    bias = (torch.randn(N, generator=gen, device="cuda") * 0.02).bfloat16()
    packed = mflux_amd.quantize(w, gs, bits)
    wide = mflux_amd.dequantize(*packed, gs, bits, dtype=torch.float32).double()
    return x, packed, bias, x.double() @ wide.t()


def _close(y, ref):
    err = (y.double() - ref).abs().amax(dim=1) / ref.abs().amax(dim=1)
    assert float(err.max()) <= 1e-2


# K: 5, 10, 7 and 37 scale periods (groups of 64; half or twice that for 128 and 32) against any number of ranges.  With
# columns that are a multiple of 8 the sliced kernel takes these; with 4 more this one does.
@pytest.mark.parametrize("bits,gs", [(4, 64), (8, 64), (6, 64), (3, 128), (4, 128), (8, 32)])
@pytest.mark.parametrize("M,K,N", [(17, 1280, 64), (129, 2560, 392), (300, 1792, 1000), (513, 9472, 128), (1000, 1280, 264),
                                   (17, 1280, 68), (129, 2560, 396), (300, 1792, 1004), (513, 9472, 132), (1000, 1280, 268)])
def test_unequal_k_ranges(M, K, N, bits, gs):
    import mflux_amd
    from gpu_util import kernel_of
    from mflux_amd import _lib

    if K % (4 * gs):
        K += 4 * gs - K % (4 * gs)
    if N % 8:
        kernel, ranges = kernel_of(M, K, N, bits, gs)
        assert kernel == _lib.KERNEL_TILES_128 and ranges > 1
    x, packed, bias, ref = _operands(M, K, N, bits, gs, 71)
    _close(mflux_amd.quantized_matmul(x, *packed, group_size=gs, bits=bits, bias=bias), ref + bias.double())
    _close(mflux_amd.quantized_matmul(x.float(), *packed, group_size=gs, bits=bits), ref)


# on the sliced kernel, and on this one: 128-row tiles and 256-row ones, few ranges and many
@pytest.mark.parametrize("M,K,N,bits,here", [
    (40, 1280, 256, 4, False), (300, 1280, 256, 4, False), (520, 1280, 256, 4, False), (70, 2560, 12296, 4, True),
    (200, 9728, 3072, 8, True), (256, 12288, 3072, 4, True), (1030, 1280, 264, 4, True), (1100, 2560, 392, 5, True)])
def test_unequal_k_ranges_with_update_and_epilogue(M, K, N, bits, here):
    """The low-rank update enters once, with the first range; GELU and gate are the reduction's."""
    import mflux_amd
    from gpu_util import kernel_of
    from mflux_amd import _lib, core

    kernel, ranges = kernel_of(M, K, N, bits, 64)
    assert (kernel == _lib.KERNEL_TILES_128 and ranges > 1) == here
    x, packed, bias, ref = _operands(M, K, N, bits, 64, 72)
    t, bs = torch.randn(M, 16, device="cuda").bfloat16(), (torch.randn(N, 16, device="cuda") * 0.02).bfloat16()
    y = mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=bits, bias=bias, low_rank=(t, bs))
    _close(y, ref + bias.double() + t.double() @ bs.double().t())
    plain = mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=bits, bias=bias)
    gate, res = torch.randn(N, device="cuda").bfloat16(), torch.randn(M, N, device="cuda").bfloat16()
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="gate_residual", group_size=64, bits=bits, bias=bias, gate=gate, residual=res)
    assert torch.equal(y, res + gate * plain)
    y = core.quantized_matmul_epilogue(x, *packed, epilogue="gelu", group_size=64, bits=bits, bias=bias)
    # the linear's 1e-2 of ITS largest output in the row, through a slope of at most 1.13, and one more rounding
    lin = ref + bias.double()
    want = torch.nn.functional.gelu(lin, approximate="tanh")
    bound = 1.13e-2 * lin.abs().amax(dim=1) + 2.0 ** -9 * want.abs().amax(dim=1)
    assert bool(((y.double() - want).abs().amax(dim=1) <= bound).all())


@pytest.mark.parametrize("M,K,N,bits", [(320, 512, 33024, 4), (600, 512, 12288, 8)])
def test_shapes_between_the_two_tile_sizes(M, K, N, bits):
    """Rows that fill 128-row tiles and leave 256-row ones half empty, on enough columns for the large tiles."""
    import mflux_amd

    x, packed, bias, ref = _operands(M, K, N, bits, 64, 73)
    _close(mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=bits, bias=bias), ref + bias.double())


def test_planes_of_every_cut_fit_the_static_scratch():
    """No plan asks for more float32 planes than mfq_qmm_t_static's buffer holds (32 MiB), so what it
    accepted it accepts."""
    from mflux_amd import _lib

    need = _lib.load().mfq_qmm_t_workspace_bytes
    for M in (17, 64, 128, 129, 200, 256, 300, 384, 400, 512):
        for K in (256, 1280, 2560, 3072, 9728, 12288, 18944):
            for N in (64, 512, 1024, 2560, 3072, 4304, 9216, 12288):
                assert need(M, K, N, 64, 4) <= 32 << 20
