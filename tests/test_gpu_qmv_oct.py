"""GPU parity: the matvec kernels that take eight weight rows at a time on the
int8 matrix instruction (csrc/qmv_oct.hip for 8-bit codes, csrc/qmv_oct4.hip
for 4-bit codes: groups of 64, one to sixteen activation rows, K of 256, 1024,
2048, 2560, 3072, 3840, 4096 and 6144, N a multiple of 8) against the float64
oracle on MLX-format operands, through the C ABI.

Tolerance of this path: max |y - y_ref| <= 1e-2 * max|y_ref row| per output
row; the cases with float32 output show how far inside it the kernel is.
"""
import numpy as np
import pytest
import torch

from conftest import seeded
from test_gpu_qmm import TOL, _assert_close, _case, _ref, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("K", [1024, 2048, 3072, 4096])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_oct_vs_f64(oracle, K, M, bits):
    """Every K the kernel is built for (one to four 128-byte steps per
    wavefront), every number of activation rows, runs of blocks that are not
    whole trips of three (N = 8 * 53 rows: some workgroups get one block, some
    two), with the layer bias."""
    o = oracle
    args = _case(o, 61, M, K, 8 * 53 if K != 3072 else 8 * 530, bits)
    _assert_close(_run(o, *args, bits), _ref(o, *args, bits))


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("N", [8, 16, 24, 72, 8 * 257, 8 * 256 * 4 + 8, 8 * 256 * 12 + 16])
def test_oct_run_lengths(oracle, N, bits):
    """One block in all; fewer blocks than compute units; one, four and five
    blocks to a workgroup; and past twelve blocks to a compute unit, where the
    weight is cut into runs of nine blocks for as many workgroups as it takes."""
    o = oracle
    args = _case(o, 62, 2 if bits == 8 else 3, 1024, N, bits)
    _assert_close(_run(o, *args, bits), _ref(o, *args, bits))


@pytest.mark.parametrize("bits", [8, 4])
def test_oct_through_the_c_abi_f16_f32_no_bias(oracle, bits):
    """mfq_qmm_t through ctypes: float16 operands, float32 output, no bias; and
    bfloat16 with bias, bit for bit what the Python level returns."""
    import mflux_amd
    from gpu_util import to_dev, u32_to_dev
    from mflux_amd import _lib

    o = oracle
    lib = _lib.load()
    M, K, N = 3, 2048, 8 * 130
    x = o._from_f32(seeded(63, 0, (M, K), 1.0), o.F16)
    w = o._from_f32(seeded(63, 1, (N, K), 0.02), o.F16)
    wq, s, b = o.c_quantize(w, o.F16, 64, bits)
    xd, wd, sd, bd = to_dev(x, o.F16), u32_to_dev(wq), to_dev(s, o.F16), to_dev(b, o.F16)
    y = torch.empty(M, N, device="cuda", dtype=torch.float32)
    stream = torch.cuda.current_stream().cuda_stream
    rc = lib.mfq_qmm_t(xd.data_ptr(), _lib.F16, M, K, wd.data_ptr(), sd.data_ptr(), bd.data_ptr(), _lib.F16, None,
                       N, 64, bits, y.data_ptr(), _lib.F32, stream)
    assert rc == 0, rc
    torch.cuda.synchronize()
    ref = o.quantized_matmul_f64(o._to_f32(x, o.F16).astype(np.float64), wq, s, b, o.F16, 64, bits)
    _assert_close(y, ref, tol=2e-3)  # nothing is rounded to 16 bits on this path
    args = _case(o, 64, 4, 3072, 8 * 100, bits)
    y_py = _run(o, *args, bits)
    xb, wqb, sb, bb, bias = args
    xd, wd, sd, bd, biasd = (to_dev(xb, o.BF16), u32_to_dev(wqb), to_dev(sb, o.BF16), to_dev(bb, o.BF16),
                             to_dev(bias, o.BF16))
    y2 = torch.empty(4, 8 * 100, device="cuda", dtype=torch.bfloat16)
    rc = lib.mfq_qmm_t(xd.data_ptr(), _lib.BF16, 4, 3072, wd.data_ptr(), sd.data_ptr(), bd.data_ptr(), _lib.BF16,
                       biasd.data_ptr(), 8 * 100, 64, bits, y2.data_ptr(), _lib.BF16, stream)
    assert rc == 0, rc
    torch.cuda.synchronize()
    assert torch.equal(y2, y_py)
    _assert_close(y2, _ref(o, *args, bits), tol=TOL)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M", [1, 4])
def test_oct_one_hot_rows_return_weight_columns(oracle, M, bits):
    """One-hot activation rows return columns of the weight: every byte of a
    wavefront's 128-byte steps, both halves of a step (the two halves of the
    matrix instruction's A operand), every eighth of K, against scale * code +
    bias to a thousandth of a code step (float32 output: nothing is rounded)."""
    import mflux_amd
    from gpu_util import to_dev, u32_to_dev

    o = oracle
    K, N = 3072, 64
    w = o.f32_to_bf16_bits(seeded(65, 1, (N, K), 0.02))
    wq, s, b = o.c_quantize(w, o.BF16, 64, bits)
    exact = o.dequantize_exact(wq, s, b, o.BF16, 64, bits).astype(np.float64)
    step = np.abs(o.bf16_bits_to_f32(s).astype(np.float64))
    ks = list(range(0, 260)) + [383, 384, 385, 447, 448, 1023, 1024, 1535, 1536, 2687, 2688, 3008, 3071]
    for k0 in ks:
        cols = [(k0 + 389 * m) % K for m in range(M)]
        xf = np.zeros((M, K), dtype=np.float32)
        for m, k in enumerate(cols):
            xf[m, k] = 1.0
        y = mflux_amd.quantized_matmul(to_dev(o.f32_to_bf16_bits(xf), o.BF16).float(), u32_to_dev(wq),
                                       to_dev(s, o.BF16), to_dev(b, o.BF16), group_size=64, bits=bits)
        got = y.cpu().numpy().astype(np.float64)
        for m, k in enumerate(cols):
            assert np.all(np.abs(got[m] - exact[:, k]) <= 1e-3 * step[:, k // 64]), (k0, m)


def test_oct_unit_weight_is_exact(oracle):
    """Codes 1 on the diagonal and 0 elsewhere, scale 1, bias 0: y = x exactly
    (float32 output), although every code enters the matrix instruction as
    code - 128 -- the 128 * sum(xq) that this takes out is put back as an
    integer, before anything is rounded."""
    import mflux_amd
    from gpu_util import to_dev, u32_to_dev

    o = oracle
    K = N = 1024
    n = np.arange(N)
    wq = np.zeros((N, K // 4), dtype=np.uint32)
    wq[n, n // 4] = np.uint32(1) << (8 * (n % 4)).astype(np.uint32)
    one = o.f32_to_bf16_bits(np.ones((N, K // 64), np.float32))
    zero = o.f32_to_bf16_bits(np.zeros((N, K // 64), np.float32))
    x = o.f32_to_bf16_bits(np.abs(seeded(66, 0, (2, K), 1.0)) + np.float32(1.0))   # all positive: sum(xq) is large
    y = mflux_amd.quantized_matmul(to_dev(x, o.BF16).float(), u32_to_dev(wq), to_dev(one, o.BF16),
                                   to_dev(zero, o.BF16), group_size=64, bits=8)
    got = y.cpu().numpy().astype(np.float64)
    xf = o.bf16_bits_to_f32(x).astype(np.float64)
    # 15-bit fixed point of each eighth of a row: 2^-15 of the eighth's largest magnitude
    assert np.all(np.abs(got - xf) <= 2.0 ** -14 * np.abs(xf).max())


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("K", [256, 1024, 2048, 2560, 3072, 3840, 4096, 6144])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
def test_oct_row_lengths_and_eights_of_rows(oracle, K, M, bits):
    """Every split of K over the wavefronts, and activation rows on two, three and
    four workgroups of four or one and two of eight (the last with one row and full)."""
    o = oracle
    args = _case(o, 64, M, K, 8 * 261, bits)
    _assert_close(_run(o, *args, bits), _ref(o, *args, bits))


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("N", [8, 8 * 255, 8 * 256 * 11, 8 * 256 * 13 + 8])
@pytest.mark.parametrize("M", [7, 16])
def test_oct_run_lengths_of_eight_rows(oracle, N, bits, M):
    """Runs of one block, and past what the partial sums of a workgroup hold (two rounds of workgroups)."""
    o = oracle
    args = _case(o, 65, M, 1024 if bits == 4 else 2048, N, bits)
    _assert_close(_run(o, *args, bits), _ref(o, *args, bits))


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M,inf,nan", [(6, 1, 4), (16, 12, 15)])
def test_oct_infinity_and_nan_stay_in_their_rows(oracle, bits, M, inf, nan):
    """More than four rows: an infinity in x gives what the product with the
    dequantised weights gives (its own sign times the weight's), a NaN gives
    NaN, and the other rows are what they are without either."""
    import mflux_amd

    torch.manual_seed(66)
    K, N = 3072, 8 * 40
    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    wq, s, b = mflux_amd.quantize(w, 64, bits)
    x = torch.randn(M, K, device="cuda").bfloat16()
    clean = mflux_amd.quantized_matmul(x, wq, s, b, group_size=64, bits=bits)
    x[inf, 700] = float("inf")
    x[nan, 3] = float("nan")
    y = mflux_amd.quantized_matmul(x, wq, s, b, group_size=64, bits=bits)
    # (in float32: a weight that is zero only after the product's own rounding is not zero to the fma of a matmul)
    column = mflux_amd.dequantize(wq, s, b, 64, bits, dtype=torch.float32)[:, 700]
    torch.testing.assert_close(y[inf].float(), column * float("inf"), rtol=0, atol=0, equal_nan=True)
    assert bool(torch.isnan(y[nan]).all())
    keep = [m for m in range(M) if m not in (inf, nan)]
    assert torch.equal(y[keep], clean[keep])


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("K", [2560, 3840, 6144])
@pytest.mark.parametrize("silu", [False, True])
def test_oct_infinity_of_two_rows_on_the_other_row_lengths(oracle, K, bits, silu):
    """Two to four rows on row lengths that are no multiple of 1024, or above 4096: the same."""
    import mflux_amd

    torch.manual_seed(67)
    w = (torch.randn(8 * 20, K, device="cuda") * 0.02).bfloat16()
    wq, s, b = mflux_amd.quantize(w, 64, bits)
    x = torch.randn(3, K, device="cuda").bfloat16()
    x[1, 600] = float("inf")
    f = mflux_amd.silu_quantized_matmul if silu else mflux_amd.quantized_matmul
    y = f(x, wq, s, b, group_size=64, bits=bits)
    column = mflux_amd.dequantize(wq, s, b, 64, bits, dtype=torch.float32)[:, 600]
    torch.testing.assert_close(y[1].float(), column * float("inf"), rtol=0, atol=0, equal_nan=True)
    assert bool(torch.isfinite(y[[0, 2]]).all())


@pytest.mark.parametrize("K,bits,nan", [(256, 8, True), (256, 4, False), (512, 8, True), (512, 4, True), (1024, 8, True)])
@pytest.mark.parametrize("M", [2, 4])
def test_infinity_of_two_to_four_rows(oracle, K, bits, nan, M):
    """An infinity makes its row NaN in the kernels that hold x in 15 bits, and gives
    the dequantised weights' infinities in the others."""
    import mflux_amd

    torch.manual_seed(68)
    packed = mflux_amd.quantize((torch.randn(8 * 20, K, device="cuda") * 0.02).bfloat16(), 64, bits)
    x = torch.randn(M, K, device="cuda").bfloat16()
    x[1, 100] = float("inf")
    y = mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=bits)
    if nan:
        assert bool(torch.isnan(y[1]).all())
    else:
        column = mflux_amd.dequantize(*packed, 64, bits, dtype=torch.float32)[:, 100]
        torch.testing.assert_close(y[1].float(), column * float("inf"), rtol=0, atol=0, equal_nan=True)
    assert bool(torch.isfinite(y[[m for m in range(M) if m != 1]]).all())


# K, M, bits of the calls whose rows enter as 23-bit fixed point (the kernels that took them before kept x in
# its 16-bit type)
_WIDE = [(K, M, bits) for bits in (4, 8) for K in (256, 1024, 2048, 2560, 3072, 3840, 4096, 6144)
         for M in (2, 4, 5, 8, 9, 16)
         if M > 4 and (bits == 4 or K > 1024) or M <= 4 and (K in (2560, 3840, 6144) or (K, bits) == (256, 4))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,M,bits", _WIDE)
def test_oct_rows_with_outliers_in_float32(K, M, bits, dtype):
    """One element of every 128 at 300 times the others: the float32 output against
    float64.  An element enters with an error of 2^-23 of its part's largest at
    most, as a float32 sum over it would round; 0.6 * 2^-23 * sqrt(128) in the
    2-norm of a sum that this largest dominates, plus a float32 rounding for
    each of the partial sums: 2^-18.  (With 15 bits it was 2^-11.5, with weights
    rounded to 16 bits 2^-9 and 2^-12.)"""
    import mflux_amd

    torch.manual_seed(70)
    N = 8 * 33
    packed = mflux_amd.quantize((torch.randn(N, K, device="cuda") * 0.02).to(dtype), 64, bits)
    x = torch.randn(M, K, device="cuda")
    x[:, 5::128] = x[:, 5::128].sign() * 300
    x = x.to(dtype)
    y = mflux_amd.quantized_matmul(x.float(), *packed, group_size=64, bits=bits)
    assert y.dtype == torch.float32 and y.shape == (M, N)
    ref = x.double() @ mflux_amd.dequantize(*packed, 64, bits, dtype=torch.float32).double().t()
    # (dequantize rounds in float32 only: 2^-24 of a weight)
    for m in range(M):
        assert float((y[m].double() - ref[m]).norm() / ref[m].norm()) <= 2.0 ** -18, m


@pytest.mark.parametrize("K,N,M,bits", [(3072, 18432, 8, 8), (3072, 9216, 5, 4), (6144, 36864, 3, 8)])
def test_oct_time_with_an_infinity(K, N, M, bits):
    """A row with an infinity is walked again on the dequantised weights, by whole
    wavefronts: some times the finite call, not the 32 to 50 of a lane to each row."""
    import mflux_amd

    packed = mflux_amd.quantize((torch.randn(N, K, device="cuda") * 0.02).bfloat16(), 64, bits)
    x = torch.randn(M, K, device="cuda").bfloat16()

    def us(x):
        f = lambda: mflux_amd.quantized_matmul(x, *packed, group_size=64, bits=bits)
        f()
        best = 1e9
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                f()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        return best

    finite = us(x)
    x[1, 3] = float("inf")
    assert us(x) < 15 * finite
