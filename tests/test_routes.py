"""Which kernel a quantized product runs on and the workspace it asks for, as the library answers without a GPU (it then
counts 256 compute units, which is what the shapes below are for)."""
import ctypes

import pytest

from mflux_amd import _lib

GROUPS = ((4, 64), (4, 32), (4, 128), (8, 64), (8, 128), (3, 64), (5, 32), (6, 64))
ROWS = (2, 16, 17, 64, 129, 256, 300, 512, 640, 1000, 1024, 1030, 2100, 4608)
SIZES = ((256, 64), (768, 3072), (1280, 264), (2560, 4096), (3072, 3072), (3072, 12288), (12288, 3072), (3584, 37888), (18944, 520),
         (2080, 1000))


def route(M, K, N, bits, gs):
    ranges = ctypes.c_int()
    kernel = _lib.load().mfq_qmm_t_kernel(M, K, N, gs, bits, ctypes.byref(ranges))
    assert kernel > 0, (kernel, M, K, N, bits, gs)
    return kernel, ranges.value


def workspace(M, K, N, bits, gs):
    return _lib.load().mfq_qmm_t_workspace_bytes(M, K, N, gs, bits)


def test_arguments_are_checked():
    f = _lib.load().mfq_qmm_t_kernel
    assert f(4, 128, 8, 48, 4, None) == -2 and f(4, 128, 8, 64, 7, None) == -3
    for bad in ((0, 128, 8), (4, 100, 8), (4, 128, 0), (1 << 31, 128, 8)):
        assert f(*bad, 64, 4, None) == -4
    assert f(1, 8192, 64, 64, 3, None) == _lib.KERNEL_MATVEC and f(1, 8256, 64, 64, 3, None) == _lib.MFQ_EUNSUPPORTED
    assert f(16, 3072, 64, 64, 4, None) == _lib.KERNEL_MATVEC


@pytest.mark.parametrize("bits,gs", GROUPS)
def test_the_workspace_is_what_the_kernel_uses(bits, gs):
    """Planes for the ranges of K the kernel named takes and for no other kernel's, the 16-bit copy where that is made."""
    for M in ROWS:
        for K, N in SIZES:
            if K % gs:
                continue
            kernel, ranges = route(M, K, N, bits, gs)
            need = workspace(M, K, N, bits, gs)
            if kernel == _lib.KERNEL_MATVEC:
                assert need == 0
            elif kernel in (_lib.KERNEL_SLICED, _lib.KERNEL_WIDE, _lib.KERNEL_TILES_128):
                assert need == (ranges * M * N * 4 if ranges > 1 else 0), (M, K, N)
            else:
                copy = -(-N // 16) * 16 * K * 2 // 256 * 256 if kernel == _lib.KERNEL_TWO_KERNELS else 0
                planes = need - copy
                assert planes % (ranges * 256 * 256 * 4) == 0 and (planes > 0) == (ranges > 1), (M, K, N)


@pytest.mark.parametrize("M,K,N", [(256, 3072, 3072), (512, 3072, 3072), (300, 2560, 4096)])
def test_shapes_that_run_in_one_launch_ask_for_no_planes(M, K, N):
    for bits, gs in ((4, 64), (4, 128)):
        assert route(M, K, N, bits, gs) == (_lib.KERNEL_SLICED, 1)
        assert workspace(M, K, N, bits, gs) == 0


# measured on 256 units, us on the sliced and on the 128-column tiles
@pytest.mark.parametrize("M,K,N,bits,gs", [
    (33, 768, 37888, 6, 64),    # 27.3, 19.8
    (76, 3072, 12288, 6, 64),   # 33.0, 28.8
    (4, 768, 37888, 6, 128),    # 25.5, 20.9
    (128, 2560, 9216, 6, 128),  # 30.1, 26.4
    (442, 768, 3072, 5, 64),    # 15.4, 13.6
    (358, 1152, 4096, 4, 64),   # 19.7, 17.9
    (432, 2560, 3840, 4, 64),   # 28.3, 26.6
])
def test_the_sliced_kernel_is_left_where_it_is_the_slower(M, K, N, bits, gs):
    assert route(M, K, N, bits, gs)[0] == _lib.KERNEL_TILES_128


@pytest.mark.parametrize("M,K,N,bits,gs", [
    (840, 3072, 512, 5, 64), (16, 3072, 3072, 6, 64), (2, 2560, 4096, 3, 64), (256, 3072, 3072, 4, 64), (300, 2560, 4096, 6, 64),
    (208, 6144, 64, 5, 64),     # 11.5, 16.0
    (159, 3584, 4096, 6, 32),   # 23.5, 27.4
])
def test_the_sliced_kernel_is_kept_where_it_is_the_faster(M, K, N, bits, gs):
    assert route(M, K, N, bits, gs)[0] == _lib.KERNEL_SLICED


# measured on 256 units, us on the kernel named and on the other one
@pytest.mark.parametrize("M,K,N,bits,gs,wide", [
    (627, 18944, 3072, 4, 64, True),    # 87, 101
    (135, 3840, 12288, 4, 128, True),   # 42, 46
    (320, 3584, 37888, 4, 64, True), (320, 3584, 37888, 8, 64, True), (320, 18944, 3584, 4, 64, True), (100, 2304, 38016, 4, 64, True),
    (67, 2560, 19456, 4, 64, False),    # 29, 33
    (1019, 12288, 3072, 4, 128, False), # 89, 98
    (1024, 3072, 12288, 4, 64, False),  # 83, 89
    (879, 10240, 4096, 8, 32, False),   # 101, 163
])
def test_where_the_wide_kernel_is_taken(M, K, N, bits, gs, wide):
    assert (route(M, K, N, bits, gs)[0] == _lib.KERNEL_WIDE) == wide


def plan(M, K, N, bits, gs, epilogue):
    ranges, need = ctypes.c_int(), ctypes.c_size_t()
    kernel = _lib.load().mfq_qmm_t_plan(M, K, N, gs, bits, epilogue, ctypes.byref(ranges), None, None, ctypes.byref(need))
    return kernel, ranges.value, need.value


# measured on 256 units between a block's other kernels, us with the copy of the weights and without
@pytest.mark.parametrize("M,K,N,bits,gs,kernel", [
    (1600, 3840, 20480, 4, 64, _lib.KERNEL_TILES_256),     # 419, 407
    (1792, 3840, 20480, 8, 64, _lib.KERNEL_TILES_256),     # 444, 434
    (1600, 3072, 12288, 4, 64, _lib.KERNEL_TILES_256),
    (1793, 3840, 20480, 4, 64, _lib.KERNEL_TWO_KERNELS),   # 443, 458 (1850 rows)
    (2000, 3072, 21504, 8, 64, _lib.KERNEL_TWO_KERNELS),   # 479, 506
    (1281, 3840, 15360, 4, 128, _lib.KERNEL_TWO_KERNELS),  # K not whole scale periods: 208, 288 by itself
    (1600, 3072, 12288, 6, 64, _lib.KERNEL_TILES_128),
])
def test_where_calls_with_an_epilogue_copy_the_weights(M, K, N, bits, gs, kernel):
    """From 1281 to 1792 rows the two-kernel path is taken for its rounds of 192-column tiles, which have no epilogue: calls with
    one stay with the fused kernel, and ask for its planes only."""
    assert route(M, K, N, bits, gs)[0] == _lib.KERNEL_TWO_KERNELS
    for epilogue in (_lib.EPILOGUE_GELU, _lib.EPILOGUE_GATE_RESIDUAL, _lib.EPILOGUE_SWIGLU):
        got, ranges, need = plan(M, K, N, bits, gs, epilogue)
        assert got == kernel
        copy = N * K * 2 if kernel == _lib.KERNEL_TWO_KERNELS else 0
        tail = -(-M // 256) * -(-N // 256) % 256 * ranges * 256 * 256 * 4 if ranges > 1 else 0
        assert need == copy + (ranges * M * N * 4 if kernel == _lib.KERNEL_TILES_128 and ranges > 1 else tail)


@pytest.mark.parametrize("bits,gs", GROUPS)
def test_plans_agree_with_the_general_answers(bits, gs):
    for M in (*ROWS, 1281, 1600, 1900, 6889):
        for K, N in SIZES:
            if K % gs:
                continue
            kernel, ranges = route(M, K, N, bits, gs)
            most = workspace(M, K, N, bits, gs)
            for epilogue in range(4):
                got, r, need = plan(M, K, N, bits, gs, epilogue)
                if epilogue and (M <= 16 or (epilogue == _lib.EPILOGUE_SWIGLU and N % 64)):
                    assert got < 0 and need == 0
                    continue
                assert got > 0 and need <= most
                if not epilogue and need != most:  # whole 192-column tiles in the place of the cut
                    assert got == kernel == _lib.KERNEL_TWO_KERNELS and r == 1 < ranges and need == -(-N // 16) * 16 * K * 2
                elif not epilogue:
                    assert (got, r, need) == (kernel, ranges, most)
                elif kernel != _lib.KERNEL_TWO_KERNELS:
                    assert (got, r, need) == (kernel, ranges, most)


def test_whole_192_column_tiles_ask_for_no_planes():
    """Calls without an epilogue, the input gradient and prepared copies: of the copy, or of nothing, where the tail's cut is not run."""
    lib = _lib.load()
    copy = 3072 * 3072 * 2
    assert plan(6889, 3072, 3072, 4, 64, 0) == (_lib.KERNEL_TWO_KERNELS, 1, copy)
    assert plan(6889, 3072, 3072, 4, 64, _lib.EPILOGUE_GELU) == (_lib.KERNEL_TWO_KERNELS, 3, copy + 68 * 3 * 256 * 256 * 4)
    assert lib.mfq_qmm_n_workspace_bytes(6889, 3072, 3072, 64, 4) == copy
    assert lib.mfq_qmm_t_prepared_workspace_bytes(6889, 3072, 3072) == 0
    # a cut that is run: its planes
    assert plan(2100, 2048, 7440, 4, 64, 0) == (_lib.KERNEL_TWO_KERNELS, 8, 7440 * 2048 * 2 + 14 * 8 * 256 * 256 * 4)
    assert lib.mfq_qmm_n_workspace_bytes(4700, 1024, 3520, 64, 4) > 3520 * 1024 * 2
    assert lib.mfq_qmm_t_prepared_workspace_bytes(2100, 2048, 7440) > 0


@pytest.mark.parametrize("M,K,N,bits,gs,epilogue,tile", [
    (16, 3072, 64, 4, 64, 0, (0, 0)), (100, 2304, 38016, 4, 64, 0, (128, 256)), (256, 12288, 3072, 4, 64, 0, (256, 128)),
    (70, 3072, 12288, 4, 64, 0, (64, 96)), (17, 3072, 3072, 4, 64, 0, (32, 32)), (512, 3072, 2560, 4, 64, 0, (64, 80)),
    (1024, 3072, 21504, 4, 64, 0, (256, 256)), (6889, 3072, 3072, 4, 64, 0, (256, 192)), (6889, 3072, 3072, 4, 64, 2, (256, 256)),
    (4608, 3072, 21504, 4, 64, 0, (256, 256)), (4096, 3072, 3072, 4, 64, 0, (256, 192))])
def test_tiles_of_a_plan(M, K, N, bits, gs, epilogue, tile):
    rows, columns = ctypes.c_int(-1), ctypes.c_int(-1)
    assert _lib.load().mfq_qmm_t_plan(M, K, N, gs, bits, epilogue, None, ctypes.byref(rows), ctypes.byref(columns), None) > 0
    assert (rows.value, columns.value) == tile


def test_plan_checks_its_arguments():
    assert plan(4, 128, 8, 4, 48, 0) == (-2, 0, 0) and plan(40, 128, 64, 4, 64, 4)[0] == -4 and plan(40, 128, 64, 4, 64, -1)[0] == -4
    assert plan(40, 128, 12, 4, 64, _lib.EPILOGUE_GELU)[0] == _lib.MFQ_EUNSUPPORTED
    assert plan(16, 3072, 64, 4, 64, 0) == (_lib.KERNEL_MATVEC, 1, 0)
