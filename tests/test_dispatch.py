"""Which kernel the matmul entries choose (no GPU: the choice depends on the shape and on
256 compute units alone).  Each line was measured on both sides; the times stand at the
rules in capi.hip and gemm_kslice.hip."""
if __name__ == "__main__":  # `python tests/<file>.py`, as the reference runs its tests
    import sys as _sys

    import pytest as _pytest
    _sys.exit(_pytest.main([__file__, "-q"]))
import ctypes

import pytest

from jjjetson_ops_amd import capi

BOTH = (False, True)


@pytest.mark.parametrize("K,N,M,layouts", [
    (4096, 4096, 2048, BOTH), (3072, 4096, 2048, BOTH), (5632, 8192, 2048, BOTH),  # full rounds of 128 x 128
    (4096, 14336, 2048, BOTH), (11008, 4096, 2048, (True,)),
    (128, 8192, 65, BOTH), (256, 2048, 512, BOTH), (768, 11008, 129, BOTH),  # short rows
    (1024, 20480, 80, BOTH), (1024, 1024, 4096, BOTH),
])
def test_tiled(K, N, M, layouts):
    for split in layouts:
        assert capi.mm_auto_kernel(K, N, M, split) in (capi.ALGO_MFMA, capi.ALGO_MFMA64, capi.ALGO_MFMA32,
                                                       capi.ALGO_MFMA_W32)


@pytest.mark.parametrize("K,N,M,form", [
    (4096, 4096, 48, 0), (11008, 4096, 24, 0), (4096, 4096, 100, 1), (4096, 8192, 128, 2), (4096, 14336, 100, 3),
    (4096, 4096, 512, 3), (11008, 4096, 777, 3), (11008, 4096, 1024, 3), (4096, 11008, 640, 3),
])
def test_kslice(K, N, M, form):
    for split in BOTH:
        assert capi.mm_auto_kernel(K, N, M, split) == capi.KERNEL_KSLICE + form


@pytest.mark.parametrize("K,N,M", [(1536, 1 << 28, 17), (1536, 1 << 28, 32), (2048, 1 << 27, 64), (256, 1 << 28, 20)])
def test_launch_fits_the_grid(K, N, M):
    """A launch holds less than 2^32 threads in x; a K-sliced tile is a workgroup of 512
    threads (forms 0..2) or 256, in multiples of eight workgroups."""
    tile = ((32, 32, 512), (32, 64, 512), (64, 64, 512), (64, 64, 256))
    for split in BOTH:
        form = capi.mm_auto_kernel(K, N, M, split) - capi.KERNEL_KSLICE
        if form >= 0:
            rows, toks, threads = tile[form]
            assert (-(-N // rows) * -(-M // toks) + 7) // 8 * 8 * threads < 1 << 32
    a16 = ctypes.c_void_p(16)  # refused before any device is touched
    assert capi.lib().jjo_mm_kernel_device(a16, a16, a16, 1536, 1 << 28, 17, 0, capi.KERNEL_KSLICE,
                                           None) == capi.JJO_ERR_INVALID_ARG
    assert capi.mm_auto_kernel(1536, (1 << 28) - 256, 17) == capi.KERNEL_KSLICE  # the most that fits


@pytest.mark.parametrize("K,N,R,E,kernel", [
    (4096, 256, 48, 8, "gemv"), (14336, 256, 48, 8, "gemv"),
    (2048, 2816, 800, 64, 1), (1408, 2048, 800, 64, 1),  # 100 tokens, 64 experts top-8: gate|up, down
    (4096, 28672, 49, 8, 1), (4096, 1024, 48 * 8, 8, 1), (2048, 256, 80 * 8, 8, 1),
    (4096, 28672, 40 * 8, 8, 2), (14336, 4096, 40 * 8, 8, 2), (2048, 2816, 48 * 64, 64, 2),
    (4096, 28672, 1024, 8, "tiles"), (14336, 4096, 1024, 8, "tiles"), (4096, 1024, 81 * 8, 8, "tiles"),
    # tiles that fill the chip, many routes or short rows
    (2048, 2816, 80 * 64, 64, "tiles"), (128, 14336, 7 * 64, 64, "tiles"), (128, 14336, 80 * 8, 8, "tiles"),
    (256, 4096, 16 * 64, 64, "tiles"), (256, 4096, 64 * 64, 64, "tiles"), (512, 8192, 64 * 64, 64, "tiles"),
])
def test_grouped(K, N, R, E, kernel):
    want = {"gemv": capi.ALGO_GEMV, "tiles": capi.ALGO_MFMA}.get(kernel)
    assert capi.grouped_auto_kernel(K, N, R, E) == (capi.KERNEL_KSLICE + kernel if want is None else want)


def test_invalid_calls_are_refused():
    for bad in ((96, 64, 64, 4), (128, 0, 64, 4), (128, 64, 0, 4), (128, 64, 64, 0), (128, 64, 64, 4097)):
        with pytest.raises(capi.JJOError):
            capi.grouped_auto_kernel(*bad)
    i0 = ctypes.c_void_p(16)
    for kernel in (0, capi.ALGO_GEMV, capi.KERNEL_KSLICE, capi.KERNEL_KSLICE + 3):
        assert capi.lib().jjo_grouped_kernel_device(i0, i0, i0, 4, None, i0, 128, 64, 64, 0, kernel,
                                                    None) == capi.JJO_ERR_INVALID_ARG
    with pytest.raises(capi.JJOError):
        capi.mm_auto_kernel(96, 4, 1)
    a16 = ctypes.c_void_p(16)
    for kernel in (-1, 0, capi.ALGO_GEMV, 8, capi.KERNEL_KSLICE - 1, capi.KERNEL_KSLICE + 4):
        assert capi.lib().jjo_mm_kernel_device(a16, a16, a16, 128, 4, 40, 0, kernel, None) == capi.JJO_ERR_INVALID_ARG
    assert capi.lib().jjo_mm_kernel_device(ctypes.c_void_p(8), a16, a16, 128, 4, 40, 1, capi.ALGO_MFMA64,
                                           None) == capi.JJO_ERR_INVALID_ARG
