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


def test_invalid_calls_are_refused():
    with pytest.raises(capi.JJOError):
        capi.mm_auto_kernel(96, 4, 1)
    a16 = ctypes.c_void_p(16)
    for kernel in (-1, 0, capi.ALGO_GEMV, 8, capi.KERNEL_KSLICE - 1, capi.KERNEL_KSLICE + 4):
        assert capi.lib().jjo_mm_kernel_device(a16, a16, a16, 128, 4, 40, 0, kernel, None) == capi.JJO_ERR_INVALID_ARG
    assert capi.lib().jjo_mm_kernel_device(ctypes.c_void_p(8), a16, a16, 128, 4, 40, 1, capi.ALGO_MFMA64,
                                           None) == capi.JJO_ERR_INVALID_ARG
