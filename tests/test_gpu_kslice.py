"""The K-sliced mid-batch GEMM, both weight layouts, against the CPU oracle: each of its
tile forms at row and token tails, fewer 128-value stages than waves and uneven slices,
asked for by name; the form the entries choose, with 4-byte-aligned weights; the grouped
form.  The layouts share every instruction after the operand expansion, so their results
are equal bit for bit."""
if __name__ == "__main__":  # `python tests/<file>.py`, as the reference runs its tests
    import sys as _sys

    import pytest as _pytest
    _sys.exit(_pytest.main([__file__, "-q"]))
import numpy as np
import pytest

from jjjetson_ops_amd import capi
from oracle import c_oracle

pytestmark = pytest.mark.gpu
RTOL, ATOL = 1e-3, 1e-4  # the repository's bar against the oracle's fp64 sums


def _case(K, N, M, dev):
    """(expected, block_q4_0 weights, the same in the split layout, activation blocks)"""
    import torch
    rng = np.random.default_rng(K + N * M)
    w = c_oracle.quantize_q4_0((rng.standard_normal((N, K)) * 0.02).astype(np.float32))
    xq = c_oracle.quantize_q8_1(rng.standard_normal((M, K)).astype(np.float32), [K, M])
    w_d = torch.from_numpy(w).to(dev)
    ws = torch.empty(w.size, dtype=torch.uint8, device=dev)
    capi.q4_0_to_split(w_d, ws, N, K)
    return c_oracle.matmul(w, xq, K, N, M), w_d, ws, torch.from_numpy(xq).to(dev)


def _run(fn, M, N, dev):
    """fn(y); the result, after a look at what lies past it."""
    import torch
    y = torch.full((M * N + 64,), float("nan"), dtype=torch.float32, device=dev)
    fn(y)
    torch.cuda.synchronize()
    assert torch.isnan(y[M * N:]).all()
    return y[:M * N].cpu().numpy().reshape(M, N)


@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("K,N,M", [
    (128, 1, 1), (128, 33, 65),      # one stage for four or eight waves; one row or token in a tile
    (384, 95, 31), (640, 130, 97),   # 3 and 5 stages; tails of 31 and 2 rows, 31 and 33 tokens
    (1152, 161, 64), (1280, 64, 33), # 9 and 10 stages; N % 4 == 1; full tiles
    (2176, 127, 130), (4096, 66, 32),
])
def test_kslice_forms(K, N, M, form, dev):
    """Forms 0..3: 32 x 32, 32 x 64 and 64 x 64 tiles of eight waves, 64 x 64 of four."""
    print(f"[case] kslice form={form} K={K} N={N} M={M}", flush=True)
    exp, w, ws, xq = _case(K, N, M, dev)
    kernel = capi.KERNEL_KSLICE + form
    got = [_run(lambda y: capi.mm_kernel(wt, xq, y, K, N, M, kernel, split), M, N, dev)
           for wt, split in ((w, False), (ws, True))]
    np.testing.assert_allclose(got[0], exp, rtol=RTOL, atol=ATOL)
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("K,N,M,form", [
    (128, 33, 31, 0), (384, 95, 33, 0), (4096, 64, 65, 0), (2944, 4106, 33, 1), (768, 6325, 97, 2),
    (640, 3591, 199, 3), (640, 8095, 98, 3),
])
def test_kslice_chosen(K, N, M, form, dev):
    """Shapes that the entries give to each form, with weights at the least alignment."""
    import torch
    print(f"[case] kslice K={K} N={N} M={M}", flush=True)
    for split in (False, True):
        assert capi.mm_auto_kernel(K, N, M, split) == capi.KERNEL_KSLICE + form
    exp, w, ws, xq = _case(K, N, M, dev)
    w_pad = torch.zeros(w.numel() + 16, dtype=torch.uint8, device=dev)
    w_pad[4:4 + w.numel()] = w
    got = [_run(lambda y: run(wt, xq, y, K, N, M), M, N, dev)
           for run, wt in ((capi.mat_mul, w), (capi.mat_mul, w_pad[4:4 + w.numel()]), (capi.mat_mul_split, ws))]
    np.testing.assert_allclose(got[0], exp, rtol=RTOL, atol=ATOL)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


def test_kslice_special_scales(dev):
    """A token with an all-zero group (d = +inf, its products NaN) makes its whole output
    row NaN and no other; a zero weight scale gives zeros from that block."""
    import torch
    K, N, M = 512, 70, 40
    rng = np.random.default_rng(3)
    wf = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    wf[5, 32:64] = 0.0
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[7, 96:128] = 0.0
    w = c_oracle.quantize_q4_0(wf)
    xq = c_oracle.quantize_q8_1(x, [K, M])
    exp = c_oracle.matmul(w, xq, K, N, M)
    y = torch.empty(M * N, dtype=torch.float32, device=dev)
    capi.mat_mul(torch.from_numpy(w).to(dev), torch.from_numpy(xq).to(dev), y, K, N, M)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(M, N)
    assert np.isnan(got[7]).all() and np.isnan(exp[7]).all()
    rest = [m for m in range(M) if m != 7]
    np.testing.assert_allclose(got[rest], exp[rest], rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("counts,N,K", [
    # full tiles, tails, empty and single-route experts; with two column tiles, tails that run
    # the one-column loop
    ([32, 0, 1, 33, 31, 5, 64], 96, 384), ([20] * 3, 65, 128), ([2] * 30 + [70], 257, 1152),
    ([64, 65, 1, 0, 96, 97, 32, 33], 130, 640), ([128, 31], 64, 256),
])
def test_kslice_grouped(counts, N, K, dev):
    """The grouped form with one and two column tiles at its tile edges, scattered outputs,
    both layouts (equal bits in all four), and what the entry chooses for the shape."""
    import torch
    E, R = len(counts), sum(counts)
    assert R > 48  # below, the grouped entry is a GEMV
    print(f"[case] kslice grouped E={E} R={R} N={N} K={K}", flush=True)
    rng = np.random.default_rng(R + N)
    ws = [c_oracle.quantize_q4_0((rng.standard_normal((N, K)) * 0.02).astype(np.float32)) for _ in counts]
    xq = c_oracle.quantize_q8_1(rng.standard_normal((R, K)).astype(np.float32), [K, R])
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    dst = rng.permutation(R).astype(np.int32)
    exp = np.empty((R, N), np.float32)
    blocks = xq.reshape(K // 128, R, 144)
    for e, n in enumerate(counts):
        if n:
            rows = np.ascontiguousarray(blocks[:, off[e]:off[e + 1]]).reshape(-1)
            exp[dst[off[e]:off[e + 1]]] = c_oracle.matmul(ws[e], rows, K, N, n)
    w = torch.from_numpy(np.concatenate(ws)).to(dev)
    w_split = torch.empty_like(w)
    capi.q4_0_to_split(w, w_split, E * N, K)
    xq, off, dst = (torch.from_numpy(v).to(dev) for v in (xq, off, dst))
    got = []
    for split in (False, True):
        wt = w_split if split else w
        for cols in (1, 2):
            got.append(_run(lambda y: capi.grouped_kernel(wt, xq, off, y, K, N, R, capi.KERNEL_KSLICE + cols,
                                                          route_dst=dst, split=split), R, N, dev))
            np.testing.assert_allclose(got[-1], exp, rtol=RTOL, atol=ATOL)
        chosen = _run(lambda y: capi.grouped_mat_mul(wt, xq, off, y, K, N, R, route_dst=dst, split=split), R, N, dev)
        np.testing.assert_allclose(chosen, exp, rtol=RTOL, atol=ATOL)
    assert all(np.array_equal(got[0], g) for g in got[1:])
