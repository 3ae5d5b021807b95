"""The K-sliced mid-batch GEMM through the AUTO entries, both weight layouts, against
the CPU oracle: each of its tile shapes (chosen by the output's size), row and token
tails, fewer 128-value stages than waves, uneven slices and 4-byte-aligned weights.
The layouts share every instruction after the operand expansion, so their results are
equal bit for bit."""
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


@pytest.mark.parametrize("K,N,M", [
    # 32 x 32 tiles, 8 waves: one stage for 8 waves; 3, 9 and 32 stages; tails
    (128, 1, 17), (128, 33, 31), (384, 95, 33), (1152, 160, 64), (4096, 64, 65), (1152, 257, 32),
    # 32 x 64, 8 waves
    (256, 2077, 129), (1280, 2080, 160),
    # 64 x 64, 8 waves
    (256, 2075, 389), (1152, 2080, 400),
    # 64 x 64, 4 waves
    (256, 4070, 500), (640, 4096, 512),
])
def test_kslice_shapes(K, N, M, dev):
    import torch
    print(f"[case] kslice K={K} N={N} M={M}", flush=True)
    rng = np.random.default_rng(K + N * M)
    w = c_oracle.quantize_q4_0((rng.standard_normal((N, K)) * 0.02).astype(np.float32))
    xq = c_oracle.quantize_q8_1(rng.standard_normal((M, K)).astype(np.float32), [K, M])
    exp = c_oracle.matmul(w, xq, K, N, M)
    xq_d = torch.from_numpy(xq).to(dev)
    w_pad = torch.zeros(w.size + 16, dtype=torch.uint8, device=dev)
    w_pad[4:4 + w.size] = torch.from_numpy(w).to(dev)
    ws = torch.empty(w.size, dtype=torch.uint8, device=dev)
    capi.q4_0_to_split(torch.from_numpy(w).to(dev), ws, N, K)
    got = []
    for run, wt in ((capi.mat_mul, torch.from_numpy(w).to(dev)), (capi.mat_mul, w_pad[4:4 + w.size]),
                    (capi.mat_mul_split, ws)):
        y = torch.full((M * N + 64,), float("nan"), dtype=torch.float32, device=dev)
        run(wt, xq_d, y, K, N, M)
        torch.cuda.synchronize()
        assert torch.isnan(y[M * N:]).all()  # nothing past the output
        got.append(y[:M * N].cpu().numpy().reshape(M, N))
        np.testing.assert_allclose(got[-1], exp, rtol=RTOL, atol=ATOL)
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
