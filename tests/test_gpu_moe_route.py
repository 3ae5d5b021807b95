"""The FFN's batched routing (top-k, then one launch that sorts, quantizes and
permutes) writes the tables and bytes of the separate oracle stages."""
import numpy as np
import pytest

from jjjetson_ops_amd import capi
from oracle import c_oracle, oracle_np

pytestmark = pytest.mark.gpu


def to_dev(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).reshape(-1)).to(dev)


@pytest.mark.parametrize("T,H,E,top_k", [
    (17, 128, 1, 1),       # one expert
    (100, 2048, 64, 6),
    (33, 4224, 3, 2),      # a row in two column chunks
    (512, 128, 65, 8),     # 4096 routes, the most sorted in the quantizing launch
    (513, 128, 64, 8),     # one token more: the dispatch kernel's tables
    (300, 256, 1024, 8),   # the most experts
    (130, 128, 40, 32),    # the largest top_k
])
def test_ffn_routing_tables(T, H, E, top_k, dev):
    import torch
    print(f"[case] moe route T={T} H={H} E={E} k={top_k}", flush=True)
    I, R = 128, T * top_k
    rng = np.random.default_rng(T + H + E)
    x = rng.standard_normal((T, H)).astype(np.float32)
    x[0, :32] = 0.0
    lg = rng.standard_normal((T, E)).astype(np.float32)
    lg[1] = np.round(lg[1])  # ties, and zeros of both signs
    lg[2, 1:] = -np.inf
    lg[3, 0] = np.nan
    ids, w = oracle_np.moe_top_k(lg, top_k)
    off, src, dst = oracle_np.moe_dispatch(ids.reshape(-1), E)
    xq = c_oracle.quantize_q8_1(x, [H, T])
    xp = oracle_np.gather_q8_1(xq, src, T, top_k, H)

    zeros = torch.zeros(E * I * H // 32 * 18, dtype=torch.uint8, device=dev)
    ws = torch.full((capi.moe_ffn_workspace_bytes(T, H, I, E, top_k),), 0xA5, dtype=torch.uint8, device=dev)
    y = torch.empty(T * H, device=dev)
    capi.moe_ffn(to_dev(x, dev), to_dev(lg, dev), zeros, zeros, zeros, y, T, H, I, E, top_k, ws)
    # the workspace's leading tables, each 256-byte aligned
    sizes = [R * 4, R * 4, (E + 1) * 4, R * 4, R * 4, T * H // 128 * 144, R * H // 128 * 144]
    parts, o = [], 0
    for n in sizes:
        parts.append(ws[o:o + n].cpu().numpy())
        o += -(-n // 256) * 256
    np.testing.assert_allclose(parts[0].view(np.float32).reshape(T, top_k), w, rtol=2e-6, atol=1e-7, equal_nan=True)
    for got, want in zip(parts[1:5], (ids, off, src, dst)):
        assert np.array_equal(got.view(np.int32), want.reshape(-1))
    assert np.array_equal(parts[6], xp.reshape(-1))
