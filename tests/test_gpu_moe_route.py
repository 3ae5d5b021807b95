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


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("T,H,I,E,top_k", [
    (2, 256, 5120, 4, 2),      # mean one, two routes at most; a workgroup per route; one and two K slices
    (4, 4096, 12416, 8, 2),    # mean one: four routes of one expert; four K slices
    (5, 2176, 128, 4, 2),      # mean above two
    (8, 4224, 128, 8, 2),      # mean two: chunks of two
    (16, 256, 128, 64, 2),     # mean one, sixteen routes on one expert
])
def test_ffn_decode_chunks(T, H, I, E, top_k, split, dev):
    """A token's row does not depend on how its expert's routes are chunked: it is that of
    the call with the token alone (one route per expert, at more routes an instance
    that sums a wave's lanes in another order).  Bound: the fp32 sums differ by about 1e-6, which moves a
    SwiGLU value across a Q8_1 step in at most a few of a row's elements; a step (a group's
    largest |mid| / 127, about 4/127 of the rms) times the largest weight (0.064, against
    an rms of 0.028) is 2e-3 of a row's largest output at I = 128, less for longer sums;
    two such steps are allowed."""
    import torch
    print(f"[case] moe chunks T={T} H={H} I={I} E={E} k={top_k} split={split}", flush=True)
    rng = np.random.default_rng(T + I)
    lg = rng.standard_normal((T, E)).astype(np.float32)
    lg[:, 1] += 8.0  # every token takes expert 1
    x = to_dev(rng.standard_normal((T, H)).astype(np.float32), dev)
    lg = to_dev(lg, dev)
    ws = []
    for rows, cols in ((E * I, H), (E * I, H), (E * H, I)):
        w = torch.empty((rows * cols // 32, 18), dtype=torch.uint8, device=dev)
        w[:, 2:] = to_dev(rng.integers(0, 256, (rows * cols // 32, 16), dtype=np.uint8), dev).view(-1, 16)
        d = (rng.random((rows * cols // 32, 1)) * 0.004 + 0.004).astype(np.float16)
        w[:, :2] = to_dev(d, dev).view(torch.uint8).view(-1, 2)
        w = w.reshape(-1)
        if split:
            s = torch.empty_like(w)
            capi.q4_0_to_split(w, s, rows, cols)
            w = s
        ws.append(w)

    def ffn(i, n):
        work = torch.empty(capi.moe_ffn_workspace_bytes(n, H, I, E, top_k), dtype=torch.uint8, device=dev)
        y = torch.empty(n * H, device=dev)
        capi.moe_ffn(x[i * H:(i + n) * H], lg[i * E:(i + n) * E], *ws, y, n, H, I, E, top_k, work, split=split)
        return y.view(n, H)

    got = ffn(0, T)
    assert torch.isfinite(got).all()
    for i in range(T):
        one = ffn(i, 1)[0]
        assert (got[i] - one).abs().max() <= 4e-3 * one.abs().max()
