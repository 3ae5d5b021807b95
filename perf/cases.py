"""The workloads this framework's speed is measured on, through its public entry points.

They are what an inference engine with Q4_0 weights has it do: the linear layers of
a decode step, of a small batch of sequences and of a prompt (each weight layout),
the mixture-of-experts FFN at decode and prompt sizes, and the quantization of a
weight matrix when a checkpoint is loaded.  Layer sizes are those of bench.py and of
the tests (hidden 2048 and 4096, intermediate 1408, 11008 and 14336).

A decode-sized case keeps several copies of its weights and goes on to the next copy
at each pass, as a model goes on to its next layer: over 512 MB together, so that the
256 MB Infinity Cache does not serve them.
"""
import math

import torch

from jjjetson_ops_amd import capi
from jjjetson_ops_amd import weights as q4_weights

ROTATE_BYTES = 512 << 20  # weights of one state that is bound by reading them
SMALL_TOKENS = 64  # up to this many tokens reading the weights is what a linear layer costs


def _linear(name, tokens, k, n, split):
    return {"name": name, "kind": "linear", "tokens": tokens, "k": k, "n": n, "split": split}


def _moe(name, tokens, experts, top_k, hidden, inter, split):
    return {"name": name, "kind": "moe", "tokens": tokens, "experts": experts, "top_k": top_k, "hidden": hidden,
            "inter": inter, "split": split}


def listed():
    return [
        # One token through an attention projection: the smallest call, launch-bound.
        _linear("decode_k4096_n4096_split", 1, 4096, 4096, True),
        # One token through the MLP's up projection (the repository's headline step).
        _linear("decode_k4096_n11008_split", 1, 4096, 11008, True),
        # One token through the MLP's down projection, weights as the checkpoint holds them.
        _linear("decode_k11008_n4096_block", 1, 11008, 4096, False),
        # Seven sequences decoded together (a ragged batch).
        _linear("batch7_k4096_n14336_split", 7, 4096, 14336, True),
        # Twenty-four sequences decoded together, long rows.
        _linear("batch24_k11008_n4096_block", 24, 11008, 4096, False),
        # A short prompt.
        _linear("prompt100_k4096_n14336_block", 100, 4096, 14336, False),
        # A prompt of an odd length through a down projection.
        _linear("prompt777_k11008_n4096_split", 777, 11008, 4096, True),
        # A long prompt (or one chunk of it) through an up projection: the largest linear.
        _linear("prompt2048_k4096_n14336_split", 2048, 4096, 14336, True),
        # Four tokens through a mixture-of-experts FFN: decode, all experts' weights read.
        _moe("moe4_e8_h4096_i14336_split", 4, 8, 2, 4096, 14336, True),
        # A batch of prompt tokens through many small experts, a few routes for each.
        _moe("moe100_e64_h2048_i1408_split", 100, 64, 8, 2048, 1408, True),
        # A prompt through the mixture-of-experts FFN: the largest case.
        _moe("moe512_e8_h4096_i14336_block", 512, 8, 2, 4096, 14336, False),
        # Loading a checkpoint: one fp32 projection to Q4_0.
        {"name": "load_14336x4096", "kind": "load", "rows": 14336, "cols": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "moe", "moe", "load"))
    split = rng.random() < 0.5
    if kind == "linear":
        k = 128 * _log(rng, 8, 112)
        n = _log(rng, 1024, 14336)
        most = min(2048, 2048 * 4096 * 14336 // (k * n))
        tokens = 1 if rng.random() < 0.25 else _log(rng, 1, most)
        return {"kind": kind, "tokens": tokens, "k": k, "n": n, "split": split}
    if kind == "moe":
        experts, top_k = rng.choice(((8, 2), (16, 2), (16, 4), (64, 8)))
        hidden = 128 * _log(rng, 8, 32)
        inter = 128 * _log(rng, 8, min(112, 8 * 32 * 112 // (experts * hidden // 128)))
        most = min(512, 1024 * 4096 * 14336 // (top_k * hidden * inter))
        return {"kind": kind, "tokens": _log(rng, 1, most), "experts": experts, "top_k": top_k, "hidden": hidden,
                "inter": inter, "split": split}
    return {"kind": kind, "rows": _log(rng, 256, 14336), "cols": 32 * _log(rng, 16, 128)}


# ------------------------------------------------------------------------- inputs
def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + what)


def _weights_f32(rows, cols, seed, what):
    return torch.randn(rows, cols, generator=_gen(seed, what), device="cuda") * 0.02


def _pack_q4_0(wf):
    """Q4_0 bytes [rows * cols/32 * 18] of fp32 weights: d = (value of largest magnitude) / -8
    as fp16, nibble = clamp(int(v/d + 8.5), 0, 15), element j low and j+16 high in byte j."""
    g = wf.reshape(-1, 32)
    mx = torch.gather(g, 1, g.abs().argmax(dim=1, keepdim=True))
    d = mx / -8.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    nib = torch.clamp(torch.trunc(g * inv + 8.5), 0, 15).to(torch.uint8)
    out = torch.empty((g.shape[0], 18), dtype=torch.uint8, device=wf.device)
    out[:, 0:2] = d.to(torch.float16).view(torch.uint8)
    out[:, 2:18] = nib[:, :16] | (nib[:, 16:] << 4)
    return out.reshape(-1)


def _block_weights(rows, cols, seed, what):
    return _pack_q4_0(_weights_f32(rows, cols, seed, what))


def _experts(experts, rows, cols, seed, what):
    return torch.cat([_block_weights(rows, cols, seed, what + e) for e in range(experts)])


def _laid_out(w, rows, cols, split):
    """The weights in the layout the case calls for, repacked once as at load time."""
    if not split:
        return w
    out = torch.empty_like(w)
    capi.q4_0_to_split(w, out, rows, cols)
    return out


def _activation(tokens, k, seed):
    """Hidden states: N(0, 1) with one channel in a thousand twenty times larger."""
    g = _gen(seed, 1)
    x = torch.randn(tokens, k, generator=g, device="cuda")
    x[:, torch.randperm(k, generator=g, device="cuda")[:max(1, k // 1000)]] *= 20.0
    return x


def _logits(case, seed):
    return torch.randn(case["tokens"], case["experts"], generator=_gen(seed, 2), device="cuda")


def prepare(case, seed):
    if case["kind"] == "load":
        rows, cols = case["rows"], case["cols"]
        copies = max(1, min(16, math.ceil(ROTATE_BYTES / (4 * rows * cols))))
        w = _weights_f32(rows, cols, seed, 3)
        return {"case": case, "w": [w] + [w.clone() for _ in range(copies - 1)], "at": 0,
                "out": torch.empty(rows * cols // 32 * 18, dtype=torch.uint8, device="cuda")}
    if case["kind"] == "linear":
        t, k, n = case["tokens"], case["k"], case["n"]
        w = _laid_out(_block_weights(n, k, seed, 3), n, k, case["split"])
        copies = max(1, math.ceil(ROTATE_BYTES / w.numel())) if t <= SMALL_TOKENS else 1
        return {"case": case, "w": [w] + [w.clone() for _ in range(copies - 1)], "at": 0,
                "x": _activation(t, k, seed),
                "ws": torch.empty(capi.linear_q4_0_workspace_bytes(k, t), dtype=torch.uint8, device="cuda"),
                "y": torch.empty(t, n, dtype=torch.float32, device="cuda")}
    t, e, top_k, h, i = (case[v] for v in ("tokens", "experts", "top_k", "hidden", "inter"))
    mats = [_laid_out(_experts(e, rows, cols, seed, what), e * rows, cols, case["split"])
            for rows, cols, what in ((i, h, 100), (i, h, 300), (h, i, 500))]
    copies = max(1, math.ceil(ROTATE_BYTES / sum(m.numel() for m in mats)))
    return {"case": case, "w": [mats] + [[m.clone() for m in mats] for _ in range(copies - 1)], "at": 0,
            "x": _activation(t, h, seed), "logits": _logits(case, seed),
            "ws": torch.empty(capi.moe_ffn_workspace_bytes(t, h, i, e, top_k), dtype=torch.uint8, device="cuda"),
            "y": torch.empty(t, h, dtype=torch.float32, device="cuda")}


# --------------------------------------------------------------------------- pass
def run(state):
    case = state["case"]
    w = state["w"][state["at"]]
    state["at"] = (state["at"] + 1) % len(state["w"])
    if case["kind"] == "load":
        q4_weights.quantize_q4_0_device(w, state["out"], case["rows"], case["cols"])
        return state["out"]
    if case["kind"] == "linear":
        linear = capi.linear_q4_0_split if case["split"] else capi.linear_q4_0
        linear(state["x"], w, state["y"], case["k"], case["n"], case["tokens"], ws=state["ws"])
        return state["y"]
    capi.moe_ffn(state["x"], state["logits"], w[0], w[1], w[2], state["y"], case["tokens"], case["hidden"],
                 case["inter"], case["experts"], case["top_k"], state["ws"], split=case["split"])
    return state["y"]


# --------------------------------------------------------------------- what it needs
def work(case):
    if case["kind"] == "load":
        values = case["rows"] * case["cols"]
        return {"bytes": 4 * values + values // 32 * 18, "flops": 0}
    if case["kind"] == "linear":
        t, k, n = case["tokens"], case["k"], case["n"]
        return {"bytes": n * k // 32 * 18 + 4 * t * k + 4 * t * n, "flops": 2 * t * k * n}
    t, e, top_k, h, i = (case[v] for v in ("tokens", "experts", "top_k", "hidden", "inter"))
    active = e * (1.0 - (1.0 - top_k / e) ** t)  # experts with a route, for a balanced router
    return {"bytes": int(active * 3 * h * i // 32 * 18) + 4 * t * (2 * h + e), "flops": 6 * t * top_k * h * i}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "linear":
        # fp32 sums over up to 448 blocks: 0.8e-7 to 4.5e-7 from the exact result, measured.
        return {"rel": 4e-6, "max": 2e-4}
    # The intermediate activation is quantized to 8 bits again: a value next to a
    # rounding boundary may land on either side of it.  1.4e-4 to 3.5e-4 from the result
    # whose intermediate is computed in 64 bits, measured.
    return {"rel": 1.2e-3, "max": 2e-2}


# -------------------------------------------------------------------------- in 64 bits
def _unpack_q4_0(w, rows, cols):
    """Unsigned nibbles [rows, cols/32, 32] and scales [rows, cols/32] in fp64."""
    b = w.reshape(rows, cols // 32, 18)
    d = b[:, :, 0:2].contiguous().view(torch.float16)[..., 0].double()
    return torch.cat([b[:, :, 2:] & 15, b[:, :, 2:] >> 4], dim=2).double(), d


def _quantize_q8_1(x):
    """The Q8_1 values of fp32 rows: q [T, K/32, 32], d and s [T, K/32] (both fp16 in the
    format), in fp64.  The format's own rounding steps are in fp32, its sum's order fixed."""
    g = x.float().reshape(x.shape[0], -1, 8, 4)
    amax = g.abs().amax(dim=(2, 3))
    inv = torch.where(amax > 0, (127.0 / amax.double()).float(), torch.zeros_like(amax))
    v = (g * inv[..., None, None]).double()
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    d = (1.0 / inv.double()).float().half().double()
    s = ((g[..., 0] + g[..., 1]) + g[..., 2]) + g[..., 3]
    s = s[..., :4] + s[..., 4:]
    s = s[..., :2] + s[..., 2:]
    s = (s[..., 0] + s[..., 1]).half().double()
    return q.reshape(*q.shape[:2], 32), d, s


def _matmul(x, w, rows, cols):
    """sum over blocks of d_w * (d_x * sum(nibble * q) - 8 * s_x), for rows x of fp32."""
    nib, dw = _unpack_q4_0(w, rows, cols)
    q, dx, sx = _quantize_q8_1(x)
    t = x.shape[0]
    a = (q * dx[..., None]).reshape(t, cols)
    y = a @ (nib * dw[..., None]).reshape(rows, cols).t().contiguous()
    return y - 8.0 * (sx @ dw.t().contiguous())


def exact(case, seed):
    if case["kind"] == "load":
        return None
    if case["kind"] == "linear":
        t, k, n = case["tokens"], case["k"], case["n"]
        return _matmul(_activation(t, k, seed), _block_weights(n, k, seed, 3), n, k)
    t, e, top_k, h, i = (case[v] for v in ("tokens", "experts", "top_k", "hidden", "inter"))
    x = _activation(t, h, seed)
    top, ids = torch.topk(_logits(case, seed).double(), top_k, dim=1)
    share = torch.softmax(top, dim=1)
    y = torch.zeros(t, h, dtype=torch.float64, device="cuda")
    for expert in range(e):
        tok, slot = torch.nonzero(ids == expert, as_tuple=True)
        if tok.numel() == 0:
            continue
        gate = _matmul(x[tok], _block_weights(i, h, seed, 100 + expert), i, h)
        up = _matmul(x[tok], _block_weights(i, h, seed, 300 + expert), i, h)
        mid = (gate * torch.sigmoid(gate) * up).float()
        y.index_add_(0, tok, share[tok, slot][:, None] * _matmul(mid, _block_weights(h, i, seed, 500 + expert), h, i))
    return y
