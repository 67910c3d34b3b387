"""The calls this library is timed on: what its users run, through its public entry points.

Three kinds of call: the MHA forward (fused_attention), the GQA/MQA forward
(fused_gqa_attention) and a training step (forward, then the backward through autograd,
fused_attention_autograd or fused_gqa_attention_autograd).  Sizes are those of the benchmark
scripts, the correctness suites and bench.py, plus ragged lengths; inputs are N(0, 1), as in
all of those (the long MQA forward scales them by 0.5).
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "fused-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
TILES = ((64, 64), (64, 128), (128, 64), (128, 128))


def _case(call, dtype, B, H, H_kv, S, D, tile_m=64, tile_n=64, sigma=1.0, name=None):
    case = dict(call=call, dtype=dtype, B=B, H=H, H_kv=H_kv, S=S, D=D, tile_m=tile_m, tile_n=tile_n, sigma=sigma)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the command-line tools' plumbing workload: one short call, bound by latency
        _case("fwd", "fp16", 1, 4, 4, 256, 64, name="fwd_B1_H4_S256_D64"),
        # a training step on short sequences (the benchmark sweep's small end, default tiles)
        _case("train", "fp16", 2, 8, 8, 512, 64, name="train_B2_H8_S512_D64"),
        # the middle of the benchmark sweep: few heads, medium length
        _case("fwd", "fp16", 2, 8, 8, 2048, 128, name="fwd_B2_H8_S2048_D128"),
        # a training step whose length is no multiple of any tile, with an odd head count
        _case("train", "bf16", 3, 5, 5, 1000, 128, name="train_B3_H5_S1000_D128"),
        # one prompt of odd length through grouped heads: prefill of a single request
        _case("fwd", "bf16", 1, 32, 8, 1531, 128, name="fwd_gqa_B1_H32_S1531_D128"),
        # the correctness suites' largest batch of short sequences, at their largest tile
        _case("fwd", "bf16", 16, 32, 32, 512, 32, 128, 128, name="fwd_B16_H32_S512_D32"),
        # the headline workload: forward, and forward + backward, at the benchmark's tile
        _case("fwd", "bf16", 4, 32, 32, 4096, 128, 128, 64, name="fwd_B4_H32_S4096_D128"),
        _case("train", "bf16", 4, 32, 32, 4096, 128, 128, 64, name="train_B4_H32_S4096_D128"),
        # grouped heads at long context
        _case("fwd", "bf16", 2, 32, 8, 8192, 128, name="fwd_gqa_B2_H32_S8192_D128"),
        # one K/V head at the longest context in use
        _case("fwd", "fp16", 1, 32, 1, 16384, 64, sigma=0.5, name="fwd_mqa_B1_H32_S16384_D64"),
        # a training step at the smaller head size
        _case("train", "fp16", 2, 16, 16, 4096, 64, name="train_B2_H16_S4096_D64"),
        # a training step through grouped heads
        _case("train", "bf16", 2, 32, 8, 4096, 128, name="train_gqa_B2_H32_S4096_D128"),
    ]


def draw(rng):
    """One more call: forward or training step, MHA or grouped, S from 128 to 16384 of any
    residue, every head size, type and tile, and no more work than the largest listed case."""
    limit = max(work(c)["flops"] for c in listed())
    while True:
        call = rng.choice(("fwd", "train"))
        H_kv = rng.choice((1, 2, 4, 5, 8, 16, 32))
        group = rng.choice((1, 1, 1, 2, 4, 8))
        if H_kv * group > 32:
            continue
        S = int(round(math.exp(rng.uniform(math.log(128), math.log(16384)))))
        if rng.random() < 0.5:
            S = max(128, S // 64 * 64)
        tile_m, tile_n = rng.choice(TILES)
        case = _case(call, rng.choice(("fp16", "bf16")), rng.choice((1, 2, 3, 4, 8, 16)), H_kv * group, H_kv, S,
                     rng.choice((32, 64, 128)), tile_m, tile_n)
        if work(case)["flops"] <= limit and case["B"] * case["H"] * S * case["D"] <= 4 * 32 * 4096 * 128:
            return case


def _inputs(case, seed):
    """Q, K, V (and dO for a training step) on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, H, H_kv, S, D = (case[k] for k in ("B", "H", "H_kv", "S", "D"))
    heads = [H, H_kv, H_kv] + ([H] if case["call"] == "train" else [])
    scales = [case["sigma"]] * 3 + [1.0]
    return [(torch.randn((B, h, S, D), generator=g, device="cuda") * s).to(dt) for h, s in zip(heads, scales)]


def prepare(case, seed):
    from attention.backward.fused_backward import fused_attention_autograd
    from attention.fused.fused import fused_attention
    from attention.gqa.fused_gqa import fused_gqa_attention, fused_gqa_attention_autograd
    mha = case["H"] == case["H_kv"]
    state = dict(call=case["call"], tiles=(case["tile_m"], case["tile_n"]), inputs=_inputs(case, seed))
    if case["call"] == "train":
        for t in state["inputs"][:3]:
            t.requires_grad_(True)
        state["fn"] = fused_attention_autograd if mha else fused_gqa_attention_autograd
    else:
        state["fn"] = fused_attention if mha else fused_gqa_attention
    return state


def run(state):
    if state["call"] == "fwd":
        return state["fn"](*state["inputs"], *state["tiles"])
    q, k, v, do = state["inputs"]
    for t in (q, k, v):
        t.grad = None
    o = state["fn"](q, k, v, *state["tiles"])
    o.backward(do)
    return o.detach(), q.grad, k.grad, v.grad


def work(case):
    """Causal FLOPs (2 B H S^2 D forward, 2.5x that for the backward, as the benchmark scripts
    count them); Q, K, V (dO) read once and O (dQ, dK, dV) written once."""
    B, H, H_kv, S, D = (case[k] for k in ("B", "H", "H_kv", "S", "D"))
    train = case["call"] == "train"
    q_rows, kv_rows = B * H * S, B * H_kv * S
    return {"bytes": 2 * D * ((4 if train else 2) * q_rows + (4 if train else 2) * kv_rows),
            "flops": (3.5 if train else 1.0) * 2.0 * B * H * float(S) * S * D}


def tolerance(case):
    """Rounding of the 16-bit operands P and dS, of O and of the outputs themselves (2^-9 of a
    bf16 value, 2^-12 of an fp16 one, each): about four times the distance from the float64
    formula, 2.0e-3 to 2.6e-3 in bf16 and 2.4e-4 to 3.2e-4 in fp16."""
    return {"rel": 1e-2, "max": 1e-1} if case["dtype"] == "bf16" else {"rel": 1.25e-3, "max": 2e-2}


def exact(case, seed):
    """The causal formula and its closed-form gradients in float64, a head at a time and in
    blocks of query rows."""
    x = [t.double() for t in _inputs(case, seed)]
    q, k, v = x[:3]
    train = case["call"] == "train"
    B, H, S, D = q.shape
    group = H // k.shape[1]
    scale = 1.0 / math.sqrt(D)
    rows = 2048
    o = torch.empty_like(q)
    if train:
        do = x[3]
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for b in range(B):
        for h in range(H):
            hk = h // group
            for r0 in range(0, S, rows):
                r1 = min(S, r0 + rows)
                kk, vv = k[b, hk, :r1], v[b, hk, :r1]
                s = torch.mm(q[b, h, r0:r1], kk.t()).mul_(scale)
                keys = torch.arange(r1, device=s.device)
                s.masked_fill_(keys[None, :] > keys[r0:, None], float("-inf"))
                p = torch.softmax(s, dim=-1)
                o[b, h, r0:r1] = torch.mm(p, vv)
                if train:
                    g = do[b, h, r0:r1]
                    delta = (g * o[b, h, r0:r1]).sum(dim=-1, keepdim=True)
                    dv[b, hk, :r1] += torch.mm(p.t(), g)
                    ds = p.mul_(torch.mm(g, vv.t()).sub_(delta)).mul_(scale)
                    dq[b, h, r0:r1] = torch.mm(ds, kk)
                    dk[b, hk, :r1] += torch.mm(ds.t(), q[b, h, r0:r1])
    return (o, dq, dk, dv) if train else o
