"""The forward on grids that leave the GPU idle: the keys of every tile split over groups of
waves, each with a reference point and sums of its own, merged through LDS at the end.

Up to three 64-row workgroups per CU may take it (256 CUs: B * H * ceil(S / 64) <= 768), each
band of the grid from its own length on: 32 or 64 rows x 4 groups over 128-key tiles up to one per CU
(at D = 128 and S >= 4096 up to two), 64 x 2 over 64-key tiles above that.  Lengths here sit at the
edges of the 32-row blocks, the 64- and 128-key tiles and the groups' shares of them (groups without a
visible key), head counts at the edges of the rule, beside the float64 oracle and the fp32 reference
with the forward suites' bars."""

import numpy as np
import pytest
import torch

from attention import _lib
from attention.backward.fused_backward import _forward
from attention.gqa.fused_gqa import fused_gqa_attention
from oracle import attention_oracle as orc
from test_exact_entries_gpu import fwd
from tests.gpu_util import check_forward, log
from tests.test_fwd_gpu import LSE_ABS

pytestmark = pytest.mark.gpu

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def make(B, H, Hkv, S, D, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((B, h, S, D), generator=g, device="cuda").to(DTYPES[dt]) for h in (H, Hkv, Hkv)]


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("S", [1, 31, 32, 33, 63, 65, 96, 97, 127, 128, 129, 161, 255, 257, 700])
def test_lengths(S, D):
    S += 384 if D == 128 else 128   # (shorter calls are not split; the edges repeat every 128 rows)
    for dt, H, Hkv in (("bf16", 3, 3), ("fp16", 4, 2)):   # one 64-row workgroup per CU at most
        q, k, v = make(1, H, Hkv, S, D, dt, seed=S + D)
        out = fused_gqa_attention(q, k, v)
        torch.cuda.synchronize()
        check_forward(out, q, k, v, rows_count=min(S, 24), label=f"key split S{S} D{D} {dt}")


# 64-row workgroups per CU: 1 (the four groups' last), a little over 1, 2, 3, and past the rule
@pytest.mark.parametrize("B,H,S", [(4, 16, 256), (2, 16, 500), (1, 257, 64), (2, 16, 1000), (3, 16, 1000), (1, 769, 64), (1, 8, 4096)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_grid_sizes(B, H, S, D):
    q, k, v = make(B, H, H, S, D, "bf16", seed=B + H + S + D)
    out, lse = _forward(q, k, v, 64, 64)
    torch.cuda.synchronize()
    check_forward(out, q, k, v, rows_count=8, label=f"key split B{B} H{H} S{S} D{D}")
    for h in (0, H - 1):
        want = orc.lse_log2(*(t[-1:, h:h + 1].double().cpu().numpy() for t in (q, k)))
        err = float(np.abs(lse[-1:, h:h + 1].cpu().numpy() - want).max())
        log(f"key split B{B} H{H} S{S} D{D} head {h} lse {err:.3e}")
        assert err <= LSE_ABS["bf16"]


@pytest.mark.parametrize("D", [32, 64, 128])
def test_large_scores_and_moving_reference(D):
    """Scores that grow along the keys (every group rescales on the way, by different amounts),
    and rows one key of a late group dominates."""
    q, k, v = make(1, 4, 4, 600, D, "fp16", seed=D)
    k = (k.float() * torch.linspace(0.1, 8.0, 600, device="cuda")[:, None]).half()
    out = fused_gqa_attention(q, k, v)
    torch.cuda.synchronize()
    check_forward(out, q, k, v, rows_count=24, label=f"key split growing scores D{D}")


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("lo,hi", [(0, 32), (32, 64), (64, 128)])
def test_keys_of_minus_infinite_score(D, lo, hi):
    """Keys lo..hi-1 score -inf in every row: rows past them are the attention over the others,
    whichever group holds them (rows with no other key are undefined)."""
    S = 400
    q, k, v = make(1, 2, 2, S, D, "bf16", seed=lo + D)
    q[..., 0] = 1.0
    k[:, :, lo:hi, 0] = float("-inf")
    out = fused_gqa_attention(q, k, v).float()
    s = (q.float() @ k.float().transpose(-1, -2).contiguous()) / D ** 0.5
    s.masked_fill_(torch.ones(S, S, device="cuda", dtype=torch.bool).triu(1), float("-inf"))
    want = torch.softmax(s, -1) @ v.float()
    rows = slice(hi if lo == 0 else 0, None)
    assert torch.isfinite(out[:, :, rows]).all()
    assert float((out - want)[:, :, rows].abs().max()) <= 2e-2


def test_nan_stays_in_its_row_block():
    """A NaN key makes the rows that see it NaN.  Of the rows before it only those of its own
    32-row block may be (a row's sum of P is taken beside row + 16's, by a product with zeros)."""
    q, k, v = make(1, 2, 2, 200, 64, "bf16", seed=9)
    clean = fused_gqa_attention(q, k, v)
    k[0, 0, 100, 3] = float("nan")
    out = fused_gqa_attention(q, k, v)
    torch.cuda.synchronize()
    assert torch.isnan(out[0, 0, 100:]).all()
    assert torch.equal(out[0, 0, :96], clean[0, 0, :96]) and torch.equal(out[0, 1], clean[0, 1])


# (heads, S, D, split): both sides of each band's shortest length
ROUTES = [(4, 64, 32, False), (4, 65, 64, True), (4, 320, 128, False), (4, 321, 128, True),
          (128, 128, 64, False), (64, 129, 32, True), (64, 511, 64, False), (64, 512, 64, True),
          (27, 704, 128, False), (27, 705, 128, True), (31, 1024, 128, False), (29, 1025, 128, True),
          (42, 768, 128, False), (38, 769, 128, True), (48, 640, 128, True),
          (64, 576, 32, False), (57, 577, 32, True), (60, 576, 128, False), (52, 641, 128, True), (41, 833, 128, False),
          (64, 640, 32, False), (45, 832, 64, False), (45, 833, 64, True), (48, 769, 128, True), (37, 1025, 128, False),
          (46, 1024, 128, False), (48, 1024, 128, True), (44, 1025, 64, False), (36, 1281, 64, True), (31, 1531, 128, False)]


@pytest.mark.parametrize("H,S,D,split", ROUTES)
def test_where_keys_are_split(H, S, D, split):
    """Calls that the split makes slower run the general kernels: bitwise the exact entry's, which
    never splits.  A split call differs from it by the rounding of P somewhere."""
    lib = _lib.load()
    q, k, v = make(1, H, H, S, D, "bf16", seed=H + S)
    o, lse = fwd(lib, q, k, v, 64, 64)
    o_x, lse_x = fwd(lib, q, k, v, 64, 64, 1)
    assert (torch.equal(o, o_x) and torch.equal(lse, lse_x)) is not split
