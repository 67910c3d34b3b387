"""The backward of small grids (one launch for dQ and dK/dV, two waves to every 32 rows or
keys), and the two-kernel backward and unsplit forward just past them.

The one launch takes up to three 64-row workgroups per CU (256 CUs: B * H * ceil(S / 64) <= 768),
one at D = 128, fewer for short sequences.
Lengths sit at the edges of the 32-row halves and the 64-row tiles; head counts put the grid just
inside or just past the rule, so ragged lengths meet both kernels.  Bars of the backward suites
(tests/test_gqa_bwd_gpu.py: check)."""

import ctypes
import math

import pytest
import torch

from attention import _lib
from attention.backward.fused_backward import _forward
from tests.gpu_util import log
from tests.test_gqa_bwd_gpu import check, make
from test_exact_entries_gpu import bwd

pytestmark = pytest.mark.gpu

# Over hundreds of heads |dQ| reaches 4 to 8, where half a bf16 ulp is 1.6e-2 and the rounding of
# dS as much again: past dQ's flat bar of 2e-2 (2.5e-2 met), whichever kernel computes it.  fp16 is
# 8 times finer.
MANY_HEADS = torch.float16
LENGTHS = [1, 31, 33, 64, 65, 95, 97, 128, 129, 300]


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("S", LENGTHS)
def test_small_lengths(S, D):
    for dt, H, Hkv in ((torch.bfloat16, 2, 2), (torch.float16, 4, 1)):
        q, k, v, do = make(2, H, Hkv, S, D, dt, seed=S + D)
        check(q, k, v, do, (64, 64), f"small bwd S{S} D{D} H{H}/{Hkv} {dt}", oracle=True)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("S", LENGTHS)
def test_ragged_lengths_past_the_rule(S, D):
    tiles = (S + 63) // 64
    H = (768 // tiles + 1 + 3) // 4 * 4
    for Hkv in (H, H // 4):
        q, k, v, do = make(1, H, Hkv, S, D, MANY_HEADS, seed=S + D + Hkv)
        check(q, k, v, do, (64, 64), f"full grid S{S} D{D} H{H}/{Hkv}")


@pytest.mark.parametrize("B,H,Hkv,S,D", [(4, 64, 64, 50, 128), (4, 16, 4, 256, 128), (1, 256, 256, 64, 128),
                                         (3, 16, 16, 1000, 64), (2, 12, 6, 2000, 64), (4, 48, 48, 250, 32)])
def test_edges_of_the_rule(B, H, Hkv, S, D):
    q, k, v, do = make(B, H, Hkv, S, D, MANY_HEADS, seed=B + H + S)
    check(q, k, v, do, (128, 64), f"small bwd edge B{B} H{H}/{Hkv} S{S} D{D}")


# (heads, K/V heads, S, D, one launch): both sides of each bound
ROUTES = [(128, 128, 64, 128, True), (129, 129, 64, 128, False), (128, 128, 128, 128, True), (129, 129, 100, 128, False),
          (218, 109, 64, 128, True), (220, 110, 64, 128, False), (256, 64, 64, 128, True),
          (768, 768, 48, 64, True), (769, 769, 48, 64, False), (384, 384, 64, 64, True), (385, 385, 64, 64, False),
          (658, 329, 64, 64, True), (660, 330, 64, 64, False), (768, 192, 64, 64, True),
          (320, 320, 100, 64, True), (321, 321, 100, 64, False), (224, 224, 128, 64, True), (225, 225, 128, 64, False),
          (384, 192, 128, 64, True), (144, 144, 256, 64, True), (145, 145, 256, 64, False), (192, 96, 256, 64, True),
          (64, 64, 640, 64, True), (65, 65, 640, 64, False), (65, 65, 704, 64, False), (64, 64, 768, 64, True),
          (63, 63, 768, 64, False), (768, 768, 64, 32, True), (106, 106, 384, 32, True), (107, 107, 384, 32, False),
          (128, 64, 384, 32, True), (109, 109, 448, 32, True), (110, 110, 448, 32, False)]


@pytest.mark.parametrize("H,Hkv,S,D,one", ROUTES)
def test_where_the_backward_is_one_launch(H, Hkv, S, D, one):
    """Calls that the one launch makes slower run the two kernels: bitwise the exact entry's, which always
    does.  A call of one launch differs from it by the fp32 summation order somewhere."""
    lib = _lib.load()
    q, k, v, do = make(1, H, Hkv, S, D, MANY_HEADS, seed=H + S)
    o, lse = _forward(q, k, v, 64, 64)
    assert lib.fa_bwd_dkdv_split(1, H, Hkv, S, D) == 1
    got = bwd(lib, q, k, v, o, do, lse, 64, 64)
    want = bwd(lib, q, k, v, o, do, lse, 64, 64, nsplit=1)
    assert all(torch.equal(a, b) for a, b in zip(got, want)) is not one


@pytest.mark.parametrize("Hkv,S,D", [(4, 1000, 128), (1, 1200, 64), (4, 4200, 64)])
def test_entries_agree(Hkv, S, D):
    """fa_bwd_gqa without a workspace, with the row terms alone, with the whole one (a split
    where the shape asks) and gradients 16 bytes off an allocation: dQ bitwise the same in all,
    dK and dV in those that do not split."""
    lib = _lib.load()
    B, H = 1, 4
    q, k, v, do = make(B, H, Hkv, S, D, torch.bfloat16, seed=S)
    o, lse = _forward(q, k, v, 64, 64)
    rows = (8 * B * H * S + 255) // 256 * 256
    full = lib.fa_bwd_gqa_workspace_size(B, H, Hkv, S, D)
    split = lib.fa_bwd_dkdv_split(B, H, Hkv, S, D)
    log(f"small bwd entries H_kv={Hkv} S={S} D={D} split {split}")

    def run(nbytes, off=0):
        grads = []
        for t in (q, k, v):
            buf = torch.zeros(t.numel() + 16, device="cuda", dtype=t.dtype)
            grads.append(buf[off:off + t.numel()])
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda") if nbytes else None
        code = lib.fa_bwd_gqa(*(ctypes.c_void_p(t.data_ptr()) for t in (q, k, v, o, do, lse, *grads)), B, H, Hkv, S, D,
                              _lib.dtype_code(q.dtype), _lib.scale_log2(D), 1.0 / math.sqrt(D), 64, 64, _lib._ptr(ws),
                              nbytes, _lib._stream(q.device))
        _lib.check(code, "fa_bwd_gqa")
        torch.cuda.synchronize()
        return grads

    ref = run(0)
    for got, whole in ((run(rows), True), (run(full), split == 1), (run(0, off=8), True)):
        assert torch.equal(got[0], ref[0])
        for g, r in zip(got[1:], ref[1:]):
            if whole:
                assert torch.equal(g, r)
            else:
                assert float((g.float() - r.float()).abs().max()) <= 2e-2 + 1e-2 * float(r.float().abs().max())


def test_split_without_room_for_the_row_terms():
    """128 query heads to one K/V head at D = 32: a workspace 256 bytes short of the row terms (8 bytes
    per query row) still holds the sums of a three-way split (8 D bytes per key and chunk).  Same
    gradients, bitwise, as with the row terms in the workspace before the same split; with dq 8
    bytes off its alignment dK/dV forms Delta itself, in another fp32 order."""
    lib = _lib.load()
    H, S, D = 128, 100, 32
    q, k, v, do = make(1, H, 1, S, D, torch.float16, seed=7)
    o, lse = _forward(q, k, v, 64, 64)
    rows, chunk = 8 * H * S, 8 * S * D
    assert rows % 256 == 0 and rows - 256 >= 3 * chunk and lib.fa_bwd_dkdv_split(1, H, 1, S, D) > 3

    def run(nbytes, off=0):
        dq = torch.zeros(q.numel() + 16, device="cuda", dtype=q.dtype)[off:off + q.numel()]
        dk, dv = torch.zeros_like(k), torch.zeros_like(v)
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        code = lib.fa_bwd_gqa(*(ctypes.c_void_p(t.data_ptr()) for t in (q, k, v, o, do, lse, dq, dk, dv)), 1, H, 1, S, D,
                              _lib.dtype_code(q.dtype), _lib.scale_log2(D), 1.0 / math.sqrt(D), 64, 64, _lib._ptr(ws),
                              nbytes, _lib._stream(q.device))
        _lib.check(code, "fa_bwd_gqa")
        torch.cuda.synchronize()
        return dq, dk, dv

    want = run(rows + 3 * chunk)
    for got, want_t in zip(run(rows - 256), want):
        assert torch.equal(got, want_t)
    dq, dk, dv = run(rows - 256, off=4)
    assert torch.equal(dq, want[0])
    for got, want_t in ((dk, want[1]), (dv, want[2])):   # sums over 128 heads: a few fp16 units
        assert float((got.float() - want_t.float()).abs().max()) <= 8 * 2.0 ** -10 * float(want_t.float().abs().max())


@pytest.mark.parametrize("D", [32, 64, 128])
def test_one_launch_leaves_the_workspace_alone(D):
    """Both kinds of workgroup of the one launch form Delta themselves: nothing reads row terms, so
    none are written into the workspace a caller gives."""
    lib = _lib.load()
    B, H, S = 1, 3, 200
    q, k, v, do = make(B, H, H, S, D, torch.float16, seed=D)
    o, lse = _forward(q, k, v, 64, 64)
    assert lib.fa_bwd_dkdv_split(B, H, H, S, D) == 1
    n = lib.fa_bwd_gqa_workspace_size(B, H, H, S, D)
    ws = torch.full((n,), 0xA5, dtype=torch.uint8, device="cuda")
    grads = [torch.empty_like(t) for t in (q, k, v)]
    code = lib.fa_bwd_gqa(*(ctypes.c_void_p(t.data_ptr()) for t in (q, k, v, o, do, lse, *grads)), B, H, H, S, D,
                          _lib.dtype_code(q.dtype), _lib.scale_log2(D), 1.0 / math.sqrt(D), 64, 64, _lib._ptr(ws), n,
                          _lib._stream(q.device))
    _lib.check(code, "fa_bwd_gqa")
    torch.cuda.synchronize()
    assert bool((ws == 0xA5).all())
