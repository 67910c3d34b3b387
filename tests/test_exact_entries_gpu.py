"""fa_fwd_exact and fa_bwd_gqa_exact on the GPU, through the C ABI.

These entry points (used by the tile study, no reference counterpart) run kernel instances
the dispatch rules never reach: 64-row forward workgroups of one head, one, two or four GQA
heads per workgroup where the rule picks another count (two heads of 128 rows where it takes
four of 64), 64-row dQ workgroups, and any dK/dV split from 1 to 64 -- including more chunks
than the heaviest key tile has (query tile, head) pairs, where some chunks are empty and store
zero partial sums.

Claims checked:
* the workgroup shape does not change a result: a 32-row wave runs the same arithmetic over
  the same key tiles whatever its workgroup holds, so O, LSE and dQ equal the dispatching
  entries' bitwise on grids past those whose keys are split over wave groups or whose backward
  is one launch, and so do dK and dV at the same split; the 128-key forward instances, which
  no rule takes, equal each other;
* on small grids too the exact entries run the shape that is asked for: the results of the
  same heads within a full grid, bitwise;
* a split changes only the fp32 summation order of dK and dV: every split matches the
  unsplit result to that order (a few bf16 / fp16 units) and the fp32 reference within the
  suites' bars;
* without a workspace the exact entry runs the dK/dV kernel that forms Delta itself: dQ
  unchanged, dK and dV within the same bars.
"""

import ctypes
import math

import pytest
import torch

from attention import _lib
from gpu_util import check_forward, log
from oracle import cases
from oracle.cpu_reference import reference_grads_gqa

pytestmark = pytest.mark.gpu

VP = ctypes.c_void_p


def ptr(t):
    return VP(t.data_ptr()) if t is not None else VP(0)


def stream():
    return VP(torch.cuda.current_stream().cuda_stream)


def inputs(B, H, Hkv, S, D, dtype, seed):
    q, do = (torch.from_numpy(x).cuda().to(dtype) for x in cases.normal_inputs([(B, H, S, D)] * 2, seed=seed))
    k, v = (torch.from_numpy(x).cuda().to(dtype) for x in cases.normal_inputs([(B, Hkv, S, D)] * 2, seed=seed + 1))
    return q, k, v, do


def fwd(lib, q, k, v, bm, bn, gh=None):
    B, H, S, D = q.shape
    Hkv = k.shape[1]
    o = torch.full_like(q, float("nan"))
    lse = torch.full((B, H, S), float("nan"), device="cuda")
    args = [ptr(q), ptr(k), ptr(v), ptr(o), ptr(lse), B, H, Hkv, S, D, _lib.dtype_code(q.dtype), _lib.scale_log2(D),
            bm, bn]
    code = lib.fa_fwd(*args, stream()) if gh is None else lib.fa_fwd_exact(*args, gh, stream())
    assert code == _lib.FA_OK, _lib.strerror(code)
    return o, lse


def rowb_bytes(B, H, S):
    return (8 * B * H * S + 255) // 256 * 256


def bwd(lib, q, k, v, o, do, lse, bm, bn, nsplit=None, workspace=True):
    B, H, S, D = q.shape
    Hkv = k.shape[1]
    dq, dk, dv = (torch.full_like(t, float("nan")) for t in (q, k, v))
    args = [ptr(q), ptr(k), ptr(v), ptr(o), ptr(do), ptr(lse), ptr(dq), ptr(dk), ptr(dv), B, H, Hkv, S, D,
            _lib.dtype_code(q.dtype), _lib.scale_log2(D), 1.0 / math.sqrt(D), bm, bn]
    if nsplit is None:
        n = lib.fa_bwd_gqa_workspace_size(B, H, Hkv, S, D)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        code = lib.fa_bwd_gqa(*args, ptr(ws), n, stream())
    else:
        n = rowb_bytes(B, H, S) + (8 * B * Hkv * nsplit * S * D if nsplit > 1 else 0) if workspace else 0
        ws = torch.empty(n, dtype=torch.uint8, device="cuda") if workspace else None
        code = lib.fa_bwd_gqa_exact(*args, nsplit, ptr(ws), n, stream())
    assert code == _lib.FA_OK, _lib.strerror(code)
    torch.cuda.synchronize()
    return dq, dk, dv


# (B, H, H_kv, S, D, dtype): grids past 768 64-row workgroups (three per CU of 256)
FWD_CASES = [
    (2, 30, 30, 900, 128, torch.bfloat16), (1, 70, 70, 777, 64, torch.float16),
    (4, 32, 8, 500, 128, torch.bfloat16), (5, 32, 8, 333, 64, torch.float16), (5, 32, 4, 333, 32, torch.bfloat16),
]


@pytest.mark.parametrize("B,H,Hkv,S,D,dtype", FWD_CASES)
def test_forward_exact_shapes_equal_dispatch_bitwise(B, H, Hkv, S, D, dtype):
    lib = _lib.load()
    q, k, v, _ = inputs(B, H, Hkv, S, D, dtype, seed=S + D)
    o_ref, lse_ref = fwd(lib, q, k, v, 64, 64)
    g = H // Hkv
    for bm, bn, gh in [(64, 64, gh) for gh in (1, 2, 4) if g % gh == 0] + [(128, 64, gh) for gh in (1, 2) if g % gh == 0]:
        o, lse = fwd(lib, q, k, v, bm, bn, gh)
        torch.cuda.synchronize()
        log(f"fwd exact {bm}x{bn} gh={gh} B={B} H={H} H_kv={Hkv} S={S} D={D}: "
            f"O maxdiff {float((o.float() - o_ref.float()).abs().max()):.3g}")
        assert torch.equal(o, o_ref), f"O of {bm}x{bn} with {gh} heads per workgroup"
        assert torch.equal(lse, lse_ref), f"LSE of {bm}x{bn} with {gh} heads per workgroup"
    # 128-key tiles (no rule takes them) round P against another reference point: equal among
    # themselves, within the suites' bars of the oracle and the fp32 reference
    o_ref, lse_ref = fwd(lib, q, k, v, 64, 128, 1)
    check_forward(o_ref, q, k, v, rows_count=16, label=f"fwd exact 64x128 S={S} D={D}")
    for bm, bn, gh in [(128, 128, 1)] + [(64, 128, 2)] * (g % 2 == 0):
        o, lse = fwd(lib, q, k, v, bm, bn, gh)
        assert torch.equal(o, o_ref) and torch.equal(lse, lse_ref), f"{bm}x{bn} with {gh} heads per workgroup"


@pytest.mark.parametrize("B,H,Hkv,S,D,dtype", [
    (1, 4, 4, 1000, 128, torch.bfloat16), (2, 2, 2, 777, 64, torch.float16),
    (1, 8, 2, 900, 128, torch.bfloat16), (1, 8, 2, 333, 64, torch.float16), (1, 8, 1, 440, 32, torch.bfloat16),
])
def test_small_grids_run_the_shape_asked_for(B, H, Hkv, S, D, dtype):
    """The same heads, many times over in one call, make a full grid: the exact entries on the
    small one must equal it bitwise, forward and backward (the dispatching entries run other
    kernels there)."""
    lib = _lib.load()
    q, k, v, do = inputs(B, H, Hkv, S, D, dtype, seed=S + 2 * D)
    n = 769 // (B * H * ((S + 63) // 64)) + 1
    big = [t.repeat(n, 1, 1, 1) for t in (q, k, v, do)]
    o_big, lse_big = fwd(lib, *big[:3], 64, 64)
    g = H // Hkv
    for bm, gh in [(64, gh) for gh in (1, 2, 4) if g % gh == 0] + [(128, gh) for gh in (1, 2) if g % gh == 0]:
        o, lse = fwd(lib, q, k, v, bm, 64, gh)
        torch.cuda.synchronize()
        assert torch.equal(o, o_big[:B]) and torch.equal(lse, lse_big[:B]), f"{bm} rows, {gh} heads per workgroup"
    assert lib.fa_bwd_dkdv_split(n * B, H, Hkv, S, D) == 1
    want = bwd(lib, *big[:3], o_big, big[3], lse_big, 64, 64)
    for bm in (64, 128):
        got = bwd(lib, q, k, v, o, do, lse, bm, 64, nsplit=1)
        assert all(torch.equal(a, b[:B]) for a, b in zip(got, want)), f"backward, {bm} dQ rows"


@pytest.mark.parametrize("B,H,Hkv,S,D,dtype", [
    (2, 16, 4, 168, 128, torch.float16), (1, 128, 64, 65, 64, torch.bfloat16), (4, 64, 8, 150, 32, torch.float16),
    (1, 250, 250, 130, 128, torch.bfloat16),
])
def test_forward_128_row_tile_of_a_small_grid_bitwise(B, H, Hkv, S, D, dtype):
    """Up to three 64-row workgroups per CU (and not split over keys) a 128-row tile of grouped heads
    counts as 64: the same O and LSE as two heads of 128 rows, and as tile 64."""
    lib = _lib.load()
    q, k, v, _ = inputs(B, H, Hkv, S, D, dtype, seed=S + H)
    o, lse = fwd(lib, q, k, v, 128, 64)
    for want in (fwd(lib, q, k, v, 64, 64), fwd(lib, q, k, v, 128, 64, min(2, H // Hkv))):
        assert torch.equal(o, want[0]) and torch.equal(lse, want[1])


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
def test_forward_gqa_tile_as_four_heads_bitwise(D, dtype):
    """A 128-row, 64-key GQA tile runs as 64-row workgroups of four heads where the grid is large
    enough (512 workgroups here, two per CU on a 256-CU device): the same O and LSE as two heads
    of 128 rows and as four heads of 64."""
    lib = _lib.load()
    B, H, Hkv, S = 2, 8, 2, 8192
    q, k, v, _ = inputs(B, H, Hkv, S, D, dtype, seed=D)
    gh = lib.fa_fwd_heads_per_wg(B, H, Hkv, S, D, 128, 64)
    rows = lib.fa_fwd_rows_per_wg(128, 64, D, gh)
    o, lse = fwd(lib, q, k, v, 128, 64)
    for bm, g in ((128, 2), (64, 4)):
        o_x, lse_x = fwd(lib, q, k, v, bm, 64, g)
        torch.cuda.synchronize()
        log(f"fwd 128x64 dispatch ({gh} heads of {rows} rows) vs exact {g} heads of {bm} rows, D={D}: "
            f"O maxdiff {float((o.float() - o_x.float()).abs().max()):.3g}")
        assert torch.equal(o, o_x) and torch.equal(lse, lse_x), f"{g} heads of {bm} rows"


# (B, H, H_kv, S, D, dtype): paired dK/dV at D = 128, one-wave at D <= 64; grids past those that
# run as one launch (256 64-row workgroups at D = 128, else 768), whose dQ the dispatch runs at 128 rows
BWD_CASES = [
    (1, 20, 10, 1000, 128, torch.bfloat16), (1, 72, 18, 700, 64, torch.float16), (1, 80, 40, 600, 32, torch.bfloat16),
]


@pytest.mark.parametrize("B,H,Hkv,S,D,dtype", BWD_CASES)
def test_backward_exact_shapes_and_splits(B, H, Hkv, S, D, dtype):
    lib = _lib.load()
    q, k, v, do = inputs(B, H, Hkv, S, D, dtype, seed=3 * S + D)
    o, lse = fwd(lib, q, k, v, 64, 64)
    base_split = lib.fa_bwd_dkdv_split(B, H, Hkv, S, D)
    want = bwd(lib, q, k, v, o, do, lse, 64, 64)
    # dQ rows per workgroup: the exact 64-row dQ against the dispatch's (128 rows)
    got = bwd(lib, q, k, v, o, do, lse, 64, 64, nsplit=base_split)
    for name, g_, w in zip(("dQ", "dK", "dV"), got, want):
        assert torch.equal(g_, w), f"{name}: 64-row dQ workgroups at the dispatch's split {base_split}"
    # the fp32 reference (autograd of the formula on repeated K/V, group sums)
    _, rq, rk, rv = reference_grads_gqa(q, k, v, do)
    g = H // Hkv
    pairs = g * ((S + 63) // 64)  # the heaviest key tile's (query tile, head) pairs
    for nsplit in (1, 2, 7, pairs, min(64, pairs + 5), 64):
        dq, dk, dv = bwd(lib, q, k, v, o, do, lse, 64, 64, nsplit=nsplit)
        assert torch.equal(dq, want[0]), "dQ does not depend on the dK/dV split"
        dd = max(float((dk.float() - want[1].float()).abs().max()), float((dv.float() - want[2].float()).abs().max()))
        ek = float((dk.float() - rk).abs().max())
        ev = float((dv.float() - rv).abs().max())
        log(f"bwd exact split {nsplit} (heaviest tile {pairs} pairs) B={B} H={H} H_kv={Hkv} S={S} D={D} {dtype}: "
            f"vs unsplit {dd:.3g}, vs fp32 dK {ek:.3g} dV {ev:.3g}")
        # only the fp32 order of the partial sums changes: a few units of the 16-bit output
        assert dd <= 8 * 2.0 ** -7 * max(1.0, float(rk.abs().max()), float(rv.abs().max()))
        for got_t, ref in ((dk, rk), (dv, rv)):
            err = (got_t.float() - ref).abs()
            assert bool((err <= 2e-2 + 2e-2 * ref.abs()).all()), f"split {nsplit} against the fp32 reference"
    # (mixed, as for dK and dV: over tens of heads |dQ| passes 4, where half a bf16 ulp is 1.6e-2)
    assert bool(((dq.float() - rq).abs() <= 2e-2 + 2e-2 * rq.abs()).all()), "dQ against the fp32 reference"
    # no workspace: the dK/dV kernel forms each row's Delta from the O and dO tiles of every key
    # tile it meets, in another fp32 order than the dQ kernel's (and, at D = 128, from dP
    # rounded once more); dQ runs after it and is unchanged
    dq, dk, dv = bwd(lib, q, k, v, o, do, lse, 64, 64, nsplit=1, workspace=False)
    assert torch.equal(dq, want[0]), "dQ with the Delta-forming dK/dV"
    dd = max(float((dk.float() - want[1].float()).abs().max()), float((dv.float() - want[2].float()).abs().max()))
    log(f"bwd exact, no workspace B={B} H={H} H_kv={Hkv} S={S} D={D} {dtype}: vs unsplit {dd:.3g}")
    assert dd <= 8 * 2.0 ** -7 * max(1.0, float(rk.abs().max()), float(rv.abs().max()))
    for got_t, ref in ((dk, rk), (dv, rv)):
        err = (got_t.float() - ref).abs()
        assert bool((err <= 2e-2 + 2e-2 * ref.abs()).all()), "Delta-forming dK/dV against the fp32 reference"
