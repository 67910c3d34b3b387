"""Short sequences at head sizes 32 and 64 run 64-row forward and dQ workgroups.

A 32-row wave does the same work in a workgroup of any size, so O, LSE and the gradients must equal,
bitwise, those of the exact entry points at 128 rows.  Lengths: one key tile and one row past it,
an odd and an even number of 64-row tiles; both sides of each bound of the rule (three tiles; seven
or eight; heads a multiple of 8; two and a half or four and a half 128-row workgroups per CU; 15 tiles); every grid is
past those whose keys are split over wave groups."""

import pytest
import torch

from attention import _lib
from test_exact_entries_gpu import bwd, fwd, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,H_kv,S,D,dtype", [
    (16, 32, 32, 65, 64, torch.float16), (16, 32, 32, 129, 32, torch.bfloat16), (16, 20, 4, 192, 64, torch.bfloat16),
    (2, 99, 99, 193, 32, torch.float16), (2, 100, 100, 256, 64, torch.bfloat16), (8, 16, 16, 448, 64, torch.float16),
    (8, 16, 16, 449, 64, torch.bfloat16), (8, 16, 16, 512, 32, torch.float16), (8, 16, 16, 513, 32, torch.bfloat16),
    (2, 44, 44, 960, 32, torch.float16), (2, 44, 44, 960, 64, torch.bfloat16), (2, 40, 40, 960, 64, torch.float16),
    (2, 44, 44, 961, 64, torch.float16), (8, 36, 36, 449, 64, torch.float16), (16, 19, 19, 512, 64, torch.bfloat16),
])
def test_short_rows_equal_128_rows(B, H, H_kv, S, D, dtype):
    lib = _lib.load()
    q, k, v, do = inputs(B, H, H_kv, S, D, dtype, seed=S + D)
    o, lse = fwd(lib, q, k, v, 64, 64)
    o128, lse128 = fwd(lib, q, k, v, 128, 64, 1)
    assert torch.equal(o, o128) and torch.equal(lse, lse128)
    want = bwd(lib, q, k, v, o, do, lse, 128, 64, nsplit=lib.fa_bwd_dkdv_split(B, H, H_kv, S, D))
    for tile_m, tile_n in ((64, 64), (128, 128)):
        got = bwd(lib, q, k, v, o, do, lse, tile_m, tile_n)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
