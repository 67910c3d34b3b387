"""Short sequences at head sizes 32 and 64 run 64-row forward and dQ workgroups.

A 32-row wave does the same work in a workgroup of any size, so O, LSE and the gradients must equal,
bitwise, those of the exact entry points at 128 rows.  Lengths: one key tile and one row past it,
an odd and an even number of 64-row tiles, both sides of the rule's last length; every grid is
past those whose keys are split over wave groups."""

import pytest
import torch

from attention import _lib
from test_exact_entries_gpu import bwd, fwd, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,H_kv,S,D,dtype", [
    (16, 32, 32, 65, 64, torch.float16), (16, 32, 32, 129, 32, torch.bfloat16), (16, 20, 4, 192, 64, torch.bfloat16),
    (4, 17, 17, 960, 32, torch.float16), (4, 17, 17, 960, 64, torch.bfloat16), (4, 16, 16, 961, 64, torch.float16),
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
