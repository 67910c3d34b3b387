"""The C++ module's forward against the same C entry called through ctypes: the same output and
the same exceptions, whichever way the call goes."""

import pytest
import torch

from attention import _lib
from attention.fused.fused import fused_attention
from attention.gqa.fused_gqa import fused_gqa_attention

pytestmark = pytest.mark.gpu


def _qkv(B, H, H_kv, S, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    return [torch.randn((B, h, S, D), generator=g, device="cuda").to(dtype) for h in (H, H_kv, H_kv)]


@pytest.mark.parametrize("S,D,H_kv,dtype", [(1, 32, 4, torch.float16), (65, 64, 2, torch.bfloat16),
                                             (200, 128, 4, torch.float16)])
def test_same_result(monkeypatch, S, D, H_kv, dtype):
    q, k, v = _qkv(2, 4, H_kv, S, D, dtype)
    fn = fused_attention if H_kv == 4 else fused_gqa_attention
    assert _lib._forward_op()   # built beside the library
    a = fn(q, k, v)
    with torch.cuda.stream(torch.cuda.Stream()) as _:
        torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
        b = fn(q.transpose(1, 2).contiguous().transpose(1, 2), k, v)   # (a strided view)
    torch.cuda.synchronize()
    monkeypatch.setattr(_lib, "_forward", False)
    monkeypatch.setattr(_lib, "_forward_op", lambda: False)
    c = fn(q, k, v)
    assert torch.equal(a, c) and torch.equal(b, c)


@pytest.mark.parametrize("ctypes_path", (False, True))
def test_same_errors(monkeypatch, ctypes_path):
    if ctypes_path:
        monkeypatch.setattr(_lib, "_forward", False)
        monkeypatch.setattr(_lib, "_forward_op", lambda: False)
    q, k, v = _qkv(1, 2, 2, 64, 64, torch.float16)
    with pytest.raises(ValueError):   # head size
        fused_attention(q[..., :48], k[..., :48], v[..., :48])
    with pytest.raises(ValueError):   # no rows
        fused_attention(q[:, :, :0], k[:, :, :0], v[:, :, :0])
    with pytest.raises(TypeError):
        fused_attention(q.float(), k.float(), v.float())
    with pytest.raises(ValueError):   # not on the GPU
        fused_attention(q.cpu(), k.cpu(), v.cpu())
