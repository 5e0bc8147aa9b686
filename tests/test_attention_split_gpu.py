"""The key-split prefill attention (few query tiles): edges of its 32-query tiles and 32-key blocks, waves without a
block, padding rows, queries behind a cache, and the sizes on both sides of its dispatch line, against float64."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _reference(q, k, v, causal, off):
    H, G = q.shape[0], q.shape[0] // k.shape[0]
    out = torch.empty_like(q, dtype=torch.float64)
    rows, cols = torch.arange(q.shape[1], device=q.device)[:, None] + off, torch.arange(k.shape[1], device=q.device)
    for h in range(H):
        s = q[h].double() @ k[h // G].double().t() / math.sqrt(q.shape[2])
        if causal:
            s = s.masked_fill(cols > rows, -math.inf)
        out[h] = torch.softmax(s, 1) @ v[h // G].double()
    return out


@pytest.mark.parametrize("H,Hkv,Sq,Skv,causal,off,pad", [
    (8, 8, 1, 1, 1, 0, 0),  # one key: three waves without a block
    (4, 1, 31, 31, 1, 0, 33),
    (32, 8, 33, 33, 1, 0, 31),  # a tile of one row, padding rows in and past it
    (8, 2, 96, 97, 0, 0, 0),  # no mask, a last block of one key
    (16, 4, 130, 130, 1, 0, 200),  # whole tiles of padding
    (8, 2, 7, 1000, 1, 993, 0),  # a few rows behind a cache
    (3, 3, 64, 300, 1, 100, 0),  # keys past the last query, heads not a multiple of 8
    (32, 8, 1536, 1536, 1, 0, 0),  # 384 tiles of 128: the last size of the split form
    (32, 8, 1537, 1537, 1, 0, 0),  # 416: the first of the other
])
def test_prefill_split(gpu, H, Hkv, Sq, Skv, causal, off, pad):
    from iron_amd import _lib

    g = torch.Generator(device=gpu).manual_seed(Sq + Skv + H)
    q = torch.randn(H, Sq, 64, device=gpu, generator=g).to(BF16)
    k, v = (torch.randn(Hkv, Skv, 64, device=gpu, generator=g).to(BF16) for _ in range(2))
    k[:, : max(1, Skv // 3)] *= 4  # maxima that move by more than the rescaling step along a row
    rows = Sq + pad
    out = torch.full((H, rows + 1, 64), 9.0, dtype=BF16, device=gpu)
    _lib.call("iron_attention_prefill", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), H, Hkv, Sq, Skv, 64,
              Sq * 64, 64, Skv * 64, 64, (rows + 1) * 64, 64, rows, causal, off, 1 / math.sqrt(64), _lib.stream_handle(gpu))
    torch.cuda.synchronize()
    ref = _reference(q, k, v, causal, off)
    # P is rounded to bf16 before the product with V (2^-9 of each weight, whose sum is 1), then the output once
    bound = 2.0**-8 * ref.abs() + 2.0**-8 * v.abs().max().double()
    assert ((out[:, :Sq].double() - ref).abs() <= bound).all()
    assert float((out[:, :Sq].double() - ref).norm() / ref.norm()) <= 6e-3
    assert (out[:, Sq:rows] == 0).all() and (out[:, rows] == 9.0).all()


def _attend(q, k, v, causal, off):
    from iron_amd import _lib

    H, Sq, _ = q.shape
    Hkv, Skv, _ = k.shape
    out = torch.empty_like(q)
    _lib.call("iron_attention_prefill", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), H, Hkv, Sq, Skv, 64,
              Sq * 64, 64, Skv * 64, 64, Sq * 64, 64, Sq, causal, off, 0.125, _lib.stream_handle(q.device))
    return out


@pytest.mark.parametrize("H,Hkv,Sq,Skv,causal,off,split", [
    (64, 8, 640, 640, 1, 0, False),  # 320 query tiles of short walks
    (64, 8, 384, 384, 1, 0, False),
    (32, 8, 1024, 1024, 0, 0, False),  # not causal: twice the keys per query
    (16, 4, 3072, 3072, 0, 0, False),
    (32, 8, 1536, 17920, 1, 16384, False),  # behind a long cache
    (64, 8, 256, 256, 0, 0, True),  # half a tile per CU
    (40, 8, 403, 403, 1, 0, True),  # short walks, but hardly more than one turn of them
    (32, 8, 1024, 1024, 1, 0, True),
    (32, 8, 768, 4368, 1, 3600, True),
    (8, 2, 4096, 4096, 1, 0, True),
])
def test_form_by_walk(gpu, H, Hkv, Sq, Skv, causal, off, split):
    """The faster form takes the call. A head's bits say which did: they depend on the form only, the same heads many
    times over (past one and a half tiles per CU) are in the 128-query form, and one KV group alone (at most half a
    tile per CU) is in the key-split one."""
    g = torch.Generator(device=gpu).manual_seed(Sq + Skv)
    q = torch.randn(H, Sq, 64, device=gpu, generator=g).to(BF16)
    k, v = (torch.randn(Hkv, Skv, 64, device=gpu, generator=g).to(BF16) for _ in range(2))
    got, G = _attend(q, k, v, causal, off)[: H // Hkv], H // Hkv
    times = 2 * 384 // (H * ((Sq + 127) // 128)) + 1
    whole = _attend(q.repeat(times, 1, 1), k.repeat(times, 1, 1), v.repeat(times, 1, 1), causal, off)[:G]
    alone = _attend(q[:G].contiguous(), k[:1].contiguous(), v[:1].contiguous(), causal, off)
    torch.cuda.synchronize()
    assert not torch.equal(whole, alone)
    assert torch.equal(got, alone if split else whole)
