"""Operator callables check their arguments on every call against specs kept from an earlier one: what was refused
before is still refused, with its message, and a changed operator is checked against its new spec."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def test_refused_after_a_good_call(gpu):
    from iron_amd.operators import ElementwiseAdd, RoPE

    x = torch.ones(1024, dtype=BF16, device=gpu)
    y = torch.empty_like(x)
    fn = ElementwiseAdd(size=1024, num_aie_columns=1, tile_size=1024).get_callable()
    fn(x, x, y)
    for bad, err, text in (((x, x), ValueError, "takes 3 arguments"), ((x, x, y.cpu()), ValueError, "must live on the GPU"),
                           ((x.cpu(), x, y), ValueError, "must live on the GPU"), ((x, x.float(), y), ValueError, "dtype"),
                           ((x, x[:512], y), ValueError, "elements"), ((x, None, y), TypeError, "torch.Tensor"),
                           ((x, torch.ones(2048, dtype=BF16, device=gpu)[::2], y), ValueError, "contiguous")):
        with pytest.raises(err, match=text):
            fn(*bad)
    fn(x, x, y)
    torch.cuda.synchronize()
    assert (y == 2).all()

    rope = RoPE(rows=16, cols=64).get_callable()  # the table may be bf16 or fp32, nothing else
    q, out = torch.ones(16, 64, dtype=BF16, device=gpu), torch.empty(16, 64, dtype=BF16, device=gpu)
    for dt in (BF16, torch.float32):
        rope(q, torch.ones(16, 64, dtype=dt, device=gpu), out)
    with pytest.raises(ValueError, match="dtype"):
        rope(q, torch.ones(16, 64, dtype=torch.float16, device=gpu), out)


def test_changed_operator_is_checked_anew(gpu):
    from iron_amd.operators import GEMVInt4

    op = GEMVInt4(M=64, K=64)
    fn = op.get_callable()
    mk = lambda M: (torch.zeros(M, 32, dtype=torch.uint8, device=gpu), torch.ones(M, 2, dtype=BF16, device=gpu),
                    torch.ones(64, dtype=BF16, device=gpu), torch.empty(M, dtype=BF16, device=gpu))
    fn(*mk(64))
    op.M = 32
    with pytest.raises(ValueError, match="elements"):
        fn(*mk(64))
    fn(*mk(32))


def test_launches_on_the_current_stream(gpu):
    """The stream is that of the call, not of an earlier one."""
    from iron_amd.operators import ElementwiseAdd

    n = 1 << 24
    fn = ElementwiseAdd(size=n, num_aie_columns=1, tile_size=n).get_callable()
    a, b = torch.ones(n, dtype=BF16, device=gpu), torch.zeros(n, dtype=BF16, device=gpu)
    fn(a, a, b)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    c = torch.zeros(n, dtype=BF16, device=gpu)
    with torch.cuda.stream(side):
        c.fill_(3.0)
        fn(c, a, b)
        got = b.clone()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert (got == 4).all()
