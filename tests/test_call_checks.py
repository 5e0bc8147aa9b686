"""What an operator's callable refuses: an argument list that its arg spec, as it is at the call, does not describe. The
specs that a callable keeps between calls may hide no change of the operator, whatever its spec depends on. Runs without
a GPU: the tensors only say that they are on one, and nothing is launched."""

import copy
from dataclasses import dataclass, field
from typing import ClassVar

import pytest
import torch

import iron_amd.operators as ops
from iron_amd import _lib
from iron_amd.common import AIERuntimeArgSpec, HIPOperator

BF16 = torch.bfloat16


class OnGpu(torch.Tensor):
    is_cuda = property(lambda self: True)
    device = property(lambda self: torch.device("cuda", 0))

    def get_device(self):
        return 0


def _x(n, dtype=BF16):
    return torch.zeros(n, dtype=dtype).as_subclass(OnGpu)


@pytest.fixture(autouse=True)
def no_device(monkeypatch):
    monkeypatch.setattr(_lib, "load", lambda: None)
    monkeypatch.setattr(_lib, "tensor_stream", lambda t: 0)
    monkeypatch.delenv("IRON_TRACE_SIZE", raising=False)


class Counting(HIPOperator):
    """Takes one tensor of ``count()`` elements and launches nothing."""

    def __init__(self):
        HIPOperator.__init__(self)
        self.launched = 0

    def get_arg_spec(self):
        return [AIERuntimeArgSpec("in", (self.count(),))]

    def _launch(self, x, *, stream):
        assert x.numel() == self.count()
        self.__dict__["launched"] += 1


class OfList(Counting):
    def __init__(self):
        super().__init__()
        self.sizes = [16]

    def count(self):
        return self.sizes[0]

    def change(self):
        self.sizes[0] = 8


class OfConfig(OfList):
    def __init__(self):
        super().__init__()
        self.config = type("Config", (), {"n": 16})()

    def count(self):
        return self.config.n

    def change(self):
        self.config.n = 8


class OfClass(Counting):
    n = 16

    def count(self):
        return self.n

    def change(self):
        type(self).n = 8


class OfDeleted(Counting):
    n = 8

    def __init__(self):
        super().__init__()
        self.n = 16

    def count(self):
        return self.n

    def change(self):
        del self.n


class OfInherited(ops.SiLU):
    """A subclass of an operator of this package whose spec depends on more than its base's."""

    def __init__(self):
        super().__init__(size=16, num_aie_columns=1, tile_size=16)
        self.sizes, self.launched = [16], 0

    def get_arg_spec(self):
        return [AIERuntimeArgSpec("in", (self.sizes[0],))]

    def _launch(self, x, *, stream):
        pass

    def change(self):
        self.sizes[0] = 8


@pytest.mark.parametrize("cls", [OfList, OfConfig, OfClass, OfDeleted, OfInherited])
def test_changed_spec_is_checked(cls):
    op = cls()
    fn = op.get_callable()
    for _ in range(2):
        fn(_x(16))
        with pytest.raises(ValueError, match="elements"):
            fn(_x(8))
    op.change()
    for _ in range(2):
        with pytest.raises(ValueError, match="elements"):
            fn(_x(16))
        fn(_x(8))


@dataclass
class Declared(HIPOperator):
    n: object = 16
    context: object = field(default=None, repr=False)
    _spec_fields: ClassVar[tuple] = ("n",)

    def __post_init__(self):
        self.meanwhile = None
        HIPOperator.__init__(self, context=self.context)

    def get_arg_spec(self):
        n = int(self.n)
        if self.meanwhile is not None:
            self.meanwhile()
        return [AIERuntimeArgSpec("in", (n,))]

    def _launch(self, x, *, stream):
        pass


def test_change_while_specs_are_built():
    """A field set between the read of the old value and the keeping of its spec (as by another thread)."""
    op = Declared()

    def change():
        op.__dict__["meanwhile"] = None
        op.n = 8

    op.meanwhile = change
    fn = op.get_callable()
    try:
        fn(_x(16))  # either value may be the one this call is checked against
    except ValueError:
        pass
    with pytest.raises(ValueError, match="elements"):
        fn(_x(16))
    fn(_x(8))
    op.n = 16
    fn(_x(16))
    with pytest.raises(ValueError, match="elements"):
        fn(_x(8))


def test_value_that_changes_in_place():
    op = Declared(n=torch.tensor(16))
    fn = op.get_callable()
    fn(_x(16))
    op.n.fill_(8)
    with pytest.raises(ValueError, match="elements"):
        fn(_x(16))
    fn(_x(8))


def _operators():
    flm = ops.flm
    return [
        ops.GEMM(M=64, K=64, N=128), ops.GEMM(M=64, K=64, N=128, b_col_maj=True, c_col_maj=True),
        ops.GEMMInt4(M=64, K=64, N=128), ops.GEMV(M=64, K=64, num_batches=2), ops.GEMVInt4(M=64, K=64), flm.GEMM(M=64, K=64, N=128),
        ops.MHA(num_heads=8, seq_len=100, d=64, num_KV_heads=2), ops.MHA(num_heads=8, seq_len=100, d=64, num_KV_heads=0),
        ops.GQADecode(num_heads=8, num_kv_heads=2, head_dim=64, max_len=128), ops.RoPE(rows=16, cols=64),
        ops.SiLU(size=1024, num_aie_columns=1, tile_size=1024),
        ops.GELU(size=1024, num_aie_columns=1, num_channels=1, tile_size=1024),
        ops.ElementwiseAdd(size=1024, num_aie_columns=1, tile_size=1024),
        ops.ElementwiseMul(size=1024, num_aie_columns=1, tile_size=1024),
        ops.RMSNorm(size=1024, num_aie_columns=1, num_channels=1, tile_size=64, weighted=True),
        ops.Softmax(rows=16, cols=64), ops.Transpose(M=64, N=128, num_aie_columns=1, num_channels=1, m=64, n=64, s=8),
        ops.Repeat(rows=4, cols=64, repeat=2), ops.Dequant(size=1024, num_aie_columns=1, num_channels=1, tile_size=1024),
        ops.StridedCopy(input_sizes=[4], input_strides=[1], input_offset=0, output_sizes=[4], output_strides=[1],
                        output_offset=0, input_buffer_size=16, output_buffer_size=16),
    ]


@pytest.mark.parametrize("i", range(20))
def test_declared_fields_are_all_the_spec_reads(i):
    """Any attribute whose change moves the spec moves the values that the kept specs are compared by."""
    op = _operators()[i]
    values = type(op)._spec_values
    shape = lambda o: [(s.dtype, s.numel) for s in o.get_arg_spec()]
    assert op._keep_specs() == shape(op)
    moved = 0
    for name, v in list(vars(op).items()):
        if name == "_spec_kept":
            continue
        other = copy.copy(op)
        new = (not v) if isinstance(v, bool) else v * 2 + 64 if isinstance(v, int) else torch.float32 if v is BF16 else None
        if new is None:
            continue
        setattr(other, name, new)
        if shape(other) != shape(op):
            moved += 1
            assert values(other) != values(op), name
        assert other._keep_specs() == shape(other), name
    assert moved > 0
