"""ArgCheck refuses what check_args refuses, with the same error, and follows the operator's fields."""

import pytest
import torch

from iron_amd.common.base import ArgCheck, check_args
from iron_amd.operators import RMSNorm, RoPE


def _error(fn):
    with pytest.raises((TypeError, ValueError)) as e:
        fn()
    return type(e.value), str(e.value)


@pytest.mark.parametrize("args", [
    (),                                              # too few
    tuple(torch.zeros(64) for _ in range(4)),        # too many
    (1.0, torch.zeros(64), torch.zeros(64)),         # not a tensor
    tuple(torch.zeros(4096) for _ in range(3)),      # not on the GPU
])
def test_same_errors(args):
    op = RoPE(rows=4, cols=32)
    assert _error(lambda: ArgCheck(op)(args)) == _error(lambda: check_args(op, args))


class _Gpu(torch.Tensor):
    """A CPU tensor that says it is on the GPU."""

    @property
    def is_cuda(self):
        return True


def _gpu(n):
    return torch.zeros(n, dtype=torch.bfloat16).as_subclass(_Gpu)


def test_sizes_follow_the_fields():
    op = RMSNorm(size=64, num_aie_columns=1, num_channels=1, tile_size=32)
    check = ArgCheck(op)
    args = (_gpu(64), _gpu(64))
    assert check(args) is args
    short, strided = (_gpu(63), _gpu(64)), (_gpu(128)[::2], _gpu(64))
    for bad in (short, strided):
        with pytest.raises(ValueError):
            check(bad)
    assert check(args) is args
    op.size = 96                       # larger: what passed is now too short
    with pytest.raises(ValueError):
        check(args)
    op.weighted = True                 # and one argument more
    with pytest.raises(ValueError, match="expected 3 arguments"):
        check((_gpu(96), _gpu(96)))
    assert len(check((_gpu(96), _gpu(32), _gpu(96)))) == 3


class _Lists(RMSNorm):
    """An operator whose sizes hang on a field that is changed in place."""

    def get_arg_spec(self):
        specs = super().get_arg_spec()
        return specs[:1] * len(self.inputs) + specs[1:]


def test_fields_that_are_no_plain_values():
    op = _Lists(size=64, num_aie_columns=1, num_channels=1, tile_size=32)
    op.inputs = [0]
    check = ArgCheck(op)
    assert len(check((_gpu(64), _gpu(64)))) == 2
    op.inputs.append(1)                # the same list, one argument more
    with pytest.raises(ValueError, match="expected 3 arguments"):
        check((_gpu(64), _gpu(64)))
    op = RMSNorm(size=64, num_aie_columns=1, num_channels=1, tile_size=32)
    check = ArgCheck(op)
    for note in (0, torch.zeros(2), torch.ones(2), "text"):   # tensors compare to no truth value
        op.note = note
        assert len(check((_gpu(64), _gpu(64)))) == 2


def test_field_changed_while_the_sizes_are_read():
    op = RMSNorm(size=64, num_aie_columns=1, num_channels=1, tile_size=32)
    spec = op.get_arg_spec

    def meanwhile():                   # another thread's change between the sizes and their record
        sizes = spec()
        object.__setattr__(op, "size", 96)
        return sizes

    check = ArgCheck(op)
    type(op).get_arg_spec, kept = lambda self: meanwhile(), type(op).get_arg_spec
    try:
        check((_gpu(64), _gpu(64)))
    finally:
        type(op).get_arg_spec = kept
    with pytest.raises(ValueError):
        check((_gpu(64), _gpu(64)))
