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
