"""near_math.h's square root, reciprocal and quotient against the IEEE forms on
the GPU at hand: every float32 in range, and 4e9 quotients."""
import pytest
import torch

from diffsph_amd import _lib

pytestmark = pytest.mark.gpu


def _differ(op, first, n, seed=0):
    c = torch.zeros(1, dtype=torch.int64, device="cuda")
    _lib.check(_lib.lib().dsph_near_check(op, first, n, seed, _lib.ptr(c), _lib.stream_handle(c.device)), "near_check")
    return int(c)


@pytest.mark.parametrize("name,op,exponent", [("sqrt", 0, 96), ("rcp", 1, 60)])
def test_every_value_in_range_is_correctly_rounded(name, op, exponent):
    print(f"case {name}", flush=True)
    first, last = (127 - exponent) << 23, (127 + exponent) << 23
    assert _differ(op, first, last - first + 1) == 0
    if op == 0:
        assert _differ(0, 0, 1) == 0                       # zero
    else:
        assert _differ(1, first + (1 << 31), last - first + 1) == 0


@pytest.mark.parametrize("seed", [1, 2])
def test_drawn_quotients_are_correctly_rounded(seed):
    print(f"case quotients {seed}", flush=True)
    assert _differ(2, 0, 2_000_000_000, seed) == 0
