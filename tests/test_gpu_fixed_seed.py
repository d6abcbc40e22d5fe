"""Fixed calls give the recorded bits (fixed_seed.py)."""
import json

import pytest

import fixed_seed

pytestmark = pytest.mark.gpu

with open(fixed_seed.GOLDEN) as _f:
    RECORDED = json.load(_f)


@pytest.mark.parametrize("name", sorted(fixed_seed.cases()))
def test_recorded_bits(ctx, torch_gpu, name):
    assert fixed_seed.cases()[name](ctx, torch_gpu) == RECORDED[name]
