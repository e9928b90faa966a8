"""Gated activations at the edges of how lanes are dealt through the rows, against
fp64: the result is rounded to bf16 once (2^-8 of itself), 2^-18 for 32-bit
functions and products."""
import math

import pytest
import torch

from xllm_service_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["silu", "gelu"])
@pytest.mark.parametrize("T", [1, 3, 33, 257])
@pytest.mark.parametrize("inner", [8, 24, 1408, 2040, 2048, 2056, 14336])
def test_rows(kind, T, inner):
    g = torch.Generator().manual_seed(T + inner)
    x = torch.randn(T, 2 * inner, generator=g).to(torch.bfloat16)
    a, b = x.double().chunk(2, 1)
    if kind == "silu":
        want = a * torch.sigmoid(a) * b
    else:
        want = b * 0.5 * a * (1 + torch.tanh(
            math.sqrt(2 / math.pi) * (a + 0.044715 * a ** 3)))
    got = getattr(ops, kind + "_and_mul")(x.cuda()).double().cpu()
    assert got.shape == want.shape
    # what is left of 1 + tanh near -1 is a difference of 32-bit numbers
    off = (got - want).abs() - 2.0 ** -8 * want.abs() \
        - 2.0 ** -18 * (a * b).abs()
    assert off.max() <= 0, f"over by {off.max():.3g}"
