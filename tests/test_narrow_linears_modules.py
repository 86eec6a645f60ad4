"""``narrow_linears`` with modules in place of plain ``nn.Linear`` layers: adapters,
modules without a tensor ``weight``, weights of a tensor subclass.  They are
called, as ``in_proj_b(x)`` and ``in_proj_a(x)`` are (linear_attention.py:311-314)."""
import pytest
import torch
from torch import nn

from tokenfactory_amd.fp8_linear import _narrow_pair, narrow_linears


class LowRank(nn.Module):
    """A linear and its low-rank update, without a ``weight`` of its own."""

    def __init__(self, base):
        super().__init__()
        self.base = base
        self.down, self.up = nn.Linear(64, 2, bias=False), nn.Linear(2, 8, bias=False)

    def forward(self, x):
        return self.base(x) + self.up(self.down(x))


class WeightMethod(nn.Module):
    def __init__(self, base):
        super().__init__()
        self.base = base

    def weight(self):
        return self.base.weight

    def forward(self, x):
        return 2 * self.base(x)


class Tagged(torch.Tensor):
    pass


def tagged():
    lin = nn.Linear(64, 8, bias=False)
    lin.weight = nn.Parameter(lin.weight.detach().as_subclass(Tagged))
    return lin


@pytest.mark.parametrize("make", [
    lambda: LowRank(nn.Linear(64, 8, bias=False)),
    lambda: WeightMethod(nn.Linear(64, 8, bias=False)),
    lambda: nn.Sequential(nn.Linear(64, 8, bias=False)),
    lambda: (lambda x: x[:, :8] * 2),
    tagged,
], ids=["adapter", "weight-method", "sequential", "function", "subclass"])
@pytest.mark.parametrize("place", [0, 1])
def test_other_modules_are_called(make, place):
    x = torch.randn(5, 64)
    pair = [nn.Linear(64, 8, bias=False), nn.Linear(64, 8, bias=False)]
    pair[place] = make()
    assert _narrow_pair(x, *pair) is None
    first, second, partials = narrow_linears(x, *pair)
    assert partials is None
    assert torch.equal(first, pair[0](x)) and torch.equal(second, pair[1](x))
