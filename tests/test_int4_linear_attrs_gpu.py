"""XPUInt4Linear whose weight or bias is not where the constructor registered it: replaced by a parameter,
parametrized, or swapped in by functional_call.  Every one computes what the plain layer computes."""

import pytest
import torch
from torch import nn

from anna_amd.quantization import XPUInt4Linear

pytestmark = pytest.mark.gpu


class Doubled(nn.Module):
    def forward(self, t):
        return 2 * t


def make(gpu, bias=True):
    torch.manual_seed(3)
    dense = nn.Linear(256, 96, bias=bias)
    return XPUInt4Linear.from_linear(dense, group_size=128, compute_dtype=torch.bfloat16, device=gpu)


@pytest.mark.parametrize("name", ["qweight", "qscale", "qzeros"])
@torch.no_grad()
def test_buffer_replaced_by_a_parameter(gpu, name):
    layer = make(gpu)
    x = torch.randn(5, 256, device=gpu, dtype=torch.bfloat16)
    want = layer(x)
    setattr(layer, name, nn.Parameter(getattr(layer, name).clone(), requires_grad=False))
    assert torch.equal(layer(x), want)


@torch.no_grad()
def test_parametrized_bias(gpu):
    layer = make(gpu)
    x = torch.randn(5, 256, device=gpu, dtype=torch.bfloat16)
    torch.nn.utils.parametrize.register_parametrization(layer, "bias", Doubled())
    plain = make(gpu)
    plain.bias.mul_(2)
    assert torch.equal(layer(x), plain(x))


@torch.no_grad()
def test_bias_as_a_plain_attribute_and_functional_call(gpu):
    layer, x = make(gpu), torch.randn(5, 256, device=gpu, dtype=torch.bfloat16)
    want = layer(x)
    bias = layer.bias.detach().clone()
    del layer.bias
    layer.bias = bias
    assert torch.equal(layer(x), want)
    other = make(gpu)
    state = {"bias": bias * 3, "qzeros": other.qzeros + 1}
    got = torch.func.functional_call(other, state, (x,))
    other.bias.mul_(3)
    other.qzeros.add_(1)
    assert torch.equal(got, other(x))
