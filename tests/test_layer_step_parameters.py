"""One token through a ``Mamba2Layer`` whose parameters are not plain ones: parametrised, or replaced by a tensor.
Such a layer's step takes the general path and gives its results."""

import copy

import pytest
import torch
import torch.nn as nn
from torch.nn.utils import parametrize

from mamformer_amd.layers import Mamba2Layer

OWN = ["conv_weight", "A_log", "dt_bias", "D"]
BF = torch.bfloat16


class Same(nn.Module):
    def forward(self, t):
        return t + 0


def replace(lay, name, how):
    """``name`` (of the layer or, with a dot, of a projection) parametrised or a plain tensor of the same values."""
    mod, leaf = lay.get_submodule(name.rpartition(".")[0]), name.rpartition(".")[2]
    if how == "parametrised":
        parametrize.register_parametrization(mod, leaf, Same())
    else:
        t = getattr(mod, leaf).detach().clone()
        delattr(mod, leaf)
        if how == "buffer":
            mod.register_buffer(leaf, t)
        else:
            setattr(mod, leaf, t)


@pytest.mark.parametrize("how", ["parametrised", "tensor", "buffer"])
@pytest.mark.parametrize("name", OWN + ["in_proj.weight", "out_proj.bias", "dt_proj.0.weight", "conv_bias"])
def test_plain_parameters_only(name, how):
    lay = Mamba2Layer(64, bias=True, dtype=BF)
    assert lay._step_parameters() is not None
    replace(lay, name, how)
    assert lay._step_parameters() is None


def test_replaced_projections():
    lay = Mamba2Layer(64, dtype=BF)
    del lay.out_proj
    lay.out_proj = lambda t: t
    assert lay._step_parameters() is None


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["parametrised", "tensor", "buffer"])
@pytest.mark.parametrize("name", OWN + ["out_proj.bias"])
def test_step_of_replaced_parameters(name, how):
    torch.manual_seed(1)
    lay = Mamba2Layer(64, bias=True, device="cuda", dtype=BF)
    with torch.no_grad():
        for p in lay.parameters():
            if p.dim() >= 2:
                p.normal_(std=0.2)
        lay.out_proj.bias.fill_(1.0)
    u = torch.randn(2, 1, 64, device="cuda").to(BF)
    cache = {"conv_state": torch.randn(2, 3, 64, device="cuda").to(BF), "ssm_state": torch.randn(2, 64, 128, device="cuda")}
    plain = copy.deepcopy(lay)
    plain.in_proj.register_forward_hook(lambda *a: None)       # the general path
    replace(lay, name, how)
    with torch.no_grad():
        out, new = lay(u, use_cache=True, cache=cache)
        want, wnew = plain(u, use_cache=True, cache=cache)
    assert torch.equal(out, want)
    assert all(torch.equal(new[k], wnew[k]) for k in wnew)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["in_proj", "dt_proj.1", "C_proj", "out_proj"])
def test_a_bias_of_another_size_is_left_to_the_general_path(name):
    lay = Mamba2Layer(64, bias=True, device="cuda", dtype=BF)
    u = torch.randn(2, 1, 64, device="cuda").to(BF)
    cache = {"conv_state": torch.randn(2, 3, 64, device="cuda").to(BF), "ssm_state": torch.randn(2, 64, 128, device="cuda")}
    lin = lay.get_submodule(name)
    with torch.no_grad():
        one = torch.full((1,), 0.5, device="cuda", dtype=BF)
        lin.bias.copy_(one.expand_as(lin.bias))
        want = lay(u, use_cache=True, cache=cache, return_h_states=True)[0]      # (the general path)
        lin.bias = nn.Parameter(one)                       # broadcast there; the kernel reads a value per row
        out = lay(u, use_cache=True, cache=cache)[0]
    assert (out.float() - want.float()).norm() <= 1e-2 * want.float().norm()
