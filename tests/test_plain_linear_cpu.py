"""What keeps the hand-written products from reading a module's weight in place of calling it."""
import torch
import torch.nn as nn

from timeviper_amd.model.plain_linear import plain_linear, unhooked


def linear(bias=True):
    return nn.Linear(16, 8, bias=bias)


X = torch.randn(3, 16)


def test_a_linear_as_it_is():
    assert plain_linear(linear(), X) and plain_linear(linear(False), X) and unhooked(nn.Identity())
    lin = linear()
    lin.weight.requires_grad_(False)
    assert plain_linear(lin, X)


def test_hooks_of_the_module_and_of_all_modules():
    lin = linear()
    for register in (lin.register_forward_hook, lin.register_forward_pre_hook):
        handle = register(lambda *a: None)
        assert not plain_linear(lin, X)
        handle.remove()
        assert plain_linear(lin, X)
    for register in (nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook):
        handle = register(lambda *a: None)
        assert not plain_linear(lin, X) and not unhooked(lin)
        handle.remove()
        assert plain_linear(lin, X)


def test_a_forward_of_its_own():
    lin = linear()
    real = lin.forward
    lin.forward = lambda x: 2 * real(x)
    assert not plain_linear(lin, X) and not unhooked(lin)
    del lin.forward
    assert plain_linear(lin, X)


def test_subclasses_of_the_module_and_of_its_tensors():
    class Mine(nn.Linear):
        pass

    class Packed(torch.Tensor):
        pass

    assert not plain_linear(Mine(16, 8), X)
    lin = linear()
    lin.weight = nn.Parameter(lin.weight.detach().as_subclass(Packed), requires_grad=False)
    assert isinstance(lin.weight, Packed) and not plain_linear(lin, X)
    lin = linear()
    nn.utils.parametrizations.weight_norm(lin)
    assert not plain_linear(lin, X)


def test_tensors_that_are_no_longer_its_parameters():
    for name in ("weight", "bias"):
        lin = linear()
        t = getattr(lin, name).detach()
        delattr(lin, name)
        setattr(lin, name, t)
        assert not plain_linear(lin, X)


def test_biases_of_another_dtype():
    lin = linear()
    lin.bias = nn.Parameter(lin.bias.detach().double())
    assert not plain_linear(lin, X)
