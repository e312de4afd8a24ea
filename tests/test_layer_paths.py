"""When the layer may take its native paths (CPU): only where calling its modules one by one would do nothing else."""
import contextlib

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.utils._python_dispatch import TorchDispatchMode
from torch.overrides import TorchFunctionMode

from fla_hip import _lib
from fla_hip.layers import GatedDeltaNet
from fla_hip.layers.gated_deltanet import LayerCache
from fla_hip.ops.backends import BackendRegistry, BaseBackend


class _Host:
    """In the place of the host extension: says which path was taken."""

    def layer_train(self, *a):
        return 'native'

    def layer_step(self, *a):
        return 'native'


@pytest.fixture
def layer(monkeypatch):
    monkeypatch.setattr(_lib, 'host', lambda: _Host())
    return GatedDeltaNet(hidden_size=64, head_dim=32, num_heads=2, expand_v=1, layer_idx=0)


def paths(layer):
    cache = LayerCache()
    cache.update(layer_idx=0, recurrent_state=torch.zeros(1), conv_state=(torch.zeros(1),) * 3)
    return layer._train(torch.zeros(1, 8, 64)), layer._step(torch.zeros(1, 1, 64), cache)


class _Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Function(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _replace_forward(name):
    def change(layer, stack, monkeypatch):
        m = layer._modules[name]
        m.forward = lambda *a, _own=m.forward, **k: _own(*a, **k)
    return change


def _global_hook(register):
    return lambda layer, stack, monkeypatch: stack.callback(register(lambda *a: None).remove)


def _class_forward(cls):
    return lambda layer, stack, monkeypatch: monkeypatch.setattr(cls, 'forward', lambda self, *a, **k: None)


def _module_call(layer, stack, monkeypatch):
    monkeypatch.setattr(nn.Module, '__call__', lambda self, *a, **k: None)


CHANGES = {
    'linear.forward': _replace_forward('q_proj'),
    'o_proj.forward': _replace_forward('o_proj'),
    'conv.forward': _replace_forward('k_conv1d'),
    'norm.forward': _replace_forward('o_norm'),
    'conv.step': lambda layer, stack, monkeypatch: setattr(layer.v_conv1d, 'step', lambda *a, **k: None),
    'Linear.forward': _class_forward(nn.Linear),
    'Module.__call__': _module_call,
    'F.linear': lambda layer, stack, monkeypatch: monkeypatch.setattr(F, 'linear', lambda *a: None),
    'compiled module': lambda layer, stack, monkeypatch: setattr(layer.q_proj, '_compiled_call_impl', lambda *a: None),
    'forward hook': lambda layer, stack, monkeypatch: layer.g_proj.register_forward_hook(lambda *a: None),
    'global forward hook': _global_hook(nn.modules.module.register_module_forward_hook),
    'global pre hook': _global_hook(nn.modules.module.register_module_forward_pre_hook),
    'global backward hook': _global_hook(nn.modules.module.register_module_full_backward_hook),
    'dispatch mode': lambda layer, stack, monkeypatch: stack.enter_context(_Dispatch()),
    'function mode': lambda layer, stack, monkeypatch: stack.enter_context(_Function()),
    'other class': lambda layer, stack, monkeypatch: setattr(layer, 'q_proj', nn.Linear(64, 64, bias=True)),
}


@pytest.mark.parametrize('change', CHANGES)
def test_a_replaced_call_is_made(layer, monkeypatch, change):
    assert paths(layer) == ('native', 'native')
    with contextlib.ExitStack() as stack:
        CHANGES[change](layer, stack, monkeypatch)
        assert paths(layer) == (None, None)


def test_a_default_device_changes_nothing(layer):
    with torch.device('cpu'):
        assert paths(layer) == ('native', 'native')


@pytest.mark.parametrize('variable', ['FLA_HIP_SCAN_MODE', 'FLA_HIP_BWD_SCAN_MODE'])
def test_forms_of_the_scans_reach_the_operator(layer, monkeypatch, variable):
    monkeypatch.setenv(variable, 'wide')
    assert paths(layer) == (None, 'native')


def test_a_backend_of_the_operator_is_asked_in_training(layer, monkeypatch):
    monkeypatch.setattr(BackendRegistry, '_registries', dict(BackendRegistry._registries))
    registry = BackendRegistry('gated_delta_rule')
    registry.register(type('Other', (BaseBackend,), dict(backend_type='other'))())
    assert paths(layer) == (None, 'native')


def test_a_parametrised_gate_goes_through_its_modules(layer, monkeypatch):
    torch.nn.utils.parametrize.register_parametrization(layer, 'A_log', nn.Identity())
    seen = []
    monkeypatch.setattr(_Host, 'layer_train', lambda self, *a: seen.append(a[9]))
    layer._train(torch.zeros(1, 8, 64))
    assert seen == [None]
