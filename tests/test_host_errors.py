"""What the native host path does with calls it cannot finish: an exception that the caller can catch, of the type the call would raise
in Python, and never the end of the process."""
import os
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# Tensors without memory (tracing): every entry in a process of its own, because an exception that leaves native code ends it.
_FAKE = r'''
import sys
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from fla_hip import _lib
from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
entry = sys.argv[1]
bf = torch.bfloat16
with FakeTensorMode(allow_non_fake_inputs=True):
    def e(*s, dtype=bf):
        return torch.empty(*s, dtype=dtype, device='cuda')
    q, k, v, g, b = e(1, 128, 2, 128), e(1, 128, 2, 128), e(1, 128, 2, 128), e(1, 128, 2, dtype=torch.float32), e(1, 128, 2)
    lin = [e(*s) for s in ((256, 256), (256, 256), (256, 256), (2, 256), (2, 256), (256, 256), (256, 256))]
    gate, norm = [e(2, dtype=torch.float32) for _ in range(2)], e(128)
    conv = tuple(e(256, 1, 4) for _ in range(3))
    native = _lib.host()
    try:
        if entry == 'fused_recurrent':
            fused_recurrent_gated_delta_rule(q, k, v, g, beta=b)
        elif entry == 'chunk_fwd':
            with torch.no_grad():
                chunk_gated_delta_rule(q, k, v, g, b)
        elif entry == 'chunk_train':
            chunk_gated_delta_rule(q.requires_grad_(), k, v, g, b)
        elif entry == 'layer_step':
            out = native.layer_step(e(3, 1, 256), *lin, *gate, conv, (None,) * 3, tuple(e(3, 256, 4) for _ in range(3)),
                                    e(3, 2, 128, 128, dtype=torch.float32), norm, 1e-5, False, 2)
            raise RuntimeError(f'not taken: {out}')
        else:
            out = native.layer_train(e(1, 128, 256).requires_grad_(), *lin, conv, *gate, norm, 1e-5, False, 2)
            raise RuntimeError(f'not taken: {out}')
    except Exception as exc:
        print('caught', type(exc).__name__, exc)
'''


@pytest.mark.parametrize('entry', ['fused_recurrent', 'chunk_fwd', 'chunk_train', 'layer_step', 'layer_train'])
def test_tensors_without_memory_raise(entry):
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, 'flash-linear-attention_amd'))
    r = subprocess.run([sys.executable, '-c', _FAKE, entry], env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith('caught'), f'exit {r.returncode}\n{r.stdout}\n{r.stderr[-2000:]}'


def _operands(T=4096, grad=False):
    gen = torch.Generator(device='cuda').manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=gen, device='cuda')
    q, k = (torch.nn.functional.normalize(rn(1, T, 2, 128), dim=-1).bfloat16() for _ in range(2))
    x = [q, k, rn(1, T, 4, 128).bfloat16(), -rn(1, T, 4).abs(), rn(1, T, 4).sigmoid()]
    return [t.requires_grad_(grad) for t in x]


@pytest.mark.gpu
@pytest.mark.parametrize('entry', ['fused_recurrent', 'chunk_fwd', 'chunk_train', 'layer_step', 'layer_train'])
def test_out_of_memory_can_be_caught(entry):
    """No room for outputs and workspaces: torch.OutOfMemoryError, as from any operator of torch, and the same call succeeds afterwards."""
    from fla_hip.layers import GatedDeltaNet
    from fla_hip.layers.gated_deltanet import LayerCache
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
    if entry.startswith('layer'):
        layer = GatedDeltaNet(hidden_size=2048, head_dim=128, expand_v=1, num_heads=16, layer_idx=0).cuda().bfloat16().train(entry == 'layer_train')
        x = torch.randn(128, 1, 2048, device='cuda').bfloat16() if entry == 'layer_step' else torch.randn(1, 8192, 2048, device='cuda').bfloat16()
        cache = LayerCache()
        cache.update(layer_idx=0, recurrent_state=torch.zeros(128, 16, 128, 128, device='cuda'),
                     conv_state=tuple(torch.zeros(128, 2048, 4, device='cuda', dtype=torch.bfloat16) for _ in range(3)))
        call = (lambda: layer._step(x, cache)) if entry == 'layer_step' else lambda: layer._train(x)
    else:
        q, k, v, g, b = _operands(16384, grad=entry == 'chunk_train')
        if entry == 'fused_recurrent':
            call = lambda: fused_recurrent_gated_delta_rule(q, k, v, g, beta=b)[0]
        else:
            call = lambda: chunk_gated_delta_rule(q, k, v, g, b)[0]
    want = call()
    assert want is not None
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-9)
    try:
        held = []                                       # (blocks that were reserved before still serve small requests)
        with pytest.raises(torch.OutOfMemoryError):
            for _ in range(4096):
                held.append(call())
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    held.clear()
    again = call()
    assert again.shape == want.shape and bool(again.isfinite().all())
    if not entry.startswith('layer'):
        assert torch.equal(again, want)


@pytest.mark.gpu
@pytest.mark.parametrize('op', ['recurrent', 'chunk'])
@pytest.mark.parametrize('form', ['vmap', 'func_grad', 'sparse', 'fake'])
def test_tensors_without_plain_memory_raise_on_the_gpu(op, form):
    from torch._subclasses.fake_tensor import FakeTensorMode
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
    q, k, v, g, b = _operands(64)
    call = (lambda x: fused_recurrent_gated_delta_rule(x, k, v, g, beta=b)[0]) if op == 'recurrent' else lambda x: chunk_gated_delta_rule(x, k, v, g, b)[0]
    want = call(q)
    with pytest.raises(Exception):
        if form == 'vmap':
            torch.vmap(call)(torch.stack([q, q]))
        elif form == 'func_grad':
            torch.func.grad(lambda x: call(x).float().sum())(q)
        elif form == 'sparse':
            call(q.to_sparse())
        else:
            with FakeTensorMode(allow_non_fake_inputs=True) as mode:
                call(mode.from_tensor(q))
    assert torch.equal(call(q), want)


class _Switch:
    """A truth value that takes the interpreter to find out."""

    def __init__(self, value):
        self.value = value

    def __bool__(self):
        if self.value is None:
            raise ValueError('no truth in it')
        return sum([bool(self.value)] * 3) == 3


def test_a_switch_without_truth_raises():
    from fla_hip import _lib
    with pytest.raises(ValueError, match='no truth'):
        _lib.host().fused_recurrent(*[None] * 10, _Switch(None), *[None] * 9)


@pytest.mark.gpu
@pytest.mark.parametrize('neg', [False, True])
def test_switches_are_read_with_the_interpreter_held(neg):
    from fla_hip.layers import GatedDeltaNet
    torch.manual_seed(0)
    layer = GatedDeltaNet(hidden_size=256, head_dim=64, expand_v=1, num_heads=4, allow_neg_eigval=neg).cuda().bfloat16().train()
    x = torch.randn(1, 130, 256, device='cuda').bfloat16()
    want = layer._train(x)
    layer.allow_neg_eigval = _Switch(neg)
    assert torch.equal(layer._train(x), want)
    layer.allow_neg_eigval = _Switch(None)
    with pytest.raises(ValueError, match='no truth'):
        layer._train(x)


@pytest.mark.gpu
def test_a_refused_layer_step_leaves_the_states_alone():
    """33024 value columns a head: more than the norm takes.  No launch may have moved the convolutions' states on by then."""
    from fla_hip.layers import GatedDeltaNet
    from fla_hip.layers.gated_deltanet import LayerCache
    layer = GatedDeltaNet(hidden_size=256, head_dim=64, expand_v=516, num_heads=1, layer_idx=0).cuda().bfloat16().eval()
    cache = LayerCache()
    cache.update(layer_idx=0, recurrent_state=torch.randn(1, 1, 33024, 64, device='cuda'),
                 conv_state=tuple(torch.randn(1, d, 4, device='cuda', dtype=torch.bfloat16) for d in (64, 64, 33024)))
    states = [cache[0]['recurrent_state'], *cache[0]['conv_state']]
    before = [s.clone() for s in states]
    assert layer._step(torch.randn(1, 1, 256, device='cuda', dtype=torch.bfloat16), cache) is None
    assert all(torch.equal(a, b) for a, b in zip(before, states))
