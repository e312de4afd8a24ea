"""Every call into the library is made with the tensors' device as the current one (CPU: the library and the device guard are stand-ins
that keep record; on one GPU the two devices cannot differ)."""
import contextlib

import pytest
import torch

from fla_hip import _lib
from fla_hip.modules import convolution, fused_norm_gate
from fla_hip.ops.comba import chunk as comba_chunk, fused_recurrent as comba_recurrent
from fla_hip.ops.delta_rule import fused_recurrent as delta_recurrent
from fla_hip.ops.gated_delta_rule import _common, chunk_bwd
from fla_hip.ops.kda import chunk as kda_chunk

HOST_ONLY = ('workspace_bytes', 'value_block')          # (entries that launch nothing)


class Library:
    def __init__(self):
        self.calls, self.inside = [], 0

    def __getattr__(self, name):
        if name.endswith(HOST_ONLY):
            return lambda *a: 256
        return lambda *a: self.calls.append((name, self.inside > 0)) or 0

    @contextlib.contextmanager
    def device(self, dev):
        self.inside += 1
        yield
        self.inside -= 1


@pytest.fixture
def lib(monkeypatch):
    lib = Library()
    monkeypatch.setattr(_lib, 'load', lambda: lib)
    monkeypatch.setattr(torch.cuda, 'device', lib.device)
    monkeypatch.setattr(_common, 'current_device', lambda: 7)
    for m in (_common, convolution, fused_norm_gate):
        monkeypatch.setattr(m, 'current_stream_ptr', lambda dev: 0)
    for m in (_common, chunk_bwd, convolution, fused_norm_gate, kda_chunk, comba_chunk, comba_recurrent, delta_recurrent):
        monkeypatch.setattr(m, 'require_gpu', lambda x, *_: x.device)
    return lib


def _conv_bwd(q, k, v, g, beta, gk):
    x = torch.zeros(2, 70, 24)
    convolution.causal_conv1d_bwd(x, x, None, torch.zeros(24, 4), torch.zeros(24, dtype=torch.float64))


def _norm(q, k, v, g, beta, gk):
    x = torch.zeros(5, 64)
    y, mean, rstd, r = fused_norm_gate.layer_norm_gated_fwd(x, x, torch.ones(64), None)
    fused_norm_gate.layer_norm_gated_bwd(x, x, x, torch.ones(64), None, 'swish', 1e-6, mean, rstd, None, False, True)


CALLS = {
    'causal_conv1d_bwd': _conv_bwd,
    'norm': _norm,
    'sum_rows': lambda q, k, v, g, beta, gk: _common.sum_rows(torch.zeros(3, 8), torch.bfloat16),
    'gate_bwd': lambda q, k, v, g, beta, gk: chunk_bwd.gate_bwd(g, beta, g, beta, torch.zeros(2), None, 1.0),
    'l2norm_fwd': lambda q, k, v, g, beta, gk: chunk_bwd.l2norm_fwd(q),
    'chunk_bwd': lambda q, k, v, g, beta, gk: chunk_bwd.chunk_gated_delta_rule_bwd(q, k, v, g, beta, 1.0, None, v, None, q_rstd=g, k_rstd=g),
    'kda_fwd': lambda q, k, v, g, beta, gk: kda_chunk.chunk_kda_fwd(q, k, v, gk, beta, 1.0, None, True),
    'kda_bwd': lambda q, k, v, g, beta, gk: kda_chunk.chunk_kda_bwd(q, k, v, gk, beta, 1.0, None, v, None),
    'comba_fwd': lambda q, k, v, g, beta, gk: comba_chunk.chunk_comba_fwd(q, k, v, k, g, beta, 1.0, None, True),
    'comba_bwd': lambda q, k, v, g, beta, gk: comba_chunk.chunk_comba_bwd(q, k, v, k, g, beta, 1.0, None, v, None, qk_l2norm=True),
    'comba_recurrent': lambda q, k, v, g, beta, gk: comba_recurrent.fused_recurrent_comba_fwd(q, k, k, v, g, beta, 1.0, None, True),
    'delta_bwd': lambda q, k, v, g, beta, gk: delta_recurrent.fused_recurrent_delta_rule_bwd(q, k, v, beta, None, v, 1.0, None),
}


@pytest.mark.parametrize('call', CALLS)
def test_launches_are_made_on_the_tensors_device(lib, call):
    q, k = torch.zeros(1, 70, 2, 64), torch.zeros(1, 70, 2, 64)
    v, g, gk = torch.zeros(1, 70, 2, 64), torch.zeros(1, 70, 2), torch.zeros(1, 70, 2, 64)
    CALLS[call](q, k, v, g, torch.ones(1, 70, 2), gk)
    assert lib.calls and all(inside for _, inside in lib.calls), lib.calls


def test_no_guard_where_the_device_is_current(lib, monkeypatch):
    monkeypatch.setattr(_common, 'current_device', lambda: None)         # (the index of the CPU device the tensors are on)
    _common.sum_rows(torch.zeros(3, 8), torch.bfloat16)
    assert lib.calls == [('gdn_sum_rows', False)]


def test_sums_of_partial_rows_in_any_type(lib):
    assert _common.sum_rows(torch.zeros(3, 8), torch.float64).dtype == torch.float64
