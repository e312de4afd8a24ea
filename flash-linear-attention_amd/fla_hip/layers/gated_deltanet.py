"""Gated DeltaNet layer: projections, causal short convolutions, the gated delta rule, gated RMS
norm, output projection - the immediate caller of this package's kernels, with the constructor arguments,
parameter names (so upstream checkpoints load with ``load_state_dict``) and call signature of the reference's
``GatedDeltaNet`` (fla/layers/gated_deltanet.py:28-364), and its cache contract: ``past_key_values[layer_idx]``
is a dict with ``recurrent_state`` ``[N, HV, V, K]`` fp32 and ``conv_state`` (three ``[N, D, W]`` tensors);
``past_key_values.update(layer_idx=..., recurrent_state=..., conv_state=..., offset=...)`` stores them
(fla/layers/utils.py:271-293, fla/models/utils.py:42-118).  ``LayerCache`` is a minimal cache with that contract;
upstream's ``fla.models.utils.Cache`` objects are used the same way.

Prompts longer than 64 tokens run the chunk kernels, shorter calls (decode) the token recurrence; both read and
write the same state layout, so a prefill hands over to decode through the cache without any conversion.
The linear projections are torch matmuls; everything between them runs in this package's HIP kernels.
In training mode (``.train()``) the call is differentiable: the convolutions, the chunked operator and the gated norm
each have backward kernels, and every call runs the chunk kernels as in the reference (fla/layers/gated_deltanet.py:237-239).
In eval mode no autograd graph is built (the token recurrence of decode has no backward)."""
from __future__ import annotations

import math
import os
import warnings

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules.module import _has_any_global_hook
from torch.utils._device import DeviceContext

from fla_hip import _lib
from fla_hip.modules import FusedRMSNormGated, ShortConvolution
from fla_hip.ops.backends import has_backends
from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule


_STEP_LINEARS = ('q_proj', 'k_proj', 'v_proj', 'a_proj', 'b_proj', 'g_proj', 'o_proj')
_STEP_CONVS = ('q_conv1d', 'k_conv1d', 'v_conv1d')
_PARTS = ((nn.Linear, _STEP_LINEARS), (ShortConvolution, _STEP_CONVS), (FusedRMSNormGated, ('o_norm',)))


def _calls() -> tuple:
    return nn.Module.__call__, F.linear, nn.Linear.forward, ShortConvolution.forward, ShortConvolution.step, FusedRMSNormGated.forward


# The calls that the native paths stand for.  Where a caller has replaced one of them - here, on a module or around every module - the
# layer runs module by module and makes it.
_CALLS = _calls()


def _watched() -> bool:
    """Whether something looks at, or stands in for, the calls between all modules: hooks on every module, torch's dispatch and
    function modes (a default device is none of those), one of ``_CALLS`` patched."""
    n = torch._C._len_torch_function_stack()
    return (_has_any_global_hook() or torch._C._len_torch_dispatch_stack() > 0 or _calls() != _CALLS
            or (n > 0 and any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(n))))


class LayerCache:
    """Per-layer states of a stack of layers: ``cache[i]`` is layer i's dict, ``update`` replaces entries in it."""

    def __init__(self):
        self.states: list[dict] = []
        self._seen_tokens = 0

    def __len__(self) -> int:
        return len(self.states)

    def __getitem__(self, layer_idx: int) -> dict:
        return self.states[layer_idx]

    def update(self, *, layer_idx: int, recurrent_state=None, conv_state=None, offset: int = 1, **_) -> dict:
        while len(self.states) <= layer_idx:
            self.states.append(dict(recurrent_state=None, attn_state=None, conv_state=None, ffn_state=None))
        entry = self.states[layer_idx]
        if recurrent_state is not None:
            entry['recurrent_state'] = recurrent_state
        if conv_state is not None:
            entry['conv_state'] = conv_state
        if layer_idx == 0:
            self._seen_tokens += offset
        return entry

    def get_seq_length(self, layer_idx: int = 0) -> int:
        return self._seen_tokens if len(self.states) > layer_idx else 0


def _unpad(hidden_states, attention_mask, q_len):
    """[B, T, ...] with a 0/1 mask -> ([1, total, ...], flat indices of the kept tokens, cu_seqlens)."""
    mask = attention_mask[:, -q_len:].to(torch.bool)
    lens = mask.sum(-1, dtype=torch.int32)
    cu_seqlens = F.pad(lens.cumsum(0, dtype=torch.int32), (1, 0))
    indices = mask.flatten().nonzero(as_tuple=False).flatten()
    flat = hidden_states.reshape(-1, *hidden_states.shape[2:])
    return flat.index_select(0, indices).unsqueeze(0), indices, cu_seqlens


class GatedDeltaNet(nn.Module):

    def __init__(
        self,
        hidden_size: int = 2048,
        expand_v: float = 2,
        head_dim: int = 256,
        num_heads: int = 6,
        num_v_heads: int | None = None,
        mode: str = 'chunk',
        use_gate: bool = True,
        use_short_conv: bool = True,
        allow_neg_eigval: bool = False,
        conv_size: int = 4,
        conv_bias: bool = False,
        layer_idx: int | None = None,
        norm_eps: float = 1e-5,
        **kwargs,
    ):
        super().__init__()
        assert mode in ['chunk', 'fused_recurrent'], f'Not supported mode `{mode}`.'
        self.mode, self.allow_neg_eigval, self.hidden_size, self.expand_v = mode, allow_neg_eigval, hidden_size, expand_v
        self.use_gate, self.use_short_conv, self.conv_size, self.conv_bias = use_gate, use_short_conv, conv_size, conv_bias
        self.head_dim = self.head_k_dim = head_dim
        self.num_heads = num_heads
        self.num_v_heads = num_heads if num_v_heads is None else num_v_heads
        self.head_v_dim = int(head_dim * expand_v)
        self.key_dim = num_heads * head_dim
        self.value_dim = self.num_v_heads * self.head_v_dim
        self.layer_idx = layer_idx
        if not math.isclose(head_dim * expand_v, self.head_v_dim, rel_tol=1e-5):
            raise ValueError(f'expand_v={expand_v} times head_dim={head_dim} is not an integer head size')
        if self.num_v_heads > num_heads and self.num_v_heads % num_heads != 0:
            raise ValueError(f'num_v_heads={self.num_v_heads} must be divisible by num_heads={num_heads}.')

        self.q_proj = nn.Linear(hidden_size, self.key_dim, bias=False)
        self.k_proj = nn.Linear(hidden_size, self.key_dim, bias=False)
        self.v_proj = nn.Linear(hidden_size, self.value_dim, bias=False)
        self.a_proj = nn.Linear(hidden_size, self.num_v_heads, bias=False)
        self.b_proj = nn.Linear(hidden_size, self.num_v_heads, bias=False)
        # decay rate and step-size bias per value head, initialised as the reference does (:153-170)
        self.A_log = nn.Parameter(torch.log(torch.empty(self.num_v_heads, dtype=torch.float32).uniform_(0, 16)))
        dt = torch.exp(torch.rand(self.num_v_heads) * (math.log(0.1) - math.log(0.001)) + math.log(0.001)).clamp(min=1e-4)
        self.dt_bias = nn.Parameter(dt + torch.log(-torch.expm1(-dt)))           # inverse of softplus
        self.A_log._no_weight_decay = self.dt_bias._no_weight_decay = True
        if use_short_conv:
            self.q_conv1d = ShortConvolution(self.key_dim, conv_size, bias=conv_bias, activation='silu')
            self.k_conv1d = ShortConvolution(self.key_dim, conv_size, bias=conv_bias, activation='silu')
            self.v_conv1d = ShortConvolution(self.value_dim, conv_size, bias=conv_bias, activation='silu')
        else:
            warnings.warn('ShortConvolution is crucial to the performance. Do not turn it off, i.e., setting '
                          '`use_short_conv=False` unless you know what you are doing.')
        if use_gate:
            self.g_proj = nn.Linear(hidden_size, self.value_dim, bias=False)
            self.o_norm = FusedRMSNormGated(self.head_v_dim, eps=norm_eps)
        else:
            self.o_norm = nn.RMSNorm(self.head_v_dim, eps=norm_eps, dtype=torch.float32)
        self.o_proj = nn.Linear(self.value_dim, hidden_size, bias=False)

    def forward(
        self,
        hidden_states: torch.Tensor,
        attention_mask: torch.Tensor | None = None,
        past_key_values=None,
        use_cache: bool | None = False,
        output_attentions: bool | None = False,
        **kwargs,
    ):
        if self.training:
            return self._forward(hidden_states, attention_mask, past_key_values, use_cache, **kwargs)
        with torch.no_grad():
            return self._forward(hidden_states, attention_mask, past_key_values, use_cache, **kwargs)

    def _plain(self):
        """(weights of the projections, the convolutions and the norm; the convolutions; the norm) where the layer is its plain self, or
        None: another module in a projection's place or another forward in a module's, hooks, modes, autocast."""
        if not (self.use_gate and self.use_short_conv) or torch.is_autocast_enabled() or _watched():
            return None
        mods = self._modules
        weights = []
        # (one loop over the modules' own dictionaries: a step asks this every time, and an attribute of a module takes half a microsecond)
        for cls, names in _PARTS:
            for name in names:
                m = mods[name]
                d = m.__dict__
                # calling m is cls.forward and nothing else: no other class, no hooks, no `forward` of its own, not compiled
                if (type(m) is not cls or d['_forward_hooks'] or d['_forward_pre_hooks'] or d['_backward_hooks'] or d['_backward_pre_hooks']
                        or 'forward' in d or 'step' in d or '_compiled_call_impl' in d):
                    return None
                params = d['_parameters']
                w = params.get('weight')
                if type(w) is not nn.Parameter or (cls is nn.Linear and params.get('bias') is not None):
                    return None
                weights.append(w)
        convs, norm = [mods[name] for name in _STEP_CONVS], mods['o_norm']
        if norm.activation == 'sigmoid' or any(m.activation is None for m in convs):
            return None
        return weights, convs, norm

    def _train(self, hidden_states):
        """Whole dense sequences without a cache through the native training path (``gdn_host.layer_train``), or None (a backend is
        registered for the operator, or a form of its scans is asked for, too)."""
        if has_backends('gated_delta_rule') or os.environ.get('FLA_HIP_SCAN_MODE') or os.environ.get('FLA_HIP_BWD_SCAN_MODE'):
            return None
        plain = self._plain()
        if plain is None or any(m._parameters.get('bias') is not None for m in plain[1]):
            return None
        w, _, norm = plain
        return _lib.host().layer_train(hidden_states, *w[:7], tuple(w[7:10]), self._parameters.get('A_log'), self._parameters.get('dt_bias'), w[10], norm.eps,
                                       self.allow_neg_eigval, self.num_heads)

    def _step(self, hidden_states, past_key_values):
        """One token per sequence on a filled cache through the native host path (``gdn_host.layer_step``: four launches), or None
        where the layer is not its plain self (``_plain``) or a state has to be converted."""
        if past_key_values is None or len(past_key_values) <= self.layer_idx:
            return None
        entry = past_key_values[self.layer_idx]
        state, conv = entry.get('recurrent_state'), entry.get('conv_state')
        if state is None or conv is None:
            return None
        plain = self._plain()
        if plain is None:
            return None
        weights, convs, norm = plain
        o = _lib.host().layer_step(
            hidden_states, *weights[:7], self._parameters.get('A_log'), self._parameters.get('dt_bias'), tuple(weights[7:10]),
            tuple(m._parameters['bias'] for m in convs), tuple(conv), state, weights[10], norm.eps, self.allow_neg_eigval, self.num_heads)
        if o is not None:
            past_key_values.update(layer_idx=self.layer_idx, recurrent_state=state, conv_state=conv, offset=1)
        return o

    def _forward(self, hidden_states, attention_mask, past_key_values, use_cache, **kwargs):
        if attention_mask is not None:
            assert attention_mask.dim() == 2, 'attention_mask must be a 0-1 matrix [batch_size, seq_len] (0 = padding)'
        if past_key_values is not None and self.layer_idx is None:
            raise ValueError(f'{self.__class__.__name__} requires `layer_idx` when `past_key_values` is provided.')
        batch_size, q_len, _ = hidden_states.shape
        mode = 'fused_recurrent' if (q_len <= 64 and not self.training) else self.mode
        if self.training and mode != 'chunk':
            raise AssertionError('Only chunk mode is supported in training.')

        if q_len == 1 and not self.training and use_cache and attention_mask is None and kwargs.get('cu_seqlens') is None:
            o = self._step(hidden_states, past_key_values)
            if o is not None:
                return o, None, past_key_values
        if self.training and past_key_values is None and not use_cache and attention_mask is None and kwargs.get('cu_seqlens') is None \
                and torch.is_grad_enabled():
            o = self._train(hidden_states)
            if o is not None:
                return o, None, None
        last_state = None
        if past_key_values is not None and len(past_key_values) > self.layer_idx:
            last_state = past_key_values[self.layer_idx]
        cu_seqlens, indices = kwargs.get('cu_seqlens'), None
        if cu_seqlens is None and attention_mask is not None:
            hidden_states, indices, cu_seqlens = _unpad(hidden_states, attention_mask, q_len)

        q, k, v = self.q_proj(hidden_states), self.k_proj(hidden_states), self.v_proj(hidden_states)
        conv_state = None
        if self.use_short_conv:
            cq, ck, cv = last_state['conv_state'] if last_state is not None and last_state.get('conv_state') is not None else (None,) * 3
            q, cq = self.q_conv1d(x=q, cache=cq, output_final_state=use_cache, cu_seqlens=cu_seqlens)
            k, ck = self.k_conv1d(x=k, cache=ck, output_final_state=use_cache, cu_seqlens=cu_seqlens)
            v, cv = self.v_conv1d(x=v, cache=cv, output_final_state=use_cache, cu_seqlens=cu_seqlens)
            conv_state = (cq, ck, cv)
        else:
            q, k, v = F.silu(q), F.silu(k), F.silu(v)
        q = q.unflatten(-1, (self.num_heads, self.head_k_dim))
        k = k.unflatten(-1, (self.num_heads, self.head_k_dim))
        v = v.unflatten(-1, (self.num_v_heads, self.head_v_dim))

        recurrent_state = last_state['recurrent_state'] if last_state is not None else None
        op = chunk_gated_delta_rule if mode == 'chunk' else fused_recurrent_gated_delta_rule
        extra = {}
        if (mode == 'fused_recurrent' and use_cache and recurrent_state is not None and recurrent_state.dtype == torch.float32
                and recurrent_state.is_contiguous()):
            # decode: the cached state is updated where it is - no allocation per step, and a step captured in a
            # HIP graph keeps reading and writing the same buffers on every replay
            extra['inplace_final_state'] = True
        o, recurrent_state = op(
            q=q, k=k, v=v, g=self.a_proj(hidden_states), beta=self.b_proj(hidden_states),
            A_log=self.A_log, dt_bias=self.dt_bias, initial_state=recurrent_state, output_final_state=use_cache,
            use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, use_beta_sigmoid_in_kernel=True,
            allow_neg_eigval=self.allow_neg_eigval, state_v_first=True, cu_seqlens=cu_seqlens, **extra)

        if past_key_values is not None:
            past_key_values.update(layer_idx=self.layer_idx, recurrent_state=recurrent_state,
                                   conv_state=conv_state if self.use_short_conv else None, offset=q_len)
        if self.use_gate:
            o = self.o_norm(o, self.g_proj(hidden_states).unflatten(-1, (self.num_v_heads, self.head_v_dim)))
        else:
            o = self.o_norm(o.float()).to(o.dtype)
        o = self.o_proj(o.flatten(-2))
        if indices is not None:                               # back to the padded [B, T, hidden] layout
            padded = o.new_zeros(batch_size * q_len, o.shape[-1])
            padded[indices] = o.squeeze(0)
            o = padded.view(batch_size, q_len, -1)
        return o, None, past_key_values
