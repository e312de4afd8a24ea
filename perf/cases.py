"""The work that users of this framework have it do, as cases that can be prepared, run and compared.

Five kinds of work, each through the public entry points that a user's program calls:
  decode       one token for each of N sequences on their states: fused_recurrent_gated_delta_rule
  prefill      prompts of any length, dense or packed: chunk_gated_delta_rule, forward
  train        a forward and backward pass of a chunked operator through autograd: chunk_gated_delta_rule, chunk_kda
  layer_step   one decode step of the whole GatedDeltaNet layer on a cache
  layer_train  a forward and backward pass of the whole layer

Two kinds of log decay occur.  "even": logsigmoid(N(0,1)) / 16 in every head, the benchmark's configurations.  "heads":
what the layer makes from its own initialisation, -exp(A_log) softplus(x + dt_bias) with a rate per head, so that some
heads forget within a chunk and others hardly at all."""
import importlib
import math
import random

import torch
import torch.nn.functional as F

importlib.import_module('flash-linear-attention_amd')
from fla_hip.layers import GatedDeltaNet  # noqa: E402
from fla_hip.layers.gated_deltanet import LayerCache  # noqa: E402
from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule  # noqa: E402
from fla_hip.ops.kda import chunk_kda  # noqa: E402

DTYPES = {'bf16': torch.bfloat16, 'f16': torch.float16}
CHUNK = 64
MOST_UNITS = 96 * 8192              # (token, value head) pairs of 128 x 128 state of the largest training step
MOST_PREFILL_UNITS = 32 * 65536     # ... and of the largest prefill


def listed():
    return [
        # One user, one token at a time, states handed on from call to call (as transformers calls the operator for a
        # Qwen3-Next style head shape: fp32 gates, bf16 betas, l2 norm inside).  4 MB of state: latency and host time.
        dict(name='decode_1', kind='decode', style='functional', N=1, H=16, HV=32, D=128, dtype='bf16', states='f32'),
        # The benchmark's decode step: 256 sequences, states updated in place, 1 GB of state traffic.
        dict(name='decode_256', kind='decode', style='inplace', N=256, H=16, HV=32, D=128, dtype='bf16', states='f32'),
        # A serving engine's step: the sequences of the moment are slots of a pool kept value-first, the gate and the
        # beta come as the projections leave them.
        dict(name='decode_pool_48', kind='decode', style='pool', N=48, H=16, HV=32, D=128, dtype='bf16', states='f32'),
        # A short question, of no round length, before the first token can be answered.
        dict(name='prefill_short', kind='prefill', B=1, T=333, seqs=0, H=16, HV=32, K=128, V=128, dtype='bf16', gates='heads', l2norm=True, h0=False),
        # One long document: the benchmark's default workload.
        dict(name='prefill_long', kind='prefill', B=1, T=32768, seqs=0, H=16, HV=32, K=128, V=128, dtype='bf16', gates='even', l2norm=False, h0=True),
        # Many prompts of different lengths packed into one call, each continuing a state: the benchmark's packed workload.
        dict(name='prefill_packed', kind='prefill', B=1, T=65536, seqs=32, H=16, HV=32, K=128, V=128, dtype='bf16', gates='even', l2norm=False, h0=True),
        # Training steps of the operator at published shapes of small and of wide heads ...
        dict(name='train_d64', kind='train', op='gdn', B=8, T=1024, seqs=0, H=8, HV=8, D=64, dtype='bf16', gates='even'),
        dict(name='train_d256', kind='train', op='gdn', B=8, T=2048, seqs=0, H=32, HV=32, D=256, dtype='bf16', gates='even'),
        # ... on packed documents with grouped value heads (fine-tuning), and of the operator with a decay per key feature.
        dict(name='train_packed', kind='train', op='gdn', B=1, T=16000, seqs=12, H=16, HV=32, D=128, dtype='bf16', gates='heads'),
        dict(name='train_kda', kind='train', op='kda', B=1, T=8192, seqs=0, H=96, HV=96, D=128, dtype='bf16', gates='even'),
        # The layer in its default size: a decode step of a small batch, and a training step.
        dict(name='layer_step_16', kind='layer_step', N=16, hidden=2048, heads=6, D=256, expand=2, dtype='bf16'),
        dict(name='layer_train', kind='layer_train', B=4, T=2048, hidden=2048, heads=6, D=256, expand=2, dtype='bf16'),
    ]


def _log_int(rng, lo, hi):
    """A whole number in [lo, hi], its logarithm spread evenly."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(['decode', 'prefill', 'train', 'layer_step', 'layer_train'], [3, 4, 4, 1, 1])[0]
    dtype = rng.choices(['bf16', 'f16'], [4, 1])[0]
    if kind == 'decode':
        HV = rng.choice([8, 16, 32])
        style = rng.choice(['functional', 'inplace', 'pool'])
        states = 'bf16' if style == 'inplace' and rng.random() < 0.25 else 'f32'
        return dict(kind=kind, style=style, N=_log_int(rng, 1, 256), H=HV // rng.choice([1, 2]), HV=HV, D=128, dtype=dtype, states=states)
    if kind == 'prefill':
        K, V = rng.choices([(64, 64), (128, 128), (256, 256), (256, 512)], [2, 6, 1, 1])[0]
        HV = rng.choice([4, 8, 16, 32])
        H = HV // rng.choice([1, 1, 2, 4])
        per_token = HV * max(1.0, K * V / 128 ** 2)
        packed = rng.random() < 0.4
        B = 1 if packed else rng.choice([1, 1, 2, 4, 8])
        T = _log_int(rng, 65, max(128, min(65536 if packed else 32768, int(MOST_PREFILL_UNITS / per_token / B))))
        seqs = _log_int(rng, 2, min(48, max(2, T // 40))) if packed else 0
        return dict(kind=kind, B=B, T=T, seqs=seqs, H=H, HV=HV, K=K, V=V, dtype=dtype, gates=rng.choice(['even', 'heads']),
                    l2norm=rng.random() < 0.6, h0=rng.random() < 0.5)
    if kind == 'train':
        op = rng.choices(['gdn', 'kda'], [3, 1])[0]
        D = 128 if op == 'kda' else rng.choices([64, 128, 256], [2, 4, 1])[0]
        HV = rng.choice([8, 16, 32, 64])
        H = HV // rng.choice([1, 1, 2])
        packed = rng.random() < 0.4
        B = 1 if packed else rng.choice([1, 2, 4, 8])
        # (wide heads: the listed 8 x 2048 tokens on 32 heads; others: 8192 tokens on 96 heads)
        most = 8 * 2048 * 32 * 3 // 4 if D == 256 else MOST_UNITS * 3 // 4
        T = _log_int(rng, 200, max(256, min(32768, most // (HV * B))))
        seqs = _log_int(rng, 2, min(32, max(2, T // 100))) if packed else 0
        return dict(kind=kind, op=op, B=B, T=T, seqs=seqs, H=H, HV=HV, D=D, dtype=dtype, gates=rng.choice(['even', 'heads']))
    shape = rng.choice([dict(hidden=2048, heads=6, D=256, expand=2), dict(hidden=1024, heads=4, D=256, expand=1), dict(hidden=1024, heads=8, D=128, expand=1)])
    if kind == 'layer_step':
        return dict(kind=kind, N=_log_int(rng, 1, 128), dtype='bf16', **shape)
    B = rng.choice([1, 2, 4])
    return dict(kind=kind, B=B, T=_log_int(rng, 200, 8192 // B), dtype='bf16', **shape)


def _boundaries(T, seqs):
    """T tokens in `seqs` sequences: lengths spread over a factor of sixteen, as prompts are (the same for every seed: they
    are part of the shape)."""
    r = random.Random(1000 * seqs + T)
    w = [r.uniform(1, 16) for _ in range(seqs)]
    lens = [max(1, int(T * x / sum(w))) for x in w]
    lens[lens.index(max(lens))] += T - sum(lens)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


def _gate(gen, kind, shape, HV, heads_dim=2):
    """Log decays in fp32; `heads_dim`: where the value heads are in `shape`."""
    x = torch.randn(shape, generator=gen, device='cuda')
    if kind == 'even':
        return F.logsigmoid(x) / 16
    rate = torch.rand(HV, generator=gen, device='cuda') * 16
    bias = torch.exp(torch.rand(HV, generator=gen, device='cuda') * math.log(100.0) + math.log(1e-3))
    bias = bias + torch.log(-torch.expm1(-bias))
    view = [1] * len(shape)
    view[heads_dim] = HV
    return -rate.view(view) * F.softplus(x + bias.view(view))


def _layer(case, seed):
    torch.manual_seed(seed)
    with torch.device('cuda'):
        layer = GatedDeltaNet(hidden_size=case['hidden'], expand_v=case['expand'], head_dim=case['D'], num_heads=case['heads'], layer_idx=0)
    return layer.to(DTYPES[case['dtype']])


def prepare(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(seed)
    dt = DTYPES[case['dtype']]

    def randn(*shape):
        return torch.randn(shape, generator=gen, device='cuda')

    s = dict(case=case)
    kind = case['kind']
    if kind == 'decode':
        N, H, HV, D = case['N'], case['H'], case['HV'], case['D']
        s.update(q=randn(N, 1, H, D).to(dt), k=randn(N, 1, H, D).to(dt), v=randn(N, 1, HV, D).to(dt))
        b = randn(N, 1, HV)
        state = 0.1 * randn(2 * N if case['style'] == 'pool' else N, HV, D, D)
        if case['style'] == 'pool':
            s.update(g=randn(N, 1, HV).to(dt), beta=b.to(dt), slots=torch.randperm(2 * N, generator=gen, device='cuda')[:N].to(torch.int32),
                     A_log=torch.log(torch.rand(HV, generator=gen, device='cuda') * 15.9 + 0.1), dt_bias=randn(HV) - 4)
        else:
            s.update(g=F.logsigmoid(randn(N, 1, HV)), beta=torch.sigmoid(b))
            if case['style'] == 'functional':
                s['beta'] = s['beta'].to(dt)
            else:               # the benchmark's step: rows normalised by the caller
                s['q'], s['k'] = (F.normalize(s[n].float(), dim=-1).to(dt) for n in 'qk')
        s['state'] = state.bfloat16() if case['states'] == 'bf16' else state
        return s
    if kind == 'prefill':
        B, T, H, HV, K, V = (case[n] for n in ('B', 'T', 'H', 'HV', 'K', 'V'))
        q, k = randn(B, T, H, K), randn(B, T, H, K)
        if not case['l2norm']:
            q, k = F.normalize(q, dim=-1), F.normalize(k, dim=-1)
        s.update(q=q.to(dt), k=k.to(dt), v=randn(B, T, HV, V).to(dt), g=_gate(gen, case['gates'], (B, T, HV), HV), beta=torch.sigmoid(randn(B, T, HV)))
        s.update(cu=None, cu_cpu=None)
        if case['seqs']:
            s['cu_cpu'] = torch.tensor(_boundaries(T, case['seqs']), dtype=torch.int64)
            s['cu'] = s['cu_cpu'].cuda()
        s['h0'] = 0.1 * randn(case['seqs'] or B, HV, K, V) if case['h0'] else None
        return s
    if kind == 'train':
        B, T, H, HV, D = (case[n] for n in ('B', 'T', 'H', 'HV', 'D'))
        leaves = dict(q=randn(B, T, H, D).to(dt), k=randn(B, T, H, D).to(dt), v=randn(B, T, HV, D).to(dt))
        if case['op'] == 'kda':
            leaves['g'] = F.logsigmoid(randn(B, T, HV, D)) / 4
            if case['gates'] == 'heads':
                leaves['g'] = leaves['g'] * (torch.rand(HV, 1, generator=gen, device='cuda') * 2)
        else:
            leaves['g'] = _gate(gen, case['gates'], (B, T, HV), HV)
        leaves['beta'] = torch.sigmoid(randn(B, T, HV))
        s['leaves'] = {n: x.requires_grad_(True) for n, x in leaves.items()}
        s['do'] = randn(B, T, HV, D).to(dt)
        s.update(cu=None, cu_cpu=None)
        if case['seqs']:
            s['cu_cpu'] = torch.tensor(_boundaries(T, case['seqs']), dtype=torch.int64)
            s['cu'] = s['cu_cpu'].cuda()
        return s
    s['layer'] = layer = _layer(case, seed)
    if kind == 'layer_step':
        N = case['N']
        layer.eval()
        s['x'] = randn(N, 1, case['hidden']).to(dt)
        s['cache'] = cache = LayerCache()
        conv = tuple(randn(N, d, layer.conv_size).to(dt) for d in (layer.key_dim, layer.key_dim, layer.value_dim))
        cache.update(layer_idx=0, recurrent_state=0.1 * randn(N, layer.num_v_heads, layer.head_v_dim, layer.head_k_dim), conv_state=conv)
        return s
    layer.train()
    s['x'] = randn(case['B'], case['T'], case['hidden']).to(dt).requires_grad_(True)
    s['dy'] = randn(case['B'], case['T'], case['hidden']).to(dt)
    return s


def run(s):
    case = s['case']
    kind = case['kind']
    if kind == 'decode':
        if case['style'] == 'functional':
            o, state = fused_recurrent_gated_delta_rule(s['q'], s['k'], s['v'], g=s['g'], beta=s['beta'], initial_state=s['state'],
                                                        output_final_state=True, use_qk_l2norm_in_kernel=True)
        elif case['style'] == 'inplace':
            o, state = fused_recurrent_gated_delta_rule(s['q'], s['k'], s['v'], s['g'], beta=s['beta'], initial_state=s['state'],
                                                        output_final_state=True, inplace_final_state=True)
        else:
            o, state = fused_recurrent_gated_delta_rule(
                s['q'], s['k'], s['v'], s['g'], beta=s['beta'], initial_state=s['state'], output_final_state=True,
                use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True, A_log=s['A_log'], dt_bias=s['dt_bias'],
                use_beta_sigmoid_in_kernel=True, state_v_first=True, inplace_final_state=True, ssm_state_indices=s['slots'])
        return dict(o=o, state=state)
    if kind == 'prefill':
        with torch.no_grad():
            o, state = chunk_gated_delta_rule(s['q'], s['k'], s['v'], s['g'], s['beta'], initial_state=s['h0'], output_final_state=True,
                                              use_qk_l2norm_in_kernel=case['l2norm'], cu_seqlens=s['cu'], cu_seqlens_cpu=s['cu_cpu'])
        return dict(o=o, state=state)
    if kind == 'train':
        leaves = s['leaves']
        op = chunk_kda if case['op'] == 'kda' else chunk_gated_delta_rule
        o, _ = op(leaves['q'], leaves['k'], leaves['v'], leaves['g'], leaves['beta'], use_qk_l2norm_in_kernel=True,
                  cu_seqlens=s['cu'], cu_seqlens_cpu=s['cu_cpu'])
        grads = torch.autograd.grad(o, list(leaves.values()), s['do'])
        return dict(o=o.detach(), **{'d' + n: g for n, g in zip(leaves, grads)})
    layer = s['layer']
    if kind == 'layer_step':
        o, _, cache = layer(s['x'], past_key_values=s['cache'], use_cache=True)
        return dict(o=o, recurrent=cache[0]['recurrent_state'], conv=cache[0]['conv_state'])
    o, _, _ = layer(s['x'])
    names, params = zip(*layer.named_parameters())
    grads = torch.autograd.grad(o, [s['x'], *params], s['dy'])
    return dict(o=o.detach(), dx=grads[0], grads=dict(zip(names, grads[1:])))


def _forward_flops(units, K, V):
    """Chunks of 64 tokens, per (token, value head): K K^T, q k^T, w; u, P v_new; w S, k^T v_new, q S."""
    return units * 2.0 * (3 * CHUNK * K + 2 * CHUNK * V + 3 * K * V)


def work(case):
    """Each input read once, each output written once; a backward pass costs each product of the forward two more."""
    kind, e = case['kind'], 2
    if kind == 'decode':
        N, H, HV, D = case['N'], case['H'], case['HV'], case['D']
        state = N * HV * D * D
        return dict(bytes=2 * state * (2 if case['states'] == 'bf16' else 4) + N * (2 * H * D + 2 * HV * D) * e + N * HV * 8, flops=7.0 * state)
    if kind == 'prefill':
        B, T, H, HV, K, V = (case[n] for n in ('B', 'T', 'H', 'HV', 'K', 'V'))
        states = (case['seqs'] or B) * HV * K * V * 4 * (2 if case['h0'] else 1)
        return dict(bytes=B * T * (2 * H * K * e + 2 * HV * V * e + 8 * HV) + states, flops=_forward_flops(B * T * HV, K, V))
    if kind == 'train':
        B, T, H, HV, D = (case[n] for n in ('B', 'T', 'H', 'HV', 'D'))
        gate = HV * (D if case['op'] == 'kda' else 1) * 4
        per_token = 2 * (2 * H * D * e + gate + 4 * HV) + 4 * HV * D * e         # q, k, g, beta and their gradients; v, do, o, dv
        return dict(bytes=B * T * per_token, flops=3 * _forward_flops(B * T * HV, D, D))
    hidden, heads, K = case['hidden'], case['heads'], case['D']
    V = K * case['expand']
    weights = hidden * heads * (2 * K + 3 * V + 2)
    channels = heads * (2 * K + V)
    if kind == 'layer_step':
        N = case['N']
        state = N * heads * K * V
        return dict(bytes=weights * e + 8 * state + 2 * N * channels * 4 * e + 2 * N * hidden * e, flops=2.0 * N * weights + 7.0 * state)
    tokens = case['B'] * case['T']
    return dict(bytes=2 * weights * e + 4 * tokens * hidden * e, flops=6.0 * tokens * weights + 3 * _forward_flops(tokens * heads, K, V))


def tolerance(case):
    """Operands and results of 16 bits, sums in fp32: about 1e-2.  The layer's gradients pass through eight such stages."""
    return dict(rel=2e-2) if case['kind'] == 'layer_train' else dict(rel=1e-2)
