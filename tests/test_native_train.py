"""The native training path against the Python path behind it: the operator (same kernels, same bits), the layer (one product for the
projections instead of six: same numbers up to rounding), and the kernels of its backward - the gate's, the sums of partial rows, runs
of the convolution that end inside a sequence."""
import contextlib

import pytest
import torch
import torch.nn.functional as F

from oracle import gdn_oracle as O
from oracle import modules_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('K,V,H,HV,cu,raw', [(128, 128, 2, 4, None, False), (64, 64, 3, 3, [0, 5, 70, 70, 190], True), (256, 384, 1, 2, None, True),
                                             (128, 128, 2, 2, [10, 100, 180], True)])
def test_operator_gives_the_python_path_s_bits(K, V, H, HV, cu, raw):
    from fla_hip.ops.gated_delta_rule import chunk as C
    from fla_hip.ops.gated_delta_rule.chunk_bwd import ChunkGatedDeltaRuleFunction
    gen = torch.Generator(device='cuda').manual_seed(K)
    B, T = (2, 190) if cu is None else (1, 190)
    N = B if cu is None else len(cu) - 1
    rn = lambda *s: torch.randn(*s, generator=gen, device='cuda')
    x = [rn(B, T, H, K).bfloat16(), rn(B, T, H, K).bfloat16(), rn(B, T, HV, V).bfloat16(), rn(B, T, HV), rn(B, T, HV).bfloat16(), rn(N, HV, V, K)]
    gate = (torch.rand(HV, generator=gen, device='cuda'), rn(HV)) if raw else (None, None)
    if not raw:
        x[3], x[4] = F.logsigmoid(x[3]), x[4].sigmoid()
    cu_t = None if cu is None else torch.tensor(cu, device='cuda')
    do, dht = rn(B, T, HV, V).bfloat16(), rn(N, HV, V, K)
    out = []
    for native in (True, False):
        q, k, v, g, beta, h0 = leaves = [t.clone().requires_grad_(True) for t in x]
        A, dt = (t.clone().requires_grad_(True) if t is not None else None for t in gate)
        if native:
            o, ht = C._native_fwd(q, k, v, g, beta, 0.1, h0, True, True, cu_t, None, A, dt, True, raw, raw, train=True)
        else:
            o, ht = ChunkGatedDeltaRuleFunction.apply(q, k, v, g, beta, 0.1, h0, True, True, cu_t, None, None, True, raw, A, dt, raw, raw, 64)
        ins = leaves + ([A, dt] if raw else [])
        inside = slice(None) if cu is None else slice(cu[0], cu[-1])
        out.append((o[:, inside], ht, *torch.autograd.grad([o, ht], ins, [do, dht])))
    for i, (a, b) in enumerate(zip(*out)):
        if i < 8:
            assert torch.equal(a, b), f'output {i}'
        else:
            assert O.get_err_ratio(b, a) < 1e-5, f'output {i}'


@pytest.mark.parametrize('B,T,hidden,heads,D,expand,HV,neg', [(2, 130, 256, 2, 64, 1, 2, False), (1, 65, 1024, 2, 256, 2, 4, True), (1, 700, 256, 3, 128, 1, 3, False)])
def test_layer_against_its_parts(B, T, hidden, heads, D, expand, HV, neg):
    from fla_hip.layers import GatedDeltaNet
    torch.manual_seed(1)
    layer = GatedDeltaNet(hidden_size=hidden, expand_v=expand, head_dim=D, num_heads=heads, num_v_heads=HV, allow_neg_eigval=neg).cuda().bfloat16().train()
    x = torch.randn(B, T, hidden, device='cuda').bfloat16().requires_grad_(True)
    dy = torch.randn(B, T, hidden, device='cuda').bfloat16()
    names, params = zip(*layer.named_parameters())
    assert layer._train(x) is not None
    native = (layer(x)[0], *torch.autograd.grad(layer(x)[0], [x, *params], dy))
    hook = layer.q_proj.register_forward_hook(lambda *a: None)           # (a hooked projection: the layer goes through its modules)
    assert layer._train(x) is None
    parts = (layer(x)[0], *torch.autograd.grad(layer(x)[0], [x, *params], dy))
    hook.remove()
    for name, a, b in zip(('o', 'dx', *names), native, parts):
        assert a.shape == b.shape and a.dtype == b.dtype
        # (the gate parameters' gradients are sums over all tokens of products of rounded factors)
        assert O.get_err_ratio(b.float(), a.float()) < (3e-2 if name in ('A_log', 'dt_bias') else 1.2e-2), name


@pytest.mark.parametrize('rows,HV,beta_max', [(1, 1, 1.0), (333, 6, 2.0), (700, 300, 0.0)])
def test_gate_backward(rows, HV, beta_max):
    from fla_hip.ops.gated_delta_rule.chunk_bwd import gate_bwd
    gen = torch.Generator().manual_seed(rows)
    rn = lambda *s: torch.randn(*s, generator=gen)
    g, b, A, dt, dg, db = rn(1, rows, HV), rn(1, rows, HV).bfloat16(), rn(HV) * 0.3, rn(HV), rn(1, rows, HV), rn(1, rows, HV)
    leaves = [t.double().requires_grad_(True) for t in (g, b, A, dt)]
    gate = -leaves[2].exp() * F.softplus(leaves[0] + leaves[3])
    beta = leaves[1].sigmoid() * beta_max if beta_max else leaves[1] * 1
    ref = torch.autograd.grad([gate, beta], leaves, [dg.double(), db.double()])
    out = gate_bwd(dg.cuda(), db.cuda(), g.cuda(), b.cuda(), A.cuda(), dt.cuda(), beta_max)
    sums = out[2].double().sum(0).cpu()
    for r, o, bar in ((ref[0], out[0], 1e-5), (ref[1], out[1], 4e-3), (ref[2], sums[0], 1e-4), (ref[3], sums[1], 1e-4)):
        assert O.get_err_ratio(r, o.double().cpu()) < bar


@pytest.mark.parametrize('what', ['operator', 'layer'])
def test_saved_tensors_may_come_back_in_another_layout_and_place(what):
    """Saved-tensor hooks: every tensor goes to the host and comes back strided, in fp32 where it was of 16 bits."""
    from fla_hip.layers import GatedDeltaNet
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule
    gen = torch.Generator(device='cuda').manual_seed(2)
    rn = lambda *s: torch.randn(*s, generator=gen, device='cuda')
    if what == 'operator':
        leaves = [rn(1, 130, 2, 128).bfloat16(), rn(1, 130, 2, 128).bfloat16(), rn(1, 130, 4, 128).bfloat16(), rn(1, 130, 4), rn(1, 130, 4).bfloat16(),
                  rn(2, 4, 128, 128), rn(4), rn(4)]
        leaves = [x.requires_grad_() for x in leaves]
        cu = torch.tensor([0, 60, 130], device='cuda')
        call = lambda: chunk_gated_delta_rule(*leaves[:5], initial_state=leaves[5], cu_seqlens=cu, use_qk_l2norm_in_kernel=True, use_gate_in_kernel=True,
                                              A_log=leaves[6], dt_bias=leaves[7], use_beta_sigmoid_in_kernel=True)[0]
    else:
        torch.manual_seed(3)
        layer = GatedDeltaNet(hidden_size=256, head_dim=64, expand_v=1, num_heads=4).cuda().bfloat16().train()
        x = rn(1, 130, 256).bfloat16().requires_grad_()
        leaves = [x, *layer.parameters()]
        call = lambda: layer(x)[0]

    def unpack(x):
        x = x.cuda()
        if x.dtype == torch.bfloat16:
            x = x.float()
        return torch.stack([x, torch.zeros_like(x)], -1)[..., 0]

    def grads(*hooks):
        with torch.autograd.graph.saved_tensors_hooks(*hooks) if hooks else contextlib.nullcontext():
            o = call()
        return torch.autograd.grad(o, leaves, torch.ones_like(o))
    for i, (a, b) in enumerate(zip(grads(), grads(lambda x: x.cpu(), unpack))):
        assert a.dtype == b.dtype and O.get_err_ratio(a.float(), b.float()) < 1e-3, f'gradient {i}'


def _layer_in_float64(layer, x, dy):
    """The layer's output and gradients by the oracle, from its (16-bit) weights and input in 64 bits."""
    p = {n: t.detach().double().cpu().requires_grad_(True) for n, t in layer.named_parameters()}
    xd = x.detach().double().cpu().requires_grad_(True)
    B, T, _ = xd.shape
    heads = dict(q=layer.num_heads, k=layer.num_heads, v=layer.num_v_heads)
    q, k, v = (M.causal_conv1d(xd @ p[f'{n}_proj.weight'].t(), p[f'{n}_conv1d.weight'].squeeze(1), activation='silu', dtype=torch.float64)[0]
               .view(B, T, h, -1) for n, h in heads.items())
    o, _ = O.recurrent_gated_delta_rule(q, k, v, xd @ p['a_proj.weight'].t(), xd @ p['b_proj.weight'].t(), use_qk_l2norm_in_kernel=True,
                                        use_gate_in_kernel=True, A_log=p['A_log'], dt_bias=p['dt_bias'], use_beta_sigmoid_in_kernel=True,
                                        allow_neg_eigval=layer.allow_neg_eigval, dtype=torch.float64)
    gate = (xd @ p['g_proj.weight'].t()).view(o.shape)
    y = M.norm_gated(o.reshape(-1, o.shape[-1]), gate.reshape(-1, o.shape[-1]), p['o_norm.weight'], eps=layer.o_norm.eps, is_rms_norm=True,
                     dtype=torch.float64)[0]
    out = y.view(B, T, -1) @ p['o_proj.weight'].t()
    return (out.detach(), *torch.autograd.grad(out, [xd, *p.values()], dy.double().cpu()))


@pytest.mark.parametrize('B,T,hidden,heads,D,expand,HV,neg', [(2, 130, 256, 2, 64, 1, 2, False), (1, 65, 1024, 2, 256, 2, 4, True), (1, 300, 256, 3, 128, 1, 3, False)])
def test_layer_against_float64(B, T, hidden, heads, D, expand, HV, neg):
    """Output and gradients of the native step, and of the same step module by module, against 64 bits."""
    from fla_hip.layers import GatedDeltaNet
    torch.manual_seed(1)
    layer = GatedDeltaNet(hidden_size=hidden, expand_v=expand, head_dim=D, num_heads=heads, num_v_heads=HV, allow_neg_eigval=neg).cuda().bfloat16().train()
    x = torch.randn(B, T, hidden, device='cuda').bfloat16().requires_grad_(True)
    dy = torch.randn(B, T, hidden, device='cuda').bfloat16()
    names, params = zip(*layer.named_parameters())

    def step():
        o = layer(x)[0]
        return [t.double().cpu() for t in (o, *torch.autograd.grad(o, [x, *params], dy))]
    ref = _layer_in_float64(layer, x, dy)
    assert layer._train(x) is not None
    native = step()
    hook = layer.q_proj.register_forward_hook(lambda *a: None)
    parts = step()
    hook.remove()
    for name, r, a, b in zip(('o', 'dx', *names), ref, native, parts):
        # A value rounded to bf16 is off by 2^-9 / sqrt(3) = 1.1e-3 on average, and a gradient passes through some twenty such roundings
        # in a row (the layer's eight stages and the chunked operator's operands): 5e-3, twice that allowed.  The gradients of A_log and
        # dt_bias are sums over all tokens of terms of both signs: twice that again.
        native_err, parts_err = O.get_err_ratio(r, a), O.get_err_ratio(r, b)
        assert native_err < (2e-2 if name in ('A_log', 'dt_bias') else 1e-2), f'{name}: {native_err:.2e}'
        assert native_err < 1.05 * parts_err, f'{name}: {native_err:.2e}, module by module {parts_err:.2e}'
