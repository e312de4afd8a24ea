"""The training gradients of the chunked operators against 64 bits, in units of the operand type's rounding step: 16-bit operands, and every sum, decay and
weight held in 32 bits."""
import pytest
import torch
import torch.nn.functional as F

from oracle import gdn_oracle as O

# A rounding to 16 bits is off by 0.29 steps (rms of an even spread over one).  From the inputs to a gradient some eight such roundings follow one another (k, S, v_new, dS,
# dv_new, A, dw, the result), independent ones: sqrt(8) x 0.29 = 0.8 steps of the gradient.
# dg of a token is a sum over the tokens from there to the end of its chunk of (q . dq) - (k . dk), which cancel for the greater part where heads forget quickly; each
# carries what dq and dk carry, 0.8 steps of the root of the sum of their squares; in the last chunk, where the state's gradient comes from outside, of the products in <S, dS> too.
# (With a decay per feature the sums are per feature and cancel little: in steps of dg itself.)  The others' 0.8 is a mean over thousands of errors, its bar twice that less a
# little; dg's largest part is one number a chunk and head, a dozen draws here: three times 0.8.
BARS = dict(dq=1.5, dk=1.5, dv=1.5, dg=2.4, dbeta=1.5, dh0=1.5)


def _cancelling(q, k, grads, ht, dht):
    """Norm, over tokens and heads, of the terms that dg adds up."""
    x = (q.double() * grads['dq']).sum(-1) ** 2 + (k.double() * grads['dk']).sum(-1) ** 2
    T = x.shape[1]
    last = (T - 1) % 64 + 1
    return (sum(x[:, i:i + 64].flip(1).cumsum(1).sum() for i in range(0, T, 64)) + last * ((ht * dht).double() ** 2).sum()).sqrt()


@pytest.mark.gpu
@pytest.mark.parametrize('op,H,D,gates', [
    ('gdn', 4, 64, 'even'), ('gdn', 4, 64, 'heads'), ('gdn', 4, 128, 'even'), ('gdn', 4, 128, 'heads'), ('gdn', 2, 256, 'even'), ('gdn', 2, 256, 'heads'),
    ('kda', 3, 128, 1 / 16), ('kda', 3, 128, 1.0), ('kda', 3, 128, 30.0),       # (30: blocks of 16 rows decay beyond what a 16-bit factor holds)
])
@pytest.mark.parametrize('dtype,step', [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize('l2', [False, True])
def test_gradients_are_as_exact_as_their_operands(op, H, D, gates, dtype, step, l2):
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule
    from fla_hip.ops.kda import chunk_kda
    T = 333
    gen = torch.Generator().manual_seed(D + H)
    rn = lambda *s: torch.randn(*s, generator=gen)
    q, k = rn(1, T, H, D), rn(1, T, H, D)
    if not l2:
        q, k = F.normalize(q, dim=-1), F.normalize(k, dim=-1)
    q, k, v, do = q.to(dtype), k.to(dtype), rn(1, T, H, D).to(dtype), rn(1, T, H, D).to(dtype)
    if op == 'kda':
        g = F.logsigmoid(rn(1, T, H, D)) * gates
    else:       # 'heads': from heads that hardly forget to heads that forget within a few tokens
        g = F.logsigmoid(rn(1, T, H)) / 16 * (1.0 if gates == 'even' else torch.logspace(-1, 1.5, H))
    beta, h0, dht = torch.rand(1, T, H, generator=gen), 0.3 * rn(1, H, D, D), rn(1, H, D, D)
    ref = (O.kda_grads if op == 'kda' else O.gated_delta_rule_grads)(q, k, v, g, beta, do, dht, initial_state=h0, use_qk_l2norm_in_kernel=l2, dtype=torch.float64)
    leaves = {n: x.cuda().requires_grad_(True) for n, x in dict(dq=q, dk=k, dv=v, dg=g, dbeta=beta, dh0=h0).items()}
    o, ht = (chunk_kda if op == 'kda' else chunk_gated_delta_rule)(*(leaves[n] for n in ('dq', 'dk', 'dv', 'dg', 'dbeta')), initial_state=leaves['dh0'],
                                                                   output_final_state=True, use_qk_l2norm_in_kernel=l2)
    torch.autograd.backward([o, ht], [do.cuda(), dht.cuda()])
    norms = {n: x.norm() for n, x in ref.items() if x is not None}
    if op == 'gdn':
        qn, kn = (O.l2norm(q.double()), O.l2norm(k.double())) if l2 else (q, k)
        norms['dg'] = _cancelling(qn, kn, O.gated_delta_rule_grads(qn, kn, v, g, beta, do, dht, initial_state=h0, dtype=torch.float64), ht.detach().cpu(), dht)
    off = {n: float((x.grad.cpu().double() - ref[n]).norm() / norms[n]) / step for n, x in leaves.items()}
    print({n: round(x, 2) for n, x in off.items()})
    assert all(off[n] <= bar for n, bar in BARS.items()), off
