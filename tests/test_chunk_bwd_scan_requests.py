"""The backward scans at 128 and 256 key features ask for the next chunk's tiles in two ways, by the sequences' average length (eight chunks at 128 features, sixteen in
the gated form beyond 64 runs; 256 features four up to 32 runs, 32 with 64 columns beyond 64): the same bits either way, at every split of the value columns, with sequences of one token, of no token and of ragged ends among them."""
import pytest
import torch
import torch.nn.functional as F


def _grads(op, x, do, cu, h0, dht):
    from fla_hip.ops.comba import chunk_comba
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule
    from fla_hip.ops.kda import chunk_kda
    leaves = [t.detach().requires_grad_(True) for t in (*x, h0)]
    o, ht = dict(gdn=chunk_gated_delta_rule, kda=chunk_kda, comba=chunk_comba)[op](*leaves[:-1], initial_state=leaves[-1], output_final_state=True, use_qk_l2norm_in_kernel=True,
                                                       cu_seqlens=torch.tensor(cu, device='cuda'))
    return torch.autograd.grad([o, ht], leaves, [do, dht])


@pytest.mark.gpu
@pytest.mark.parametrize('op,D,H', [(op, 128, H) for op in ('gdn', 'kda', 'comba') for H in (2, 10, 14, 26)]       # 10, 50, 70 and 130 runs: 32, 64, 128 and 64, 128 value columns to a workgroup
                         + [('gdn', 256, 2), ('gdn', 256, 9)])                                                      # 20 and 90 runs: 32, 64
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
def test_both_ways_of_asking_give_the_same_bits(op, D, H, dtype):
    # 1, 2, 0, 13 chunks and as many more as make the average, in five sequences
    chunks = 5 * ((32 if H == 9 else 4) if D == 256 else 16 if op == 'gdn' and H > 12 else 8)
    cu = [3, 4, 69, 69, 900, 880 + 64 * (chunks - 16)]
    T, N = cu[-1] + 4, 5
    gen = torch.Generator(device='cuda').manual_seed(H)
    rn = lambda *s: torch.randn(*s, generator=gen, device='cuda')
    q, k, p, v, do = (rn(1, T, H, D).to(dtype) for _ in range(5))
    g = F.logsigmoid(rn(1, T, H, D) if op == 'kda' else rn(1, T, H)) / 4
    beta = rn(1, T, H).sigmoid()
    h0, dht = 0.3 * rn(N + 1, H, D, D), rn(N + 1, H, D, D)
    x = (q, k, p, v, g, beta) if op == 'comba' else (q, k, v, g, beta)
    ahead = _grads(op, x, do, cu, h0[:N], dht[:N])
    # (a sixth sequence, without tokens: fewer chunks on average)
    masked = _grads(op, x, do, [*cu, cu[-1]], h0, dht)
    for n, a, b in zip(('q', 'k', *('p' if op == 'comba' else []), 'v', 'g', 'beta', 'h0'), ahead, masked):
        assert torch.isfinite(a).all(), n
        assert torch.equal(a, b[:N] if n == 'h0' else b), n
