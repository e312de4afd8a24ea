"""The backward's chunk-parallel kernel with the l2 normalisation of q and k inside where value heads share a q/k head (one to four of
them, and head dims above 128, whose value columns count as heads) and the two scans in one launch with the longest sequence first."""
import pytest
import torch
import torch.nn.functional as F

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,T,H,HV,K,V,cu,dtype', [
    (1, 130, 2, 4, 128, 128, None, torch.bfloat16),
    (1, 200, 1, 4, 96, 128, [0, 1, 1, 130, 200], torch.float16),        # one token, an empty sequence, the longest in the middle
    (2, 65, 1, 1, 256, 256, None, torch.bfloat16),
    (1, 190, 1, 3, 200, 160, [0, 63, 190], torch.bfloat16),
    (3, 64, 50, 50, 128, 128, None, torch.bfloat16),                    # 150 runs: more workgroups than CUs in the launch of the scans
    (1, 500, 36, 72, 64, 64, [0, 20, 300, 500], torch.bfloat16),
])
def test_grouped_backward_with_l2norm(B, T, H, HV, K, V, cu, dtype):
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule
    gen = torch.Generator().manual_seed(11)
    N = B if cu is None else len(cu) - 1
    q, k = (torch.randn(B, T, H, K, generator=gen).to(dtype) for _ in range(2))
    v, do = (torch.randn(B, T, HV, V, generator=gen).to(dtype) for _ in range(2))
    g, beta = F.logsigmoid(torch.randn(B, T, HV, generator=gen)) / 2, torch.rand(B, T, HV, generator=gen)
    h0, dht = 0.5 * torch.randn(N, HV, K, V, generator=gen), torch.randn(N, HV, K, V, generator=gen)
    ref = O.gated_delta_rule_grads(q, k, v, g, beta, do, dht, initial_state=h0, cu_seqlens=cu, use_qk_l2norm_in_kernel=True, dtype=torch.float32)
    leaves = {n: x.cuda().requires_grad_(True) for n, x in dict(dq=q, dk=k, dv=v, dg=g, dbeta=beta, dh0=h0).items()}
    o, ht = chunk_gated_delta_rule(*(leaves[n] for n in ('dq', 'dk', 'dv', 'dg', 'dbeta')), initial_state=leaves['dh0'], output_final_state=True,
                                   cu_seqlens=None if cu is None else torch.tensor(cu, device='cuda'), use_qk_l2norm_in_kernel=True)
    torch.autograd.backward([o, ht], [do.cuda(), dht.cuda()])
    for n, bar in dict(dq=0.008, dk=0.008, dv=0.008, dg=0.02, dbeta=0.02, dh0=0.008).items():
        err = O.get_err_ratio(ref[n], leaves[n].grad.float().cpu())
        assert err <= bar, f'{n}: rel-rmse {err:.3e}'
