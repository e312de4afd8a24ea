"""The backward's last kernel walks over (chunk, q/k head) items with one workgroup per CU (64 key features: two): more items than workgroups, counts that
wrap around heads, sequences and parts, chunks of every length among them."""
import pytest
import torch
import torch.nn.functional as F

from oracle import gdn_oracle as O


@pytest.mark.gpu
@pytest.mark.parametrize('B,T,H,HV,D,cu,dtype', [
    (3, 70, 43, 43, 128, None, torch.bfloat16),                             # 258 items on 256 workgroups, a sequence's second chunk of 6 tokens
    (2, 129, 90, 180, 128, None, torch.float16),                            # 540: three rounds, two value heads each
    (1, 300, 70, 70, 128, [0, 1, 65, 65, 190, 290], torch.bfloat16),        # packed, 1 .. 64 tokens a chunk, an empty sequence, tokens outside
    (5, 65, 53, 53, 64, None, torch.bfloat16),                              # 530 on 512
    (1, 200, 260, 260, 64, [3, 60, 61, 200], torch.float16),                # 1300, packed
    (1, 300, 140, 140, 256, [3, 66, 66, 67, 280], torch.bfloat16),          # 256 features: rows normalised a tile of q's at a time; tokens outside
    (2, 130, 43, 129, 256, None, torch.float16),                            # ... three value heads each, 258 items
    # groups in five parts (tests/test_chunk_bwd_parts.py), of which no round of workgroups is a multiple: from one item to the next the part wraps around, and with it head and chunk
    (1, 630, 10, 50, 128, None, torch.bfloat16),                            # 500 items on 256
    (1, 440, 10, 50, 128, [2, 70, 70, 71, 300, 430], torch.float16),        # ... packed
    (2, 310, 20, 100, 64, None, torch.float16),                             # 1000 items on 512
])
@pytest.mark.parametrize('l2', [False, True])
def test_more_items_than_workgroups(B, T, H, HV, D, cu, dtype, l2):
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule
    gen = torch.Generator().manual_seed(B + T)
    N = B if cu is None else len(cu) - 1
    q, k = (torch.randn(B, T, H, D, generator=gen) for _ in range(2))
    if not l2:
        q, k = F.normalize(q, dim=-1), F.normalize(k, dim=-1)
    q, k = q.to(dtype), k.to(dtype)
    v, do = (torch.randn(B, T, HV, D, generator=gen).to(dtype) for _ in range(2))
    g, beta = F.logsigmoid(torch.randn(B, T, HV, generator=gen)) / 2, torch.rand(B, T, HV, generator=gen)
    h0, dht = 0.5 * torch.randn(N, HV, D, D, generator=gen), torch.randn(N, HV, D, D, generator=gen)
    G = HV // H
    # (the oracle on heads apart from one another: the first, the last, and those where a round of workgroups ends)
    parts = 5 if G == 5 else 1
    heads = sorted({0, H - 1, *(i // parts % H for i in (255, 256, 511, 512))})
    vheads = [h * G + i for h in heads for i in range(G)]
    ref = O.gated_delta_rule_grads(q[:, :, heads], k[:, :, heads], v[:, :, vheads], g[:, :, vheads], beta[:, :, vheads], do[:, :, vheads], dht[:, vheads],
                                   initial_state=h0[:, vheads], cu_seqlens=cu, use_qk_l2norm_in_kernel=l2, dtype=torch.float32)
    leaves = {n: x.cuda().requires_grad_(True) for n, x in dict(dq=q, dk=k, dv=v, dg=g, dbeta=beta, dh0=h0).items()}
    o, ht = chunk_gated_delta_rule(*(leaves[n] for n in ('dq', 'dk', 'dv', 'dg', 'dbeta')), initial_state=leaves['dh0'], output_final_state=True,
                                   cu_seqlens=None if cu is None else torch.tensor(cu, device='cuda'), use_qk_l2norm_in_kernel=l2)
    torch.autograd.backward([o, ht], [do.cuda(), dht.cuda()])
    for n in leaves:
        x = leaves[n].grad.float().cpu()
        assert torch.isfinite(x).all(), n
        x = x[:, vheads] if n == 'dh0' else x[:, :, heads if n in ('dq', 'dk') else vheads]
        r = O.get_err_ratio(ref[n], x)                                       # operands of 16 bits, sums in fp32
        assert r <= (0.02 if n in ('dg', 'dbeta') else 0.008), f'{n}: rel-rmse {r:.3e}'
