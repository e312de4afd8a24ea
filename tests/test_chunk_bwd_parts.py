"""The backward where a q/k head's value heads (or a wide head's blocks of value columns) are dealt out to several workgroups, whose rows of
dq and dk and sums of dg and dbeta are added up in fp32."""
import pytest
import torch
import torch.nn.functional as F

from oracle import gdn_oracle as O


@pytest.mark.parametrize('num_chunks,H,HV,K,V,parts', [
    (16, 2, 16, 128, 128, 8),                   # 32 workgroups' worth of chunks: a value head each
    (32, 4, 32, 128, 128, 2),                   # half the chip: two workgroups a group fill it
    (4, 16, 32, 128, 128, 1),                   # one head saved is not worth a launch in a call this short
    (4, 2, 16, 128, 128, 8),
    (32, 8, 32, 128, 128, 1),                   # enough as it is
    (16, 2, 16, 64, 64, 8),
    (4, 6, 6, 256, 512, 4),                     # the blocks of a head apart: dg and dbeta in four parts as well
    (4, 3, 6, 128, 384, 6),
    (64, 2, 4, 128, 128, 1),                    # two parts would fill the chip: fp32 rows cost as much as the head saved
    (16, 16, 32, 64, 64, 1),
    (32, 4, 4, 256, 256, 2),                    # ... not at 256 features
    (12, 10, 30, 128, 128, 1),
    (10, 10, 50, 128, 128, 5),                  # more than fill it (tests/test_chunk_bwd_items.py)
    (10, 20, 100, 64, 64, 5),
])
def test_parts_are_reserved_in_the_workspace(num_chunks, H, HV, K, V, parts):
    from fla_hip import _lib
    ws = _lib.load().gdn_chunk_bwd_heads_workspace_bytes
    tokens, align = 64 * num_chunks - 5, lambda n: (n + 255) // 256 * 256
    nb = V // (64 if K == 64 else 128)
    units = num_chunks * HV
    plain = sum(map(align, (units * 256, units * 256, units * 8192, units * 8192, *[units * nb * 128 * (V // nb)] * 2,
                            *[units * nb * K * (V // nb) * 2] * 2, units * 4)))
    split = max(1, nb * parts // (HV // H * nb))
    want = 0 if parts == 1 else 2 * align(tokens * H * parts * K * 4) + (2 * align(tokens * HV * split * 4) if split > 1 else 0)
    assert ws(num_chunks, H, HV, K, V, tokens, 0) - plain == want


@pytest.mark.gpu
@pytest.mark.parametrize('B,T,H,HV,K,V,cu,dtype', [
    (1, 1024, 2, 16, 128, 128, None, torch.bfloat16),
    (2, 70, 1, 6, 64, 64, None, torch.bfloat16),
    (1, 500, 1, 6, 128, 256, [7, 20, 20, 300, 480], torch.float16),      # tokens outside, an empty sequence, ragged chunks
    (2, 70, 2, 2, 256, 512, None, torch.bfloat16),                       # parts of one value head
    (1, 300, 2, 4, 256, 256, None, torch.float16),
])
@pytest.mark.parametrize('l2', [False, True])
def test_parts_against_the_oracle(B, T, H, HV, K, V, cu, dtype, l2):
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule
    gen = torch.Generator().manual_seed(5)
    N = B if cu is None else len(cu) - 1
    q, k = (torch.randn(B, T, H, K, generator=gen) for _ in range(2))
    if not l2:
        q, k = F.normalize(q, dim=-1), F.normalize(k, dim=-1)
    q, k = q.to(dtype), k.to(dtype)
    v, do = (torch.randn(B, T, HV, V, generator=gen).to(dtype) for _ in range(2))
    g, beta = F.logsigmoid(torch.randn(B, T, HV, generator=gen)) / 2, torch.rand(B, T, HV, generator=gen)
    h0, dht = 0.5 * torch.randn(N, HV, K, V, generator=gen), torch.randn(N, HV, K, V, generator=gen)
    ref = O.gated_delta_rule_grads(q, k, v, g, beta, do, dht, initial_state=h0, cu_seqlens=cu, use_qk_l2norm_in_kernel=l2, dtype=torch.float32)
    runs = []
    for _ in range(2):
        leaves = {n: x.cuda().requires_grad_(True) for n, x in dict(dq=q, dk=k, dv=v, dg=g, dbeta=beta, dh0=h0).items()}
        o, ht = chunk_gated_delta_rule(*(leaves[n] for n in ('dq', 'dk', 'dv', 'dg', 'dbeta')), initial_state=leaves['dh0'], output_final_state=True,
                                       cu_seqlens=None if cu is None else torch.tensor(cu, device='cuda'), use_qk_l2norm_in_kernel=l2)
        torch.autograd.backward([o, ht], [do.cuda(), dht.cuda()])
        runs.append({n: x.grad for n, x in leaves.items()})
    inside = slice(None) if cu is None else slice(cu[0], cu[-1])
    # (bars: those of the same kernels with all heads in one workgroup, tests/test_chunk_bwd_grouped.py)
    for n, bar in dict(dq=0.008, dk=0.008, dv=0.008, dg=0.02, dbeta=0.02, dh0=0.008).items():
        got = runs[0][n]
        assert torch.equal(got, runs[1][n]), f'{n}: two runs differ'
        if cu is not None and n != 'dh0':
            assert not got[:, :cu[0]].any() and not got[:, cu[-1]:].any(), f'{n}: tokens outside every sequence'
        at = (lambda x: x) if n == 'dh0' else lambda x: x[:, inside]
        err = O.get_err_ratio(at(ref[n]), at(got.float().cpu()))
        assert err <= bar, f'{n}: rel-rmse {err:.3e}'


@pytest.mark.gpu
def test_a_workspace_without_room_for_parts_is_enough():
    """The C entry with the workspace of the call's other arrays alone: all heads of a group in one workgroup, the same gradients."""
    from fla_hip import _lib
    lib = _lib.load()
    B, T, H, HV, D = 1, 300, 2, 8, 128
    nc = 5
    gen = torch.Generator(device='cuda').manual_seed(7)
    rn = lambda *s: torch.randn(*s, generator=gen, device='cuda')
    q, k = (F.normalize(rn(B, T, H, D), dim=-1).bfloat16() for _ in range(2))
    v, do = rn(B, T, HV, D).bfloat16(), rn(B, T, HV, D).bfloat16()
    g, beta = F.logsigmoid(rn(B, T, HV)), rn(B, T, HV).sigmoid()
    full, least = (lib.gdn_chunk_bwd_heads_workspace_bytes(nc, h, HV, D, D, B * T, 0) for h in (H, HV))
    assert full > least
    out = []
    for size, status in ((full, 0), (least, 0), (least - 256, _lib.GDN_ERR_WORKSPACE)):
        ws = torch.empty(size, dtype=torch.uint8, device='cuda')
        grads = [torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v), torch.zeros_like(g), torch.zeros_like(beta)]
        rc = lib.gdn_chunk_bwd_heads(
            *(x.data_ptr() for x in (q, k, v, g, beta)), None, None, None, do.data_ptr(), None, *(x.data_ptr() for x in grads), None,
            None, None, None, ws.data_ptr(), size, B, T, H, HV, D, D, B, nc, D ** -0.5, _lib.DTYPE_BF16, _lib.DTYPE_F32, 0,
            torch.cuda.current_stream().cuda_stream)
        assert rc == status
        out.append(grads)
    # (dq and dk: the same fp32 sums in another order, each rounded to bf16 once; the rest: the same bits)
    for a, b, bar in zip(out[0], out[1], (1e-3, 1e-3, 0, 0, 0)):
        assert (torch.equal(a, b) if bar == 0 else O.get_err_ratio(b.float(), a.float()) < bar)
