"""The native host path and the decode kernels behind it: blocks of 32 (16) value columns at the edges of their range, gates and betas of
different types, and the same bits as the general Python path where both can run a call."""
import pytest
import torch

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N,T,H,HV,K,V,vfirst', [
    (1, 1, 1, 1, 128, 32, False), (1, 1, 1, 1, 128, 32, True), (1, 3, 16, 32, 128, 128, True), (70, 1, 16, 32, 128, 128, True),
    (70, 1, 16, 32, 128, 128, False), (2, 2, 2, 4, 256, 96, False), (3, 1, 6, 6, 256, 512, True), (20, 1, 6, 6, 256, 512, True)])
def test_decode_blocks(N, T, H, HV, K, V, vfirst):
    from fla_hip.ops.gated_delta_rule import fused_recurrent_gated_delta_rule
    q, k, v, g, beta, h0 = O.make_inputs(N, T, H, HV, K, V, seed=N + K, gate_div=2.0, h0_std=0.3, dtype=torch.bfloat16)
    beta = beta.bfloat16()
    ref_o, ref_h = O.recurrent_gated_delta_rule(q, k, v, g, beta.float(), None, h0, True)
    h = h0.transpose(-1, -2).contiguous() if vfirst else h0.clone()
    o, ht = fused_recurrent_gated_delta_rule(q.cuda(), k.cuda(), v.cuda(), g.cuda(), beta=beta.cuda(), initial_state=h.cuda(),
                                             output_final_state=True, state_v_first=vfirst)
    ht = ht.transpose(-1, -2) if vfirst else ht
    assert O.get_err_ratio(ref_o, o.float().cpu()) < 5e-3
    assert O.get_err_ratio(ref_h, ht.cpu()) < 1e-5


@pytest.mark.parametrize('cu', [None, [0, 5, 70, 70, 200]])
def test_native_path_gives_the_general_path_s_bits(cu):
    from fla_hip.ops.gated_delta_rule import chunk as C
    from fla_hip.ops.gated_delta_rule import fused_recurrent as R
    N = 2 if cu is None else len(cu) - 1
    q, k, v, g, beta, h0 = (x.cuda() for x in O.make_inputs(2 if cu is None else 1, 200, 2, 4, 128, 128, seed=3, gate_div=4.0, h0_std=0.3, N=N,
                                                            dtype=torch.bfloat16))
    cu_t = None if cu is None else torch.tensor(cu, device='cuda', dtype=torch.int32)
    args = (q, k, v, g, beta, 0.1, h0, True, False, cu_t)
    kw = dict(use_qk_l2norm_in_kernel=True)
    native = C._native_fwd(*args, None, None, None, True, False, False)
    assert native is not None
    general = C._chunk_fwd_general(*args, **kw)
    assert all(torch.equal(a, b) for a, b in zip(native, general))
    rargs = (q, k, v, g, None, None, beta, None, None, 0.1, h0, True)
    native, general = R.fused_recurrent_gated_delta_rule_fwd(*rargs, cu_seqlens=cu_t, **kw), R._fused_recurrent_general(*rargs, cu_seqlens=cu_t, **kw)
    assert all(torch.equal(a, b) for a, b in zip(native, general))


@pytest.mark.parametrize('N,hidden,heads,v_heads,D,expand,conv,neg', [
    (1, 256, 2, 2, 128, 1, 4, False), (3, 512, 2, 4, 128, 2, 3, True), (16, 2048, 6, 6, 256, 2, 4, False), (17, 1024, 4, 4, 256, 1, 4, False),
    (33, 1024, 8, 8, 128, 1, 4, True), (65, 512, 4, 4, 64, 1, 4, False), (128, 512, 4, 4, 128, 1, 2, False)])
def test_layer_step_in_four_launches(N, hidden, heads, v_heads, D, expand, conv, neg, monkeypatch, dtype=torch.bfloat16):
    """The native decode step of the layer against the same step module by module: output and every state, two steps in a row."""
    from fla_hip.layers import GatedDeltaNet
    from fla_hip.layers.gated_deltanet import LayerCache
    torch.manual_seed(N)
    layer = GatedDeltaNet(hidden_size=hidden, expand_v=expand, head_dim=D, num_heads=heads, num_v_heads=v_heads, conv_size=conv, conv_bias=neg,
                          allow_neg_eigval=neg, layer_idx=0).cuda().to(dtype).eval()
    caches = []
    state = 0.1 * torch.randn(N, v_heads, layer.head_v_dim, D, device='cuda')
    convs = [torch.randn(N, d, conv, device='cuda', dtype=dtype) for d in (layer.key_dim, layer.key_dim, layer.value_dim)]
    for _ in range(2):
        caches.append(LayerCache())
        caches[-1].update(layer_idx=0, recurrent_state=state.clone(), conv_state=tuple(c.clone() for c in convs))
    for step in range(2):
        x = torch.randn(N, 1, hidden, device='cuda', dtype=dtype)
        assert layer._step(x, None) is None
        got = layer._step(x, caches[0])
        assert got is not None
        with monkeypatch.context() as m:
            m.setattr(GatedDeltaNet, '_step', lambda *a: None)
            want, _, _ = layer(x, past_key_values=caches[1], use_cache=True)
        assert O.get_err_ratio(want.float(), got.float()) < 5e-3
        assert O.get_err_ratio(caches[1][0]['recurrent_state'], caches[0][0]['recurrent_state']) < 2e-3
        for a, b in zip(caches[1][0]['conv_state'], caches[0][0]['conv_state']):
            assert O.get_err_ratio(a.float(), b.float()) < 2e-3


@pytest.mark.parametrize('N', [128, 129, 255, 257])
def test_layer_step_beyond_one_tile_of_rows(N, monkeypatch):
    test_layer_step_in_four_launches(N, 512, 2, 4, 64, 1, 4, False, monkeypatch)


@pytest.mark.parametrize('N,hidden,heads,v_heads,D,expand', [
    (1, 4096, 4, 4, 64, 1), (16, 768, 3, 6, 64, 2), (7, 256, 8, 8, 32, 1), (15, 512, 3, 3, 256, 4), (2, 256, 8, 8, 256, 2), (16, 256, 1, 32, 64, 0.625)])
def test_layer_step_of_few_sequences(N, hidden, heads, v_heads, D, expand, monkeypatch):
    """The projections' kernel for up to 16 rows: fewer steps than waves, more than it requests at once, hidden sizes that are no power of two,
    one to three tiles of columns to a workgroup, segments of a few columns."""
    test_layer_step_in_four_launches(N, hidden, heads, v_heads, D, expand, 4, False, monkeypatch)


@pytest.mark.parametrize('N,heads,v_heads,expand,dtype', [(16, 3, 6, 1, torch.bfloat16), (5, 4, 4, 2, torch.bfloat16), (13, 4, 4, 2, torch.float16),
                                                          (3, 3, 6, 1, torch.float16)])
def test_layer_step_of_few_sequences_in_two_tiles_of_columns(N, heads, v_heads, expand, dtype, monkeypatch):
    """Two tiles in sixteen waves (a contraction of more than 1024): projections of 4620 columns, 24 to a workgroup, and of 6152, 32 to one."""
    test_layer_step_in_four_launches(N, 2048, heads, v_heads, 256, expand, 4, False, monkeypatch, dtype)


def test_layer_step_leaves_many_sequences_of_a_large_layer_to_its_modules():
    from fla_hip.layers import GatedDeltaNet
    from fla_hip.layers.gated_deltanet import LayerCache
    layer = GatedDeltaNet(hidden_size=2048, layer_idx=0).cuda().bfloat16().eval()
    for N, native in ((192, True), (256, False)):
        cache = LayerCache()
        cache.update(layer_idx=0, recurrent_state=torch.zeros(N, 6, 512, 256, device='cuda'),
                     conv_state=tuple(torch.zeros(N, d, 4, device='cuda', dtype=torch.bfloat16) for d in (1536, 1536, 3072)))
        x = torch.randn(N, 1, 2048, device='cuda', dtype=torch.bfloat16)
        assert (layer._step(x, cache) is not None) == native
