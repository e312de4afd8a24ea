"""The scan in halves of 64 value columns (whole sequences, up to 128 runs of 128 x 128) and its form for whole runs of 64 x 64: one chunk and
less, remainders, the last run count that takes it and the first that does not, packed sequences with an empty one, states in both layouts."""
import pytest
import torch

from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,T,H,HV,cu,dtype,vfirst,l2', [
    (1, 1, 1, 1, None, torch.bfloat16, False, False), (1, 63, 2, 6, None, torch.float16, True, True), (2, 64, 4, 4, None, torch.bfloat16, True, True),
    (8, 65, 16, 16, None, torch.bfloat16, False, True), (3, 129, 43, 43, None, torch.bfloat16, False, True), (1, 449, 2, 4, None, torch.bfloat16, False, True),
    (1, 700, 2, 4, [0, 1, 65, 65, 193, 700], torch.bfloat16, False, True), (1, 2304, 1, 2, None, torch.bfloat16, True, False),
    (1, 2305, 1, 2, None, torch.bfloat16, True, True)])
def test_halves(B, T, H, HV, cu, dtype, vfirst, l2, D=128):
    from fla_hip.ops.gated_delta_rule import chunk_gated_delta_rule
    N = B if cu is None else len(cu) - 1
    q, k, v, g, beta, h0 = O.make_inputs(B, T, H, HV, D, D, seed=T, gate_div=4.0, h0_std=0.3, N=N, dtype=dtype)
    qr, kr = (O.l2norm(q), O.l2norm(k)) if l2 else (q, k)
    ref_o, ref_h = O.chunk_gated_delta_rule(qr, kr, v, g, beta, None, h0, True, cu_seqlens=cu)
    h = h0.transpose(-1, -2).contiguous() if vfirst else h0
    o, ht = chunk_gated_delta_rule(q.cuda(), k.cuda(), v.cuda(), g.cuda(), beta.cuda(), initial_state=h.cuda(), output_final_state=True, state_v_first=vfirst,
                                   use_qk_l2norm_in_kernel=l2, cu_seqlens=None if cu is None else torch.tensor(cu, device='cuda'))
    ht = ht.transpose(-1, -2) if vfirst else ht
    assert O.get_err_ratio(ref_o.float(), o.float().cpu()) < 5e-3
    assert O.get_err_ratio(ref_h, ht.cpu()) < 5e-3


@pytest.mark.parametrize('B,T,H,HV,cu,dtype,vfirst,l2', [
    (1, 1, 1, 1, None, torch.bfloat16, False, False), (1, 63, 2, 6, None, torch.float16, True, True), (2, 64, 4, 4, None, torch.bfloat16, True, True),
    (8, 65, 16, 16, None, torch.bfloat16, False, True), (3, 129, 43, 43, None, torch.bfloat16, False, True), (1, 449, 2, 4, None, torch.float16, False, False),
    (1, 700, 2, 4, [0, 1, 65, 65, 193, 700], torch.bfloat16, False, True), (1, 1984, 1, 2, None, torch.bfloat16, True, False),
    (1, 1985, 1, 2, None, torch.bfloat16, True, True)])
def test_whole_runs_of_64(B, T, H, HV, cu, dtype, vfirst, l2):
    test_halves(B, T, H, HV, cu, dtype, vfirst, l2, D=64)


@pytest.mark.parametrize('l2', [False, True])
@pytest.mark.parametrize('D,dtype', [(128, torch.bfloat16), (128, torch.float16), (64, torch.bfloat16), (64, torch.float16)])
def test_records_of_many_units(D, dtype, l2):
    """64 runs of 13 chunks: 832 units, which the kernel with one wave to a unit prepares, P with them."""
    test_halves(4, 829, 8, 16, None, dtype, False, l2, D=D)
