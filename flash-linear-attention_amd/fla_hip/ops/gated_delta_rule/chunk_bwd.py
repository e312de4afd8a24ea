"""Backward of ``chunk_gated_delta_rule``: ``chunk_gated_delta_rule_bwd`` with the argument meaning of
fla/ops/gated_delta_rule/chunk.py:125-257 and the autograd function around forward and backward
(chunk.py:260-395) for calls that the native one (csrc/host/gdn_host_train.h) leaves.  One call into libgdn_hip.so
(``gdn_chunk_bwd_heads``) replaces the reference's seven launches and, with the in-kernel l2 norm, the four around them
(chunk.py:278-288, 385-393); nothing is kept from the forward call but its inputs (A, P, the per-chunk states and v_new are computed
again).  The derivatives of the gate and of beta's sigmoid are one more kernel (``gate_bwd``)."""
from __future__ import annotations

import os

import torch
import torch.nn.functional as F

from fla_hip import _lib
from fla_hip.ops.gated_delta_rule._common import aligned16, as_f32, check_operand_shapes, dtype_code, launch, pad_last_two, ptr, require_gpu
from fla_hip.ops.utils.index import check_cu_seqlens, cu_bounds, prepare_chunk_indices, prepare_scan_tables

_CHUNK = 64
_DIM = 128          # block of value columns of the backward kernels


def _pad_last(x: torch.Tensor, size: int) -> torch.Tensor:
    return x if x.shape[-1] == size else F.pad(x, (0, size - x.shape[-1]))


def chunk_gated_delta_rule_bwd(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    g: torch.Tensor | None,
    beta: torch.Tensor,
    scale: float,
    initial_state: torch.Tensor | None,
    do: torch.Tensor,
    dht: torch.Tensor | None,
    state_v_first: bool = False,
    cu_seqlens: torch.Tensor | None = None,
    cu_seqlens_cpu: torch.Tensor | None = None,
    chunk_indices: torch.Tensor | None = None,
    chunk_size: int = 64,
    q_rstd: torch.Tensor | None = None,
    k_rstd: torch.Tensor | None = None,
    qk_l2norm: bool = False,
    A_log: torch.Tensor | None = None,
    dt_bias: torch.Tensor | None = None,
    beta_sigmoid: bool = False,
    neg_eigval: bool = False,
):
    """q, k ``[B,T,H,K]``, v, do ``[B,T,HV,V]``, g (log decay), beta ``[B,T,HV]`` as the recurrence uses them.
    Returns ``(dq, dk, dv, dbeta, dg, dh0)``: dq, dk, dv in q's dtype, dbeta, dg fp32, dh0 fp32 (None without
    ``initial_state``).  With ``q_rstd``, ``k_rstd`` (the factors ``l2norm_fwd`` returns next to the normalised rows
    passed as q and k) dq and dk are the gradients of the rows before normalisation: the reference's ``l2norm_bwd``
    (chunk.py:385-387) in a kernel of its own.  With ``qk_l2norm`` q and k
    are the rows BEFORE their l2 normalisation and dq, dk the gradients of those: one C call
    (``gdn_chunk_bwd_heads``), which also adds up the value heads of a q/k head.  With ``A_log`` (and ``dt_bias``, both ``[HV]`` fp32)
    or ``beta_sigmoid`` g and beta are the inputs of those activations; dg and dbeta stay the gradients of their results
    (``gate_bwd`` goes on from there)."""
    dev = require_gpu(q, k, v, beta, do)
    check_operand_shapes(q, k, v, g=g, beta=beta)
    if do.shape != v.shape:
        raise ValueError(f'do must have the shape of v, got {tuple(do.shape)} and {tuple(v.shape)}')
    B, T, H, K = k.shape
    HV, V = v.shape[2], v.shape[3]
    if K > 2 * _DIM:
        raise NotImplementedError(f'the backward kernels cover key head dims up to {2 * _DIM} (got K={K})')
    # the kernels' dims: 64 x 64, or 128 or 256 key features with value columns in blocks of 128
    KD, VD = (64, 64) if K <= 64 and V <= 64 else (_DIM if K <= _DIM else 2 * _DIM, (V + _DIM - 1) // _DIM * _DIM)
    N = B if cu_seqlens is None else len(cu_seqlens) - 1

    out_dtype = q.dtype
    work = q.dtype if q.dtype in (torch.bfloat16, torch.float16) else torch.bfloat16
    qw, kw = (aligned16(_pad_last(x.to(work), KD).contiguous()) for x in (q, k))
    vw, dow = (aligned16(_pad_last(x.to(work), VD).contiguous()) for x in (v, do))
    gw = None if g is None else as_f32(g).contiguous()
    bw = as_f32(beta).contiguous()

    def state_in(s):
        if s is None:
            return None
        want = (N, HV, V, K) if state_v_first else (N, HV, K, V)
        if tuple(s.shape) != want:
            raise ValueError(f'initial_state and dht must have shape {want}, got {tuple(s.shape)}')
        s = as_f32(s)
        if state_v_first:
            s = s.transpose(-1, -2)
        return aligned16(pad_last_two(s, KD, VD).contiguous())
    h0, dhtw = state_in(initial_state), state_in(dht)

    # FLA_HIP_BWD_SCAN_MODE forces one form of the two scans (default: automatic): whole sequences ('wide') or time segments
    # wherever they are possible at all ('segments')
    flags = {'wide': _lib.FLAG_SCAN_WIDE, 'segments': _lib.FLAG_SCAN_SEGMENTS}.get(os.environ.get('FLA_HIP_BWD_SCAN_MODE', 'auto'), 0)
    chunk_table = chunk_offsets = None
    if cu_seqlens is not None:
        if cu_seqlens.dtype not in (torch.int32, torch.int64):
            cu_seqlens = cu_seqlens.long()
        cu_seqlens = cu_seqlens.to(dev)
        if cu_seqlens.dtype == torch.int32:
            flags |= _lib.FLAG_CU_INT32
        check_cu_seqlens(cu_seqlens, T, cu_seqlens_cpu)
        chunk_indices = prepare_chunk_indices(cu_seqlens, _CHUNK, cu_seqlens_cpu=cu_seqlens_cpu)      # (derived here, never taken over)
        chunk_table = chunk_indices.to(device=dev, dtype=cu_seqlens.dtype).contiguous()
        flags |= _lib.FLAG_SEQ_ORDER
        chunk_offsets = prepare_scan_tables(cu_seqlens, _CHUNK, cu_seqlens_cpu=cu_seqlens_cpu)
        num_chunks = chunk_table.shape[0]
    else:
        num_chunks = B * ((T + _CHUNK - 1) // _CHUNK)

    # The kernels write the tokens inside [cu_seqlens[0], cu_seqlens[-1]) only.  Tokens of a packed tensor outside every
    # sequence get zero gradients (what autograd hands on, e.g. to a projection's weight gradient, must not be
    # uninitialised memory); the boundaries are known from the host summary that check_cu_seqlens has just memoised.
    alloc = torch.empty
    if cu_seqlens is not None:
        first, last = cu_bounds(cu_seqlens, cu_seqlens_cpu)
        if first != 0 or last != T:
            alloc = torch.zeros
    dq = alloc(B, T, H, KD, dtype=work, device=dev)
    dk = alloc(B, T, H, KD, dtype=work, device=dev)
    dv = alloc(B, T, HV, VD, dtype=work, device=dev)
    dg = alloc(B, T, HV, dtype=torch.float32, device=dev)
    db = alloc(B, T, HV, dtype=torch.float32, device=dev)
    dh0 = torch.empty(N, HV, KD, VD, dtype=torch.float32, device=dev) if initial_state is not None else None
    lib = _lib.load()
    if qk_l2norm:
        flags |= _lib.FLAG_QK_L2NORM
    if beta_sigmoid:
        flags |= _lib.FLAG_BETA_SIGMOID | (_lib.FLAG_NEG_EIGVAL if neg_eigval else 0)
    ws_bytes = lib.gdn_chunk_bwd_heads_workspace_bytes(num_chunks, H, HV, KD, VD, B * T, flags)
    workspace = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=dev)
    launch(
        lib.gdn_chunk_bwd_heads, dev, ptr(qw), ptr(kw), ptr(vw), ptr(gw), ptr(bw), ptr(A_log), ptr(dt_bias), ptr(h0), ptr(dow), ptr(dhtw),
        ptr(dq), ptr(dk), ptr(dv), ptr(dg), ptr(db), ptr(dh0),
        ptr(cu_seqlens), ptr(chunk_table), ptr(chunk_offsets), ptr(workspace), ws_bytes,
        B, T, H, HV, KD, VD, N, num_chunks, float(scale), dtype_code(work), _lib.DTYPE_F32, flags)
    dq = _finish(lib, dq, qw, q_rstd, H, K, out_dtype)
    dk = _finish(lib, dk, kw, k_rstd, H, K, out_dtype)
    dv = dv[..., :V].to(out_dtype)
    if dh0 is not None:
        dh0 = dh0[..., :K, :V]
        dh0 = (dh0.transpose(-1, -2) if state_v_first else dh0).contiguous()
    return dq, dk, dv, db, dg, dh0


def gate_bwd(dgate, dbeta, g, beta, A_log, dt_bias, beta_max):
    """The gradients of the gate ``-exp(A_log) softplus(g + dt_bias)`` (``g`` None: of no gate, ``dgate`` comes back) and of
    ``beta_max sigmoid(beta)`` (0: none) with respect to g and beta, in their types; and ``[parts, 2, HV]`` partial sums of the
    gradients of A_log and dt_bias (fla/ops/gated_delta_rule/gate.py:109-160)."""
    dev = dbeta.device
    HV = dbeta.shape[-1]
    rows = dbeta.numel() // HV
    with_gate = g is not None
    if with_gate:
        g = g if g.dtype in (torch.bfloat16, torch.float16, torch.float32) else g.float()
        g = g.contiguous()
    beta = beta if beta.dtype in (torch.bfloat16, torch.float16, torch.float32) else beta.float()
    beta = beta.contiguous()
    parts = max(1, min(256, rows * HV // 256))
    dg = torch.empty_like(g) if with_gate else None
    db = torch.empty_like(beta)
    part = torch.empty(parts, 2, HV, dtype=torch.float32, device=dev) if with_gate else None
    launch(
        _lib.load().gdn_gate_bwd, dev, ptr(dgate) if with_gate else None, ptr(dbeta), ptr(g) if with_gate else None, ptr(beta), ptr(A_log) if with_gate else None,
        ptr(dt_bias), ptr(dg), ptr(db), ptr(part), rows, HV, parts, HV, HV, HV, HV, 0, 0,
        dtype_code(g.dtype) if with_gate else _lib.DTYPE_F32, dtype_code(beta.dtype), beta_max)
    return dg if with_gate else dgate, db, part


def _finish(lib, dxh: torch.Tensor, y: torch.Tensor, rstd: torch.Tensor | None, H: int, K: int, out_dtype) -> torch.Tensor:
    """dq or dk per value head (or already per q/k head) ``[B,T,HV,KD]`` -> per q/k head ``[B,T,H,K]``: the sum over the value heads of a
    q/k head and, with ``rstd``, the way back through the l2 normalisation (``y``: the normalised rows, KD wide)."""
    B, T, HV, D = dxh.shape
    if rstd is None and HV == H and K == D:
        return dxh.to(out_dtype)
    dx = torch.empty(B, T, H, K, dtype=dxh.dtype, device=dxh.device)
    if K % 8:                                       # (rows of the kernel are multiples of 8 elements)
        KP = (K + 7) // 8 * 8
        dx = torch.empty(B, T, H, KP, dtype=dxh.dtype, device=dxh.device)
    launch(lib.gdn_l2norm_bwd, dxh.device, ptr(dxh), ptr(y) if rstd is not None else None, ptr(rstd), ptr(dx), B * T * H, HV // H, D,
           dx.shape[-1], dtype_code(dxh.dtype))
    return dx[..., :K].to(out_dtype)


def l2norm_fwd(x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """Rows divided by sqrt(sum x^2 + 1e-6), in x's dtype (fp32 input: bf16), and the factors ``[..., 1]`` fp32
    (fla/modules/l2norm.py:222-262).  Rows whose length is not a multiple of 8 come back zero-padded to one."""
    require_gpu(x)
    work = x.dtype if x.dtype in (torch.bfloat16, torch.float16) else torch.bfloat16
    if x.shape[-1] > 256:
        raise NotImplementedError('l2norm_fwd: rows of up to 256 elements')
    x = _pad_last(x, (x.shape[-1] + 7) // 8 * 8)
    D = x.shape[-1]
    xw = aligned16(x.to(work).contiguous())
    y = torch.empty_like(xw)
    rstd = torch.empty(*x.shape[:-1], 1, dtype=torch.float32, device=x.device)
    launch(_lib.load().gdn_l2norm_fwd, x.device, ptr(xw), ptr(y), ptr(rstd), xw.numel() // D, D, D, dtype_code(work))
    return y, rstd


class ChunkGatedDeltaRuleFunction(torch.autograd.Function):
    """Forward through the fused inference kernels, backward through ``gdn_chunk_bwd_heads``."""

    @staticmethod
    def forward(ctx, q, k, v, g, beta, scale, initial_state, output_final_state, state_v_first, cu_seqlens,
                cu_seqlens_cpu, chunk_indices, use_qk_l2norm_in_kernel, use_gate_in_kernel, A_log, dt_bias,
                use_beta_sigmoid_in_kernel, allow_neg_eigval, chunk_size):
        from fla_hip.ops.gated_delta_rule.chunk import chunk_gated_delta_rule_fwd
        o, ht = chunk_gated_delta_rule_fwd(
            q, k, v, g, beta, scale, initial_state, output_final_state, state_v_first, cu_seqlens, cu_seqlens_cpu,
            chunk_indices, chunk_size, A_log if use_gate_in_kernel else None, dt_bias if use_gate_in_kernel else None,
            use_qk_l2norm_in_kernel, use_beta_sigmoid_in_kernel, allow_neg_eigval)
        ctx.save_for_backward(q, k, v, g, beta, initial_state, cu_seqlens, cu_seqlens_cpu, chunk_indices, A_log, dt_bias)
        ctx.opts = (scale, state_v_first, use_qk_l2norm_in_kernel, use_gate_in_kernel, use_beta_sigmoid_in_kernel,
                    allow_neg_eigval, chunk_size)
        return o, ht

    @staticmethod
    def backward(ctx, do, dht):
        q, k, v, g, beta_raw, h0, cu_seqlens, cu_seqlens_cpu, chunk_indices, A_log, dt_bias = ctx.saved_tensors
        scale, state_v_first, l2, gate, bsig, neg, chunk_size = ctx.opts
        K = q.shape[-1]
        A32 = A_log.float().reshape(-1).contiguous() if gate else None
        dt32 = dt_bias.float().reshape(-1).contiguous() if gate and dt_bias is not None else None
        dq, dk, dv, db, dg, dh0 = chunk_gated_delta_rule_bwd(
            q, k, v, g, beta_raw, scale, h0, do.contiguous(), dht, state_v_first, cu_seqlens, cu_seqlens_cpu,
            chunk_indices, chunk_size, qk_l2norm=l2, A_log=A32, dt_bias=dt32, beta_sigmoid=bsig, neg_eigval=neg)
        dA_log = ddt_bias = None
        if gate or bsig:
            dg, db, part = gate_bwd(dg, db, g if gate else None, beta_raw, A32, dt32, (2.0 if neg else 1.0) if bsig else 0.0)
            if gate:
                sums = part.sum(0)
                dA_log = sums[0].to(A_log.dtype).reshape(A_log.shape)
                if dt_bias is not None:
                    ddt_bias = sums[1].to(dt_bias.dtype).reshape(dt_bias.shape)
        if g is not None:
            dg = dg.to(g.dtype)
        else:
            dg = None
        return (dq[..., :K].to(q.dtype), dk[..., :K].to(k.dtype), dv.to(v.dtype), dg, db.to(beta_raw.dtype), None, dh0, None, None, None,
                None, None, None, None, dA_log, ddt_bias, None, None, None)
