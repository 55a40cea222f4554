"""The DSQG block's forward with the phase-probe features inside the kernels.

``DSQGAttentionV19.forward`` (kernels/dsqg_attention_v22.py:3144-3284) forms
the MOVT phase features y (from q) and z (from k) with an einsum over fp32
copies of q and k (dsqg:3231-3254) and hands them to the op as y_pre and
z_pre; their backward is a second pass over q and k.  ``dsqg_block_forward``
is a forward for that module: the same attributes, the same arguments and
the same result, with the op called in its probe form
(``dsqg_attention_with_probes``): y formed in the forward kernel from the q
rows it loads, z from the phase-probe kernel over k, and dy / dz added to dq
/ dk inside the backward kernels.  A maintainer binds it as the method::

    DSQGAttentionV19.forward = amd.dsqg_block_forward

Module attributes read (all set by DSQGAttentionV19.__init__, dsqg:2790-2978):
num_heads, head_dim, minimum_offset, support_crop_projections,
support_crop_min_offset, qkvg_proj, npci_theta_k, npci_theta_v,
npci_strength_tau, query_probes, key_probes, phase_gate, pos_bias,
centered_scale_embed, phase_base, phase_gain, j_val, j_small, j_large,
offsets_dev, the five sparse-plan buffers, k_group_size, grouped_mode_id,
verify_mode, max_group_spread_observed, plane_shift, backend,
online_softmax, if_gain, out_proj, dropout.

Under bf16 autocast, without kv_inject and without support cropping (the
trainer's blocks), the whole block is one autograd Function
(``_DSQGBlockFn``): the attention reads q, k and v as views of the fused
projection [B, N, 4D], the per-head gain and the content gate are one launch
after it (csrc/block.hip), the backward writes dq, dk, dv and the gate's
gradient straight into one [B, N, 4D] gradient, and the projections' weight
gradients are split over the tokens (csrc/wgrad.hip).  Each product is
rounded where the unfused expression rounds it, with two roundings fewer:
the weight and bias gradients stay fp32 (autocast's products give bf16), and
the gate's gradient is rounded once after the sigmoid's derivative (PyTorch's
bf16 sigmoid backward rounds g (1 - s) and then that times s).  Against 64
bits at B15 H8 T2048: qkvg weight 5.3e-3 (unfused 5.6e-3), its bias 3.9e-3
(4.2e-3), output weight 4.6e-3 (4.9e-3), dx 5.79e-3 (5.82e-3).
"""

from __future__ import annotations

import ctypes

import torch
import torch.nn.functional as F

from . import _lib
from .dsqg import (HEAD_DIM, _check_call, _planes, _rows_ok, _stream, dsqg_attention_with_probes, dsqg_backward,
                   dsqg_forward, normalize_inputs, normalized_probe_banks, schedule_for)
from .npci import npci_rotate
from .probe import probe_forward

_WGRAD_MAX_STRIDE = 1 << 22
_AUTOCAST_TYPES = (torch.bfloat16, torch.float16, torch.float32)
NPCI_THETA_MAX = 0.25   # bound of the NPCI rotation angle, theta = 0.25 tanh(raw) (dsqg:71, 3216, 3222)


def _cropped_projections(block, x: torch.Tensor, query_start: int, key_end: int):
    """q, k, v and the content gate, each [B, N, D], under support cropping (dsqg:3158-3187).

    Only the rows that can take part are projected: q and the gate for rows
    >= query_start (no offset reaches an earlier query), k and v for rows
    < key_end (no query reaches a later source); the other rows are zero.
    """
    D = x.shape[-1]
    w, b = block.qkvg_proj.weight, block.qkvg_proj.bias
    q, k, v, gate = (x.new_zeros(x.shape) for _ in range(4))
    tail, head = x[:, query_start:], x[:, :key_end]
    q[:, query_start:] = F.linear(tail, w[:D], b[:D])
    gate[:, query_start:] = F.linear(tail, w[3 * D:], b[3 * D:])
    kv = F.linear(head, w[D:3 * D], b[D:3 * D])
    k[:, :key_end], v[:, :key_end] = kv[..., :D], kv[..., D:]
    return q, k, v, gate


def _heads(t: torch.Tensor, heads: int) -> torch.Tensor:
    """[B, N, H*64] -> [B, H, N, 64] view."""
    B, N, D = t.shape
    return t.reshape(B, N, heads, D // heads).permute(0, 2, 1, 3)


def _expect(ok: bool, what: str) -> None:
    """The kernels take shapes and types as given: a raw launch on others would read out of range."""
    if not ok:
        raise ValueError(f"the raw launch expects {what}")


def _check_gate(out, gain, gate, *rows) -> None:
    B, H, N, hd = out.shape
    _expect(hd == HEAD_DIM and out.dtype == torch.bfloat16, "out bf16 [B,H,N,64]")
    _expect(gain.shape == (H,) and gain.dtype == torch.float32 and gain.is_contiguous(), "gain fp32 [H], contiguous")
    _expect(all(t.shape == (B, N, H * hd) and t.dtype == torch.bfloat16 for t in (gate, *rows)),
            "gate and its gradients bf16 [B,N,H*64]")


def _fill_gate(a: _lib.HeadGateFwdArgs, out, gain, gate) -> None:
    a.B, a.H, a.N = out.shape[:3]
    a.out, a.out_stride = out.data_ptr(), _lib.i64_array(out.stride())
    a.gain = gain.data_ptr()
    a.gate, a.gate_stride = gate.data_ptr(), _lib.i64_array(gate.stride())


def head_gate_forward(out: torch.Tensor, gain: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    """Raw launch: bf16((out * gain[h]) * bf16(sigmoid(gate))) as [B,N,H*64]; out bf16 [B,H,N,64], gain fp32
    [H], gate bf16 [B,N,H*64]."""
    _check_gate(out, gain, gate)
    return _gate_forward(out, gain, gate)


def _gate_forward(out, gain, gate):
    lib = _lib.load()
    B, H, N, hd = out.shape
    gated = torch.empty((B, N, H * hd), device=out.device, dtype=out.dtype)
    a = _lib.HeadGateFwdArgs()
    _fill_gate(a, out, gain, gate)
    a.gated, a.gated_stride = gated.data_ptr(), _lib.i64_array(gated.stride())
    _lib.check(lib.dwarf_head_gate_fwd(ctypes.byref(a), _stream(out.device)), "dwarf_head_gate_fwd")
    return gated


def head_gate_backward(dgated, out, gain, gate, dgate, *, lse=None, query_start=0, pairs=0):
    """Raw launch: (dout like out, dgain fp32 [H]); the gate's gradient goes into ``dgate``.  pairs: address
    of the [B,H,N] (delta, lse) pairs to write as well, 0 for none."""
    _check_gate(out, gain, gate, dgated, dgate)
    _expect(not pairs or (lse.shape == out.shape[:3] and lse.dtype == torch.float32), "lse fp32 [B,H,N] for the pairs")
    return _gate_backward(dgated, out, gain, gate, dgate, lse, query_start, pairs)


def _gate_backward(dgated, out, gain, gate, dgate, lse, query_start, pairs):
    lib = _lib.load()
    dout = torch.empty_like(out)
    dgain = torch.empty(gain.shape, device=out.device, dtype=torch.float32)
    a = _lib.HeadGateBwdArgs()
    _fill_gate(a.fwd, out, gain, gate)
    a.dgated, a.dgated_stride = dgated.data_ptr(), _lib.i64_array(dgated.stride())
    a.dout, a.dout_stride = dout.data_ptr(), _lib.i64_array(dout.stride())
    a.dgate, a.dgate_stride = dgate.data_ptr(), _lib.i64_array(dgate.stride())
    a.dgain = dgain.data_ptr()
    if pairs:
        a.delta_pairs, a.query_start = pairs, int(query_start)
        a.lse, a.lse_stride = lse.data_ptr(), _lib.i64_array(lse.stride())
    ws = torch.empty(max(int(lib.dwarf_head_gate_bwd_workspace_bytes(ctypes.byref(a))), 16), device=out.device,
                     dtype=torch.uint8)
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    _lib.check(lib.dwarf_head_gate_bwd(ctypes.byref(a), _stream(out.device)), "dwarf_head_gate_bwd")
    return dout, dgain


def linear_wgrad(dy: torch.Tensor, x: torch.Tensor, bias: bool) -> tuple[torch.Tensor, torch.Tensor | None]:
    """Raw launch: (dW [O,I], db [O] or None) fp32 of y = x W^T + b from dy [..., O] and x [..., I] bf16."""
    dy, x = (t.reshape(-1, t.shape[-1]) for t in (dy, x))
    _expect(dy.shape[0] == x.shape[0] and dy.dtype == x.dtype == torch.bfloat16, "as many bf16 rows of dy as of x")
    # the kernel reads a split's rows with 32-bit offsets: rows at most 2^22 elements apart
    dy, x = (t if _rows_ok(t) and t.shape[1] <= t.stride(0) <= _WGRAD_MAX_STRIDE
             else t.clone(memory_format=torch.contiguous_format) for t in (dy, x))
    lib = _lib.load()
    dw = torch.empty((dy.shape[1], x.shape[1]), device=dy.device, dtype=torch.float32)
    db = torch.empty(dy.shape[1], device=dy.device, dtype=torch.float32) if bias else None
    a = _lib.LinearWgradArgs()
    a.M, a.O, a.I = dy.shape[0], dy.shape[1], x.shape[1]
    a.dy, a.dy_stride, a.x, a.x_stride = dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0)
    a.dw, a.db = dw.data_ptr(), None if db is None else db.data_ptr()
    ws = torch.empty(max(int(lib.dwarf_linear_wgrad_workspace_bytes(ctypes.byref(a))), 16), device=dy.device,
                     dtype=torch.uint8)
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    _lib.check(lib.dwarf_linear_wgrad(ctypes.byref(a), _stream(dy.device)), "dwarf_linear_wgrad")
    return dw, db


def _check_block(qkvg, gain, heads) -> None:
    _expect(qkvg.dim() == 3 and qkvg.dtype == torch.bfloat16 and qkvg.shape[2] == 4 * HEAD_DIM * heads
            and gain.shape == (heads,), "qkvg bf16 [B,N,4*64*H] and gain [H]")


def block_forward(qkvg, pos_bias, scale_embed, phase_base, phase_gain, query_probes, key_probes, gain, offsets, heads,
                  j_small, j_large, plane_shift, query_start, schedule):
    """Raw launches from the fused projection [B,N,4D] (bf16, contiguous) to the gated heads [B,N,D]: returns
    (gated, out [B,N,H,64], lse, y, z)."""
    _check_block(qkvg, gain, heads)
    qkvg = qkvg if qkvg.is_contiguous() and _rows_ok(qkvg) else qkvg.clone(memory_format=torch.contiguous_format)
    B, N, D4 = qkvg.shape
    q, k, v, gate = qkvg.split(D4 // 4, dim=-1)
    q, k, v = (_heads(t, heads) for t in (q, k, v))
    z = probe_forward(k, key_probes, 0, N)
    t = normalize_inputs(q, k, v, pos_bias, scale_embed, phase_base, phase_gain, None, z, offsets, j_small + j_large)
    out = torch.empty((B, N, heads, HEAD_DIM), device=qkvg.device, dtype=qkvg.dtype)
    _, lse, y = dsqg_forward(*t, j_small, j_large, plane_shift, query_start, schedule=schedule,
                             query_probes=_planes(query_probes.float()), out=out.permute(0, 2, 1, 3))
    gated = _gate_forward(out.permute(0, 2, 1, 3), gain.float().contiguous(), gate)
    return gated, out, lse, y, z


def block_backward(dgated, qkvg, pos_bias, scale_embed, phase_base, phase_gain, query_probes, key_probes, gain, offsets,
                   out, lse, y, z, heads, j_small, j_large, plane_shift, query_start, schedule):
    """Raw launches: (dqkvg [B,N,4D], dpos_bias, dscale_embed, dphase_base, dphase_gain, dgain)."""
    _check_block(qkvg, gain, heads)
    B, N = qkvg.shape[:2]
    _expect(out.shape == (B, N, heads, HEAD_DIM) and dgated.shape == (B, N, heads * HEAD_DIM)
            and out.dtype == torch.bfloat16 and lse.shape == (B, heads, N) and lse.dtype == torch.float32
            and y.shape == z.shape == (B, heads, N, 4),
            "out bf16 [B,N,H,64], dgated [B,N,H*64], lse fp32 [B,H,N] and y, z [B,H,N,4]")
    qkvg = qkvg if qkvg.is_contiguous() and _rows_ok(qkvg) else qkvg.clone(memory_format=torch.contiguous_format)
    D = qkvg.shape[-1] // 4
    dgated = dgated.to(qkvg.dtype)
    dgated = dgated if _rows_ok(dgated) else dgated.clone(memory_format=torch.contiguous_format)
    dqkvg = torch.empty_like(qkvg)
    q, k, v, gate = qkvg.split(D, dim=-1)
    dq, dk, dv, dgate = dqkvg.split(D, dim=-1)
    q, k, v, dq, dk, dv = (_heads(t, heads) for t in (q, k, v, dq, dk, dv))
    o = out.contiguous().permute(0, 2, 1, 3)
    lse = lse.contiguous()
    t = normalize_inputs(q, k, v, pos_bias, scale_embed, phase_base, phase_gain, y, z, offsets, j_small + j_large)
    gain = gain.float().contiguous()
    dgain = None

    def gate_launch(pairs):
        nonlocal dgain
        dout, dgain = _gate_backward(dgated, o, gain, gate, dgate, lse, query_start, pairs)
        return dout

    g = dsqg_backward(gate_launch, *t, o, lse, j_small, j_large, plane_shift, query_start, schedule=schedule,
                      query_probes=_planes(query_probes.float()), key_probes=_planes(key_probes.float()),
                      into=(dq, dk, dv))
    return (dqkvg, *g[3:7], dgain)


class _OnceOnly(torch.autograd.Function):
    """The gradients as they are, with a graph whose only use is to raise (``anchor``: any tensor with a gradient)."""

    @staticmethod
    def forward(ctx, anchor, *grads):
        return grads

    @staticmethod
    def backward(ctx, *_):
        raise RuntimeError("the DSQG block has no second derivative")


class _DSQGBlockFn(torch.autograd.Function):
    """The block from its input to its output projection as one node (bf16): the two projections, and between them
    the custom ops ``torch.ops.dwarf.dsqg_block_fwd`` / ``dsqg_block_bwd``; the projections' weight and bias
    gradients come from ``torch.ops.dwarf.linear_wgrad`` (all registered in ``ops.py``) in fp32.  Probes:
    normalised fp32 [4,64], without gradient; a projection's bias may be None."""

    @staticmethod
    def forward(ctx, x, w_in, b_in, w_out, b_out, pos_bias, scale_embed, phase_base, phase_gain, gain, query_probes,
                key_probes, offsets_dev, heads, j_small, j_large, plane_shift, query_start, schedule, bwd_schedule):
        args = (int(heads), int(j_small), int(j_large), int(plane_shift), int(query_start))
        ctx.args = (*args, int(bwd_schedule))
        bf16 = torch.bfloat16
        x16, wi, wo = x.to(bf16), w_in.to(bf16), w_out.to(bf16)
        qkvg = F.linear(x16, wi, None if b_in is None else b_in.to(bf16))
        gated, out, lse, y, z = torch.ops.dwarf.dsqg_block_fwd(qkvg, pos_bias, scale_embed, phase_base, phase_gain,
                                                               query_probes, key_probes, gain, offsets_dev, *args,
                                                               int(schedule))
        result = F.linear(gated, wo, None if b_out is None else b_out.to(bf16))
        ctx.save_for_backward(x16, wi, wo, qkvg, gated, pos_bias, scale_embed, phase_base, phase_gain, gain,
                              query_probes, key_probes, offsets_dev, out, lse, y, z)
        ctx.dtypes = tuple(None if t is None else t.dtype for t in (x, w_in, b_in, w_out, b_out))
        return result

    @staticmethod
    def backward(ctx, dy):
        x16, wi, wo, qkvg, gated, pb, se, pbase, pgain, gain, qp, kp, offsets, out, lse, y, z = ctx.saved_tensors
        dt_x, dt_wi, dt_bi, dt_wo, dt_bo = ctx.dtypes
        need = ctx.needs_input_grad
        dy = dy.to(torch.bfloat16)

        def weights(grad, inp, dt_w, dt_b, need_w, need_b):
            if not (need_w or need_b):
                return None, None
            dw, db = torch.ops.dwarf.linear_wgrad(grad, inp, dt_b is not None)
            return dw.to(dt_w), None if dt_b is None else db.to(dt_b)

        dwo, dbo = weights(dy, gated, dt_wo, dt_bo, need[3], need[4])
        g = torch.ops.dwarf.dsqg_block_bwd(torch.matmul(dy, wo), qkvg, pb, se, pbase, pgain, qp, kp, gain, offsets, out,
                                           lse, y, z, *ctx.args)
        dqkvg, dpb, dse, dpbase, dpgain, dgain = g
        dwi, dbi = weights(dqkvg, x16, dt_wi, dt_bi, need[1], need[2])
        dx = torch.matmul(dqkvg, wi).to(dt_x) if need[0] else None
        grads = (dx, dwi, dbi, dwo, dbo, dpb, dse, dpbase, dpgain, dgain.reshape(gain.shape))
        if torch.is_grad_enabled() and not torch.compiler.is_compiling():
            # create_graph: the saved intermediates carry no graph, so a second derivative would lack their terms
            grads = _OnceOnly.apply(torch.empty(0, device=dy.device, requires_grad=True), *grads)
        return grads + (None,) * 10


def _plain_linear(m):
    """(weight, bias) of an nn.Linear nothing hooks into, of whole 16-byte rows and plain parameters, whose forward is
    F.linear on them; else None.  Hooks of its own, hooks on every module and a forward set on the instance (module
    trackers, adapters, offloading) need the call, and so does a weight or bias of a class of its own."""
    every = torch.nn.modules.module
    if (type(m) is not torch.nn.Linear or m.in_features % 8 or m.out_features % 8
            or m._forward_pre_hooks or m._forward_hooks or m._backward_hooks or m._backward_pre_hooks
            or every._global_forward_pre_hooks or every._global_forward_hooks
            or every._global_backward_hooks or every._global_backward_pre_hooks or "forward" in m.__dict__):
        return None
    w, b = m.weight, m.bias
    plain = (torch.nn.Parameter, torch.Tensor)
    return (w, b) if type(w) in plain and (b is None or type(b) in plain) else None


def _one_node(block, x: torch.Tensor) -> bool:
    """Whether the block runs as ``_DSQGBlockFn``: bf16 autocast (both projections read and write bf16), plain
    linear projections, frozen phase probes, the fp32 gain of the module."""
    if not (x.is_cuda and torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16):
        return False
    if torch.is_grad_enabled() and (block.query_probes.requires_grad or block.key_probes.requires_grad):
        return False
    proj, out, gain, D = block.qkvg_proj, block.out_proj, block.if_gain, block.num_heads * HEAD_DIM
    given, taken = _plain_linear(proj), _plain_linear(out)
    if given is None or taken is None or x.dtype not in _AUTOCAST_TYPES:
        return False
    for t in (*given, *taken):
        # what autocast casts; float64 it leaves as it is, for the projections to keep or to refuse
        if t is not None and (t.dtype not in _AUTOCAST_TYPES or t.device != x.device):
            return False
    return (block.head_dim == HEAD_DIM
            and proj.in_features == x.shape[-1] == D and proj.out_features == 4 * D and out.in_features == D
            and gain.dtype == torch.float32 and gain.numel() == block.num_heads and gain.device == x.device
            and str(block.backend).lower() in ("auto", "triton", "hip"))


def _block_node(block, x: torch.Tensor, query_start: int) -> torch.Tensor:
    H, N = block.num_heads, x.shape[1]
    # the op's own checks, on the shapes its q, k and v views will have
    probe = torch.empty(1, device=x.device, dtype=torch.bfloat16).expand(x.shape[0], H, N, HEAD_DIM)
    _check_call(probe, probe, probe, None, None, block.j_val, block.j_small, block.j_large, block.offsets_dev,
                block.grouped_mode_id)
    qp, kp = normalized_probe_banks(block.query_probes, block.key_probes, x.device)
    phase_gate = torch.sigmoid(block.phase_gate)[:, None, None]
    proj, out = block.qkvg_proj, block.out_proj
    return _DSQGBlockFn.apply(
        x, proj.weight, proj.bias, out.weight, out.bias, block.pos_bias.float(), block.centered_scale_embed.float(),
        (block.phase_base * phase_gate).float(), (block.phase_gain * phase_gate).float(), block.if_gain.reshape(-1), qp,
        kp, block.offsets_dev, H, int(block.j_small), int(block.j_large), int(block.plane_shift),
        max(0, min(int(query_start), N)),
        *(schedule_for(block.grouped_mode_id, bool(block.online_softmax), int(block.j_small), back)
          for back in (False, True)))


def _inject(block, k: torch.Tensor, v: torch.Tensor, kv_inject, key_end: int):
    """NPCI rotation of the live key/value prefix by the injected deltas (dsqg:3196-3229).

    The deltas are full [B,H,N,hd] tensors (their first key_end rows are
    used) or exactly the live prefix [B,H,key_end,hd]; anything else raises
    ValueError.  Rows >= key_end are kept as they are.
    """
    dk, dv = kv_inject
    B, H, N, hd = k.shape
    if dk.shape == k.shape and dv.shape == k.shape:
        dk, dv = dk[:, :, :key_end], dv[:, :, :key_end]
    elif not (dk.shape == (B, H, key_end, hd) and dv.shape == (B, H, key_end, hd)):
        raise ValueError("kv_inject must contain full [B,H,N,HD] tensors or the "
                         "exact live source prefix [B,H,N-min_offset,HD]")
    tau = block.npci_strength_tau
    rk = npci_rotate(k[:, :, :key_end], dk, NPCI_THETA_MAX * torch.tanh(block.npci_theta_k), strength_tau=tau)
    rv = npci_rotate(v[:, :, :key_end], dv, NPCI_THETA_MAX * torch.tanh(block.npci_theta_v), strength_tau=tau)
    if key_end == N:
        return rk, rv
    return torch.cat((rk, k[:, :, key_end:]), dim=2), torch.cat((rv, v[:, :, key_end:]), dim=2)


def dsqg_block_forward(block, x: torch.Tensor, kv_inject=None) -> torch.Tensor:
    """DSQGAttentionV19.forward (dsqg:3144-3284) with y/z and their gradients inside the kernels.

    x [B, N, D] -> [B, N, D].  When no offset has a source at this length the
    result is zeros (dsqg:3153-3156).
    """
    B, N, D = x.shape
    H, hd = block.num_heads, block.head_dim
    query_start = min(block.minimum_offset, N)
    if query_start >= N:
        return torch.zeros_like(x)
    key_end = max(0, N - query_start)
    if block.support_crop_projections and query_start >= block.support_crop_min_offset:
        q, k, v, gate = _cropped_projections(block, x, query_start, key_end)
    elif kv_inject is None and _one_node(block, x):
        return block.dropout(_block_node(block, x, query_start))
    else:
        q, k, v, gate = block.qkvg_proj(x).split(D, dim=-1)
    # [B, N, H*hd] -> [B, H, N, hd] views over the projection rows
    q, k, v = (t.reshape(B, N, H, hd).permute(0, 2, 1, 3) for t in (q, k, v))
    if kv_inject is not None:
        k, v = _inject(block, k, v, kv_inject, key_end)
    phase_gate = torch.sigmoid(block.phase_gate)[:, None, None]
    out = dsqg_attention_with_probes(
        q, k, v, block.pos_bias, block.centered_scale_embed, block.phase_base * phase_gate,
        block.phase_gain * phase_gate, block.query_probes, block.key_probes, block.j_val, block.j_small,
        block.j_large, block.offsets_dev, block.sparse_order_dev, block.group_start_dev, block.group_len_dev,
        block.group_dmin_dev, block.group_dmax_dev, block.k_group_size, block.grouped_mode_id, block.verify_mode,
        block.max_group_spread_observed, block.plane_shift, query_start, backend=block.backend,
        online_softmax=block.online_softmax)
    out = out * block.if_gain.reshape(1, H, 1, 1)
    merged = out.permute(0, 2, 1, 3).reshape(B, N, D)
    return block.dropout(block.out_proj(merged * torch.sigmoid(gate)))
