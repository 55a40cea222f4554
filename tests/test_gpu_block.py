"""GPU parity of ``dsqg_block_forward``, the DSQG block's forward with y/z inside the kernels (MI355X).

The module is a stand-in that carries the attributes DSQGAttentionV19 sets
(dsqg:2790-2978) with seeded values; the block runs in bf16 as under the
trainer's autocast (train:1128).  The oracle restates DSQGAttentionV19.forward
(dsqg:3144-3284) on the CPU in float64: the projections (cropped to the
support rows when the minimum offset reaches support_crop_min_offset,
dsqg:3158-3187), rounded to bf16 as the GPU's bf16 projections are; the NPCI
rotation of the live key/value prefix (``oracle/npci_ref.py``); the block's
y/z einsum (``dsqg_ref.probe_features``); the op (``dsqg_ref.dsqg_forward``,
bf16 scale embeddings); the head gain, the content gate and the output
projection.  Gradients come from autograd through that restatement.

The fp32 block (no autocast) takes the op's fp32 route and is held to 1e-5
relative on everything; the bf16 block to 2e-2 max-abs on the output and dx
and 2e-2 of the largest magnitude on the parameter gradients (sums over every
token).
"""

from __future__ import annotations

import pytest
import torch
import torch.nn as nn

from oracle import dsqg_ref, npci_ref
from tests.dsqg_cases import orthogonal_probes

pytestmark = pytest.mark.gpu


class StandInBlock(nn.Module):
    """The attributes DSQGAttentionV19.forward reads, with seeded values."""

    def __init__(self, D, H, offsets, js, shift, crop_min, seed):
        super().__init__()
        g = torch.Generator().manual_seed(seed)
        hd = D // H
        J, jl = len(offsets), max(len(offsets) - js, 1)
        self.num_heads, self.head_dim = H, hd
        self.minimum_offset = min(offsets)
        self.support_crop_projections, self.support_crop_min_offset = True, crop_min
        self.qkvg_proj = nn.Linear(D, 4 * D, bias=True)
        self.out_proj = nn.Linear(D, D, bias=False)
        with torch.no_grad():
            self.qkvg_proj.weight.copy_(torch.randn(4 * D, D, generator=g) / D ** 0.5)
            self.qkvg_proj.bias.copy_(0.1 * torch.randn(4 * D, generator=g))
            self.out_proj.weight.copy_(torch.randn(D, D, generator=g) / D ** 0.5)
        self.npci_theta_k = nn.Parameter(0.8 * torch.randn(H, generator=g))
        self.npci_theta_v = nn.Parameter(0.8 * torch.randn(H, generator=g))
        self.npci_strength_tau = 0.25
        qp, kp = orthogonal_probes(hd, shift)
        self.query_probes = nn.Parameter(qp + 0.2 * torch.randn(qp.shape, generator=g), requires_grad=False)
        self.key_probes = nn.Parameter(kp + 0.2 * torch.randn(kp.shape, generator=g), requires_grad=False)
        self.phase_gate = nn.Parameter(torch.randn(jl, generator=g))
        self.pos_bias = nn.Parameter(0.02 * torch.randn(J, H, generator=g))
        self.centered_scale_embed = nn.Parameter(0.01 * torch.randn(J, hd, generator=g))
        self.phase_base = nn.Parameter(0.05 * torch.randn(jl, H, 4, generator=g))
        self.phase_gain = nn.Parameter(4.0 * torch.randn(jl, H, 4, generator=g))
        self.if_gain = nn.Parameter(1.0 + 0.2 * torch.randn(H, generator=g))
        self.j_val, self.j_small, self.j_large = J, js, J - js
        self.register_buffer("offsets_dev", torch.tensor(offsets, dtype=torch.int32))
        self.sparse_order_dev = self.group_start_dev = self.group_len_dev = None
        self.group_dmin_dev = self.group_dmax_dev = None
        self.k_group_size, self.grouped_mode_id, self.verify_mode, self.max_group_spread_observed = 3, 0, False, 0
        self.plane_shift, self.backend, self.online_softmax = shift, "auto", True
        self.dropout = nn.Dropout(0.0)


PARAMS = ("qkvg_proj.weight", "qkvg_proj.bias", "out_proj.weight", "npci_theta_k", "npci_theta_v", "phase_gate",
          "pos_bias", "centered_scale_embed", "phase_base", "phase_gain", "if_gain")


def _round(t, bf16):
    """bf16 rounding with a straight-through gradient where the GPU's bf16 autocast rounds; else t."""
    return t + (t.to(torch.bfloat16).to(t.dtype) - t).detach() if bf16 else t


def block_oracle(p, x, kv, blk, bf16):
    """DSQGAttentionV19.forward (dsqg:3144-3284) in float64 from the parameter dict p; with bf16, the
    roundings of bf16 autocast: linear layers take bf16 weights and inputs and give bf16 outputs, the
    sigmoid of the bf16 gate is bf16, and the op and the NPCI rotation return bf16."""
    def _bf16(t):
        return _round(t, bf16)

    B, N, D = x.shape
    H, hd = blk.num_heads, blk.head_dim
    qs = min(blk.minimum_offset, N)
    ke = N - qs
    W, b = _bf16(p["qkvg_proj.weight"]), _bf16(p["qkvg_proj.bias"])
    full = _bf16(x) @ W.t() + b
    q, k, v, gate = (_bf16(t) for t in full.split(D, dim=-1))
    if blk.support_crop_projections and qs >= blk.support_crop_min_offset:
        rows = torch.arange(N).view(1, N, 1)
        q, gate = q * (rows >= qs), gate * (rows >= qs)
        k, v = k * (rows < ke), v * (rows < ke)
    q, k, v = (t.reshape(B, N, H, hd).permute(0, 2, 1, 3) for t in (q, k, v))
    if kv is not None:
        kd, vd = kv[0].double()[:, :, :ke], kv[1].double()[:, :, :ke]
        rk = _bf16(npci_ref.npci_rotate(k[:, :, :ke], kd, 0.25 * torch.tanh(p["npci_theta_k"]), 0.25))
        rv = _bf16(npci_ref.npci_rotate(v[:, :, :ke], vd, 0.25 * torch.tanh(p["npci_theta_v"]), 0.25))
        k, v = torch.cat((rk, k[:, :, ke:]), 2), torch.cat((rv, v[:, :, ke:]), 2)
    y = dsqg_ref.probe_features(q, blk.query_probes.detach().double())
    z = dsqg_ref.probe_features(k, blk.key_probes.detach().double())
    pg = torch.sigmoid(p["phase_gate"])[:, None, None]
    out = dsqg_ref.dsqg_forward(q, k, v, p["pos_bias"], p["centered_scale_embed"], p["phase_base"] * pg,
                                p["phase_gain"] * pg, y, z, blk.offsets_dev.tolist(), blk.j_small,
                                plane_shift=blk.plane_shift, query_start=qs, round_se=bf16)
    out = _bf16(out) * p["if_gain"].reshape(1, H, 1, 1)
    merged = out.permute(0, 2, 1, 3).reshape(B, N, D)
    return _bf16(_bf16(merged * _bf16(torch.sigmoid(gate))) @ _bf16(p["out_proj.weight"]).t())


def _lattice(pkg, name):
    if name == "canonical":
        return list(pkg.ALL_OFFSETS), 17, 3
    return [64, 96, 128, 200, 333], 0, 5


def _compare(pkg, device, lattice, inject, dtype, bar_out, bar_param):
    offsets, js, shift = _lattice(pkg, lattice)
    B, N, D, H = 2, 300, 256, 4
    blk = StandInBlock(D, H, offsets, js, shift, 64, seed=90 + js)   # for the oracle's settings
    g = torch.Generator().manual_seed(91)
    x = torch.randn(B, N, D, generator=g).to(dtype)
    dy = torch.randn(B, N, D, generator=g).to(dtype)
    kv = None
    if inject:
        kv = (torch.randn(B, H, N, 64, generator=g).to(dtype), torch.randn(B, H, N, 64, generator=g).to(dtype))
    bf16 = dtype == torch.bfloat16
    # the GPU block: fp32 parameters; bf16 runs under bf16 autocast (the trainer's setting, train:1128)
    gblk = StandInBlock(D, H, offsets, js, shift, 64, seed=90 + js).to(device)
    xg = x.to(device).requires_grad_(True)
    kvg = None if kv is None else tuple(t.to(device) for t in kv)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=bf16):
        out = pkg.dsqg_block_forward(gblk, xg, kvg)
    out.backward(dy.to(device))
    torch.cuda.synchronize()
    assert out.dtype == dtype
    # the oracle on the same parameters, in float64
    named = dict(gblk.named_parameters())
    p = {n: named[n].detach().double().cpu().requires_grad_(True) for n in PARAMS}
    xo = x.double().requires_grad_(True)
    ro = block_oracle(p, xo, kv, blk, bf16)
    (ro * dy.double()).sum().backward()

    def rel(a, b):
        return float((a - b).abs().max() / b.abs().max().clamp_min(1e-30))

    errs = {"out": (out.detach().double().cpu(), ro.detach()), "dx": (xg.grad.double().cpu(), xo.grad)}
    for n, (a, b) in errs.items():
        e = float((a - b).abs().max()) if bf16 else rel(a, b)
        assert e < bar_out, (n, e)
    for n in PARAMS:
        ref = p[n].grad
        if named[n].grad is None:   # a parameter that takes no part (NPCI angles without kv_inject)
            assert ref is None or not bool(ref.any()), n
            continue
        e = rel(named[n].grad.double().cpu(), ref)
        assert e < bar_param, (n, e)


@pytest.mark.parametrize("lattice", ["canonical", "far"])
def test_block_forward_bf16_probes_in_kernels(pkg, device, lattice):
    """bf16 under autocast: the op in its probe form (y/z and their gradients inside the kernels).
    canonical: the 96-offset lattice (minimum offset 1, no cropping).  far: offsets >= 64 only (support
    cropping on: q/gate rows before 64 and k/v rows past N - 64 are never projected).  Bars: out and dx 2e-2
    max-abs; parameter gradients 2e-2 of their largest magnitude."""
    _compare(pkg, device, lattice, False, torch.bfloat16, 2e-2, 2e-2)


def test_block_forward_fp32_crop_and_kv_inject(pkg, device):
    """fp32 (the phase-probe kernels and the fp32 op), the far lattice with support cropping and a full-shape
    kv_inject through the NPCI rotation of the live key/value prefix: out, dx and every parameter gradient
    within 1e-5 relative of the float64 restatement."""
    _compare(pkg, device, "far", True, torch.float32, 1e-5, 1e-5)


def _ulp(x):
    """bf16 spacing at |x|."""
    return torch.exp2(torch.floor(torch.log2(x.abs().clamp_min(1e-30)))) * 2.0 ** -7


@pytest.mark.parametrize("B,H,N,pairs", [(1, 1, 1, False), (2, 3, 37, True), (1, 40, 33, False), (3, 8, 700, True)])
def test_head_gate_against_the_expression(pkg, device, B, H, N, pairs):
    """The gain-and-gate launches against the expression in float64 with its bf16 roundings: one item, heads that do
    not divide a workgroup's items (3), more heads than items (40), several grid strides; the gate and dout as strided
    views.  bf16 results within one spacing (a float32 product on the other side of a rounding boundary; a bf16
    sigmoid likewise moves one spacing, so two for what it multiplies); dgain: B N 64 float32 products, bounded by
    2e-6 of the sum of their magnitudes.  The (delta, lse) pairs against the sum over the rounded dout."""
    block = pkg.block
    g = torch.Generator().manual_seed(7 * N + H)
    D = 64 * H
    qkvg = torch.randn(B, N, 4 * D, generator=g).to(torch.bfloat16).to(device)
    gate = qkvg[..., 3 * D:]
    out = torch.randn(B, N, H, 64, generator=g).to(torch.bfloat16).to(device).permute(0, 2, 1, 3)
    gain = (1 + 0.3 * torch.randn(H, generator=g)).to(device)
    dg = torch.randn(B, N, D, generator=g).to(torch.bfloat16).to(device)
    lse = torch.randn(B, H, N, generator=g).to(device)
    lse[:, :, :1] = float("-inf")
    got = block.head_gate_forward(out, gain, gate)
    dgate = torch.empty_like(qkvg)[..., 3 * D:]
    ws = torch.full((B, H, N, 2), float("nan"), device=device)
    dout, dgain = block.head_gate_backward(dg, out, gain, gate, dgate, lse=lse, query_start=2,
                                           pairs=ws.data_ptr() if pairs else 0)
    torch.cuda.synchronize()

    def r16(t):
        return t.to(torch.bfloat16).double()

    o = out.double().cpu().permute(0, 2, 1, 3).reshape(B, N, D)
    s, d, gn = r16(torch.sigmoid(gate.double().cpu())), dg.double().cpu(), gain.double().cpu().repeat_interleave(64)
    want = o * gn * s
    assert ((got.double().cpu() - want).abs() <= 2 * _ulp(want)).all()
    wd = d * s * gn
    gd = dout.double().cpu().permute(0, 2, 1, 3).reshape(B, N, D)
    assert ((gd - wd).abs() <= 2 * _ulp(wd)).all()
    ds = r16(d * o * gn)
    wg = ds * (1 - s) * s
    # dgate multiplies s and 1 - s, each a bf16 spacing off at most: 2^-7 (1 - s) + 2^-8 s of ds beside its own rounding
    assert ((dgate.double().cpu() - wg).abs() <= 2 * _ulp(wg) + ds.abs() * 2.0 ** -7).all()
    wgain = (d * s * o).reshape(B * N, H, 64)
    err = (dgain.double().cpu() - wgain.sum((0, 2))).abs()
    # a sigmoid on the other side of its rounding boundary (one in 10^4) shifts its own term by 2^-8
    assert (err <= 2e-6 * wgain.abs().sum((0, 2)) + 2.0 ** -8 * wgain.abs().amax((0, 2))).all()
    if pairs:
        p = ws.double().cpu()
        wdelta = (gd * o).reshape(B, N, H, 64).sum(-1).permute(0, 2, 1)
        bound = 1e-6 * (gd * o).abs().reshape(B, N, H, 64).sum(-1).permute(0, 2, 1)
        assert ((p[..., 0] - wdelta).abs() <= bound).all()
        live = (torch.arange(N) >= 2) & torch.isfinite(lse.cpu())
        want2 = torch.where(live, lse.double().cpu() * 1.4426950408889634, torch.tensor(float("inf"), dtype=torch.double))
        assert torch.equal(torch.isinf(p[..., 1]), torch.isinf(want2))
        assert ((p[..., 1] - want2).abs()[live] <= 1e-6).all() if live.any() else True


@pytest.mark.parametrize("H,N,lattice,ones", [(3, 65, "third1", False), (8, 301, "third2", True), (4, 130, "canonical", False)])
def test_block_as_one_node_equals_the_composed_block(pkg, device, H, N, lattice, ones):
    """The one-node block (bf16 autocast) against the composed one, which a forward hook on the output projection
    selects: out, dx and every parameter gradient.  Both round the same products, in the same places; the bars are
    two bf16 spacings of the largest magnitude (2^-7), for sums over tokens of terms rounded a spacing apart."""
    offsets = list(pkg.ALL_OFFSETS) if lattice == "canonical" else list(pkg.lattice.build_offset_groups(2048)[int(lattice[-1])])
    js = sum(d <= 28 for d in offsets)
    blk = StandInBlock(64 * H, H, offsets, js, 4, 64, seed=H + N).to(device)
    g = torch.Generator().manual_seed(N)
    x = torch.randn(2, N, 64 * H, generator=g).to(torch.bfloat16).to(device).requires_grad_(True)
    dy = torch.randn(2, N, 64 * H, generator=g).to(torch.bfloat16).to(device)
    named = [(n, p) for n, p in blk.named_parameters() if p.requires_grad and not n.startswith("npci")]

    def both():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = pkg.dsqg_block_forward(blk, x)
        loss = out.float().sum() if ones else (out * dy).float().sum()
        return [out.detach()] + list(torch.autograd.grad(loss, [x] + [p for _, p in named]))

    one = both()
    blk.out_proj.register_forward_hook(lambda m, i, o: None)
    composed = both()
    for n, a, b in zip(["out", "x"] + [n for n, _ in named], one, composed):
        assert a.dtype == b.dtype and a.shape == b.shape, n
        scale = float(b.abs().max())
        assert float((a.double() - b.double()).abs().max()) <= 2.0 ** -7 * scale, n


@pytest.mark.parametrize("M,O,I,bias", [(1, 8, 8, True), (65, 136, 264, True), (127, 128, 256, False),
                                        (129, 2048, 64, True), (700, 72, 520, True), (9000, 512, 512, True)])
def test_linear_wgrad(pkg, device, M, O, I, bias):
    """dY^T X and the column sums of dY against float64: one row, rows past a 64-row step by one, outputs and inputs
    past a 128 x 256 tile by 8, several splits; dY and X as column blocks of wider rows.  Products of bf16 values are
    exact in float32; M summands in float32 give at most M 2^-24 of the magnitudes' sum, and a random walk of
    roundings far less: the bar is 2e-6 of that sum."""
    g = torch.Generator().manual_seed(M + O)
    dy = torch.randn(M, O + 24, generator=g).to(torch.bfloat16).to(device)[:, 8:8 + O]
    x = torch.randn(M, I + 8, generator=g).to(torch.bfloat16).to(device)[:, :I]
    dw, db = pkg.block.linear_wgrad(dy, x, bias)
    again, _ = pkg.block.linear_wgrad(dy, x, bias)
    a, b = dy.double().cpu(), x.double().cpu()
    assert torch.equal(dw, again)
    assert ((dw.double().cpu() - a.t() @ b).abs() <= 2e-6 * (a.abs().t() @ b.abs())).all()
    if bias:
        assert ((db.double().cpu() - a.sum(0)).abs() <= 2e-6 * a.abs().sum(0)).all()
    else:
        assert db is None


@pytest.mark.parametrize("frozen", ["x", "weights"])
def test_block_node_with_frozen_parts(pkg, device, frozen):
    """Gradients that are not needed are not formed and change no other: a block input without gradient, frozen
    projections; an input in fp32 gets its gradient in fp32."""
    offsets = list(pkg.lattice.build_offset_groups(2048)[1])
    blk = StandInBlock(128, 2, offsets, sum(d <= 28 for d in offsets), 2, 64, seed=5).to(device)
    g = torch.Generator().manual_seed(2)
    x = torch.randn(2, 70, 128, generator=g).to(device).requires_grad_(True)
    dy = torch.randn(2, 70, 128, generator=g).to(torch.bfloat16).to(device)

    def step():
        for p in [x] + list(blk.parameters()):
            p.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = pkg.dsqg_block_forward(blk, x)
        out.backward(dy)
        return {n: p.grad for n, p in [("x", x)] + list(blk.named_parameters())}

    full = {n: None if t is None else t.clone() for n, t in step().items()}
    assert full["x"].dtype == torch.float32 and full["qkvg_proj.weight"].dtype == torch.float32
    gone = ["x"] if frozen == "x" else ["qkvg_proj.weight", "qkvg_proj.bias", "out_proj.weight"]
    for n in gone:
        (x if n == "x" else dict(blk.named_parameters())[n]).requires_grad_(False)
    part = step()
    for n, t in full.items():
        if n in gone:
            assert part[n] is None
        elif t is not None:
            assert torch.equal(part[n], t), n


def test_block_one_node_compiles(pkg, device):
    """torch.compile traces the block's node with fullgraph; out and dx have the eager bits (the same launches)."""
    offsets = list(pkg.lattice.build_offset_groups(2048)[0])
    blk = StandInBlock(256, 4, offsets, sum(d <= 28 for d in offsets), 2, 64, seed=3).to(device)
    x = torch.randn(2, 96, 256, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(device)

    def step(inp):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return pkg.dsqg_block_forward(blk, inp)

    a, b = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    ea = step(a)
    eb = torch.compile(step, fullgraph=True)(b)
    ea.float().sum().backward()
    eb.float().sum().backward()
    assert torch.equal(ea, eb) and torch.equal(a.grad, b.grad)


@pytest.mark.parametrize("inner", ["tables", "nothing"])
def test_block_second_backward_is_refused(pkg, device, inner):
    """A gradient taken with create_graph cannot be differentiated again: the second backward raises, also where
    only the projections and the input have gradients (the tables frozen), and does not give a partial gradient."""
    offsets = list(pkg.lattice.build_offset_groups(2048)[0])
    blk = StandInBlock(128, 2, offsets, sum(d <= 28 for d in offsets), 2, 64, seed=6).to(device)
    if inner == "nothing":
        for n, p in blk.named_parameters():
            p.requires_grad_("proj" in n)
    x = torch.randn(1, 70, 128, generator=torch.Generator().manual_seed(3)).to(device).requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = pkg.dsqg_block_forward(blk, x)
    (dx,) = torch.autograd.grad(out.float().sum(), x, create_graph=True)
    assert dx.requires_grad
    with pytest.raises(RuntimeError):
        (out.float().sum() + dx.square().sum()).backward()


@pytest.mark.parametrize("H,N,lattice", [(8, 1025, "canonical"), (3, 700, "far")])
def test_block_schedules_give_the_same_bits(pkg, device, monkeypatch, H, N, lattice):
    """The block's backward with the gate launch's (delta, lse) pairs beside two streams, and with one stream, where
    the dQ launch forms them: every gradient bit for bit.  "far": queries before the smallest offset take no part."""
    offsets, js = (list(pkg.ALL_OFFSETS), 17) if lattice == "canonical" else ([64, 96, 128, 200, 333], 0)
    blk = StandInBlock(64 * H, H, offsets, js, 3, 10 ** 6, seed=17).to(device)   # 10^6: no support cropping
    g = torch.Generator().manual_seed(18)
    x = torch.randn(2, N, 64 * H, generator=g).to(torch.bfloat16).to(device).requires_grad_(True)
    dy = torch.randn(2, N, 64 * H, generator=g).to(torch.bfloat16).to(device)
    params = [p for n, p in blk.named_parameters() if p.requires_grad and not n.startswith("npci")]
    got = {}
    for two in (True, False):
        monkeypatch.setattr(pkg.dsqg, "_worth_two_streams", lambda q, J: two)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = pkg.dsqg_block_forward(blk, x)
        got[two] = torch.autograd.grad(out, [x] + params, dy)
    for i, (a, b) in enumerate(zip(got[True], got[False])):
        assert torch.equal(a, b), i
