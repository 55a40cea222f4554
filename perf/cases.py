"""Workloads of the library, each one pass through its public entry points.

The ranges are the shapes the library is used at: the training microbatch
(B15 H8 T2048, head_dim 64, width 512) with the whole 96-offset lattice and
with the trainer's per-block 29-offset groups, the long context (T8192),
grouped K/V heads, odd and short sequences, fp32, the width-512 scans and
rotations around the attention, and the q6 cache (write and prefill, and the
nine-layer decode step from one to 256 sequences).

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` does one pass,
``work`` is what one pass cannot do without, ``exact`` the same results in
plain 64-bit torch.

Small launches in steady loops (the decode step, the EMA scan, the packet, the
rotation) are run as a program runs them that must not pay the host for each
launch: captured once into a HIP graph over fixed buffers and replayed.  The
attention calls and the block are eager calls.
"""

from __future__ import annotations

import importlib
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

HD = 64          # head dim
R = 4            # MOVT planes
J_SMALL_MAX = 28  # offsets up to this are the near ones
CLIP = (1e-5, 0.5)  # EMA factor bounds
TABLES = ("pos_bias", "scale_embed", "phase_base", "phase_gain")


def _pkg():
    return importlib.import_module("dwarf-v2_amd")


def listed():
    return [
        # one DSQG layer of the training microbatch, forward and backward, y/z given by the caller
        dict(name="attention_microbatch", op="attention", B=15, H=8, Hkv=8, N=2048, lattice="full", shift=0,
             dtype="bf16", probes=False, grad=True),
        # the long context, probe features inside the kernels
        dict(name="attention_long", op="attention", B=4, H=8, Hkv=8, N=8192, lattice="full", shift=4,
             dtype="bf16", probes=True, grad=True),
        # grouped K/V heads at a ragged length
        dict(name="attention_gqa_ragged", op="attention", B=7, H=8, Hkv=2, N=1999, lattice="full", shift=6,
             dtype="bf16", probes=False, grad=True),
        # a short sequence through one of the trainer's 29-offset groups: launches and latency
        dict(name="attention_short", op="attention", B=2, H=8, Hkv=8, N=261, lattice="third1", shift=2,
             dtype="bf16", probes=True, grad=True),
        # fp32 training of one sequence (parity runs, fp32 fine-tuning)
        dict(name="attention_fp32", op="attention", B=1, H=8, Hkv=8, N=2048, lattice="full", shift=0,
             dtype="fp32", probes=False, grad=True),
        # a whole DSQG block of the trainer (projections, attention on a 29-offset group, gates, output projection)
        # under bf16 autocast, forward and backward
        dict(name="block_train", op="block", B=15, H=8, N=2048, lattice="third0", shift=2),
        # the causal EMA at long context, per-channel factors, forward and backward
        dict(name="ema_long", op="ema", B=4, N=8192, D=512, dtype="bf16", per_channel=True, reset=False),
        # the InterferencePacket (three scans, mix, direction, confidence, gate), forward and backward
        dict(name="packet_microbatch", op="packet", B=15, N=2048, D=512, dtype="bf16"),
        # the kv_inject rotation of one layer's keys, forward and backward
        dict(name="npci_keys", op="npci", B=15, H=8, N=2048, dtype="bf16"),
        # serving prefill: quantise the prompt's K/V into the cache and attend over it
        dict(name="q6_prefill", op="prefill", B=20, H=8, Hkv=8, N=2048, shift=0),
        # serving decode: one token for 256 sequences, nine layers
        dict(name="q6_decode_256", op="decode", S=256, L=9, H=8, Hkv=8, N=2048, shift=0),
        # serving decode for a handful of sequences
        dict(name="q6_decode_5", op="decode", S=5, L=9, H=8, Hkv=8, N=1537, shift=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["attention"] * 5 + ["block", "ema", "packet", "npci", "prefill", "decode", "decode"])
    shift = rng.randrange(0, 15)
    if op == "attention":
        fp32 = rng.random() < 0.2
        N = _log(rng, 130, 2600 if fp32 else 8192)
        if rng.random() < 0.3:
            N = max(128, N // 64 * 64)
        B = max(1, min(15, _log(rng, 1, 20), (3000 if fp32 else 32000) // N))
        Hkv = rng.choice([8, 8, 8, 4, 2, 1])
        return dict(op="attention", B=B, H=8, Hkv=Hkv, N=N, lattice=rng.choice(["full", "full", "third0", "third1", "third2"]),
                    shift=shift, dtype="fp32" if fp32 else "bf16", probes=rng.random() < 0.5, grad=rng.random() < 0.8)
    if op == "block":
        N = _log(rng, 200, 4096)
        return dict(op="block", B=max(1, min(15, 30000 // N, _log(rng, 1, 20))), H=8, N=N,
                    lattice=rng.choice(["full", "third0", "third1", "third2"]), shift=shift)
    if op == "ema":
        N = _log(rng, 100, 8192)
        return dict(op="ema", B=max(1, min(15, 32000 // N, _log(rng, 1, 20))), N=N, D=rng.choice([512, 512, 384, 1000]),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]), per_channel=rng.random() < 0.5, reset=rng.random() < 0.3)
    if op == "packet":
        N = _log(rng, 100, 2048)
        return dict(op="packet", B=max(1, min(15, 30000 // N, _log(rng, 1, 20))), N=N, D=rng.choice([512, 512, 384, 1000]),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if op == "npci":
        N = _log(rng, 100, 8192)
        return dict(op="npci", B=max(1, min(15, 32000 // N, _log(rng, 1, 20))), H=8, N=N,
                    dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if op == "prefill":
        N = _log(rng, 100, 4096)
        return dict(op="prefill", B=max(1, min(20, 40000 // N, _log(rng, 1, 24))), H=8, Hkv=rng.choice([8, 8, 2]), N=N,
                    shift=shift)
    return dict(op="decode", S=_log(rng, 1, 256), L=9, H=8, Hkv=rng.choice([8, 8, 2]), N=rng.choice([2048, 1537, 1024, 300]),
                shift=shift)


# ---- inputs ----------------------------------------------------------------------------------------------------
def _lattice(name):
    """(offsets, number of near offsets): the whole lattice, or one of the trainer's three per-block groups."""
    p = _pkg()
    off = list(p.ALL_OFFSETS) if name == "full" else list(p.lattice.build_offset_groups(2048)[int(name[-1])])
    return off, sum(d <= J_SMALL_MAX for d in off)


def _dtype(name):
    return torch.float32 if name == "fp32" else torch.bfloat16


class _Draws:
    """Seeded normal draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def __call__(self, *shape, std=1.0, dtype=torch.float32):
        return (std * torch.randn(*shape, generator=self.g, device="cuda")).to(dtype)


def _features(x, probes):
    """<x, p_r> / sqrt(|x|^2 + 1e-6 hd), as the block forms y and z."""
    return (x @ probes.t().to(x.dtype)) * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6 * HD)


def _tables(d, J, jl, H, lead=()):
    pb = d(*lead, J, H, std=0.02)
    se = d(*lead, J, HD, std=0.01)
    se = se - se.mean(-2, keepdim=True)
    return dict(pos_bias=pb, scale_embed=se, phase_base=d(*lead, jl, H, R, std=0.005),
                phase_gain=d(*lead, jl, H, R, std=0.64))


def _probes(shift):
    q, k = _pkg()._orthogonal_phase_probes(R, HD, shift)
    return q.cuda(), k.cuda()


def _attention_inputs(c, seed):
    d = _Draws(seed)
    off, js = _lattice(c["lattice"])
    dt = _dtype(c["dtype"])
    B, H, Hkv, N = c["B"], c["H"], c["Hkv"], c["N"]
    t = dict(q=d(B, H, N, HD, dtype=dt), k=d(B, Hkv, N, HD, dtype=dt), v=d(B, Hkv, N, HD, dtype=dt))
    dout = d(B, H, N, HD, dtype=dt)
    t.update(_tables(d, len(off), len(off) - js, H))
    qp, kp = _probes(c["shift"])
    if not c["probes"]:
        t["y_pre"], t["z_pre"] = _features(t["q"].float(), qp), _features(t["k"].float(), kp)
    return t, dout, off, js, qp, kp


class _Block(nn.Module):
    """The attributes the DSQG block's forward reads."""

    def __init__(self, c, d):
        super().__init__()
        off, js = _lattice(c["lattice"])
        H, D = c["H"], c["H"] * HD
        J, jl = len(off), len(off) - js
        self.num_heads, self.head_dim, self.minimum_offset = H, HD, min(off)
        self.support_crop_projections, self.support_crop_min_offset = True, 64
        self.qkvg_proj = nn.Linear(D, 4 * D, bias=True, device="cuda")
        self.out_proj = nn.Linear(D, D, bias=False, device="cuda")
        with torch.no_grad():
            self.qkvg_proj.weight.copy_(d(4 * D, D, std=D ** -0.5))
            self.qkvg_proj.bias.copy_(d(4 * D, std=0.1))
            self.out_proj.weight.copy_(d(D, D, std=D ** -0.5))
        qp, kp = _probes(c["shift"])
        self.query_probes = nn.Parameter(qp, requires_grad=False)
        self.key_probes = nn.Parameter(kp, requires_grad=False)
        t = _tables(d, J, jl, H)
        self.phase_gate = nn.Parameter(d(jl))
        self.pos_bias = nn.Parameter(t["pos_bias"])
        self.centered_scale_embed = nn.Parameter(t["scale_embed"])
        self.phase_base = nn.Parameter(2 * t["phase_base"])
        self.phase_gain = nn.Parameter(2 * t["phase_gain"])
        self.if_gain = nn.Parameter(1.0 + d(H, std=0.1))
        self.register_buffer("offsets_dev", torch.tensor(off, dtype=torch.int32, device="cuda"))
        self.j_val, self.j_small, self.j_large = J, js, jl
        self.sparse_order_dev = self.group_start_dev = self.group_len_dev = None
        self.group_dmin_dev = self.group_dmax_dev = None
        self.k_group_size, self.grouped_mode_id, self.verify_mode, self.max_group_spread_observed = 3, 0, False, 0
        self.plane_shift, self.backend, self.online_softmax = c["shift"], "auto", True
        self.dropout = nn.Dropout(0.0)

    def trained(self):
        return [(n, p) for n, p in self.named_parameters() if p.requires_grad]


def _block_inputs(c, seed):
    d = _Draws(seed)
    D = c["H"] * HD
    x = d(c["B"], c["N"], D, dtype=torch.bfloat16)
    dy = d(c["B"], c["N"], D, dtype=torch.bfloat16)
    return x, dy, _Block(c, d)


def _scan_inputs(c, seed):
    d = _Draws(seed)
    B, N, D, dt = c["B"], c["N"], c["D"], _dtype(c["dtype"])
    t = dict(x=d(B, N, D, dtype=dt), dy=d(B, N, D, dtype=dt))
    if c["op"] == "packet":
        t["gate"] = d(B, N, D, std=1.5, dtype=dt)
        t["factors"] = torch.tensor([1 / 16, 1 / 64, 1 / 256], device="cuda")
        t["mixture"] = torch.softmax(d(3, std=0.3), 0)
    else:
        u = torch.rand(D if c["per_channel"] else 1, generator=d.g, device="cuda")
        t["alpha"] = 0.001 + 0.099 * u
        t["reset"] = torch.rand(B, N, generator=d.g, device="cuda") < 1e-3 if c["reset"] else None
    return t


def _npci_inputs(c, seed):
    d = _Draws(seed)
    B, H, N, dt = c["B"], c["H"], c["N"], _dtype(c["dtype"])
    return dict(x=d(B, N, H, HD, dtype=dt).transpose(1, 2), delta=d(B, H, N, HD, std=0.3, dtype=dt),
                theta=0.25 * torch.tanh(d(H)), dy=d(B, H, N, HD, dtype=dt))


def _prefill_inputs(c, seed):
    d = _Draws(seed)
    off, js = _lattice("full")
    bf = torch.bfloat16
    t = dict(q=d(c["B"], c["H"], c["N"], HD, dtype=bf), k=d(c["B"], c["Hkv"], c["N"], HD, dtype=bf),
             v=d(c["B"], c["Hkv"], c["N"], HD, dtype=bf))
    t.update(_tables(d, len(off), len(off) - js, c["H"]))
    return t, off, js


def _decode_inputs(c, seed):
    """Query rows, positions and tables; the K/V rows of one layer come from ``_decode_rows``."""
    d = _Draws(seed)
    off, js = _lattice("full")
    t = dict(q=d(c["S"], c["L"], c["H"], HD, dtype=torch.bfloat16))
    t["pos"] = torch.randint(96, c["N"], (c["S"],), generator=d.g, device="cuda", dtype=torch.int32)
    t.update(_tables(d, len(off), len(off) - js, c["H"], lead=(c["L"],)))
    return t, off, js


def _decode_rows(c, seed, layer):
    d = _Draws(seed * 31 + 7 + layer)
    return (torch.randn(c["S"], c["Hkv"], c["N"], HD, generator=d.g, device="cuda", dtype=torch.bfloat16),
            torch.randn(c["S"], c["Hkv"], c["N"], HD, generator=d.g, device="cuda", dtype=torch.bfloat16))


# ---- one pass --------------------------------------------------------------------------------------------------
def _attention_pass(s):
    p, c, t = _pkg(), s["case"], s["t"]
    feats = (s["qp"], s["kp"]) if c["probes"] else (t["y_pre"], t["z_pre"])
    entry = p.dsqg_attention_with_probes if c["probes"] else p.dsqg_attention_v18_grouped
    js, J = s["js"], s["J"]
    with torch.set_grad_enabled(c["grad"]):
        out = entry(t["q"], t["k"], t["v"], *(t[n] for n in TABLES), *feats, J, js, J - js, s["off"], None, None, None,
                    None, None, 3, 0, False, 0, c["shift"], s["start"])
        if not c["grad"]:
            return {"out": out}
        grads = torch.autograd.grad(out, list(t.values()), s["dout"])
    return {"out": out.detach(), **dict(zip(t, grads))}


def _block_pass(s):
    p, blk = _pkg(), s["block"]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = p.dsqg_block_forward(blk, s["x"])
    named = s["named"]
    grads = torch.autograd.grad(out, [s["x"]] + [w for _, w in named], s["dy"])
    return {"out": out.detach(), "x": grads[0], **{n: g for (n, _), g in zip(named, grads[1:])}}


def _ema_pass(s):
    t = s["t"]
    y = _pkg().causal_ema_scan(t["x"], t["alpha"], *CLIP, reset_mask=t["reset"])
    dx, da = torch.autograd.grad(y, (t["x"], t["alpha"]), t["dy"])
    return {"y": y.detach(), "dx": dx, "dalpha": da}


def _packet_pass(s):
    t = s["t"]
    y = _pkg().interference_packet(t["x"], t["factors"], t["mixture"], t["gate"])
    g = torch.autograd.grad(y, (t["x"], t["factors"], t["mixture"], t["gate"]), t["dy"])
    return {"packet": y.detach(), "dx": g[0], "dfactors": g[1], "dmixture": g[2], "dgate": g[3]}


def _npci_pass(s):
    t = s["t"]
    y = _pkg().npci_rotate(t["x"], t["delta"], t["theta"])
    g = torch.autograd.grad(y, (t["x"], t["delta"], t["theta"]), t["dy"])
    return {"out": y.detach(), "dx": g[0], "ddelta": g[1], "dtheta": g[2]}


def _prefill_pass(s):
    q6, t = _pkg().q6, s["t"]
    cache = q6.pack_kv(t["k"], t["v"], s["kp"])
    out = q6.q6_prefill(t["q"], cache, *(t[n] for n in TABLES), s["qp"], s["off"], s["js"], s["J"] - s["js"],
                        s["case"]["shift"], 1)
    return {"cache": cache, "out": out}


def _decode_pass(s):
    t = s["t"]
    return {"out": _pkg().q6.q6_decode(t["q"], t["pos"], s["caches"], *(t[n] for n in TABLES), s["qps"], s["off"],
                                       s["js"], s["J"] - s["js"], s["case"]["shift"])}


PASSES = dict(attention=_attention_pass, block=_block_pass, ema=_ema_pass, packet=_packet_pass, npci=_npci_pass,
              prefill=_prefill_pass, decode=_decode_pass)
GRAPHED = ("ema", "packet", "npci", "decode")


def _leaves(t, *names):
    for n in names:
        t[n] = t[n].detach().requires_grad_(True)


def _capture(s, one_pass):
    """The pass in a HIP graph over the state's buffers."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        one_pass(s)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        s["result"] = one_pass(s)
    s["graph"] = graph


def prepare(case, seed):
    c, op = case, case["op"]
    s = {"case": c}
    if op == "attention":
        t, s["dout"], off, js, s["qp"], s["kp"] = _attention_inputs(c, seed)
        if c["grad"]:
            _leaves(t, *t)
        s.update(t=t, start=min(off))
    elif op == "block":
        s["x"], s["dy"], s["block"] = _block_inputs(c, seed)
        s["x"].requires_grad_(True)
        s["named"] = s["block"].trained()
        off = js = None
    elif op in ("ema", "packet"):
        s["t"], off, js = _scan_inputs(c, seed), None, None
        _leaves(s["t"], *(("x", "alpha") if op == "ema" else ("x", "factors", "mixture", "gate")))
    elif op == "npci":
        s["t"], off, js = _npci_inputs(c, seed), None, None
        _leaves(s["t"], "x", "delta", "theta")
    elif op == "prefill":
        s["t"], off, js = _prefill_inputs(c, seed)
        qp, kp = _probes(c["shift"])
        s["qp"], s["kp"] = F.normalize(qp, dim=-1), F.normalize(kp, dim=-1)
    else:
        s["t"], off, js = _decode_inputs(c, seed)
        qp, kp = (F.normalize(p, dim=-1) for p in _probes(c["shift"]))
        s["qps"] = torch.stack([qp] * c["L"])
        s["caches"] = torch.empty((c["L"], c["S"], c["Hkv"], c["N"], 128), dtype=torch.uint8, device="cuda")
        for layer in range(c["L"]):
            s["caches"][layer] = _pkg().q6.pack_kv(*_decode_rows(c, seed, layer), kp)
    if off is not None:
        s.update(off=torch.tensor(off, dtype=torch.int32, device="cuda"), js=js, J=len(off))
    if op in GRAPHED:
        _capture(s, PASSES[op])
    return s


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["result"]
    return PASSES[state["case"]["op"]](state)


# ---- what one pass cannot do without ---------------------------------------------------------------------------
def _pairs(off, N):
    return sum(max(0, N - d) for d in off)


def _attention_work(B, H, Hkv, N, off, js, size, probes, grad):
    J = len(off)
    rows, kv = B * H * N, B * Hkv * N
    tables = 4 * (J * H + J * HD + 2 * (J - js) * H * R)
    row = HD * size
    plane = 0 if probes else 4 * R
    bytes_ = rows * (2 * row + plane) + kv * (2 * row + plane) + tables
    flops = 4.0 * HD * B * H * _pairs(off, N)
    if grad:
        # dO in; dq, dk, dv and the plane gradients out; the table gradients out
        bytes_ += rows * (2 * row + plane) + kv * (2 * row + plane) + tables
        flops += 10.0 * HD * B * H * _pairs(off, N)
    return bytes_, flops


def work(case):
    c, op = case, case["op"]
    if op == "attention":
        off, js = _lattice(c["lattice"])
        b, f = _attention_work(c["B"], c["H"], c["Hkv"], c["N"], off, js, 4 if c["dtype"] == "fp32" else 2, c["probes"],
                               c["grad"])
        return {"bytes": b, "flops": f}
    if op == "block":
        # x and dy in, out and dx out (bf16); five D x D weights in and their gradients out (fp32)
        off, _ = _lattice(c["lattice"])
        D, rows = c["H"] * HD, c["B"] * c["N"]
        return {"bytes": 4 * rows * D * 2 + 2 * 5 * D * D * 4,
                "flops": 3 * 2.0 * rows * D * 5 * D + 14.0 * HD * c["B"] * c["H"] * _pairs(off, c["N"])}
    if op in ("ema", "packet"):
        n, size = c["B"] * c["N"] * c["D"], 4 if c["dtype"] == "fp32" else 2
        # ema: x, dy in, y, dx out; packet: x, gate, dy in, packet, dx, dgate out
        return {"bytes": n * size * (4 if op == "ema" else 6), "flops": n * (10 if op == "ema" else 60)}
    if op == "npci":
        n, size = c["B"] * c["H"] * c["N"] * HD, 4 if c["dtype"] == "fp32" else 2
        return {"bytes": n * size * 6, "flops": n * 30}
    off, js = _lattice("full")
    if op == "prefill":
        q, kv = c["B"] * c["H"] * c["N"], c["B"] * c["Hkv"] * c["N"]
        return {"bytes": q * 2 * 2 * HD + kv * (2 * 2 * HD + 128), "flops": 4.0 * HD * c["B"] * c["H"] * _pairs(off, c["N"])}
    mean = sum(max(0, c["N"] - max(d, 96)) for d in off) / (c["N"] - 96)   # valid offsets of a position in [96, N)
    tables = 4 * c["L"] * (len(off) * (c["H"] + HD) + 2 * (len(off) - js) * c["H"] * R)
    return {"bytes": c["S"] * c["L"] * (c["H"] * 4 * HD + c["Hkv"] * mean * 120) + tables,
            "flops": 4.0 * HD * c["S"] * c["L"] * c["H"] * mean}


def tolerance(case):
    """About four times the error measured against ``exact`` (the worst output of a kind): half an ulp of bf16 is 1.7e-3
    in norm; the attention's gradients reach 3.6e-2 of the rms at single elements; the packet and the block round to bf16
    several times on the way."""
    op = case["op"]
    if case.get("dtype") == "fp32":
        return {"attention": {"rel": 2e-6, "max": 2e-5}, "ema": {"rel": 1.6e-5, "max": 1e-4},
                "packet": {"rel": 3e-6, "max": 2e-5}, "npci": {"rel": 1.2e-6, "max": 4e-6}}[op]
    return {"attention": {"rel": 7e-3, "max": 0.15}, "packet": {"rel": 3e-2, "max": 0.08},
            "block": {"rel": 2.4e-2, "max": 0.2}}.get(op, {"rel": 7e-3, "max": 0.016})


# ---- the same in 64 bits ---------------------------------------------------------------------------------------
class _Attention64(torch.autograd.Function):
    """DSQG attention in float64, one offset at a time: out[n] = sum_j P[n,j] Rot(theta[n,j]) v[n - d_j], P the softmax
    of <q[n], k[n - d_j] + e_j> / 8 + pos_bias over the offsets with a source, far offsets rotated by
    theta = base + gain y[n] z[n - d_j] on the planes' channel pairs."""

    @staticmethod
    def _rotated(v, theta, ch):
        a, b = v[..., ch], v[..., ch + 1]
        c, s = torch.cos(theta), torch.sin(theta)
        w = v.clone()
        w[..., ch], w[..., ch + 1] = c * a - s * b, s * a + c * b
        return w

    @staticmethod
    def forward(ctx, q, k, v, pb, se, base, gain, y, z, off, js, shift, start):
        B, H, N, hd = q.shape
        ch = torch.arange(R, device=q.device) * (hd // R) + shift
        S = torch.full((len(off), B, H, N), -math.inf, device=q.device, dtype=q.dtype)
        for j, d in enumerate(off):
            lo = max(d, start)
            if lo < N:
                S[j, :, :, lo:] = (q[:, :, lo:] * (k[:, :, lo - d:N - d] + se[j])).sum(-1) / 8 + pb[j].view(1, H, 1)
        m = S.amax(0)
        P = torch.exp(S - torch.where(m.isinf(), 0.0, m))
        P = P / P.sum(0).clamp_min(1e-300)
        out = torch.zeros_like(q)
        for j, d in enumerate(off):
            lo = max(d, start)
            if lo < N:
                w = v[:, :, lo - d:N - d]
                if j >= js:
                    th = base[j - js].view(1, H, 1, R) + gain[j - js].view(1, H, 1, R) * y[:, :, lo:] * z[:, :, lo - d:N - d]
                    w = _Attention64._rotated(w, th, ch)
                out[:, :, lo:] += P[j, :, :, lo:, None] * w
        ctx.save_for_backward(q, k, v, se, base, gain, y, z, P, out)
        ctx.args = (off, js, start, ch)
        return out

    @staticmethod
    def backward(ctx, g):
        q, k, v, se, base, gain, y, z, P, out = ctx.saved_tensors
        off, js, start, ch = ctx.args
        B, H, N, hd = q.shape
        dq, dk, dv, dy, dz = (torch.zeros_like(t) for t in (q, k, v, y, z))
        dpb = torch.zeros(len(off), H, device=q.device, dtype=q.dtype)
        dse, dbase, dgain = torch.zeros_like(se), torch.zeros_like(base), torch.zeros_like(gain)
        delta = (g * out).sum(-1)
        for j, d in enumerate(off):
            lo = max(d, start)
            if lo >= N:
                continue
            src, p, gn = slice(lo - d, N - d), P[j, :, :, lo:], g[:, :, lo:]
            if j >= js:
                i = j - js
                bv, gv = base[i].view(1, H, 1, R), gain[i].view(1, H, 1, R)
                th = bv + gv * y[:, :, lo:] * z[:, :, src]
                w = _Attention64._rotated(v[:, :, src], th, ch)
                dth = p[..., None] * (gn[..., ch + 1] * w[..., ch] - gn[..., ch] * w[..., ch + 1])
                dbase[i] += dth.sum((0, 2))
                dgain[i] += (dth * y[:, :, lo:] * z[:, :, src]).sum((0, 2))
                dy[:, :, lo:] += dth * gv * z[:, :, src]
                dz[:, :, src] += dth * gv * y[:, :, lo:]
                dv[:, :, src] += _Attention64._rotated(p[..., None] * gn, -th, ch)
            else:
                w = v[:, :, src]
                dv[:, :, src] += p[..., None] * gn
            ds = p * ((gn * w).sum(-1) - delta[:, :, lo:])
            dpb[j] += ds.sum((0, 2))
            dq[:, :, lo:] += ds[..., None] * (k[:, :, src] + se[j]) / 8
            t = ds[..., None] * q[:, :, lo:] / 8
            dk[:, :, src] += t
            dse[j] += t.sum((0, 1, 2))
        return dq, dk, dv, dpb, dse, dbase, dgain, dy, dz, None, None, None, None


def _attention64(t, qp, kp, off, js, shift, start, round_se):
    """t: float64 leaves; y/z from the probes where t has none.  round_se: the 16-bit path reads scale_embed as bf16."""
    H, Hkv = t["q"].shape[1], t["k"].shape[1]
    y = t["y_pre"] if "y_pre" in t else _features(t["q"], qp.double())
    z = t["z_pre"] if "z_pre" in t else _features(t["k"], kp.double())
    se = t["scale_embed"]
    if round_se:
        se = se + (se.detach().to(torch.bfloat16).double() - se.detach())
    k, v, z = (x.repeat_interleave(H // Hkv, 1) if H != Hkv else x for x in (t["k"], t["v"], z))
    return _Attention64.apply(t["q"], k, v, t["pos_bias"], se, t["phase_base"], t["phase_gain"], y, z, off, js, shift, start)


def _leaf64(t):
    return t.detach().double().requires_grad_(True)


def _exact_attention(c, seed):
    t, dout, off, js, qp, kp = _attention_inputs(c, seed)
    if c["B"] * c["H"] * c["N"] * len(off) > 6e7:
        return None
    t = {n: _leaf64(x) for n, x in t.items()}
    out = _attention64(t, qp, kp, off, js, c["shift"], min(off), c["dtype"] == "bf16")
    if not c["grad"]:
        return {"out": out.detach()}
    return {"out": out.detach(), **dict(zip(t, torch.autograd.grad(out, list(t.values()), dout.double())))}


def _exact_block(c, seed):
    x, dy, blk = _block_inputs(c, seed)
    off, js = _lattice(c["lattice"])
    named = blk.trained()
    p = {n: _leaf64(w) for n, w in named}
    x = _leaf64(x)
    B, N, D = x.shape
    H = c["H"]
    q, k, v, gate = (x @ p["qkvg_proj.weight"].t() + p["qkvg_proj.bias"]).split(D, dim=-1)
    q, k, v = (t.reshape(B, N, H, HD).permute(0, 2, 1, 3) for t in (q, k, v))
    pg = torch.sigmoid(p["phase_gate"])[:, None, None]
    t = dict(q=q, k=k, v=v, pos_bias=p["pos_bias"], scale_embed=p["centered_scale_embed"],
             phase_base=p["phase_base"] * pg, phase_gain=p["phase_gain"] * pg)
    out = _attention64(t, blk.query_probes, blk.key_probes, off, js, c["shift"], min(off), True)
    out = (out * p["if_gain"].view(1, H, 1, 1)).permute(0, 2, 1, 3).reshape(B, N, D)
    out = (out * torch.sigmoid(gate)) @ p["out_proj.weight"].t()
    grads = torch.autograd.grad(out, [x] + list(p.values()), dy.double())
    return {"out": out.detach(), "x": grads[0], **dict(zip(p, grads[1:]))}


def _scan64(x, a, keep):
    """states of y[t] = a x[t] + (1 - a) keep[t] y[t-1] over dim 1; a broadcasts over the last dims."""
    s, rows = torch.zeros_like(x[:, 0] * a), []
    for t in range(x.shape[1]):
        s = torch.addcmul(a * x[:, t], (1 - a), s if keep is None else s * keep[:, t])
        rows.append(s)
    return torch.stack(rows, 1)


def _adjoint64(g, a, keep):
    """lam[t] = g[t] + (1 - a) keep[t+1] lam[t+1]."""
    s, rows = torch.zeros_like(g[:, 0] * a), []
    for t in range(g.shape[1] - 1, -1, -1):
        if keep is not None and t + 1 < g.shape[1]:
            s = s * keep[:, t + 1]
        s = torch.addcmul(g[:, t], (1 - a), s)
        rows.append(s)
    return torch.stack(rows[::-1], 1)


def _before(y, keep):
    prev = torch.cat((torch.zeros_like(y[:, :1]), y[:, :-1]), 1)
    return prev if keep is None else prev * keep


def _exact_ema(c, seed):
    t = _scan_inputs(c, seed)
    x, g, a = t["x"].double(), t["dy"].double(), t["alpha"].double()
    keep = None if t["reset"] is None else (~t["reset"]).double()[..., None]
    y = _scan64(x, a, keep)
    lam = _adjoint64(g, a, keep)
    da = (lam * (x - _before(y, keep))).sum((0, 1))
    return {"y": y, "dx": a * lam, "dalpha": da if c["per_channel"] else da.sum().reshape(1)}


def _exact_packet(c, seed):
    t = _scan_inputs(c, seed)
    x, gate, w, g = (t[n].double() for n in ("x", "gate", "mixture", "dy"))
    a = t["factors"].double().view(3, 1)
    y = _scan64(x[:, :, None], a, None)                      # [B, N, 3, D]
    u = _leaf64((y * w.view(3, 1)).sum(2))
    gate = _leaf64(gate)
    ms = u.square().mean(-1, keepdim=True)
    out = u * torch.rsqrt(ms + 1e-6) * torch.tanh(ms.sqrt() / 0.25) * torch.sigmoid(gate)
    du, dgate = torch.autograd.grad(out, (u, gate), g)
    lam = _adjoint64(du[:, :, None] * w.view(3, 1), a, None)
    return {"packet": out.detach(), "dx": (a * lam).sum(2), "dfactors": (lam * (x[:, :, None] - _before(y, None))).sum((0, 1, 3)),
            "dmixture": (du[:, :, None] * y).sum((0, 1, 3)), "dgate": dgate}


def _exact_npci(c, seed):
    t = _npci_inputs(c, seed)
    x, d, th = (_leaf64(t[n]) for n in ("x", "delta", "theta"))
    n = x.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    u = x / n
    p = d - (d * u).sum(-1, keepdim=True) * u
    m = p.norm(dim=-1, keepdim=True)
    angle = th.view(1, -1, 1, 1) * torch.tanh(m / (0.25 * n + 1e-12))
    out = torch.cos(angle) * x + torch.sin(angle) * n * p / m.clamp_min(1e-20)
    g = torch.autograd.grad(out, (x, d, th), t["dy"].double())
    return {"out": out.detach(), "dx": g[0], "ddelta": g[1], "dtheta": g[2]}


def _q6_rows(x):
    """A row's value after the cache's codec: two groups of 32, code rint(x / s) in [-31, 31], s = fp16(absmax / 31)."""
    g = x.float().reshape(*x.shape[:-1], 2, 32)
    s = (g.abs().amax(-1, keepdim=True) / 31.0).to(torch.float16).float()
    code = torch.round(g / torch.where(s == 0, 1.0, s)).clamp(-31, 31)
    return (code.double() * s.double()).reshape(x.shape)


def _exact_prefill(c, seed):
    t, off, js = _prefill_inputs(c, seed)
    if c["B"] * c["H"] * c["N"] * len(off) > 6e7:
        return None
    qp, kp = _probes(c["shift"])
    t = {n: (_q6_rows(x) if n in "kv" else x.double()) for n, x in t.items()}
    return {"cache": None, "out": _attention64(t, qp, kp, off, js, c["shift"], 1, True)}


def _exact_decode(c, seed):
    t, off, js = _decode_inputs(c, seed)
    qp, kp = (p.double() for p in _probes(c["shift"]))
    S, H, Hkv = c["S"], c["H"], c["Hkv"]
    src = t["pos"].long()[:, None] - torch.tensor(off, device="cuda")             # [S, J]
    ok = (src >= 0)[:, None]
    idx = src.clamp_min(0)[:, None, :, None].expand(S, Hkv, len(off), HD)
    head = torch.arange(H, device="cuda") // (H // Hkv)
    ch = torch.arange(R, device="cuda") * (HD // R) + c["shift"]
    outs = []
    for layer in range(c["L"]):
        k, v = (_q6_rows(x.gather(2, idx))[:, head] for x in _decode_rows(c, seed, layer))   # [S, H, J, 64]
        q = t["q"][:, layer].double()
        se = t["scale_embed"][layer].to(torch.bfloat16).double()
        score = (q[:, :, None] * (k + se)).sum(-1) / 8 + t["pos_bias"][layer].double().t()
        P = torch.softmax(score.masked_fill(~ok, -math.inf), -1)
        y, z = _features(q, qp), _features(k, kp)
        th = t["phase_base"][layer].double().transpose(0, 1) + t["phase_gain"][layer].double().transpose(0, 1) * y[:, :, None] * z[:, :, js:]
        w = torch.cat((v[:, :, :js], _Attention64._rotated(v[:, :, js:], th, ch)), 2)
        outs.append((P[..., None] * w).sum(2))
    return {"out": torch.stack(outs, 1)}


EXACT = dict(attention=_exact_attention, block=_exact_block, ema=_exact_ema, packet=_exact_packet, npci=_exact_npci,
             prefill=_exact_prefill, decode=_exact_decode)


def exact(case, seed):
    return EXACT[case["op"]](case, seed)
