"""Host-side behaviour of the Python mirror of the reference interface (no GPU).

Errors are raised with the reference's exception types before any device
work: ValueError for shapes/arguments (dsqg:2209-2225), NotImplementedError
for unsupported modes (dsqg:2217-2221), RuntimeError when no GPU tensors are
given -- this library has no CPU fallback.
"""

import importlib

import pytest
import torch


def _args(B=1, H=2, Hkv=2, N=8, hd=64, J=3, js=2):
    return dict(
        q=torch.zeros(B, H, N, hd), k=torch.zeros(B, Hkv, N, hd), v=torch.zeros(B, Hkv, N, hd),
        pos_bias=torch.zeros(J, H), scale_embed=torch.zeros(J, hd),
        phase_base=torch.zeros(max(J - js, 1), H, 4), phase_gain=torch.zeros(max(J - js, 1), H, 4),
        y_pre=torch.zeros(B, H, N, 4), z_pre=torch.zeros(B, Hkv, N, 4),
    )


def _call(pkg, a, J=3, js=2, backend="auto", mode=0):
    return pkg.dsqg_attention_v18_grouped(
        a["q"], a["k"], a["v"], a["pos_bias"], a["scale_embed"], a["phase_base"], a["phase_gain"],
        a["y_pre"], a["z_pre"], J, js, J - js, torch.tensor([1, 2, 48], dtype=torch.int32),
        None, None, None, None, None, 3, mode, False, 0, 0, 1, backend=backend,
    )


def _fn(pkg, a, mode=0):
    return pkg._DSQGV18GroupedFn.apply(
        a["q"], a["k"], a["v"], a["pos_bias"], a["scale_embed"], a["phase_base"], a["phase_gain"],
        a["y_pre"], a["z_pre"], 3, 2, 1, torch.tensor([1, 2, 48], dtype=torch.int32),
        None, None, None, None, None, 3, mode, False, 0, 0, 1, True,
    )


def test_backend_selection(pkg):
    a = _args()
    with pytest.raises(ValueError):
        _call(pkg, a, backend="cuda")
    with pytest.raises(NotImplementedError):
        _call(pkg, a, backend="eager")
    with pytest.raises(RuntimeError):
        _call(pkg, a)                 # CPU tensors: no fallback
    with pytest.raises(RuntimeError):
        _call(pkg, a, backend="triton")


def test_function_shape_errors(pkg):
    a = _args()
    a["v"] = torch.zeros(1, 2, 9, 64)
    with pytest.raises(ValueError, match="k/v shape mismatch"):
        _fn(pkg, a)
    a = _args(H=3, Hkv=2)
    with pytest.raises(ValueError, match="divisible"):
        _fn(pkg, a)
    a = _args(H=4, Hkv=2)
    with pytest.raises(NotImplementedError):
        _fn(pkg, a, mode=1)
    a = _args()
    a["y_pre"] = torch.zeros(1, 2, 7, 4)
    with pytest.raises(ValueError, match="y_pre"):
        _fn(pkg, a)
    a = _args()
    a["z_pre"] = torch.zeros(1, 1, 8, 4)
    with pytest.raises(ValueError, match="z_pre"):
        _fn(pkg, a)
    a = _args()
    with pytest.raises(RuntimeError, match="device"):
        _fn(pkg, a)


def test_ema_errors(pkg):
    x = torch.zeros(2, 5, 3)
    a = torch.tensor([0.1])
    with pytest.raises(ValueError):
        pkg.causal_ema_scan(torch.zeros(5, 3), a)
    with pytest.raises(ValueError):
        pkg.causal_ema_scan(x, torch.tensor([0.1, 0.2]))
    with pytest.raises(ValueError):
        pkg.causal_ema_scan(x, a, 0.6, 0.5)
    with pytest.raises(ValueError):   # reset_mask must be [B,N] (ema:463-464)
        pkg.causal_ema_scan(x, a, reset_mask=torch.zeros(2, 4, dtype=torch.bool))
    with pytest.raises(RuntimeError):
        pkg.causal_ema_scan(x, a, reset_mask=torch.zeros(2, 5, dtype=torch.bool))
    with pytest.raises(RuntimeError):
        pkg.causal_ema_scan(x, a)
    with pytest.raises(RuntimeError):
        pkg.causal_ema_scan(x, torch.full((3,), 0.1))   # per-channel accepted, but no CPU path


def test_interference_pool_errors(pkg):
    x = torch.zeros(2, 5, 3)
    a, w = torch.tensor([0.1, 0.01, 0.001]), torch.full((3,), 1 / 3)
    with pytest.raises(ValueError):
        pkg.interference_pool(torch.zeros(5, 3), a, w)
    with pytest.raises(ValueError):   # one weight per factor
        pkg.interference_pool(x, a, w[:2])
    with pytest.raises(ValueError):   # at most four timescales
        pkg.interference_pool(x, torch.full((5,), 0.1), torch.full((5,), 0.2))
    with pytest.raises(ValueError):
        pkg.interference_pool(x, a, w, floor=0.6, ceiling=0.5)
    with pytest.raises(RuntimeError):   # no CPU path
        pkg.interference_pool(x, a, w)


def test_q6_errors(pkg):
    with pytest.raises(ValueError):
        pkg.q6.pack_kv(torch.zeros(1, 1, 4, 64), torch.zeros(1, 1, 5, 64))
    with pytest.raises(RuntimeError):
        pkg.q6.pack_kv(torch.zeros(1, 1, 4, 64), torch.zeros(1, 1, 4, 64))
    with pytest.raises(ValueError):
        pkg.q6.unpack_kv(torch.zeros(1, 1, 4, 100, dtype=torch.uint8))


def test_library_is_the_only_path(pkg):
    """The package loads its HIP library eagerly on use and never imports the oracle."""
    import sys

    for name in list(sys.modules):
        if name.startswith("dwarf-v2_amd"):
            mod = sys.modules[name]
            src = open(mod.__file__).read() if getattr(mod, "__file__", None) else ""
            assert "import oracle" not in src and "from oracle" not in src
    assert pkg.native_library_path().endswith("libdwarf_dsqg.so")


def test_backward_sets_the_delta_stage_flag_itself(pkg, monkeypatch):
    """A caller's schedule that carries DWARF_SCHED_DELTA_STAGE does not reach the serial stages (the dQ
    launch would then skip the (delta, lse) pairs dK/dV reads and no delta launch would write them): the
    flag is cleared and set only where the delta launch runs.  The C ABI is replaced by a recorder."""
    dsqg = importlib.import_module("dwarf-v2_amd.dsqg")
    L = pkg._lib
    seen = []

    class Recorder:
        def dwarf_dsqg_bwd_workspace_bytes(self, args):
            return 256

        def __getattr__(self, name):
            def launch(args, stream):
                seen.append((name, args._obj.fwd.schedule))
                return 0
            return launch

    monkeypatch.setattr(dsqg._lib, "load", lambda: Recorder())
    monkeypatch.setattr(dsqg, "_stream", lambda device: 0)
    a = _args(N=8, J=3, js=2)
    a = {n: t.to(torch.bfloat16) if n in ("q", "k", "v") else t for n, t in a.items()}
    off = torch.tensor([1, 2, 48], dtype=torch.int32)
    out, lse = torch.zeros_like(a["q"]), torch.zeros(1, 2, 8)
    for sched in (L.DWARF_SCHED_DELTA_STAGE, L.DWARF_SCHED_BAND | L.DWARF_SCHED_DELTA_STAGE):
        seen.clear()
        dsqg.dsqg_backward(torch.zeros_like(a["q"]), a["q"], a["k"], a["v"], a["pos_bias"], a["scale_embed"],
                           a["phase_base"], a["phase_gain"], a["y_pre"], a["z_pre"], off, out, lse, 2, 1,
                           schedule=sched, overlap=False)
        assert [n for n, _ in seen] == ["dwarf_dsqg_bwd_dq", "dwarf_dsqg_bwd_params", "dwarf_dsqg_bwd_dkdv"]
        assert all(s & L.DWARF_SCHED_DELTA_STAGE == 0 for _, s in seen), seen
        assert all(s == sched & ~L.DWARF_SCHED_DELTA_STAGE for _, s in seen), seen
        seen.clear()
        dsqg.dsqg_backward(torch.zeros_like(a["q"]), a["q"], a["k"], a["v"], a["pos_bias"], a["scale_embed"],
                           a["phase_base"], a["phase_gain"], a["y_pre"], a["z_pre"], off, out, lse, 2, 1,
                           schedule=sched, overlap=True, one_call=True)
        assert seen == [("dwarf_dsqg_bwd", sched)]


def test_custom_ops_default_to_the_python_schedule(pkg):
    """dwarf::dsqg_fwd / dsqg_bwd called without a schedule run the schedule dsqg_forward/backward and the
    autograd Function run (DEFAULT_SCHEDULE), not the gather loops alone."""
    import inspect

    ops = importlib.import_module("dwarf-v2_amd.ops")
    dsqg = importlib.import_module("dwarf-v2_amd.dsqg")
    for fn in (ops.dsqg_fwd, ops.dsqg_bwd):
        schema = fn._opoverload._schema
        arg = [x for x in schema.arguments if x.name == "schedule"][0]
        assert arg.default_value == dsqg.DEFAULT_SCHEDULE
    assert inspect.signature(ops._dsqg_fwd_fake).parameters["schedule"].default == dsqg.DEFAULT_SCHEDULE


def test_schedule_by_mode_and_near_offsets(pkg):
    """The band is set for the overlap-slab modes always, for the baseline mode from the counts at which it is the
    faster schedule, and where the count is not known; the offline softmax flag is independent of it."""
    dsqg = importlib.import_module("dwarf-v2_amd.dsqg")
    L = pkg._lib
    for back, least in ((False, dsqg.BAND_MIN_FORWARD), (True, dsqg.BAND_MIN_BACKWARD)):
        for js in range(18):
            for online in (True, False):
                two = 0 if online else L.DWARF_SCHED_TWO_PASS
                assert dsqg.schedule_for(0, online, js, back) == two | (L.DWARF_SCHED_BAND if js >= least else 0)
                assert dsqg.schedule_for(1, online, js, back) == dsqg.schedule_for(3, online, js, back) \
                    == two | L.DWARF_SCHED_BAND
    assert dsqg.schedule_for(0, True) == dsqg.DEFAULT_SCHEDULE == L.DWARF_SCHED_BAND


def test_integration_guide_names_exist(pkg):
    """Every ``amd.<name>`` the drop-in guide tells a maintainer to bind exists in the package, so the
    rebinding it shows runs as written."""
    import os
    import re

    guide = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "INTEGRATION.md")).read()
    names = sorted(set(re.findall(r"\bamd\.([A-Za-z_][A-Za-z0-9_]*)", guide)))
    assert len(names) >= 15
    missing = [n for n in names if not hasattr(pkg, n)]
    assert not missing, missing


# ---- the block's one node: when it runs (no GPU: the block and a stand-in for x on the CPU) --------------------
def _node_case(pkg, monkeypatch, dtype=torch.bfloat16):
    from types import SimpleNamespace

    from tests.test_gpu_block import StandInBlock

    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *a: True)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda *a: torch.bfloat16)
    blk = StandInBlock(128, 2, [1, 2, 48, 64], 2, 3, 64, seed=1)
    x = SimpleNamespace(is_cuda=True, shape=(2, 8, 128), dtype=dtype, device=torch.device("cpu"))
    assert pkg.block._one_node(blk, SimpleNamespace(**{**vars(x), "dtype": torch.bfloat16}))
    return blk, x


@pytest.mark.parametrize("kind", ["register_module_forward_hook", "register_module_forward_pre_hook",
                                  "register_module_full_backward_hook", "register_module_full_backward_pre_hook",
                                  "instance forward", "weight subclass"])
def test_block_node_gives_way_to_what_changes_a_projection(pkg, monkeypatch, kind):
    """Hooks on every module, a forward set on the instance and a weight that answers for itself are honoured by
    calling the projection, so the block is composed then."""
    blk, x = _node_case(pkg, monkeypatch)
    if kind.startswith("register"):
        handle = getattr(torch.nn.modules.module, kind)(lambda *a: None)
        try:
            assert not pkg.block._one_node(blk, x)
        finally:
            handle.remove()
        assert pkg.block._one_node(blk, x)
    elif kind == "instance forward":
        blk.out_proj.forward = lambda inp: inp
        assert not pkg.block._one_node(blk, x)
    else:
        class Own(torch.Tensor):
            pass

        blk.qkvg_proj.weight = torch.nn.Parameter(blk.qkvg_proj.weight.detach().as_subclass(Own))
        assert not pkg.block._one_node(blk, x)


@pytest.mark.parametrize("wide", ["x", "qkvg_proj.weight", "qkvg_proj.bias", "out_proj.weight"])
def test_block_node_leaves_float64_to_the_projections(pkg, monkeypatch, wide):
    """Autocast leaves float64 alone: a projection of mixed types raises and one all in float64 stays so, which the
    node, all bf16, would not."""
    blk, x = _node_case(pkg, monkeypatch, torch.float64 if wide == "x" else torch.float32)
    if wide != "x":
        assert pkg.block._one_node(blk, x)
        p = dict(blk.named_parameters())[wide]
        p.data = p.data.double()
    assert not pkg.block._one_node(blk, x)


@pytest.mark.parametrize("name", ["if_gain", "qkvg_proj.bias", "out_proj.weight"])
def test_block_node_only_with_everything_on_one_device(pkg, monkeypatch, name):
    """The gate's launch reads if_gain by address: a gain elsewhere goes to the composed block, whose product with it
    raises."""
    blk, x = _node_case(pkg, monkeypatch)
    p = dict(blk.named_parameters())[name]
    owner = blk.get_submodule(name.rpartition(".")[0])
    setattr(owner, name.rpartition(".")[2], torch.nn.Parameter(torch.empty(p.shape, device="meta")))
    assert not pkg.block._one_node(blk, x)


def test_block_raw_launches_check_what_their_kernels_assume(pkg):
    """The raw launches (and the custom ops over them) refuse operands whose shapes or types the kernels would read
    out of range or as something else, before anything is launched."""
    b, bf = pkg.block, torch.bfloat16
    t = lambda *s, dtype=bf: torch.zeros(*s, dtype=dtype)
    bad = [
        lambda: b.linear_wgrad(t(4, 8), t(5, 8), True),                       # other row counts
        lambda: b.linear_wgrad(t(4, 8, dtype=torch.float32), t(4, 8), True),  # not bf16
        lambda: b.linear_wgrad(t(4, 8), t(4, 8, dtype=torch.float16), True),
        lambda: b.head_gate_forward(t(1, 2, 4, 64), t(1, dtype=torch.float32), t(1, 4, 128)),
        lambda: b.head_gate_forward(t(1, 2, 4, 64), t(2), t(1, 4, 128)),
        lambda: b.head_gate_forward(t(1, 2, 4, 64), t(2, dtype=torch.float32), t(1, 4, 64)),
        lambda: b.head_gate_forward(t(1, 2, 4, 32), t(2, dtype=torch.float32), t(1, 4, 64)),
        lambda: b.head_gate_backward(t(1, 4, 64), t(1, 2, 4, 64), t(2, dtype=torch.float32), t(1, 4, 128), t(1, 4, 128)),
        lambda: b.head_gate_backward(t(1, 4, 128), t(1, 2, 4, 64), t(2, dtype=torch.float32), t(1, 4, 128), t(1, 3, 128)),
        lambda: b.block_forward(t(1, 4, 256), *[None] * 6, t(2, dtype=torch.float32), None, 2, 1, 1, 0, 1, 0),
        lambda: b.block_backward(t(1, 4, 128), t(1, 4, 512), *[None] * 6, t(2, dtype=torch.float32), None, t(1, 2, 4, 64),
                                 *[None] * 3, 2, 1, 1, 0, 1, 0),
        lambda: pkg.dsqg.normalize_probes(t(3, 64, dtype=torch.float32), t(4, 64, dtype=torch.float32)),
        lambda: pkg.dsqg.normalize_probes(t(4, 64, dtype=torch.float32), t(4, 64)),
    ]
    for i, call in enumerate(bad):
        with pytest.raises(ValueError, match="expects"):
            call()


def test_linear_wgrad_takes_rows_of_any_stride(pkg, monkeypatch):
    """Rows further apart than the kernel's 32-bit offsets reach (2^22 elements) are copied together first; the
    library is replaced by a recorder."""
    b = pkg.block
    seen = {}

    class Recorder:
        def dwarf_linear_wgrad_workspace_bytes(self, args):
            return 0

        def dwarf_linear_wgrad(self, args, stream):
            seen.update(dy=args._obj.dy_stride, x=args._obj.x_stride)
            return 0

    monkeypatch.setattr(b._lib, "load", lambda: Recorder())
    monkeypatch.setattr(b, "_stream", lambda device: 0)
    far = torch.zeros(2, (1 << 22) + 8, dtype=torch.bfloat16)
    b.linear_wgrad(far[:, :16], far[:, :8], True)
    assert seen == {"dy": 16, "x": 8}
    near = torch.zeros(2, 1 << 22, dtype=torch.bfloat16)
    b.linear_wgrad(near[:, :16], near[:, :8], True)
    assert seen == {"dy": 1 << 22, "x": 1 << 22}
