"""The 16-wave scan (16-bit activations) at the shapes and layouts it takes beyond the model's
own: other d_state, head_dim and angle counts, every rank, groups, padded and reversed token
strides, calls without phases, biases or a start, and the calls at the edges of a sub-chunk.

Each is compared with the oracle run in FP32 on the same 16-bit values. The bar is 2-norm
relative: the kernel rounds q / k, the decayed weights, the scaled values, the state and the
output once each to the activation dtype, six roundings of at most u = 2^-9 (bf16) or 2^-12 (f16)
relative each, and as root of the sum of squares of uniform errors (u / sqrt 3) that is 1.5 u;
asserted at 3 u for the output and the state.
"""

from __future__ import annotations

import math

import pytest
import torch

from mamba3_amd import Mamba3, _hip, ops
from oracle import portable as op

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
BAR = {torch.bfloat16: 3 * 2.0 ** -9, torch.float16: 3 * 2.0 ** -12}


def _close(got, want, dtype):
    got, want = got.double().cpu(), want.double()
    assert got.shape == want.shape
    err = ((got - want).norm() / want.norm()).item()
    assert err <= BAR[dtype], f"relative error {err:.3e}"


def _inputs(rank, dtype, *, batch, length, heads, groups, head_dim, d_state, angles, bias,
            initial, seed):
    g = torch.Generator().manual_seed(seed)

    def rand(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g) * scale).to(dtype)

    inp = dict(q=rand(batch, length, groups, rank, d_state), k=rand(batch, length, groups, rank, d_state),
               value=rand(batch, length, heads, head_dim), gate=rand(batch, length, heads, head_dim),
               dt=torch.rand(batch, length, heads, generator=g) * 0.1 + 0.001,
               trap_logits=rand(batch, length, heads), D=torch.randn(heads, generator=g))
    inp["adt"] = -torch.rand(batch, length, heads, generator=g) * inp["dt"] * 3
    if rank > 1:
        for name in ("mimo_x", "mimo_z", "mimo_out"):
            # values of the activation dtype: the kernel rounds mimo_x and mimo_z to it
            inp[name] = rand(heads, rank, head_dim, scale=0.5).float()
    if angles:
        inp["phase"] = (torch.rand(batch, length, heads, angles, generator=g) * 2 - 1) * 6
        inp["mimo_rotation"] = rank > 1
    if bias:
        inp["q_bias"] = (1 + 0.1 * torch.randn(heads, rank, d_state, generator=g)).to(dtype).float()
        inp["k_bias"] = (1 + 0.1 * torch.randn(heads, rank, d_state, generator=g)).to(dtype).float()
    if initial:
        inp["initial_state"] = torch.randn(batch, heads, head_dim, d_state, generator=g) * 0.3
        inp["initial_k"] = rand(batch, heads, rank, d_state)
        inp["initial_value"] = rand(batch, heads, head_dim)
    return inp


def _oracle32(inp):
    return op.ssd_scan(**{n: (t.float() if isinstance(t, torch.Tensor) else t)
                          for n, t in inp.items()}, chunk_size=16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank,groups,head_dim,d_state,angles,length,bias,initial", [
    (1, 1, 64, 128, 32, 64, True, True),     # the model's shape, one full sub-chunk
    (1, 1, 64, 128, 32, 1, True, True),      # one token
    (1, 2, 36, 96, 24, 65, True, True),      # odd widths, two groups, one token over
    (1, 1, 64, 100, 13, 130, True, False),   # d_state no multiple of 8, few angles
    (1, 1, 4, 4, 1, 63, False, True),        # the narrowest rows
    (1, 1, 64, 128, 0, 200, False, False),   # no rotation at all
    (2, 1, 64, 128, 32, 33, True, True),
    (2, 3, 20, 48, 12, 95, True, True),
    (4, 1, 64, 64, 16, 17, True, False),
    (4, 2, 32, 112, 28, 81, False, True),
    (8, 1, 64, 128, 32, 9, True, True),
    (8, 1, 16, 16, 4, 40, True, True),
    (8, 1, 64, 80, 0, 23, True, False),
])
def test_hook_form_shapes(rank, groups, head_dim, d_state, angles, length, bias, initial, dtype):
    inp = _inputs(rank, dtype, batch=2, length=length, heads=6, groups=groups, head_dim=head_dim,
                  d_state=d_state, angles=angles, bias=bias, initial=initial, seed=length)
    want, want_state = _oracle32(inp)
    got, state = ops.mamba3_scan(**{n: (t.to(DEV) if isinstance(t, torch.Tensor) else t)
                                    for n, t in inp.items()})
    _close(got, want, dtype)
    _close(state, want_state, dtype)


def _odd_rows(t):
    """The same values with rows that start on odd elements."""
    wide = torch.zeros((*t.shape[:-1], t.shape[-1] + 7 - t.shape[-1] % 2), dtype=t.dtype,
                       device=t.device)
    wide[..., 1:1 + t.shape[-1]] = t
    return wide[..., 1:1 + t.shape[-1]]


def _error(got, want):
    return ((got.double().cpu() - want.double()).norm() / want.double().norm()).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank,d_state,head_dim,small_dt", [
    (1, 96, 64, False), (1, 100, 36, False), (1, 96, 64, True), (2, 112, 32, False),
    (4, 48, 64, False), (8, 80, 64, False)])
def test_widths_no_power_of_two_are_as_exact_as_the_recurrent_scan(rank, d_state, head_dim,
                                                                   small_dt, dtype):
    """d_state no power of 2: the recurrent scan (which rows on odd elements take) holds the decay
    weights and the scaled values in FP32, and the 16-wave scan must be no further from the FP32
    oracle. With the rounding of both emulated, its error is 0.88-1.00 of the recurrent scan's (the
    state's 0.71-0.93); with the weights rounded once to 16 bits 1.2 at rank 1, with the values
    1.02-1.05 (and 0.87-0.95 for the state). The bar is 1.01: 1% for the sample of some 60,000
    outputs. A small dt (1e-6) puts FP16's scaled values among its subnormal numbers, where one
    16-bit operand keeps few bits."""
    inp = _inputs(rank, dtype, batch=2, length=500, heads=4, groups=1, head_dim=head_dim,
                  d_state=d_state, angles=d_state // 4, bias=True, initial=False, seed=d_state + rank)
    if small_dt:
        inp["dt"] = inp["dt"] * 1e-4
        inp["D"] = torch.zeros_like(inp["D"])
    want, want_state = _oracle32(inp)
    dev = {n: (t.to(DEV) if isinstance(t, torch.Tensor) else t) for n, t in inp.items()}
    got, state = ops.mamba3_scan(**dev)
    odd = dict(dev, q=_odd_rows(dev["q"]), k=_odd_rows(dev["k"]))
    rec, rec_state = ops.mamba3_scan(**odd)
    e, r = _error(got, want), _error(rec, want)
    es, rs = _error(state, want_state), _error(rec_state, want_state)
    print(f"d_state {d_state} R={rank} {dtype}: output {e:.3e} (recurrent {r:.3e}), "
          f"state {es:.3e} ({rs:.3e})", flush=True)
    assert e <= 1.01 * r
    assert es <= 1.01 * rs


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank,d_state,span", [(1, 96, 30.0), (1, 96, 1e4), (2, 48, 1e6), (8, 80, 1e7)])
def test_given_phases_need_no_reduction(rank, d_state, span, dtype):
    """Given phases of many turns at a d_state that is no power of 2: cos and sin to full
    precision whatever the phase, as the recurrent scan takes them (the hardware functions alone
    are off by 2^-24 of the phase: 0.06 at 1e6, where every bar here would be missed)."""
    inp = _inputs(rank, dtype, batch=1, length=200, heads=3, groups=1, head_dim=32, d_state=d_state,
                  angles=d_state // 4, bias=True, initial=True, seed=5)
    inp["phase"] = inp["phase"] * (span / 6)
    want, want_state = _oracle32(inp)
    got, state = ops.mamba3_scan(**{n: (t.to(DEV) if isinstance(t, torch.Tensor) else t)
                                    for n, t in inp.items()})
    _close(got, want, dtype)
    _close(state, want_state, dtype)


@pytest.mark.parametrize("layout", ["padded", "head_major", "unaligned"])
def test_hook_form_layouts(layout):
    """Rows padded to a longer token stride, q / k and value / gate as slices of one buffer,
    head-major values (a token stride below the head stride), and rows that start on odd
    elements (those take the kernel that reads element by element): the same result."""
    inp = _inputs(2, torch.bfloat16, batch=2, length=70, heads=4, groups=1, head_dim=64,
                  d_state=128, angles=32, bias=True, initial=True, seed=7)
    dev = {n: (t.to(DEV) if isinstance(t, torch.Tensor) else t) for n, t in inp.items()}
    want, want_state = ops.mamba3_scan(**dev)

    def relayout(t, name):
        if layout == "head_major" and name in ("value", "gate"):
            return t.transpose(1, 2).contiguous().transpose(1, 2)
        lead, last = t.shape[:-1], t.shape[-1]
        off = 1 if layout == "unaligned" else 8
        wide = torch.full((*lead, last + 16), float("nan"), dtype=t.dtype, device=DEV)
        wide[..., off:off + last] = t
        return wide[..., off:off + last]

    for name in ("q", "k", "value", "gate"):
        dev[name] = relayout(dev[name], name)
    got, state = ops.mamba3_scan(**dev)
    _close(got, want.cpu(), torch.bfloat16)
    _close(state, want_state.cpu(), torch.bfloat16)


@pytest.mark.parametrize("rank,groups,d_state,angles,length,layout", [
    (1, 4, 64, 16, 70, "groups_first"), (2, 4, 128, 32, 70, "groups_first"),
    (2, 2, 128, 32, 45, "ranks_first"), (4, 1, 48, 12, 33, "ranks_first"),
    (8, 4, 16, 4, 19, "q_k_apart"), (4, 2, 112, 0, 40, "q_k_apart"),
    (1, 2, 100, 25, 130, "q_k_apart"), (1, 1, 128, 32, 70, "pairs_j_2s"),
    (1, 1, 128, 32, 1, "one_token"), (4, 4, 64, 16, 1, "one_token"), (1, 1, 96, 24, 1, "one_token"),
])
def test_hook_form_row_layouts(rank, groups, d_state, angles, length, layout):
    """q and k rows as they lie in the caller's buffers: groups ahead of tokens, ranks ahead of
    tokens (whose rows pass the next token's: another kernel), q and k with strides of their own,
    rank 1 with the MIMO pairs (another kernel), and one token whose stride is 0. Against the
    oracle."""
    inp = _inputs(rank, torch.bfloat16, batch=2, length=length, heads=4, groups=groups, head_dim=32,
                  d_state=d_state, angles=angles, bias=True, initial=True, seed=length)
    if layout == "pairs_j_2s":
        inp["mimo_rotation"] = True
    want, want_state = _oracle32(inp)
    dev = {n: (t.to(DEV) if isinstance(t, torch.Tensor) else t) for n, t in inp.items()}
    if layout == "q_k_apart":
        for name, extra in (("q", 4), ("k", 20)):
            t = dev[name]
            wide = torch.full((*t.shape[:2], groups + 1, rank, d_state + extra), float("nan"),
                              dtype=t.dtype, device=DEV)
            wide[:, :, :groups, :, :d_state] = t
            dev[name] = wide[:, :, :groups, :, :d_state]
    elif layout == "one_token":
        for name in ("q", "k"):
            t = dev[name]
            dev[name] = t.as_strided(t.shape, (t.stride(0), 0, *t.stride()[2:]))
    elif layout != "pairs_j_2s":
        axis = 2 if layout == "groups_first" else 3
        for name in ("q", "k"):
            dev[name] = dev[name].transpose(1, axis).contiguous().transpose(1, axis)
    got, state = ops.mamba3_scan(**dev)
    _close(got, want, torch.bfloat16)
    _close(state, want_state, torch.bfloat16)


@pytest.mark.parametrize("rank,d_model,d_state,length,reverse", [
    (1, 96, 96, 70, False), (1, 40, 96, 129, True), (2, 64, 128, 40, False),
    (4, 64, 96, 33, True), (8, 96, 128, 20, False), (4, 128, 128, 1, False),
])
def test_projection_form_shapes(rank, d_model, d_state, length, reverse):
    """The model's mixer at widths other than its own: outputs (both directions) and the cache
    against the oracle's mixer in FP32 on the same bf16 projection."""
    torch.manual_seed(length)
    model = Mamba3(d_model, d_state=d_state, depth=1, mimo_rank=rank).eval()
    params = {n: w.detach().to(torch.bfloat16).float() for n, w in model.state_dict().items()}
    model.load_state_dict(params)
    mixer = model.to(DEV).layers[0].mixer
    width = mixer.in_proj.weight.shape[0]
    proj = torch.randn(2, length, width).to(torch.bfloat16)
    src = proj.flip(1) if reverse else proj
    want, cache = op.mixer_scan(params, "layers.0.mixer.", src.float(),
                                op.Dims(d_model, d_state, rank), chunk=16)
    with torch.inference_mode():
        got, state, phase, k = ops.scan_projection(proj.to(DEV), mixer, want_cache=not reverse,
                                                   reverse=reverse)
    _close(got, want.flip(1) if reverse else want, torch.bfloat16)
    _close(state, cache[1], torch.bfloat16)
    if not reverse:
        _close(k, cache[2], torch.bfloat16)
        turns = (phase.cpu() - cache[0]) / (2 * math.pi)  # whole turns are the same phase
        assert (turns - turns.round()).abs().max() < 1e-4


def test_scan_without_room_for_rows():
    """A hook call whose q and k alone would fill m3_scan_fwd_noalloc's scratch: its rows are read as
    they lie, and the result is the workspace call's."""
    torch.manual_seed(3)
    b, l, h, n, p, r = 20, 1024, 2, 64, 16, 8  # q, k at 128 slots: 84 MB
    mk = lambda *s: torch.randn(*s, device=DEV).to(torch.bfloat16)
    q, k, v, z, tr = mk(b, l, 1, r, n), mk(b, l, 1, r, n), mk(b, l, h, p), mk(b, l, h, p), mk(b, l, h)
    dt = torch.rand(b, l, h, device=DEV) * 0.1
    adt, D = -dt, torch.ones(h, device=DEV)
    mimo = [torch.rand(h, r, p, device=DEV) for _ in range(3)]
    want, want_state = ops.mamba3_scan(q, k, v, z, adt, dt, tr, D, mimo_x=mimo[0], mimo_z=mimo[1],
                                       mimo_out=mimo[2])
    out, state = torch.empty_like(want), torch.empty_like(want_state)
    args = _hip.ScanArgs(batch=b, length=l, heads=h, groups=1, rank=r, d_state=n, head_dim=p,
                         chunk=64, act_dtype=_hip.BF16, phase_mode=_hip.PHASE_NONE, segments=1,
                         norm_eps=1e-5)
    for name, t in dict(q=q, k=k, value=v, gate=z, dt=dt, a=adt, trap=tr, D=D, mimo_x=mimo[0],
                        mimo_z=mimo[1], mimo_out=mimo[2], out=out, final_state=state).items():
        setattr(args, name, _hip.tensor(t))
    _hip.call("m3_scan_fwd_noalloc", args, DEV)
    _close(out, want.cpu(), torch.bfloat16)
    _close(state, want_state.cpu(), torch.bfloat16)


def test_reversed_call_with_far_given_phases():
    """A reversed call whose phases of one batch row span more than 2^29 bytes, with fewer angles
    than the kernel's 32: the lanes without an angle read none of them at any token. The same
    arithmetic as the forward call on flipped inputs, so the same bits."""
    torch.manual_seed(11)
    l, h, n, p, s = 40000, 2, 64, 4, 16
    rows = torch.empty(1, l, 256, s, device=DEV)  # 256 heads' worth: 16 KiB per token, 655 MB
    rows.uniform_(-3, 3)
    mk = lambda *shape: torch.randn(*shape, device=DEV).to(torch.bfloat16)
    t = dict(q=mk(1, l, 1, 1, n), k=mk(1, l, 1, 1, n), value=mk(1, l, h, p), gate=mk(1, l, h, p),
             dt=torch.rand(1, l, h, device=DEV) * 0.1, trap=mk(1, l, h), phase=rows[:, :, :h])
    t["a"] = -t["dt"]
    D = torch.ones(h, device=DEV)

    def scan(tensors, reverse):
        out = torch.empty(1, l, h, p, device=DEV, dtype=torch.bfloat16)
        state = torch.empty(1, h, p, n, device=DEV)
        args = _hip.ScanArgs(batch=1, length=l, heads=h, groups=1, rank=1, d_state=n, head_dim=p,
                             num_angles=s, chunk=64, act_dtype=_hip.BF16,
                             phase_mode=_hip.PHASE_GIVEN, norm_eps=1e-5, segments=1)
        for name, x in dict(tensors, D=D, out=out, final_state=state).items():
            setattr(args, name, _hip.tensor(x))
        if reverse:
            for name in (*tensors, "out"):
                ops._backwards(getattr(args, name), l)
        ws = _hip.scan_workspace(args, DEV)
        _hip.call("m3_scan_fwd", args, DEV)
        del ws
        return out, state

    got, state = scan(t, True)
    flipped = {name: x.flip(1) for name, x in t.items() if name != "phase"}
    flipped["phase"] = torch.empty_like(rows)[:, :, :h]
    flipped["phase"].copy_(t["phase"].flip(1))
    want, want_state = scan(flipped, False)
    assert torch.equal(got, want.flip(1))
    assert torch.equal(state, want_state)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rank,d_state", [(1, 96), (4, 48), (2, 128), (4, 128), (1, 128)])
def test_a_workspace_below_the_answer(rank, d_state, dtype):
    """A call with less workspace than the query asks for takes the routes that need less: at a
    d_state that is no power of 2 none at all; in 16 bits above rank 1, and for the model's shape,
    without the q / k rows. Below that it is refused."""
    torch.manual_seed(rank + d_state)
    mixer = Mamba3(256, d_state=d_state, depth=1, mimo_rank=rank).eval().to(DEV).layers[0].mixer
    proj = torch.randn(2, 300, mixer.in_proj.weight.shape[0], device=DEV).to(dtype)
    with torch.inference_mode():
        call = ops.ScanCall(proj, mixer, want_cache=True)
        call.launch()
        want = [t.clone() for t in (call.out, call.final_state, call.final_k)]
        full = call.args.workspace_bytes
        power = d_state & (d_state - 1) == 0
        rows = 2 * 300 * rank * 2 * (2 if rank in (1, 4) else 4) * d_state
        least = 0 if not power else full - rows if dtype == torch.bfloat16 else full
        if power and dtype == torch.bfloat16:
            least += 2 * 300 * rank * 2 * 4  # the norm factors in the rows' place
        for t in (call.out, call.final_state, call.final_k):
            t.fill_(float("nan"))
        # (each region is rounded up to 256 bytes at most)
        call.args.workspace_bytes = min(full, least + 512) if power else 0
        if not power:
            call.args.workspace = None
        call.launch()
        for got, ref in zip((call.out, call.final_state, call.final_k), want):
            if dtype == torch.bfloat16:
                # the model's shape is rounded after its norm, the others are not
                bar = 3 * 2.0 ** -9
            else:
                bar = 1e-6
            assert _error(got, ref.cpu()) <= bar
        if power:
            call.args.workspace_bytes = least // 2
            with pytest.raises(_hip.HipError, match="workspace"):
                call.launch()


def test_noalloc_keeps_the_split():
    """A call whose q / k rows outgrow the scratch (1 x 32768 tokens, rank 2, FP32 rows: 67 MB) stays
    split, reading the caller's rows: bit for bit m3_scan_fwd's result with a workspace that has no
    room for the rows, which keeps the split; an unsplit scan sums in another order."""
    torch.manual_seed(4)
    mixer = Mamba3(128, d_state=128, depth=1, mimo_rank=2).eval().to(DEV).layers[0].mixer
    proj = torch.randn(1, 32768, mixer.in_proj.weight.shape[0], device=DEV).to(torch.bfloat16)
    with torch.inference_mode():
        call = ops.ScanCall(proj, mixer, want_cache=True)
        assert call.args.workspace_bytes > _hip.SCRATCH_BYTES
        call.launch()
        out = call.out.clone()
        call.args.workspace_bytes = _hip.SCRATCH_BYTES
        call.launch()
        want = [t.clone() for t in (call.out, call.final_state, call.final_phase, call.final_k)]
        for t in (call.out, call.final_state, call.final_phase, call.final_k):
            t.fill_(float("nan"))
        args = type(call.args).from_buffer_copy(call.args)
        args.workspace, args.workspace_bytes = None, 0
        _hip.call("m3_scan_fwd_noalloc", args, DEV)
    for got, ref in zip((call.out, call.final_state, call.final_phase, call.final_k), want):
        assert torch.equal(got, ref)
    _close(call.out, out.cpu(), torch.bfloat16)


def test_noalloc_ends_at_the_recurrent_scan():
    """FP32 at a d_state that is no power of 2, more scalar blocks than the scratch holds (800 x 64
    heads x 64 tokens, 68 MB): the recurrent scan, which needs no scratch, as the workspace call."""
    torch.manual_seed(6)
    b, l, h, n, p = 800, 64, 64, 96, 4
    mk = lambda *s: torch.randn(*s, device=DEV)
    t = dict(q=mk(b, l, 1, 1, n), k=mk(b, l, 1, 1, n), value=mk(b, l, h, p), gate=mk(b, l, h, p),
             dt=torch.rand(b, l, h, device=DEV) * 0.1, trap=mk(b, l, h), D=torch.ones(h, device=DEV))
    t["a"] = -t["dt"]
    want, want_state = ops.mamba3_scan(t["q"], t["k"], t["value"], t["gate"], t["a"], t["dt"],
                                       t["trap"], t["D"])
    out, state = torch.empty_like(want), torch.empty_like(want_state)
    args = _hip.ScanArgs(batch=b, length=l, heads=h, groups=1, rank=1, d_state=n, head_dim=p,
                         chunk=64, act_dtype=_hip.F32, phase_mode=_hip.PHASE_NONE, norm_eps=1e-5)
    for name, x in dict(t, out=out, final_state=state).items():
        setattr(args, name, _hip.tensor(x))
    _hip.call("m3_scan_fwd_noalloc", args, DEV)
    assert _error(out, want.cpu()) <= 1e-6
    assert _error(state, want_state.cpu()) <= 1e-6
