"""Sequences the library splits into segments of which the last is shorter: split against
unsplit, over ranks, dtypes, walked phases (projection form), given or no phases (hook form),
starts and widths."""

from __future__ import annotations

import pytest
import torch

from mamba3_amd import Mamba3, _hip, ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
# 2-norm relative. The split sums each state in another order and, in 16 bits, rounds the state
# before another token of the same sub-chunk grid: FP32 sums of a few thousand terms agree to
# about 1e-6; a 16-bit output to one rounding (2^-9) per element at worst
BAR = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -9}


def _close(got, want, dtype):
    err = ((got.double() - want.double()).norm() / want.double().norm()).item()
    assert err <= BAR[dtype], f"relative error {err:.3e}"


def _segments(call) -> int:
    return _hip.scan_segments(call.args, 1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d_model,d_state,rank,batch,length", [
    (128, 128, 1, 1, 1777),  # 28 sub-chunks of 64 tokens in 16 bits
    (128, 128, 4, 2, 1001),
    (96, 64, 2, 1, 2049),    # one token in the last sub-chunk
    (64, 128, 8, 1, 700),
    (128, 96, 1, 3, 1500),   # d_state no power of two
    (256, 48, 4, 1, 900),
])
def test_split_matches_unsplit(d_model, d_state, rank, batch, length, dtype, monkeypatch):
    torch.manual_seed(length)
    mixer = Mamba3(d_model, d_state=d_state, depth=1, mimo_rank=rank).eval().to(DEV).layers[0].mixer
    proj = torch.randn(batch, length, mixer.in_proj.weight.shape[0], device=DEV).to(dtype)
    cache = (torch.rand(batch, mixer.nheads, mixer.num_angles, device=DEV) * 6,
             torch.randn(batch, mixer.nheads, mixer.headdim, d_state, device=DEV),
             torch.randn(batch, mixer.nheads, rank, d_state, device=DEV).to(dtype),
             torch.randn(batch, mixer.nheads, mixer.headdim, device=DEV).to(dtype))
    res = {}
    with torch.inference_mode():
        for segs in (1, 0):
            monkeypatch.setattr(ops, "SCAN_SEGMENTS", segs)
            call = ops.ScanCall(proj, mixer, cache=cache, want_cache=True)
            blocks = torch.full((batch, mixer.nheads, (length + 63) // 64, mixer.num_angles),
                                float("nan"), device=DEV)
            decay = torch.full((batch, mixer.nheads), float("nan"), device=DEV)
            call.args.block_phase = _hip.tensor(blocks)
            call.args.final_decay = _hip.tensor(decay)
            assert (_segments(call) > 1) == (segs == 0)
            call.launch()
            res[segs] = (call.out, call.final_state, call.final_phase, call.final_k, blocks, decay)
            back = ops.ScanCall(proj, mixer, reverse=True)
            back.launch()
            res[segs] += (back.out, back.final_state)
    one, split = res[1], res[0]
    for i in (0, 1, 3, 6, 7):
        _close(split[i], one[i], dtype)
    assert torch.equal(split[2], one[2]), "the phase carry differs from the unsplit scan's"
    assert torch.equal(split[4], one[4])
    _close(split[5], one[5], torch.float32)


def test_two_concurrent_calls_take_the_librarys_ragged_count():
    """A bidirectional layer asks for the split of two calls at once and passes the count back: a
    count that does not divide the sequence is accepted when it is the library's own."""
    torch.manual_seed(5)
    mixer = Mamba3(128, d_state=128, depth=1).eval().to(DEV).layers[0].mixer
    proj = torch.randn(1, 2500, mixer.in_proj.weight.shape[0], device=DEV).to(torch.bfloat16)
    with torch.inference_mode():
        call = ops.ScanCall(proj, mixer, concurrent=2)
        assert call.args.segments > 1 and 2500 % call.args.segments != 0
        call.launch()
        want = ops.scan_projection(proj, mixer)
    _close(call.out, want[0], torch.bfloat16)
    _close(call.final_state, want[1], torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d_model,d_state,rank,length", [
    (64, 128, 1, 1000), (64, 128, 4, 33), (64, 64, 2, 70), (256, 96, 1, 130)])
def test_ragged_rows_read_only_their_own(d_model, d_state, rank, length, dtype, monkeypatch):
    """A last sub-chunk that is not full reads nothing past its row: neither what a workspace held
    before (all bits set: NaN) nor the next batch row, here all NaN, reaches the first row."""
    monkeypatch.setattr(ops, "SCAN_SEGMENTS", 1)
    torch.manual_seed(length)
    mixer = Mamba3(d_model, d_state=d_state, depth=1, mimo_rank=rank).eval().to(DEV).layers[0].mixer
    proj = torch.randn(2, length, mixer.in_proj.weight.shape[0], device=DEV).to(dtype)
    with torch.inference_mode():
        want = ops.scan_projection(proj[:1].contiguous(), mixer, want_cache=True)
        proj[1] = float("nan")
        call = ops.ScanCall(proj, mixer, want_cache=True)
        call._keep[-1].fill_(255)
        call.launch()
    for got, ref in zip((call.out, call.final_state, call.final_phase, call.final_k), want):
        assert torch.equal(got[:1], ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rank,d_state,groups,length,given,initial,segments", [
    (1, 128, 1, 1777, True, True, 0),    # 64-token sub-chunks in 16 bits, 32 in FP32
    (2, 128, 1, 1000, True, False, 0),   # 32 and 16: cuts off the 64-token phase blocks
    (2, 64, 2, 1000, False, True, 10),   # a request of 100 tokens a segment, rounded up
    (4, 128, 1, 601, True, True, 0),     # 16 and 8
    (4, 64, 4, 555, False, False, 5),
    (8, 128, 1, 333, True, True, 0),     # 8 and 4
    (8, 16, 2, 260, False, True, 13),
    (1, 96, 2, 1500, True, True, 0),     # d_state no power of two
    (4, 48, 1, 700, True, True, 7),
])
def test_hook_split_matches_unsplit(rank, d_state, groups, length, given, initial, segments, dtype,
                                    monkeypatch):
    """The hook form, split (the state-only first pass, segments on sub-chunks of 64 / rank tokens)
    against unsplit: given phases or none, with and without a start, over the q / k row sources
    (2 heads to a group or 16), and by the routes without copies of the rows."""
    g = torch.Generator(DEV).manual_seed(length)
    heads, p, s = 16 if groups == 1 else 2 * groups, 32, d_state // 4
    mk = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    q, k = (mk(1, length, groups, rank, d_state).to(dtype) for _ in range(2))
    v, z, tr = mk(1, length, heads, p).to(dtype), mk(1, length, heads, p).to(dtype), mk(1, length, heads)
    dt = torch.rand(1, length, heads, generator=g, device=DEV) * 0.1
    kw = dict(phase=mk(1, length, heads, s), mimo_rotation=rank > 1) if given else {}
    if rank > 1:
        kw.update({m: mk(heads, rank, p).to(dtype).float() for m in ("mimo_x", "mimo_z", "mimo_out")})
    if initial:
        kw.update(initial_state=mk(1, heads, p, d_state), initial_k=mk(1, heads, rank, d_state).to(dtype),
                  initial_value=mk(1, heads, p).to(dtype))
    sizes = {}
    query = _hip.scan_workspace

    def scan(segs, short=0):
        monkeypatch.setattr(ops, "SCAN_SEGMENTS", segs)

        def workspace(args, device):
            ws = query(args, device)
            sizes[segs] = args.workspace_bytes
            args.workspace_bytes -= short
            return ws
        monkeypatch.setattr(_hip, "scan_workspace", workspace)
        return ops.mamba3_scan(q, k, v, z, -dt, dt, tr, torch.ones(heads, device=DEV), **kw)

    one, split = scan(1), scan(segments)
    assert sizes[segments] > sizes[1], "not split"
    for got, want in zip(split, one):
        _close(got, want, dtype)
    if dtype == torch.bfloat16 and rank > 1 and groups == 1 and d_state & (d_state - 1) == 0:
        # 256 bytes short of the copies of the rows: they are read as they lie
        for got, want in zip(scan(segments, 256), split):
            assert torch.equal(got, want)


@pytest.mark.parametrize("segments", [1, 3])
@pytest.mark.parametrize("rank,d_state,groups,length", [
    (1, 128, 1, 195), (1, 64, 4, 99), (2, 128, 4, 75), (2, 128, 1, 75), (4, 48, 2, 45), (8, 128, 1, 27),
    (1, 96, 16, 195)])
def test_hook_rows_read_only_their_own(rank, d_state, groups, length, segments, monkeypatch):
    """The hook form's rows end with their batch row and group: the next batch row all NaN, the
    other groups' q and k NaN beside the first's, the workspace all bits set before the call."""
    monkeypatch.setattr(ops, "SCAN_SEGMENTS", segments)
    g = torch.Generator(DEV).manual_seed(length)
    heads, p, s = 16, 32, d_state // 4
    mk = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    dtype = torch.bfloat16
    t = dict(q=mk(2, length, groups, rank, d_state).to(dtype), k=mk(2, length, groups, rank, d_state).to(dtype),
             value=mk(2, length, heads, p).to(dtype), gate=mk(2, length, heads, p).to(dtype),
             dt=torch.rand(2, length, heads, generator=g, device=DEV) * 0.1,
             trap_logits=mk(2, length, heads), phase=mk(2, length, heads, s))
    t["adt"] = -t["dt"]
    kw = dict(D=torch.ones(heads, device=DEV), mimo_rotation=rank > 1)
    if rank > 1:
        kw.update({m: mk(heads, rank, p) for m in ("mimo_x", "mimo_z", "mimo_out")})
    query = _hip.scan_workspace

    def dirty(args, device):
        ws = query(args, device)
        ws.fill_(255)
        return ws
    monkeypatch.setattr(_hip, "scan_workspace", dirty)
    want, want_state = ops.mamba3_scan(**{n: x[:1].contiguous() for n, x in t.items()}, **kw)
    for name, x in t.items():
        x[1] = float("nan")
        if name in ("q", "k") and groups > 1:
            x[0, :, 1:] = float("nan")
    got, state = ops.mamba3_scan(**t, **kw)
    own = heads // groups  # the heads of the first group
    assert torch.equal(got[:1, :, :own], want[:, :, :own])
    assert torch.equal(state[:1, :own], want_state[:, :own])
    assert torch.isfinite(want.float()).all()


@pytest.mark.parametrize("concurrent", [5, 7, 12])
@pytest.mark.parametrize("length", [1055, 2048])
def test_many_concurrent_calls(concurrent, length):
    """More concurrent calls than the library takes ragged counts back for: its answer is one that
    divides the sequence, or no split, and the call runs."""
    torch.manual_seed(length)
    mixer = Mamba3(256, d_state=128, depth=1).eval().to(DEV).layers[0].mixer
    proj = torch.randn(1, length, mixer.in_proj.weight.shape[0], device=DEV).to(torch.bfloat16)
    with torch.inference_mode():
        got = ops.scan_projection(proj, mixer, concurrent=concurrent)
        want = ops.scan_projection(proj, mixer)
    _close(got[0], want[0], torch.bfloat16)
    _close(got[1], want[1], torch.bfloat16)
