"""Sequences the library splits into segments of which the last is shorter: split against
unsplit, over ranks, dtypes, given and walked phases, starts and widths."""

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
    (128, 96, 1, 3, 1500),   # d_state no power of two (FP32: the recurrent scan, never split)
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
            tiled = d_state & (d_state - 1) == 0 or dtype != torch.float32
            if tiled:
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
    if tiled:
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
