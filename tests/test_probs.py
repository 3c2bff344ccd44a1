"""The probabilities' two launches (the rows' states, then the rows written over the whole chip) against
the one-launch form, which a C caller with the smaller workspace gets: the same bits."""

from __future__ import annotations

import ctypes

import pytest
import torch

from tests.parity import launches
from vinfer_amd import _lib
from vinfer_amd.registry import BackendContext
from vinfer_amd.sampler import SAMPLER
from vinfer_amd.sampling import PackedParams

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def one_launch(s, logits, params, hist_ids, hist_offsets):
    a, keep = s._args(logits, params, hist_ids, hist_offsets)  # (a workspace of vsamp_workspace_bytes())
    B, V = logits.shape
    need = int(s._lib.vsamp_workspace_bytes(B, V, a.hist_total))
    ws = torch.zeros(need + 512, dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = (ws.data_ptr() + 255) & ~255, need
    out = torch.full((B, V), -1.0, device=DEV)
    _lib.check(s._lib.vsamp_probs(ctypes.byref(a), out.data_ptr(), V, s._stream(DEV)))
    torch.cuda.synchronize()
    return out


# (2048 ids a workgroup of the second launch: one short of a tile, one tile, one past it, a large and an odd
# vocabulary, rows on both sides of the 8192 ids from which there are two launches; `offset` moves the rows off
# 16-byte alignment)
@pytest.mark.parametrize("pen", [False, True], ids=["plain", "penalties"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("V,offset", [(1, 0), (2047, 0), (2048, 0), (2049, 1), (50257, 0), (151936, 0), (151936, 3),
                                      (8192, 0), (8193, 0), (10239, 0), (10240, 0), (10241, 1)])
def test_two_launches_equal_one(V, offset, dtype, pen):
    s = SAMPLER.resolve("hip", BackendContext(DEV, dtype))
    g = torch.Generator(device=DEV).manual_seed(V + offset)
    B = 9
    x = torch.randn(B * V + offset, generator=g, device=DEV) * 3.0
    logits = x.to(dtype)[offset:].view(B, V)
    logits[1] = 0.25  # every token tied: the cutoff group splits
    logits[2, 0] = float("inf")
    logits[3, V // 2] = float("nan")
    logits[4] = float("-inf")
    f = lambda v: torch.tensor(v, dtype=torch.float32, device=DEV)  # noqa: E731
    params = PackedParams(
        temperature=f([0.8, 0.7, 0.9, 1.0, 1.0, 0.0, 1.2, 0.5, 1.0]),
        top_k=torch.tensor([0, 0, 0, 0, 0, 0, 50, 700, 0], dtype=torch.int32, device=DEV),
        top_p=f([0.95, 0.6, 0.9, 0.9, 0.9, 1.0, 0.9, 0.99, 1.0]), min_p=f([0, 0, 0, 0, 0, 0, 0, 0, 0.02]),
        repetition_penalty=f([1.1 if pen else 1.0] * B), presence_penalty=f([0.5 if pen else 0.0] * B),
        frequency_penalty=f([0.2 if pen else 0.0] * B))
    ids = off = None
    if pen:  # (one empty history, one past what the histogram path counts)
        lengths = torch.tensor([100, 40, 7, 9, 11, 500, 0, 9000, 3000])
        off = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).to(torch.int32).to(DEV)
        ids = torch.randint(0, V, (int(lengths.sum()),), generator=g, device=DEV).to(torch.int32)
    print(f"probs V={V} offset={offset} {dtype} pen={pen}", flush=True)
    got = s.probs(logits, params, ids, off)
    torch.cuda.synchronize()
    want = one_launch(s, logits, params, ids, off)
    rows = [(r, int((got[r] != want[r]).sum()), got[r][got[r] != want[r]][:3].tolist(), want[r][got[r] != want[r]][:3].tolist())
            for r in range(B) if not torch.equal(got[r], want[r])]
    assert not rows, rows


@pytest.mark.parametrize("pen", [False, True], ids=["plain", "penalties"])
def test_a_workspace_is_used_past_the_penalties_only_when_given_for_it(pen):
    # (without the flag, calls that apply no penalties may share one workspace on several streams)
    s = SAMPLER.resolve("hip", BackendContext(DEV, torch.float32))
    B, V = 5, 20000
    g = torch.Generator(device=DEV).manual_seed(3)
    logits = torch.randn(B, V, generator=g, device=DEV) * 3.0
    f = lambda v: torch.full((B,), v, device=DEV)  # noqa: E731
    params = PackedParams(temperature=f(0.8), top_k=torch.zeros(B, dtype=torch.int32, device=DEV), top_p=f(0.9), min_p=f(0.0),
                          repetition_penalty=f(1.1), presence_penalty=f(0.5), frequency_penalty=f(0.2))
    ids = torch.randint(0, V, (50 * B,), generator=g, device=DEV).to(torch.int32) if pen else None
    off = torch.arange(0, 50 * B + 1, 50, dtype=torch.int32, device=DEV) if pen else None
    want = one_launch(s, logits, params, ids, off)
    for flag in (0, _lib.VSAMP_PROBS_STATES):
        a, keep = s._args(logits, params, ids, off)
        need = int(s._lib.vsamp_probs_workspace_bytes(B, V, a.hist_total))
        kept = int(s._lib.vsamp_workspace_bytes(B, V, a.hist_total)) if pen else 0
        ws = torch.full((need + 512,), 0xA5, dtype=torch.uint8, device=DEV)
        at = (ws.data_ptr() + 255 & ~255) - ws.data_ptr()
        a.workspace, a.workspace_bytes, a.flags = ws.data_ptr() + at, need, a.flags | flag
        out = torch.empty(B, V, device=DEV)
        _lib.check(s._lib.vsamp_probs(ctypes.byref(a), out.data_ptr(), V, s._stream(DEV)))
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert bool((ws[at + kept:at + need] == 0xA5).all()) == (flag == 0)


def test_a_call_makes_one_workspace():
    # (the thread's kept workspace, which the draws use, neither grows nor is made for the probabilities)
    s = SAMPLER.resolve("hip", BackendContext(DEV, torch.float32))
    B, V = 3, 9000
    g = torch.Generator(device=DEV).manual_seed(4)
    logits = torch.randn(B, V, generator=g, device=DEV)
    f = lambda v: torch.full((B,), v, device=DEV)  # noqa: E731
    params = PackedParams(temperature=f(0.8), top_k=torch.zeros(B, dtype=torch.int32, device=DEV), top_p=f(0.9), min_p=f(0.0),
                          repetition_penalty=f(1.1), presence_penalty=f(0.5), frequency_penalty=f(0.2))
    kept = s._local.__dict__.get("workspaces", {}).get(DEV)
    most = 0 if kept is None else kept.numel() // 12
    off = torch.arange(0, 3 * (most + 4000) + 1, most + 4000, dtype=torch.int32, device=DEV)
    ids = torch.randint(0, V, (int(off[-1]),), generator=g, device=DEV).to(torch.int32)
    got = s.probs(logits, params, ids, off)
    torch.cuda.synchronize()
    after = s._local.__dict__.get("workspaces", {}).get(DEV)
    assert after is kept
    assert torch.equal(got, one_launch(s, logits, params, ids, off))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("V,pad", [(8193, 1), (10240, 7), (10007, 64)])
def test_two_launches_write_strided_rows_and_nothing_between(V, pad, dtype):
    s = SAMPLER.resolve("hip", BackendContext(DEV, dtype))
    B = 6
    g = torch.Generator(device=DEV).manual_seed(V)
    logits = (torch.randn(B, V, generator=g, device=DEV) * 3.0).to(dtype)
    f = lambda v: torch.full((B,), v, device=DEV)  # noqa: E731
    params = PackedParams(temperature=f(0.8), top_k=torch.zeros(B, dtype=torch.int32, device=DEV), top_p=f(0.9), min_p=f(0.0),
                          repetition_penalty=f(1.1), presence_penalty=f(0.5), frequency_penalty=f(0.2))
    off = torch.arange(0, 40 * B + 1, 40, dtype=torch.int32, device=DEV)
    ids = torch.randint(0, V, (40 * B,), generator=g, device=DEV).to(torch.int32)
    want = one_launch(s, logits, params, ids, off)
    a, keep = s._args(logits, params, ids, off, own_workspace=True)
    need = int(s._lib.vsamp_probs_workspace_bytes(B, V, a.hist_total))
    ws = torch.empty(need + 256, dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = (ws.data_ptr() + 255) & ~255, need
    a.flags |= _lib.VSAMP_PROBS_STATES
    out = torch.full((B, V + pad), -7.0, device=DEV)
    print(f"probs stride V={V} pad={pad} {dtype}", flush=True)
    _lib.check(s._lib.vsamp_probs(ctypes.byref(a), out.data_ptr(), V + pad, s._stream(DEV)))
    torch.cuda.synchronize()
    assert torch.equal(out[:, :V], want)
    assert bool((out[:, V:] == -7.0).all())


@pytest.mark.parametrize("V,want", [(1, 1), (2000, 1), (8192, 1), (8193, 2)])
def test_short_rows_take_one_launch(V, want):
    s = SAMPLER.resolve("hip", BackendContext(DEV, torch.bfloat16))
    logits = torch.randn(2, V, device=DEV).to(torch.bfloat16)
    f = lambda v: torch.full((2,), v, device=DEV)  # noqa: E731
    params = PackedParams(temperature=f(0.8), top_k=torch.zeros(2, dtype=torch.int32, device=DEV), top_p=f(0.9), min_p=f(0.0),
                          repetition_penalty=f(1.0), presence_penalty=f(0.0), frequency_penalty=f(0.0))
    s.probs(logits, params)
    torch.cuda.synchronize()
    assert launches(lambda: s.probs(logits, params)) == want
