"""Top-k rows with penalties that only lower values (repetition >= 1, presence and frequency >= 0): decided
from the elements above a sampled bound and their counts alone, or handed to the penalty pass. Against the
oracle, at the sizes and parameters where the route changes."""

from __future__ import annotations

import math
from dataclasses import fields

import numpy as np
import pytest
import torch

from tests.parity import compare_ids, launches, oracle
from vinfer_amd.registry import BackendContext
from vinfer_amd.sampler import SAMPLER
from vinfer_amd.sampling import PackedParams, SamplingParams, pack_history, pack_params
from vinfer_amd.workloads import Workload

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("V", [16383, 16384, 16385, 24583])  # two whole stripes of 8192 are sampled
def test_lowered_top_k_rows_match_the_oracle(V, dtype):
    s = SAMPLER.resolve("hip", BackendContext(DEV, dtype))
    rng = np.random.default_rng(V)
    x = torch.randn(24, V, generator=torch.Generator().manual_seed(V)) * 2.5
    order = x.argsort(dim=1, descending=True)
    rows, hist, draft = [], [], []

    def row(k, ids, d=0, **kw):
        rows.append(SamplingParams(**{"temperature": 0.8, "top_k": k, "top_p": 0.95, "repetition_penalty": 1.1,
                                      "presence_penalty": 0.4, "frequency_penalty": 0.2, **kw}))
        hist.append([int(i) for i in ids])
        draft.append(int(d))

    def some(n):
        return rng.integers(0, V, n)

    for k in (1, 2, 50, 191, 192, 193):  # the largest top-k served, one past it
        row(k, some(300), order[len(rows), 0])
    row(50, order[6, :10].repeat(3), order[6, 3])  # the best tokens penalised, the draft among them
    row(50, order[7, :4000], order[7, 0])  # every candidate penalised: too few stay
    row(50, order[8, ::2].repeat(2)[:9000], order[8, 1])  # every other one, a long history
    row(50, some(100), order[9, 5], repetition_penalty=0.9)  # raises values: the penalty pass
    row(50, some(100), order[10, 5], presence_penalty=-0.5)
    row(50, some(100), order[11, 5], frequency_penalty=-0.1)
    row(50, some(100), order[12, 5], repetition_penalty=1.0, presence_penalty=0.0, frequency_penalty=0.0)  # off
    row(20, [-1, -7, V, V + 5, *some(40)], order[13, 0])  # ids outside the vocabulary
    row(50, [], order[14, 0])
    row(50, some(100), order[15, 0])
    x[15, :] = (x[15] * 0.5).round()  # ties
    row(50, some(100), order[16, 0])
    x[16, 40:] = -math.inf  # fewer than k finite
    row(5, [3, 3, 4], 4)
    x[17, 100] = math.inf
    row(5, [3, 3, 4], 4)
    x[18, 100] = math.nan
    row(30, some(3000), order[19, 2], min_p=0.2)
    row(30, some(3000), order[20, 2], temperature=0.0)
    row(30, order[21, :1].repeat(5000), order[21, 0], frequency_penalty=0.01)  # one id's count
    row(30, some(20), order[22, 9], repetition_penalty=3e38)  # products overflow to -inf
    row(30, some(20), 7)
    x[23, :] = 1.5  # all tied
    pp = pack_params(rows)
    ids, off = pack_history(hist)
    logits = x.to(dtype)
    u = torch.from_numpy(rng.random(24, dtype=np.float32))
    w = Workload("lowered", logits, pp, u, ids, off, torch.tensor(draft, dtype=torch.int32))
    print(f"lowered top-k V={V} {dtype}", flush=True)
    d = w.to(DEV)
    for tiles in (False, True):  # (24 rows of this vocabulary: the row launch, then the tile pass's)
        s.tile_pass = tiles
        got, dp = s.sample_batch(d.logits, d.params, d.uniforms, d.hist_ids, d.hist_offsets, d.draft_ids)
        torch.cuda.synchronize()
        _, bad = compare_ids(got, oracle(w), dp)
        assert not bad, (tiles, bad[:8])
    s.tile_pass = True


@pytest.mark.parametrize("V", [16384, 20011])
def test_more_fp32_rows_than_cus_equal_smaller_batches(V):
    # above one row a CU the candidates' rows and the others take a launch each; the same rows in
    # batches of 200 take the one launch
    s = SAMPLER.resolve("hip", BackendContext(DEV, torch.float32))
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    g = torch.Generator(device=DEV).manual_seed(V)
    rng = np.random.default_rng(V)
    for B in (cus, cus + 1, 2 * cus + 5):
        x = torch.randn(B, V, generator=g, device=DEV) * 2.5
        x[5, V - 1] = math.nan
        rows = [SamplingParams(temperature=(0.8, 0.0, 1.1)[b % 3], top_k=(50, 20, 0, 192, 400)[b % 5], top_p=0.9,
                               repetition_penalty=(1.1, 0.95)[b % 7 == 0], presence_penalty=0.3, frequency_penalty=0.1)
                for b in range(B)]
        hist = [rng.integers(0, V, int(rng.integers(0, 400))).tolist() for _ in range(B)]
        u = torch.rand(B, generator=g, device=DEV)
        draft = torch.randint(0, V, (B,), generator=g, device=DEV).to(torch.int32)
        print(f"fp32 rows past the CUs B={B} V={V}", flush=True)

        def run(lo, hi):
            ids, off = pack_history(hist[lo:hi], DEV)
            return s.sample_batch(x[lo:hi], pack_params(rows[lo:hi]).to(DEV), u[lo:hi], ids, off, draft[lo:hi])

        got = run(0, B)
        parts = [run(lo, min(B, lo + 200)) for lo in range(0, B, 200)]
        torch.cuda.synchronize()
        assert torch.equal(got[0], torch.cat([p[0] for p in parts]))
        assert torch.equal(got[1], torch.cat([p[1] for p in parts]))


def penalised_step(s, B, V, mean=0.0, std=2.0, K=50, history=300, best=0, seed=0, **kw):
    """A prepared step of fp32 rows N(mean, std) whose histories hold random ids, the row's `best` largest
    twice among them; and its inputs as a Workload."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(B, V, generator=g, device=DEV) * std + mean
    ids = torch.randint(0, V, (B, history), generator=g, device=DEV).to(torch.int32)
    if best:
        ids[:, :2 * best] = x.topk(best, dim=1).indices.to(torch.int32).repeat(1, 2)
    off = torch.arange(0, B * history + 1, history, dtype=torch.int32, device=DEV)
    p = pack_params([SamplingParams(**{"temperature": 0.8, "top_k": K, "top_p": 0.9, "repetition_penalty": 1.05,
                                       "presence_penalty": 0.3, "frequency_penalty": 0.1, **kw})] * B).to(DEV)
    w = Workload("penalised", x, p, torch.rand(B, generator=g, device=DEV), ids.view(-1), off, None)
    return s.prepare_batch(w.logits, w.params, w.uniforms, w.hist_ids, w.hist_offsets), w


def test_two_launches_only_past_one_row_a_cu_and_from_the_sample_on():
    s = SAMPLER.resolve("hip", BackendContext(DEV, torch.float32))
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    for B, V, want in ((cus, 16384, 1), (cus + 1, 16384, 2), (cus + 1, 16383, 1), (cus + 1, 8192, 1)):
        step, _ = penalised_step(s, B, V)
        step.launch()
        torch.cuda.synchronize()
        assert launches(step.launch) == want, (B, V)


@pytest.mark.parametrize("kw,decided", [
    ({}, True), ({"K": 1}, True), ({"K": 192}, True), ({"K": 193}, False),
    # (bounds between powers of two, where values of one bin of a few key bits are many)
    ({"mean": 20.0, "std": 1.0}, True), ({"mean": 20.0, "std": 1.0, "K": 192}, True), ({"mean": -40.0, "std": 1.0}, True),
    ({"mean": 10.0, "std": 3.0, "K": 192}, True),
    # (the best tokens penalised: fewer than K stay above the sample's bound, a second pass takes the bound that
    # they give; pushed so far down that it would hold a third of the row, none does)
    ({"history": 800, "best": 400, "presence_penalty": 1.0}, True),
    ({"history": 800, "best": 400, "frequency_penalty": 3.0}, False),
    # (greedy rows: the largest penalised value, the best tokens penalised or not)
    ({"temperature": 0.0, "K": 0}, True), ({"temperature": 0.0, "history": 800, "best": 400}, True),
    ({"temperature": 0.0, "repetition_penalty": 0.95}, False), ({"K": 0}, False),
    ({"repetition_penalty": 0.95}, False), ({"std": 0.0}, False),
], ids=str)
def test_the_rows_that_the_candidates_decide(kw, decided):
    # (the first launch marks them, in the workspace's first words; the second leaves the marks)
    s = SAMPLER.resolve("hip", BackendContext(DEV, torch.float32))
    B, V = torch.cuda.get_device_properties(DEV).multi_processor_count + 8, 40000
    print(f"rows the candidates decide {kw}", flush=True)
    step, w = penalised_step(s, B, V, **kw)
    step.launch()
    torch.cuda.synchronize()
    ws = step._keep[-1]
    at = step._args.workspace - ws.data_ptr()
    marks = ws[at:at + 4 * B].view(torch.int32)
    assert bool((marks == -1).all()) == decided and bool((marks == -1).any()) == decided
    few = slice(0, 8)
    n = int(w.hist_offsets[8])
    part = Workload("part", w.logits[few], PackedParams(**{f.name: getattr(w.params, f.name)[few] for f in fields(w.params)}), w.uniforms[few],
                    w.hist_ids[:n], w.hist_offsets[:9], None)
    _, bad = compare_ids(step.ids[few], oracle(part))
    assert not bad, bad


def test_history_append_where_the_rows_take_two_launches():
    # per-row ranges with a spare entry each, rows of the first launch and rows of the second: the draws are those
    # of the same call without append, each drawn id lands behind its row's range, nothing else is written
    s = SAMPLER.resolve("hip", BackendContext(DEV, torch.float32))
    B, V, room = torch.cuda.get_device_properties(DEV).multi_processor_count + 5, 17000, 260
    g = torch.Generator(device=DEV).manual_seed(11)
    x = torch.randn(B, V, generator=g, device=DEV) * 2.5
    x[7, 100] = math.nan
    hist = torch.randint(0, V, (B * room,), generator=g, device=DEV).to(torch.int32)
    start = torch.randperm(B, generator=g, device=DEV) * room  # (the rows' regions in any order)
    length = torch.arange(B, device=DEV) % room  # 0 .. room - 1
    off = torch.stack([start, start + length], 1).to(torch.int32)
    p = pack_params([SamplingParams(temperature=(0.8, 0.0, 1.1)[b % 3], top_k=(50, 192, 400, 0)[b % 4], top_p=0.9,
                                    repetition_penalty=(1.1, 0.95)[b % 7 == 0], presence_penalty=0.3, frequency_penalty=0.1)
                     for b in range(B)]).to(DEV)
    u = torch.rand(B, generator=g, device=DEV)
    want, _ = s.sample_batch(x, p, u, hist.clone(), off)
    step = s.prepare_batch(x, p, u, grown := hist.clone(), off, append_history=True)
    step.launch()
    torch.cuda.synchronize()
    ws = step._keep[-1]
    at = step._args.workspace - ws.data_ptr()
    decided = ws[at:at + 4 * B].view(torch.int32) == -1
    assert 20 < int(decided.sum()) < B - 20
    assert torch.equal(step.ids, want)
    hist[(start + length).long()] = want
    assert torch.equal(grown, hist)
