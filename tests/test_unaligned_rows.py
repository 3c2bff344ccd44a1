"""Rows that start at any element: every entry point's outputs on them equal those on 16-byte aligned
copies of the same rows (the rows are read 16 bytes at a time at whatever address they have)."""

from __future__ import annotations

import pytest
import torch

from vinfer_amd.registry import BackendContext
from vinfer_amd.sampler import SAMPLER
from vinfer_amd.sampling import PackedParams

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def same(a, b) -> bool:
    return all((x is None and y is None) or torch.equal(x.nan_to_num(7.0), y.nan_to_num(7.0)) for x, y in zip(a, b))


# (below, at and past one 16-byte block, a tile of 128, a stripe of 8192 and the blocks whose low bytes the
# bf16 path keeps)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("V", [5, 8, 129, 8191, 8193, 50257, 155651])
def test_unaligned_rows_equal_aligned_ones(V, dtype):
    s = SAMPLER.resolve("hip", BackendContext(DEV, dtype))
    g = torch.Generator(device=DEV).manual_seed(V)
    B = 16  # odd strides: the rows take every offset
    stride = V + 1 - V % 2
    f = lambda v: torch.full((B,), float(v), device=DEV)  # noqa: E731
    temp = torch.where(torch.arange(B, device=DEV) % 4 == 0, 0.0, 0.9)
    top_k = (torch.arange(B, device=DEV) % 3 * 20).to(torch.int32)
    plain = PackedParams(temperature=temp, top_k=top_k, top_p=f(0.9), min_p=f(0), repetition_penalty=f(1),
                         presence_penalty=f(0), frequency_penalty=f(0))
    pen = PackedParams(temperature=temp, top_k=top_k, top_p=f(0.9), min_p=f(0), repetition_penalty=f(1.1),
                       presence_penalty=f(0.3), frequency_penalty=f(0.1))
    u = torch.rand(B, generator=g, device=DEV)
    ids = torch.randint(0, V, (B * 40,), generator=g, device=DEV).to(torch.int32)
    off = (torch.arange(B + 1, device=DEV) * 40).to(torch.int32)
    draft = torch.randint(0, V, (B,), generator=g, device=DEV).to(torch.int32)
    for shift in (0, 1):
        flat = torch.randn(B * stride + shift, generator=g, device=DEV).mul_(3.0).to(dtype)
        x = flat[shift:].view(B, stride)[:, :V]
        pad = torch.zeros(B, (V + 7) // 8 * 8, dtype=dtype, device=DEV)
        pad[:, :V] = x
        y = pad[:, :V]
        print(f"unaligned V={V} {dtype} shift={shift}", flush=True)
        outs = []
        for z in (x, y):
            o = [*s.sample_batch(z, pen, u, ids, off, draft), *s.sample_tile_pass(z, plain, u, None, None, draft),
                 *s.logprobs(z, draft, min(V, 20)), s.probs(z, pen, ids, off), *s.sample_states(z, plain, u)]
            if dtype == torch.bfloat16:
                o += s.tile_stats(z)
            s.tile_pass = False
            o += s.sample_batch(z, plain, u, None, None, draft)
            s.tile_pass = True
            half = PackedParams(**{k: getattr(plain, k)[: B // 2] for k in plain.__dataclass_fields__})
            # rows (b, 0), (b, 1) of the target; the drafts' rows are the same logits, one of two
            t = z.unflatten(0, (B // 2, 2)) if z is x else z.clone().view(B // 2, 2, V)
            dl = z[::2].unsqueeze(1)
            o += s.verify(t, dl, draft[: B // 2, None], half, u[: B // 2, None], u[B // 2:, None], u[: B // 2])
            outs.append(o)
        torch.cuda.synchronize()
        assert same(*outs)
