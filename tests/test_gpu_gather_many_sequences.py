"""Gathers of batches past the sequence lookup's one probe (64 + 64 * 64
sequences), or with thousands of empty sequences between two tokens: bit-exact
rows against the CPU oracle, and a time that does not grow with the number of
sequences skipped (a lookup that walks them one dependent load at a time takes
milliseconds: 2.4 ms for 16384 one-token MLA rows, against 12 us)."""

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from pipeswift_amd import cache_ops, mla_fp8
from tests.conftest import raw

pytestmark = pytest.mark.gpu

MANY = [1] * 4159 + [0, 3] * 300 + [2] * 900          # sequences past the probe's reach
EMPTY = ([1] + [0] * 700) * 6 + [4200]                # long stretches without tokens


@pytest.mark.parametrize("lens", [MANY, EMPTY])
def test_mla_rows(dev, lens):
    g = torch.Generator().manual_seed(71 + len(lens))
    P, ps, B = 40, 16, len(lens)
    E = mla_fp8.entry_bytes(512, 64)
    cache = torch.randint(0, 256, (P, ps, E), generator=g, dtype=torch.uint8)
    cache[:, :, 512:528] = (torch.randn(P, ps, 4, generator=g) * 0.02).view(torch.uint8).view(P, ps, 16)
    cache[:, :, :512] &= 0xbf                          # no NaN codes: whole rows compare as bits
    bt = torch.randint(0, P, (B, -(-max(lens) // ps)), generator=g, dtype=torch.int32)
    cu = torch.tensor(np.r_[0, np.cumsum(lens)], dtype=torch.int32)
    print(f"mla gather: {B} sequences, {int(cu[-1])} rows", flush=True)
    out = torch.full((int(cu[-1]), 576), 7.0, dtype=torch.bfloat16)
    od = out.to(dev)
    mla_fp8.gather_mla_fp8_tiles(cache.to(dev), od, bt.to(dev), cu.to(dev))
    exp = raw(out).copy()
    O.gather_mla_tiles(cache.numpy(), bt.numpy(), cu.numpy(), 512, out=exp, out_dtype="bf16")
    assert np.array_equal(raw(od), exp)


@pytest.mark.parametrize("row", [128, 512])            # packed rows (one head), a row a load
@pytest.mark.parametrize("lens", [MANY, EMPTY])
def test_rows(dev, lens, row):
    g = torch.Generator().manual_seed(72 + len(lens) + row)
    P, ps, B = 40, 16, len(lens)
    src = (torch.randn(P, ps, row, generator=g) * 2).to(torch.float8_e4m3fn)
    bt = torch.randint(0, P, (B, -(-max(lens) // ps)), generator=g, dtype=torch.int32)
    cu = torch.tensor(np.r_[0, np.cumsum(lens)], dtype=torch.int32)
    T = int(cu[-1])
    assert T >= 4096                                   # the short rows' own kernel
    print(f"gather: {B} sequences, {T} rows of {row}", flush=True)
    dst = torch.full((T, row), 7.0, dtype=torch.bfloat16)
    dd, scale = dst.to(dev), torch.tensor([0.37])
    cache_ops.gather_cache(src.to(dev), dd, bt.to(dev), cu.to(dev), scale=scale.to(dev))
    exp = raw(dst).copy()
    O.gather_cache(raw(src), bt.numpy(), cu.numpy(), out=exp, cache_dtype="fp8", out_dtype="bf16", scale=float(scale))
    assert np.array_equal(raw(dd), exp)


@pytest.mark.parametrize("kind", ["mla", "packed", "row"])
def test_time_does_not_follow_the_sequences(dev, kind):
    """16384 sequences of one token against one sequence of 16384: the lookup
    adds a search, not a walk (20x is far above the one, far below the other)."""
    T, ps, P = 16384, 16, 1100
    bt = torch.zeros(T, 1, dtype=torch.int32, device=dev)
    bt1 = torch.arange(T // ps, dtype=torch.int32, device=dev).view(1, -1)
    cu = torch.arange(T + 1, dtype=torch.int32, device=dev)
    cu1 = torch.tensor([0, T], dtype=torch.int32, device=dev)
    if kind == "mla":
        src = torch.zeros(P, ps, mla_fp8.entry_bytes(512, 64), dtype=torch.uint8, device=dev)
        out = torch.empty(T, 576, dtype=torch.bfloat16, device=dev)

        def call(b, c):
            mla_fp8.gather_mla_fp8_tiles(src, out, b, c)
    else:
        src = torch.zeros(P, ps, 128 if kind == "packed" else 512, dtype=torch.float8_e4m3fn, device=dev)
        out = torch.empty(T, src.shape[2], dtype=torch.bfloat16, device=dev)
        scale = torch.ones(1, device=dev)

        def call(b, c):
            cache_ops.gather_cache(src, out, b, c, scale=scale)

    def us(b, c):
        a, e = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        best = float("inf")
        for _ in range(5):
            call(b, c)
            torch.cuda.synchronize()
            a.record()
            for _ in range(20):
                call(b, c)
            e.record()
            e.synchronize()
            best = min(best, a.elapsed_time(e) * 50)
        return best

    one, many = us(bt1, cu1), us(bt, cu)
    print(f"{kind}: one sequence {one:.1f} us, 16384 sequences {many:.1f} us", flush=True)
    assert many <= 20 * one
