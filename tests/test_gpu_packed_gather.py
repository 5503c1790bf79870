"""GPU parity of the gather of short rows (several tokens a load from 4096
tokens up) and of the shapes next to it with the CPU oracle: bit-exact rows,
rows of no sequence untouched."""

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from pipeswift_amd import cache_ops
from tests.conftest import raw

pytestmark = pytest.mark.gpu

DT = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "f32", torch.float8_e4m3fn: "fp8"}


@pytest.mark.parametrize("lens,row,ps,cache,out,starts,two", [
    ([4096 - 7], 128, 16, torch.float8_e4m3fn, torch.bfloat16, False, True),        # 16 vectors: four tokens a load
    ([700, 0, 1, 4000], 256, 16, torch.float8_e4m3fn, torch.float16, True, True),   # 32 vectors: two
    ([3] * 1200 + [1, 0] * 900, 128, 24, torch.bfloat16, torch.bfloat16, True, True),  # a lane walks past its window
    ([0] * 70 + [4500] + [0] * 70 + [1], 8, 7, torch.float8_e4m3fn, torch.bfloat16, True, False),  # one vector a row
    ([2100, 2100], 128, 1, torch.float8_e4m3fn, torch.float32, False, True),        # 32 vectors of 4 bytes
    ([4300], 96, 16, torch.bfloat16, torch.bfloat16, False, True),                  # 12 vectors: not packed
    ([2050, 2040], 512, 64, torch.float8_e4m3fn, torch.bfloat16, True, True),       # 64 vectors: not packed
])
def test_short_rows(dev, lens, row, ps, cache, out, starts, two):
    g = torch.Generator().manual_seed(row + ps)
    P, W, B = 37, -(-max(lens) // ps) + 1, len(lens)
    src = (torch.randn(P, 2, ps, row, generator=g) * 2).to(cache)
    bt = torch.randint(0, P, (B, W), generator=g, dtype=torch.int32)
    bt[::3, 0] = P                             # no such page: zero rows
    bt[1::5, 0] = -1
    st = torch.randint(0, 3 * ps, (B,), generator=g, dtype=torch.int32)  # some rows past the table: zeros
    cu = torch.tensor(np.r_[0, np.cumsum(lens)], dtype=torch.int32) + 2   # two rows before the first sequence
    T = int(cu[-1]) + 5
    assert T >= 4096
    print(f"gather: {T} rows of {row} {cache} to {out}, {B} sequences, pages of {ps}", flush=True)
    dst = torch.full((2, T, row), 7.0, dtype=torch.float32).to(out)
    sd, dd = src.to(dev), dst.to(dev)
    fp8 = cache == torch.float8_e4m3fn
    scale = torch.tensor([0.37], dtype=torch.float32) if fp8 else None
    kw = {"src_cache_v": sd[:, 1], "dst_v": dd[1]} if two else {}
    cache_ops.gather_cache(sd[:, 0], dd[0], bt.to(dev), cu.to(dev), seq_starts=st.to(dev) if starts else None,
                           scale=scale.to(dev) if fp8 else None, **kw)
    for i in range(2):
        exp = raw(dst[i]).copy()
        if i == 0 or two:
            O.gather_cache(raw(src[:, i]), bt.numpy(), cu.numpy(), seq_starts=st.numpy() if starts else None, out=exp,
                           cache_dtype=DT[cache], out_dtype=DT[out], scale=float(scale[0]) if fp8 else None)
        assert np.array_equal(raw(dd[i]), exp)
