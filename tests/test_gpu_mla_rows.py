"""GPU parity of the tile-scaled FP8 MLA gather at the edges of its two kernels
(several tokens a wave for the 512 + 64 entry on 16-byte boundaries to bf16, one
token a wave otherwise) with the CPU oracle: bit-exact bf16 rows, rows of no
sequence untouched."""

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from pipeswift_amd import mla_fp8
from tests.conftest import raw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,ps,pad,starts", [
    ([1], 64, 0, False),                       # few tokens and sequences: one token a wave
    ([2, 0, 5], 1, 0, True), ([8], 64, 0, False), ([0, 3, 6, 0], 3, 0, True),
    ([0, 1] + [0] * 6, 64, 0, False),          # 8 sequences, one token: the wave's second has no row
    ([2, 0, 5] + [0] * 6, 1, 0, True),         # seven tokens: a workgroup that is not full
    ([0] * 7 + [8], 64, 0, False),             # a workgroup exactly
    ([0, 3, 6, 0] * 2, 3, 0, True),            # pages of three: division instead of a shift
    ([2000, 2090], 128, 0, True),              # the last of one token a wave (4095 rows with the five beside them)
    ([2000, 2091], 128, 0, True),              # 4096 rows: two tokens a wave
    ([1, 0, 2] * 30, 16, 0, True),             # 90 sequences: past the window of 64
    ([0] * 70 + [5] + [0] * 70 + [4], 4, 0, False),  # empty sequences fill whole windows
    ([3] * 63 + [1, 40], 16, 16, True),        # a wave across the end of the window; entries 672 bytes apart
    ([33, 2], 16, 4, True),                    # entries on 4-byte boundaries: the other kernel
])
def test_gather_rows(dev, lens, ps, pad, starts):
    g = torch.Generator().manual_seed(61 + len(lens) + ps)
    P, W = 24, 44
    E = mla_fp8.entry_bytes(512, 64)
    wide = torch.randint(0, 256, (P, ps, E + pad), generator=g, dtype=torch.uint8)
    # the four scales: any finite f32, and one NaN and one infinity among them
    scales = torch.randn(P, ps, 4, generator=g) * 0.02
    scales[0, 0, 0], scales[1, 0, 1] = float("nan"), float("inf")
    wide[:, :, 512:528] = scales.view(torch.uint8).view(P, ps, 16)
    bt = torch.randint(0, P, (len(lens), W), generator=g, dtype=torch.int32)
    bt[::3, 0] = P                             # no such page: zero rows
    bt[1::3, 0] = -1
    st = torch.randint(0, ps + 2, (len(lens),), generator=g, dtype=torch.int32)
    cu = torch.tensor(np.r_[0, np.cumsum(lens)], dtype=torch.int32) + 2   # two rows before the first sequence
    T = int(cu[-1]) + 3
    print(f"mla rows: {sum(lens)} tokens, {len(lens)} sequences, pages of {ps}, pad {pad}", flush=True)
    out = torch.full((T, 576), 7.0, dtype=torch.bfloat16)
    od = out.to(dev)
    mla_fp8.gather_mla_fp8_tiles(wide.to(dev)[:, :, :E], od, bt.to(dev), cu.to(dev),
                                 seq_starts=st.to(dev) if starts else None)
    exp = raw(out).copy()
    O.gather_mla_tiles(wide.numpy()[:, :, :E], bt.numpy(), cu.numpy(), 512,
                       seq_starts=st.numpy() if starts else None, out=exp, out_dtype="bf16")
    got = raw(od)
    nan = ((exp & 0x7f80) == 0x7f80) & ((exp & 0x7f) != 0)
    assert np.array_equal(got[~nan], exp[~nan])
    assert np.all(((got[nan] & 0x7f80) == 0x7f80) & ((got[nan] & 0x7f) != 0))
