"""GPU parity of the prefill-sized FP8 append at the edges of its kernels: rows
of a power of two of eight-element vectors on 16-byte boundaries (two vectors a
lane, wide or short rows) and the shapes next to them, bit-exact against the
CPU oracle, untouched slots included."""

import numpy as np
import pytest
import torch

from oracle import kv_oracle as O
from pipeswift_amd import reshape_and_cache as rc
from tests.conftest import raw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,heads,dim,ps,pad,dtype", [
    (1024, 8, 128, 16, 0, "bf16"),     # 128 vectors: a wave a row
    (1027, 16, 128, 16, 0, "f16"),     # 256: two waves a row
    (1025, 4, 128, 64, 0, "bf16"),     # 64 up to 2560 tokens: the kernel without pairs
    (2560, 4, 128, 64, 0, "bf16"),     # the same
    (2561, 4, 128, 64, 0, "bf16"),     # 64: two rows a wave, one left over
    (1024, 2, 128, 16, 0, "bf16"),     # 32 up to 1024 tokens: the kernel without pairs
    (1025, 2, 128, 16, 0, "f16"),      # 32: four rows a wave, one left over
    (1039, 1, 128, 1, 0, "bf16"),      # 16: eight rows a wave
    (1155, 1, 16, 16, 0, "f16"),       # 2: sixty-four rows a wave
    (1024, 1, 8, 16, 0, "bf16"),       # one vector: the kernel without pairs
    (1030, 3, 128, 16, 0, "bf16"),     # 48: the same
    (1030, 2, 128, 16, 8, "bf16"),     # cache rows on 8-byte boundaries: the same
    (1030, 2, 128, 24, 0, "bf16"),     # pages of 24: the general kernel
])
def test_prefill_fp8_append(dev, tokens, heads, dim, ps, pad, dtype):
    g = torch.Generator().manual_seed(tokens + heads)
    td = {"bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    P, row = max(1400, tokens + 200) // ps + 4, heads * dim
    qkv = (torch.randn(tokens, 4 * row, generator=g) * 3).to(td)
    flat = qkv.view(-1)
    flat[torch.randint(0, flat.numel(), (64,), generator=g)] = float("nan")
    flat[torch.randint(0, flat.numel(), (64,), generator=g)] = float("-inf")
    key, value = qkv[:, row:2 * row].view(tokens, heads, dim), qkv[:, 3 * row:].view(tokens, heads, dim)
    slots = torch.randperm(P * ps, generator=g)[:tokens].to(torch.int64)
    slots[::7] = -1
    slots[5::31] = P * ps
    back = torch.randint(0, 256, (P, 2, ps, row + pad), generator=g, dtype=torch.uint8)
    scales = torch.tensor([0.21, -0.037], dtype=torch.float32)
    print(f"fp8 append: {tokens} tokens, {heads} x {dim}, pages of {ps}, pad {pad}, {dtype}", flush=True)

    def views(t):
        return [t[:, i, :, :row].view(P, ps, heads, dim) for i in range(2)]

    bd, qd = back.to(dev), qkv.to(dev)
    kd, vd = qd[:, row:2 * row].view(tokens, heads, dim), qd[:, 3 * row:].view(tokens, heads, dim)
    kc, vc = views(bd.view(torch.float8_e4m3fn))
    sd = scales.to(dev)
    rc.reshape_and_cache_flash(kd, vd, kc, vc, slots.to(dev), sd[0:1], sd[1:2])
    exp = back.clone()
    ek, ev = (v.numpy() for v in views(exp))
    O.reshape_and_cache(raw(key), raw(value), ek, ev, slots.numpy(), in_dtype=dtype, cache_dtype="fp8",
                        k_scale=float(scales[0]), v_scale=float(scales[1]))
    assert np.array_equal(bd.cpu().numpy(), exp.numpy())
