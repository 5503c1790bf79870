"""GPU parity of the decode reader's balanced schedule where its runs and the
note of a sequence's first and last run can go wrong: fewer tiles than runs, a
tile more or less than the 256 runs of an MI355X, sequences without tokens
before, between and after the others, more sequences than a workgroup has
threads, and one sequence alone on 1, 2, 4 and 8 kv heads per workgroup.  The
oracle, bounds and helper are test_gpu_attention.py's."""

import pytest
import torch

from tests.test_gpu_attention import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [
    [1], [16 * 247 + 1], [16 * 248], [16 * 249 - 3],   # 8 start units and 248 tiles are 256 units
    [0, 0, 5, 0, 4000, 0], [3000, 0, 0], [17] * 40, [0] * 4 + [4001] + [1] * 30,
])
def test_runs_and_spans(dev, lens):
    _case(dev, 1500 + len(lens), len(lens), 32, 8, 16, 300, lens, "fp8", torch.float32, "per_seq_head")


@pytest.mark.parametrize("Hq,Hkv", [(8, 1), (4, 2), (12, 4), (3, 3), (16, 16)])
def test_one_sequence(dev, Hq, Hkv):
    _case(dev, 1520 + Hkv, 1, Hq, Hkv, 16, 400, [6000], "bf16", torch.float32, "per_seq_head")


def test_many_sequences(dev):
    """Two rounds of the workgroups' scan (512 sequences a round), empty ones among them."""
    lens = [(i * 37) % 90 for i in range(700)]
    _case(dev, 1530, 700, 4, 2, 16, 64, lens, "bf16", torch.bfloat16, None)
