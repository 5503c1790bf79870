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


@pytest.mark.parametrize("Hq,Hkv,lens", [(16, 1, [200]), (16, 1, [40, 0, 3000, 17]), (32, 2, [5, 900]),
                                         (64, 4, [260, 1]), (3, 1, [130, 131])])
def test_few_kv_heads(dev, Hq, Hkv, lens):
    """Workgroups whose waves share a kv head write its record together: 2 to 8
    waves a head, all their rows, every 64th column of a row that does not end
    on a wave (3 query heads: 384 columns over 8 waves)."""
    _case(dev, 1540 + Hq + Hkv, len(lens), Hq, Hkv, 16, 300, lens, "bf16", torch.float32, "per_seq_head")


def test_few_kv_heads_cost_no_more(dev):
    """200 tokens of 16 query heads over one kv head against 32 over 8: an
    eighth of the bytes.  One wave writing the workgroup's record alone took
    1.42x the time; shared by its waves it is 1.06x."""
    from pipeswift_amd import attention

    def us(Hq, Hkv, n=50):
        kv = torch.zeros(16, 2, 16, Hkv, 128, dtype=torch.float8_e4m3fn, device=dev)
        bt = torch.arange(13, dtype=torch.int32, device=dev).view(1, 13)
        lens = torch.full((1,), 200, dtype=torch.int32, device=dev)
        q = torch.zeros(1, Hq, 128, dtype=torch.float8_e4m3fn, device=dev)
        out = torch.empty(1, Hq, 128, dtype=torch.bfloat16, device=dev)
        ws = torch.empty(attention.workspace_floats(1, Hq, Hkv, 208), dtype=torch.float32, device=dev)

        def call():
            attention.paged_decode_attention(q, kv[:, 0], kv[:, 1], bt, lens, out=out, workspace=ws)

        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(n):
                call()
        a, e = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        best = float("inf")
        for _ in range(7):
            a.record()
            graph.replay()
            e.record()
            e.synchronize()
            best = min(best, a.elapsed_time(e) * 1e3 / n)
        return best

    one, eight = us(16, 1), us(32, 8)
    print(f"16 over 1: {one:.1f} us, 32 over 8: {eight:.1f} us", flush=True)
    assert one <= 1.25 * eight
