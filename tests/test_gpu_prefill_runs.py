"""GPU parity of the prefill steps that are cut into equal runs
(``csrc/prefill_runs.hip``): few query blocks, or long cached prefixes.  The
sizes are those where a run's bookkeeping can go wrong: one block over more
runs than a wave has lanes, runs of several blocks, pieces longer than a wave's
window of page ids, blocks that end inside and at a run, sequences
without keys or queries, more of them than a wave or a workgroup has threads,
pages of sizes a wave's staged keys do and do not
share, missing pages, and scores that outgrow a run's first maximum; and the
choice between the runs and a workgroup per block.  The
oracle, bounds and helper are test_gpu_attention_prefill.py's (a run's P is
rounded to fp16 under the same 2^15 headroom, by raising the maximum)."""

import numpy as np
import pytest
import torch

from pipeswift_amd import attention
from tests import prefill_schedule as S
from tests.test_gpu_attention_prefill import _prefill_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,counts,prefixes,ps,causal", [
    (8, 1, [64], [16000], 16, True),             # two blocks of 32 tokens over 64 runs: 31 and 32 records
    (8, 1, [20], [4100], 16, True),              # one partial block: waves without query rows
    (32, 8, [100, 3, 60], [1500, 7, 2900], 16, True),
    (32, 4, [70, 0, 33], [1200, 0, 1999], 24, True),   # an empty sequence, 24-token pages
    (32, 4, [70, 33], [1200, 1999], 12, True),   # pages a wave's 8 keys straddle: per-thread lookups
    (6, 2, [40, 90], [1100, 1300], 64, False),   # groups of 3, every key visible
    (32, 8, [90, 65], [1024, 1983], 128, True),  # lengths next to stage boundaries
    (16, 16, [300], [1724], 16, True),           # group 1: 256-token blocks
])
def test_runs(dev, Hq, Hkv, counts, prefixes, ps, causal):
    lens = [c + p for c, p in zip(counts, prefixes)]
    assert S.takes_runs(counts, lens, Hq, Hkv, sum(counts) + 2, causal)
    _prefill_case(dev, 1300 + Hq + ps + len(counts), lens, counts, Hq, Hkv, ps, causal, spare_rows=2)


@pytest.mark.parametrize("q_dtype,out_dtype", [(torch.float8_e4m3fn, torch.bfloat16), (torch.float16, torch.float32),
                                               (torch.float32, torch.bfloat16)])
def test_runs_dtypes(dev, q_dtype, out_dtype):
    _prefill_case(dev, 1400, [1800, 1200], [80, 200], 32, 4, 16, True, q_dtype=q_dtype, out_dtype=out_dtype)


def test_one_block_over_more_runs_than_lanes(dev):
    """A block over 136 runs: its records are found in three rounds of a wave."""
    counts, lens = [20], [70020]
    assert max(S.records(S.runs(counts, lens, 8, 1, True)).values()) == 136
    _prefill_case(dev, 1401, lens, counts, 8, 1, 16, True)


@pytest.mark.parametrize("ps,causal", [(16, True), (12, True), (24, False)])
def test_runs_of_several_long_pieces(dev, ps, causal):
    """Two runs per kv head, of three blocks each: each piece hands over to the
    next, and pieces of more than 64 stages refill their window of page ids
    (pages that a wave's keys share, and per-thread lookups)."""
    counts, lens = [20, 5, 33, 9, 12], [3000, 9, 9100, 700, 2900]
    plan = S.runs(counts, lens, 128, 128, causal)
    assert len(plan) == 2 and max(map(len, plan)) >= 3
    assert max(p.sb - p.sa for run in plan for p in run) > 64
    _prefill_case(dev, 1402 + ps, lens, counts, 128, 128, ps, causal)


@pytest.mark.parametrize("ps", [16, 12])
def test_runs_missing_pages(dev, ps):
    """Missing pages read as zero rows: in a piece's first stage, which is
    staged before its pipeline starts, and after whole stages of a run of 26
    (64 kv heads: four runs), where the later loads' count depends on it: one
    page of a stage, a whole stage, the last page."""
    _prefill_case(dev, 1410, [2300, 1100], [64, 90], 32, 8, ps, True, bad_ids=True)
    lens, counts = [3000, 2500], [60, 21]
    plan = S.runs(counts, lens, 64, 64, True)
    at = [700, *range(1920, 1984, 4), 2999]
    assert all(any(p.b == 0 and p.sa + 8 <= key // 64 < p.sb for run in plan for p in run) for key in at)
    holes = [(0, page) for page in sorted({key // ps for key in at})] + [(1, 1000 // ps)]
    _prefill_case(dev, 1411, lens, counts, 64, 64, ps, True, holes=holes)


@pytest.mark.parametrize("ps", [16, 24])
def test_runs_head_major_cache(dev, ps):
    """A cache whose heads are further apart than its rows."""
    _prefill_case(dev, 1470, [2300, 1100], [64, 90], 32, 8, ps, True, head_major=True)


def test_runs_page_stride_past_32_bits(dev):
    """Pages 4 GiB + 32 KiB apart; every table entry is one of the two, so the
    sequence of 1200 keys reads them again and again."""
    from oracle import kv_oracle as O
    from tests.conftest import raw
    from tests.test_gpu_attention_prefill import p_rounding_bound

    Hkv, Hq, ps, D, L, n = 2, 16, 16, 128, 1200, 20
    assert S.takes_runs([n], [L], Hq, Hkv)
    stride = (1 << 32) + (1 << 15)
    base = torch.zeros(stride + 2 * ps * Hkv * D * 2, dtype=torch.uint8, device=dev)
    g = torch.Generator().manual_seed(1480)
    pages = (torch.randn(2, 2, ps, Hkv, D, generator=g) * 2).to(torch.float8_e4m3fn)
    for p in range(2):
        base[p * stride: p * stride + 2 * ps * Hkv * D].copy_(pages[p].reshape(-1).view(torch.uint8).to(dev))
    kc = base.view(torch.float8_e4m3fn).as_strided((2, ps, Hkv, D), (stride, Hkv * D, D, 1))
    vc = base.view(torch.float8_e4m3fn).as_strided((2, ps, Hkv, D), (stride, Hkv * D, D, 1), ps * Hkv * D)
    q = (torch.randn(n, Hq, D, generator=g) * 3).to(torch.bfloat16)
    bt = torch.randint(0, 2, (1, L // ps), generator=g, dtype=torch.int32)
    cu = torch.tensor([0, n], dtype=torch.int32)
    print(f"prefill runs wide page stride: stride={stride}", flush=True)
    got = attention.paged_prefill_attention(q.to(dev), kc, vc, bt.to(dev), torch.tensor([L], dtype=torch.int32,
                                            device=dev), cu.to(dev), n, 128 ** -0.5,
                                            out=torch.zeros(n, Hq, D, dtype=torch.float32, device=dev))
    exp, _ = O.paged_decode_attention(raw(q), "bf16", raw(pages[:, 0]), raw(pages[:, 1]), bt.numpy(), np.array([L]),
                                      128 ** -0.5, cu_seqlens_q=cu.numpy(), causal=True)
    vmax = float(np.abs(O.e4m3fn_to_f32(raw(pages[:, 1]))).max())
    err = np.abs(got.double().cpu().numpy() - exp)
    assert (err <= 3e-4 * vmax + p_rounding_bound(L, vmax) + 1e-4 * np.abs(exp)).all(), f"max err {err.max():.3e}"


@pytest.mark.parametrize("B", [64, 65, 130, 700])
@pytest.mark.parametrize("long", [True, False])
def test_many_sequences(dev, B, long):
    """As many sequences as a wave has lanes, and more than that and than a
    workgroup has threads, empty ones among them (in keys, in queries), under a
    table of 2000 keys: with a long sequence the step is cut into runs (two
    rounds of the scan at 700), without one the device leaves the blocks in
    launch order."""
    counts = [(i * 7) % 5 for i in range(B)]
    lens = [c + (i * 13) % 40 if i % 11 else 0 for i, c in enumerate(counts)]
    counts[B // 2], lens[B // 2] = 6, 2000 if long else 70
    counts[0] = counts[B - 1] = 0
    assert S.takes_runs(counts, lens, 16, 2) == long
    _prefill_case(dev, 1490 + B, lens, counts, 16, 2, 16, True, wide=2000)


def _step(dev, counts, lens, Hq, Hkv, ps=16, seed=1500):
    g = torch.Generator(device=dev).manual_seed(seed)
    need = [-(-n // ps) for n in lens]
    P = sum(need) + 1
    kv = torch.randn(P, 2, ps, Hkv, 128, generator=g, device=dev).to(torch.float8_e4m3fn)
    perm = torch.randperm(P, generator=g, device=dev).to(torch.int32)
    bt = torch.zeros(len(lens), max(need), dtype=torch.int32, device=dev)
    at = 0
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n]
        at += n
    q = torch.randn(sum(counts), Hq, 128, generator=g, device=dev).to(torch.bfloat16)
    cu = torch.tensor(np.r_[0, np.cumsum(counts)], dtype=torch.int32, device=dev)
    return q, kv, bt, cu, torch.tensor(lens, dtype=torch.int32, device=dev)


@pytest.mark.parametrize("counts,prefixes,Hq,Hkv,runs", [
    ([500], [0], 32, 8, False), ([250, 3], [0, 0], 32, 8, False), ([3000], [0], 32, 8, False),
    ([500] * 8, [0] * 8, 32, 8, False), ([700, 40], [250, 500], 32, 4, False),
    ([500, 1], [0, 9000], 32, 8, True), ([64], [1000], 32, 8, True), ([2000], [0], 8, 1, True),
])
def test_the_lengths_choose_the_kernel(dev, counts, prefixes, Hq, Hkv, runs):
    """Not the block table's width: under a table of 32768 keys, and with and
    without a bound on the lengths, a step gives the same bits, those of a
    workgroup per block where that is its kernel."""
    lens = [c + p for c, p in zip(counts, prefixes)]
    assert S.takes_runs(counts, lens, Hq, Hkv) == runs
    q, kv, bt, cu, L = _step(dev, counts, lens, Hq, Hkv)
    wide = torch.zeros(len(lens), 2048, dtype=torch.int32, device=dev)
    wide[:, :bt.shape[1]] = bt

    def call(table, **kw):
        print(f"counts {counts} prefixes {prefixes}: table of {table.shape[1] * 16} keys {list(kw)}", flush=True)
        return attention.paged_prefill_attention(q, kv[:, 0], kv[:, 1], table, L, cu, max(counts), 128 ** -0.5,
                                                 **kw).view(torch.int16)

    tight = call(bt)
    blocks = call(bt, workspace=torch.empty(2 * len(lens) + 1, dtype=torch.int32, device=dev))
    assert torch.equal(tight, blocks) != runs
    assert torch.equal(call(wide), tight)
    assert torch.equal(call(wide, max_seqlen_k=max(lens)), tight)
    out = attention.flash_attn_varlen_func(q, kv[:, 0], kv[:, 1], max(counts), cu, max(lens), L, wide,
                                           softmax_scale=128 ** -0.5, causal=True)
    assert torch.equal(out.view(torch.int16), tight)


def test_workspace_only_where_it_is_used(dev):
    """A fresh prompt allocates nothing for partial results; a step that may
    leave them does; and on a GPU without room for them it still runs, with a
    workgroup per block."""
    counts, lens = [300], [300]
    q, kv, bt, cu, L = _step(dev, counts, lens, 32, 8)
    out = torch.empty(300, 32, 128, dtype=torch.bfloat16, device=dev)

    def grown(table, seq_lens):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        attention.paged_prefill_attention(q, kv[:, 0], kv[:, 1], table, seq_lens, cu, 300, out=out)
        return torch.cuda.max_memory_allocated() - before

    wide = torch.zeros(1, 512, dtype=torch.int32, device=dev)
    wide[:, :bt.shape[1]] = bt
    assert grown(bt, L) < 1 << 16
    assert grown(wide, L) > 60 << 20
    free, total = torch.cuda.mem_get_info()
    torch.cuda.empty_cache()
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (24 << 20)) / total)
        assert grown(wide, L) < 1 << 20
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    want = attention.paged_prefill_attention(q, kv[:, 0], kv[:, 1], bt, L, cu, 300)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


def test_runs_negative_score_scale(dev):
    _prefill_case(dev, 1430, [2400], [64], 16, 2, 16, True, k_sign=-1.0)


def test_runs_raise_their_maximum(dev):
    """Scores spread over hundreds of binary orders of magnitude: weights pass
    2^15 above the maximum of a run's first 32 keys, in every run."""
    _prefill_case(dev, 1420, [2400, 1500], [64, 130], 32, 4, 16, True, scale=4.0)


def test_runs_query_tokens_without_keys(dev):
    """A sequence shorter than its queries: zeros and lse -inf, beside one that has its keys."""
    _prefill_case(dev, 1440, [5, 3000], [20, 40], 32, 8, 16, True)


def test_runs_in_a_graph(dev):
    """Captured with the caller's workspace and replayed on changed lengths and
    inputs: every replay equals the eager call, bit for bit."""
    Hq, Hkv, ps, W = 32, 8, 16, 128
    g = torch.Generator(device=dev).manual_seed(1450)
    kv = torch.randn(2, W, 2, ps, Hkv, 128, generator=g, device=dev).to(torch.float8_e4m3fn)[0]
    bt = torch.randperm(W, generator=g, device=dev).to(torch.int32).view(1, W)
    q = torch.randn(80, Hq, 128, generator=g, device=dev).to(torch.bfloat16)
    cu = torch.tensor([0, 80], dtype=torch.int32, device=dev)
    lens = torch.tensor([1500], dtype=torch.int32, device=dev)
    out = torch.empty(80, Hq, 128, dtype=torch.bfloat16, device=dev)
    ws = torch.empty(attention.prefill_workspace_words(1), dtype=torch.int32, device=dev)

    def call(o):
        return attention.paged_prefill_attention(q, kv[:, 0], kv[:, 1], bt, lens, cu, 80, out=o, workspace=ws)

    call(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    # (81, 100 and 200 keys take a workgroup per block, the others the runs)
    for n in (1500, 100, 2048, 81, 1100, 200):
        lens.fill_(n)
        q.normal_(generator=g)
        out.zero_()
        graph.replay()
        eager = call(torch.empty_like(out))
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16)), f"replay at {n} keys"


def test_small_workspace_takes_a_workgroup_per_block(dev):
    """A workspace of the least size taken before (2 B + 1 words) is still
    taken: the step then runs without records, with the same results."""
    from pipeswift_amd import _lib

    Hq, Hkv, ps, n, L = 8, 2, 16, 40, 2000
    g = torch.Generator(device=dev).manual_seed(1460)
    W = -(-L // ps)
    kv = torch.randn(W, 2, ps, Hkv, 128, generator=g, device=dev).to(torch.float8_e4m3fn)
    bt = torch.arange(W, dtype=torch.int32, device=dev).view(1, W)
    q = torch.randn(n, Hq, 128, generator=g, device=dev).to(torch.float8_e4m3fn)
    cu = torch.tensor([0, n], dtype=torch.int32, device=dev)
    lens = torch.tensor([L], dtype=torch.int32, device=dev)
    want = attention.paged_prefill_attention(q, kv[:, 0], kv[:, 1], bt, lens, cu, n,
                                             out=torch.empty(n, Hq, 128, dtype=torch.float32, device=dev))
    got = torch.empty(n, Hq, 128, dtype=torch.float32, device=dev)
    ws = torch.empty(3, dtype=torch.int32, device=dev)
    k, v = kv[:, 0], kv[:, 1]
    st = _lib.lib().psk_paged_prefill_attention(
        q.data_ptr(), q.stride(0), q.stride(1), 3, k.data_ptr(), v.data_ptr(), _lib.i64_array(k.stride()[:3]),
        _lib.i64_array(v.stride()[:3]), bt.data_ptr(), bt.stride(0), W, lens.data_ptr(), 1, Hq, Hkv, 128, ps, W, n, n,
        cu.data_ptr(), 1, 128 ** -0.5, None, None, None, _lib.i64_array([0] * 6), got.data_ptr(), got.stride(0),
        got.stride(1), 0, None, 0, ws.data_ptr(), ws.numel(), _lib.stream_handle(q.device))
    assert st == 0, _lib.lib().psk_last_error()
    # two kernels of the same arithmetic, P rounded to fp16 about different maxima
    assert float((got - want).abs().max()) <= 2 * 2.0 ** -11 * float(v.float().abs().max())
