"""CPU checks of the equal-run prefill schedule's model (tests/prefill_schedule.py)
and of the C rule that chooses between the prefill kernels: every stage of every
block is one run's, a shared block's records are one slot each of runs that
follow each other (as the merge walks them), and the workspace query asks for
the partial results only where some length within the bound would use them."""

import random

import pytest

from pipeswift_amd._lib import lib
from tests import prefill_schedule as S

SHAPES = [(32, 8), (32, 4), (8, 1), (16, 16), (6, 2), (256, 1), (8, 8), (128, 64)]


@pytest.mark.parametrize("seed", range(60))
def test_every_stage_once_and_records_in_a_row(seed):
    r = random.Random(seed)
    Hq, Hkv = r.choice(SHAPES)
    B = r.choice([1, 1, 2, 7, 100])
    top = r.choice([40, 300, 3000])
    counts = [r.choice([0, 1, r.randint(1, top)]) for _ in range(B)]
    lens = [max(0, c + r.choice([0, 0, -5, r.randint(0, 200), r.randint(0, 60000)])) for c in counts]
    causal = r.random() < 0.7
    plan = S.runs(counts, lens, Hq, Hkv, causal)
    seen, tq = {}, S.ROWS // (Hq // Hkv)
    for j, mine in enumerate(plan):
        for k, p in enumerate(mine):
            seen.setdefault((p.b, p.i), []).append((j, k, p))
        # one piece a slot: only a run's first piece begins inside a block, only its last ends inside one
        assert all(p.sa == 0 for p in mine[1:])
        assert all(p.sb == p.ns for p in mine[:-1])
    for b, n in enumerate(counts):
        for i in range(-(-n // tq)):
            got = seen.pop((b, i))
            ns = got[0][2].ns
            assert got[0][2].sa == 0 and got[-1][2].sb == ns
            assert all(x[2].sb == y[2].sa for x, y in zip(got, got[1:]))
            if len(got) > 1:
                js = [j for j, _, _ in got]
                assert js == list(range(js[0], js[0] + len(js)))
                # the first of them in its run's slot of blocks it begins, the others in the other slot
                assert all(p.sa > 0 for _, _, p in got[1:]) and all(k == 0 for _, k, _ in got[1:])
    assert not seen


def _step_words(counts, Hq, Hkv, keys):
    return lib().psk_paged_prefill_step_workspace_len(len(counts), sum(counts), max(counts), Hq, Hkv, keys)


@pytest.mark.parametrize("counts,Hq,Hkv,keys,records", [
    ([500], 32, 8, 500, False),          # a fresh prompt under a table of its own width
    ([500], 32, 8, 32768, True),         # the same under a wide table: the device decides
    ([1800], 32, 8, 1800, True), ([2000], 32, 8, 2000, False), ([2000], 8, 1, 2000, True),
    ([8000], 32, 8, 1 << 20, True),      # 1000 workgroups: a long enough prefix would take the runs
    ([8001 * 5], 32, 8, 1 << 20, False),  # past four blocks a CU no length does
    ([100] * 1025, 32, 8, 4096, False),  # more sequences than the runs scan
    ([64], 32, 8, 979, False), ([64], 32, 8, 980, True),
    ([512], 512, 256, 65536, False),     # more kv heads than half the CUs
])
def test_workspace_follows_the_step(counts, Hq, Hkv, keys, records):
    B = len(counts)
    most = lib().psk_paged_prefill_workspace_len(B)
    words = _step_words(counts, Hq, Hkv, keys)
    assert words == (most if records else 2 * B + 1)
    assert most >= 2 * B + 1


def test_workspace_query_allows_what_the_device_takes():
    """Over random steps and lengths within the bound: where the device would
    cut the step into runs, the query has asked for their records, and where
    the query tokens are all the keys there can be it asks for no others'."""
    r, took = random.Random(5), 0
    for _ in range(6000):
        Hq, Hkv = r.choice(SHAPES)
        counts = [r.randint(1, r.choice([50, 900, 9000])) for _ in range(r.choice([1, 1, 2, r.randint(1, 9)]))]
        keys = max(counts) + r.choice([0, r.randint(0, 1500), r.randint(0, 60000)])
        lens = [r.randint(n, keys) for n in counts]
        if r.random() < 0.5:
            lens[r.randrange(len(lens))] = keys
        records = _step_words(counts, Hq, Hkv, keys) > 2 * len(counts) + 1
        if S.takes_runs(counts, lens, Hq, Hkv, causal=r.random() < 0.7):
            took += 1
            assert records, (counts, lens, Hq, Hkv, keys)
        if len(counts) == 1 and keys == counts[0]:
            assert records == S.takes_runs(counts, counts, Hq, Hkv)
    assert took > 500
    f = lib().psk_paged_prefill_step_workspace_len
    assert f(1, 500, 500, 32, 8, (1 << 63) - 1) == lib().psk_paged_prefill_workspace_len(1)  # lengths not known
    for bad in [(-1, 5, 5, 32, 8, 9), (1, -5, 5, 32, 8, 9), (1, 1 << 31, 5, 32, 8, 9), (1, 5, 0, 32, 8, 9), (1, 5, 5, 30, 8, 9),
                (1, 5, 5, 0, 8, 9), (1, 5, 5, 32, 0, 9), (1, 5, 5, 514, 2, 9)]:
        assert f(*bad) < 0


def test_more_keys_or_less_to_share_never_refuse():
    """What a longer bound and a smaller share refuse, no shorter length or
    larger share takes: what lets the host settle steps."""
    r = random.Random(6)
    for _ in range(2000):
        max_q, w = r.randint(1, 20000), r.randint(1, 2000)
        ks, c = sorted(r.randint(0, r.choice([2000, 90000])) for _ in range(6)), r.randint(0, 5000)
        got = [S.prefers_runs(k, c, max_q, w) for k in ks]
        assert got == sorted(got)
        cs = sorted(r.randint(0, 5000) for _ in range(6))
        got = [S.prefers_runs(ks[-1], c, max_q, w) for c in cs]
        assert got == sorted(got, reverse=True)
