"""CPU checks of the equal-run prefill schedule's model (tests/prefill_schedule.py):
every stage of every block is one run's, and a shared block's records are one
slot each of runs that follow each other (as the merge walks them)."""

import random

import pytest

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


def test_a_bound_on_the_keys_decides_monotonically():
    """What a longer bound refuses no shorter length takes, which is what lets
    the host leave the records out and the longest sequence's own query tokens
    settle a step."""
    r = random.Random(6)
    for _ in range(2000):
        max_q, w = r.randint(1, 20000), r.randint(1, 2000)
        ks = sorted(r.randint(0, 90000) for _ in range(6))
        got = [S.prefers_runs(k, max_q, w) for k in ks]
        assert got == sorted(got)
