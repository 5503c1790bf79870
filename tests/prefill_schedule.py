"""The equal-run schedule of a prefill step (``csrc/prefill_runs.hip``) in plain
Python: which stages of which query block each run takes, as the kernel computes
it, for the tests to check its invariants and to name what a shape reaches."""

from collections import namedtuple

KEYS, COST, SNAP, MIN_RUN, ROWS, CUS = 64, 384, 3, 512, 256, 256

Piece = namedtuple("Piece", "b i sa sb ns")  # stages [sa, sb) of block i of sequence b, of ns


def prefers_runs(keys, share, max_q, wgs, cus=CUS):
    prefix = keys >= 4 * max_q
    if wgs > cus:
        return prefix and keys >= 1024 and wgs <= 4 * cus
    if keys < 1536:
        return keys >= 980 and share <= (450 if keys < 1280 else 800)
    return prefix or keys >= 4096 or 4 * keys >= 5 * share + 1100


def wgs(counts, Hq, Hkv, total_q=None):
    tq = ROWS // (Hq // Hkv)
    return -(-(sum(counts) if total_q is None else total_q) // tq) * Hkv


def cost(counts, lens, Hq, Hkv, causal=True):
    """The step's cost per kv head."""
    tq, total = ROWS // (Hq // Hkv), 0
    for n, length in zip(counts, lens):
        nb, length = -(-n // tq), max(length, 0)
        total += nb * (COST + (max(length - n, 0) + tq if causal else length)) + (tq * nb * (nb - 1) // 2 if causal else 0)
    return total


def takes_runs(counts, lens, Hq, Hkv, total_q=None, causal=True, cus=CUS):
    """What the device decides (the host settles some steps before it, alike)."""
    keys = max((n for c, n in zip(counts, lens) if c > 0), default=0)
    share = cost(counts, lens, Hq, Hkv, causal) * Hkv // cus
    return len(lens) <= 1024 and 2 * Hkv <= cus and prefers_runs(keys, share, max(counts), wgs(counts, Hq, Hkv, total_q),
                                                                 cus)


def runs(counts, lens, Hq, Hkv, causal, cus=CUS):
    """The pieces of each run of one kv head, in the order of the keys."""
    tq, blocks, at = ROWS // (Hq // Hkv), [], 0
    for b, (n, length) in enumerate(zip(counts, lens)):
        length = max(length, 0)
        for i in range(-(-n // tq)):
            cost = COST + ((max(length - n, 0) + tq + i * tq) if causal else length)
            end = min(max(length - n + min((i + 1) * tq, n), 0), length) if causal else length
            blocks.append((b, i, at, cost, -(-end // KEYS)))
            at += cost
    T, top = at, cus // Hkv
    if T == 0:
        return []
    M = max(1, min(top, T // MIN_RUN))
    start = [(T * ((j << 16) // M)) >> 16 for j in range(M + 1)]

    def stage_at(x, at, cost, ns):
        if x <= at:
            return 0
        if x >= at + cost:
            return ns
        s = int((x - at - COST) / KEYS)  # toward zero, as in C
        return 0 if s < SNAP else ns if s > ns - SNAP else s

    out = []
    for j in range(M):
        lo, hi, mine = start[j], start[j + 1], []
        for b, i, a, cost, ns in blocks:
            x0, x1 = max(lo, a), min(hi, a + cost)
            if x0 >= x1:
                continue
            sa, sb = stage_at(x0, a, cost, ns), stage_at(x1, a, cost, ns)
            if sa < sb or (x0 == a and ns == 0):
                mine.append(Piece(b, i, sa, sb, ns))
        out.append(mine)
    return out


def records(plan):
    """{(b, i): how many runs leave a record of the block}, of blocks in several runs."""
    n = {}
    for mine in plan:
        for p in mine:
            if (p.sa, p.sb) != (0, p.ns):
                n[p.b, p.i] = n.get((p.b, p.i), 0) + 1
    return n
