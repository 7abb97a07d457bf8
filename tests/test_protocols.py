"""CPU models of the cross-work-group protocols the kernels use, run over
every interleaving of a few work-groups (exhaustive for small counts,
randomised for larger ones).  They check the design, not the GPU code:

* split-K combine (decode3.hip, the runs of prefill_block_kernel):
  every work-group stores its partial (o, m, l), waits for the stores, then
  adds one to its head's arrival counter; the one that reads n-1 resets the
  counter and merges all partials in split order, its own from registers.
  Nobody waits on another work-group, so every interleaving terminates;
  exactly one work-group merges; the counter is 0 again after the launch, so
  the next launch starts clean; the merged bytes do not depend on the order
  of arrival.
* the prefill's exchange of halves (prefill_block_kernel): each of two halves
  holds both row tiles of a wave over its own key tiles; half h leaves row tile
  1 - h in LDS, a barrier, then finishes row tile h from its own and the one it
  finds, in half order.

The merge arithmetic is the kernels' (exp2 of the difference to the running
max, fp32 throughout); a planted mistake (merging in arrival order) makes
the order-independence check fail, so the check has teeth.
"""
from __future__ import annotations

import itertools

import numpy as np
import pytest


def merge(parts, order):
    """The kernels' ordered merge of partials (m, l, o): running max M, scale
    factors exp2(M - Mn) and exp2(m - Mn), fp32."""
    f = np.float32
    M, L = f(-np.inf), f(0.0)
    acc = np.zeros_like(parts[0][2])
    for i in order:
        m, l, o = parts[i]
        Mn = max(M, m)
        fo = np.exp2(f(M - Mn)) if M != -np.inf else f(0.0)
        fs = np.exp2(f(m - Mn)) if m != -np.inf else f(0.0)
        acc = (acc * fo + o * fs).astype(np.float32)
        L = f(L * fo + l * fs)
        M = Mn
    return acc / L


def run_launch(parts, arrival, counter, merge_in_arrival_order=False):
    """One launch under a given arrival order.  Returns (who merged, result)
    and leaves the counter as the kernel would."""
    n = len(parts)
    stored = [False] * n
    mergers, result = [], None
    for s in arrival:
        stored[s] = True                      # stores acknowledged before the add
        old = counter[0]
        counter[0] += 1                       # the atomic add returns the old value
        if old == n - 1:
            counter[0] = 0                    # the merger resets it
            assert all(stored), "a partial was read before its stores were acknowledged"
            mergers.append(s)
            order = list(arrival) if merge_in_arrival_order else list(range(n))
            result = merge(parts, order)
    return mergers, result


def random_parts(rng, n, width=8, spread=2.0):
    parts = []
    for _ in range(n):
        m = np.float32(rng.normal(0, spread))
        parts.append((m, np.float32(rng.uniform(1, 50)), rng.standard_normal(width).astype(np.float32) * 30))
    return parts


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5])
def test_split_combine_every_order(n):
    rng = np.random.default_rng(n)
    parts = random_parts(rng, n)
    counter = [0]
    ref = None
    for arrival in itertools.permutations(range(n)):
        mergers, res = run_launch(parts, arrival, counter)
        assert mergers == [arrival[-1]], "exactly one merger, the last to arrive"
        assert counter[0] == 0, "the counter is back to 0 for the next launch"
        ref = res if ref is None else ref
        assert res.tobytes() == ref.tobytes(), "merged bytes depend on the arrival order"


@pytest.mark.parametrize("n", [8, 32, 64])
def test_split_combine_random_orders(n):
    rng = np.random.default_rng(100 + n)
    parts = random_parts(rng, n)
    # one split with no key (m = -inf, l = 0, o = 0), as an empty split leaves it
    parts[n // 2] = (np.float32(-np.inf), np.float32(0.0), np.zeros(8, np.float32))
    counter = [0]
    ref = merge(parts, range(n))
    for _ in range(50):
        arrival = rng.permutation(n)
        mergers, res = run_launch(parts, arrival, counter)
        assert len(mergers) == 1 and counter[0] == 0
        assert res.tobytes() == ref.tobytes()
    # against fp64 softmax-weighted sum of the same partials
    m = np.array([p[0] for p in parts], np.float64)
    w = np.where(np.isfinite(m), np.exp2(m - m[np.isfinite(m)].max()), 0.0)
    num = sum(wi * p[2].astype(np.float64) for wi, p in zip(w, parts))
    den = sum(wi * float(p[1]) for wi, p in zip(w, parts))
    assert np.allclose(ref, num / den, rtol=1e-5, atol=1e-6)


def test_planted_arrival_order_merge_is_caught():
    """Merging in arrival order instead of split order changes the rounding:
    the order-independence check above would catch it."""
    rng = np.random.default_rng(7)
    parts = random_parts(rng, 6)
    counter = [0]
    outs = {run_launch(parts, p, counter, merge_in_arrival_order=True)[1].tobytes()
            for p in itertools.permutations(range(6))}
    assert len(outs) > 1


def test_consecutive_launches_start_clean():
    """Launches back to back on the same counter (stream order): each one's
    merger is its own last arrival and the counter is 0 between them."""
    rng = np.random.default_rng(3)
    counter = [0]
    for launch in range(20):
        n = int(rng.integers(1, 9))
        parts = random_parts(rng, n)
        mergers, res = run_launch(parts, rng.permutation(n), counter)
        assert len(mergers) == 1 and counter[0] == 0
        assert res.tobytes() == merge(parts, range(n)).tobytes()


def exchange(st, order, wrong_tile=False):
    """Two halves' (m, l, o) of row tiles 0 and 1, st[half][tile]: the LDS
    exchange with the halves' steps run in `order`, a barrier between the
    stores and the merges.  Returns the finished row tiles."""
    lds, out = {}, {}
    for half in order:
        lds[half] = st[half][half if wrong_tile else 1 - half]   # the tile the other one finishes
    for half in order:
        own, other = st[half][half], lds[1 - half]
        out[half] = merge([own, other], [0, 1] if half == 0 else [1, 0])
    return out


def exact_tiles(st):
    """The merged row tiles in fp64, and the bound of the fp32 merge: factors,
    products, sums and the quotient are each rounded once, a few 2^-24 of the
    terms."""
    for tile in (0, 1):
        m = np.array([st[h][tile][0] for h in (0, 1)], np.float64)
        w = np.exp2(m - m.max())
        den = sum(w[h] * float(st[h][tile][1]) for h in (0, 1))
        o = [st[h][tile][2].astype(np.float64) for h in (0, 1)]
        yield (w[0] * o[0] + w[1] * o[1]) / den, 8 * 2.0 ** -24 * (w[0] * np.abs(o[0]) + w[1] * np.abs(o[1])) / den


EMPTY = (np.float32(-np.inf), np.float32(0.0), np.zeros(8, np.float32))


def test_halves_exchange_row_tiles():
    """Every row tile is finished once, with both halves' parts of that tile in
    half order, whichever half is first; a half with no key (a run of one tile)
    leaves the other's rows exactly as they were."""
    rng = np.random.default_rng(9)
    for _ in range(20):
        st = [random_parts(rng, 2), random_parts(rng, 2)]
        out = exchange(st, [0, 1])
        for tile, (exact, bound) in enumerate(exact_tiles(st)):
            assert (np.abs(out[tile] - exact) <= bound).all()
        again = exchange(st, [1, 0])
        assert all(again[t].tobytes() == out[t].tobytes() for t in (0, 1))
        lone = exchange([st[0], [EMPTY, EMPTY]], [0, 1])
        for tile in (0, 1):
            m, l, o = st[0][tile]
            assert lone[tile].tobytes() == (o / l).astype(np.float32).tobytes()


def test_planted_wrong_tile_is_caught():
    """A half that leaves the row tile it finishes itself: beyond the bound."""
    rng = np.random.default_rng(10)
    st = [random_parts(rng, 2), random_parts(rng, 2)]
    out = exchange(st, [0, 1], wrong_tile=True)
    for tile, (exact, bound) in enumerate(exact_tiles(st)):
        assert not (np.abs(out[tile] - exact) <= bound).all()
