"""The units of the dK + dV launch (tests/key_units.py restates the plan of bwd.hip): every tile of keys, or both of
its halves, is one unit of every kv-head, the longest units come first, and the plan of each case of
test_gpu_backward_units.py is the one that its comment states."""
import random

import pytest

from tests.key_units import MAX_BATCH, MAX_LEVELS, Plan
from tests.test_gpu_backward_units import CASES


def _check(p):
    got = [p.unit_at(u) for u in range(p.units())]
    want = {(b, h, t, half) for b, n in enumerate(p.tiles) for t in range(n) for h in range(p.hkv)
            for half in ((0, 1) if n - 1 - t >= p.split_from else (-1,))}
    assert len(got) == len(set(got)) and set(got) == want
    assert p.unit_at(p.units()) is None and p.unit_at(p.units() + 255) is None
    if p.causal:
        costs = [p.cost(u) for u in got]
        assert costs == sorted(costs, reverse=True)


def test_every_unit_once_and_the_longest_first():
    rng = random.Random(9)
    for _ in range(300):
        longest = rng.choice([1, 64, 65, 129, 300, 2000, 9000])
        lens = [rng.choice([0, 1, longest, rng.randint(0, longest)]) for _ in range(rng.choice([1, 2, 5, 17, 64]))]
        hkv = rng.choice([1, 2, 3, 8])
        p = Plan(lens, hkv * rng.choice([1, 2, 4]), hkv, rng.random() < 0.8, rng.choice([8, 64, 256]))
        if rng.random() < 0.5:
            p.split_from = rng.randint(0, p.levels)
        _check(p)


# of CASES, in their order: dealt, halved levels out of all levels; None: more sequences or levels than the plan holds
PLANS = [(True, (1, 2)), (True, (2, 27)), (True, (11, 32)), (True, (0, 67)), (True, (0, 6)), None, (True, (8, 8)),
         (False, None), (True, (7, 16)), (True, (2, 2)), (False, None), None, (True, (0, 64))]


@pytest.mark.parametrize("case,want", list(zip(CASES, PLANS)))
def test_plans_of_the_device_test(case, want):
    lens, Hq, Hkv, _, _, causal = case
    lens = [lens[1]] * lens[0] if isinstance(lens, tuple) else lens
    if want is None:
        assert len(lens) > MAX_BATCH or -(-max(lens) // 128) > MAX_LEVELS
        return
    p = Plan(lens, Hq, Hkv, causal)
    dealt, halved = want
    assert p.dealt == dealt
    if dealt:
        assert (p.levels - p.split_from, p.levels) == halved


@pytest.mark.parametrize("lens,heads,heads_kv,dealt", [
    ([60] * 64, 2, 2, False), ([100] * 64, 4, 4, False), ([512] * 8, 8, 8, False), ([1024] * 2, 16, 16, False),   # nothing to gain
    ([256], 8, 8, False), ([512], 8, 8, True), ([512] * 4, 8, 8, True),                                         # chains of four and eight
    ([64], 8, 1, False), ([65], 8, 1, True),                                                                    # a second half
    ([512] * 8, 32, 8, False), ([4096], 32, 8, True), ([2048], 16, 2, True),
    ([512] * 8, 16, 16, True),                                                                                  # more than a round
    ([3000] * 43, 4, 1, False), ([3000] * 42, 4, 1, True),                                                      # four rounds
    ([4096] + [100] * 63, 16, 16, False), ([4096] + [100] * 63, 10, 10, True),
])
def test_which_launches_deal_their_units(lens, heads, heads_kv, dealt):
    assert Plan(lens, heads, heads_kv).dealt == dealt
