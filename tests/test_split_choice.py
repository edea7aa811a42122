"""The split choice's shortcuts against the definitions they stand for (CPU):
select_splits scores each length class once, balanced_split_keys bisects its
grid instead of scanning it."""
import math
import random

import pytest

from fgw_amd.operators.mha import split_cost_model as M


class Device:
    num_cus = 256
    wg_per_cu = (2, 1, 1)
    wg_per_cu_key_single = 2


def _select_by_scoring_every_time(batch, sq, heads, dim, capacity, lengths):
    model = M.load_model()
    costs = {s: M.predict(batch, sq, heads, dim, lengths, s, 256, Device.wg_per_cu, model)
             for s in M.SPLITS if s <= max(1, math.ceil(capacity / 32))}
    best = min(costs.values())
    limit = best + max(abs(best) * model["selection_tolerance"], model.get("absolute_margin_us", 0.0))
    return min(s for s, c in costs.items() if c <= limit)


def _balanced_by_scan(lengths, splits, capacity):
    batch, longest = len(lengths), max(lengths)
    if splits < 2 or batch < 2 or batch > M.MAX_BALANCED_BATCH or len(set(lengths)) < 2 or longest <= 0:
        return None
    keys = next((k for k in M._KEY_GRID
                 if sum(max(1, -(-n // k)) for n in lengths) <= batch * splits), None)
    rounds = lambda n: -(-n // M.KEYS_PER_ROUND)  # noqa: E731
    if keys is None or rounds(-(-longest // splits)) - rounds(keys) < M.MIN_ROUNDS_SAVED:
        return None
    slots = 1
    while slots < -(-longest // keys):
        slots *= 2
    slots = min(slots, 128, max(1, -(-capacity // 32)))
    return (slots, keys) if slots >= 2 else None


@pytest.mark.parametrize("seed", range(4))
def test_choices_equal_their_definitions(seed):
    r = random.Random(seed)
    for _ in range(300):
        batch = r.choice([1, 2, 3, 8, 64, 300])
        capacity = int(32 * 2 ** (r.random() * 11))
        lengths = [r.randint(0, capacity) for _ in range(batch)] if r.random() < 0.9 else [0] * batch
        sq, heads, dim = r.choice([1, 16, 32, 33, 128]), r.choice([1, 8, 32]), r.choice([64, 128, 256])
        got = M.select_splits(batch, sq, heads, dim, capacity, lengths, Device)
        assert got == _select_by_scoring_every_time(batch, sq, heads, dim, capacity, lengths)
        splits = r.choice(M.SPLITS)
        assert M.balanced_split_keys(lengths, splits, capacity) == _balanced_by_scan(lengths, splits,
                                                                                     capacity)
