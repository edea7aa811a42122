"""Which kernel variant a planned call launches (CPU: the choice is host arithmetic)."""
import random

import pytest

from fgw_amd import _lib

DEVICE = _lib.DeviceInfo(256, (_lib.c_int32 * 3)(2, 1, 1), 1, 2)


@pytest.fixture(scope="module", autouse=True)
def lib():
    if not _lib.LIBRARY.exists():
        from fgw_amd import build
        build.build(verbose=False)
    return _lib.load()


def launch(b=2, sq=1, h=8, d=128, kv=2048, page=64, causal=0, layout=-1, splits=0, programs=-1,
           split_keys=0, stages=0):
    width = -(-kv // page)
    shape = _lib.Shape(b, sq, h, d, b * width * page, width, page, causal, _lib.DTYPE_BFLOAT16)
    plan = _lib.plan(shape, _lib.Request(splits, programs, layout, split_keys, stages), DEVICE)
    return plan, _lib.launch_info(shape, plan)


@pytest.mark.parametrize("name,kwargs", [
    ("decode", dict()), ("decode", dict(d=96, page=16)), ("key", dict(page=6)),
    ("key", dict(sq=4)), ("key_groups", dict(sq=4, page=16)), ("key_groups", dict(sq=4, d=80)),
    ("query", dict(sq=64)), ("query_groups", dict(sq=64, page=16)),
    ("query_groups", dict(sq=64, d=192)), ("query_eight_waves", dict(sq=64, d=256, splits=1)),
    ("query", dict(sq=64, d=256, kv=512, splits=1)),
    ("prefill", dict(sq=4096)), ("prefill_groups", dict(sq=4096, page=16)),
    ("prefill_padded", dict(sq=4096, d=96)), ("half_tiles", dict(b=1, h=16, sq=1536, kv=1024)),
    ("half_tiles_padded", dict(b=8, sq=257, d=96, kv=1152)), ("prefill", dict(sq=4096, page=6))])
def test_variant_of_a_plan(name, kwargs):
    plan, info = launch(**kwargs)
    assert info.name == name
    assert (info.grid, info.threads) == (plan.grid, plan.threads)
    assert info.threads == (512 if name[:4] in ("deco", "pref", "half") or "eight" in name else 256)
    if not name.startswith("half"):
        assert (info.q_tiles, info.work_items) == (plan.q_tiles, plan.work_items)


MIB = 1 << 20


@pytest.mark.parametrize("name,stream,kwargs", [
    # Whole blocks at tile 128: the key kernel from 128 MiB of K/V, past the cache above 256.
    ("decode", 0, dict(kv=16383 // 64 * 64)), ("key", 0, dict(kv=16384)), ("key", 0, dict(kv=32768)),
    ("key_stream", 256, dict(kv=32832)), ("key_stream", 256, dict(sq=8, kv=32832)),
    ("key", 0, dict(sq=8, kv=32768)),
    # Tile 64: the single-token kernel below the cache's size.
    ("decode", 0, dict(d=64, kv=65472)), ("key", 0, dict(d=64, kv=65536)),
    ("key_stream", 256, dict(d=64, kv=65600)),
    # A few long items: the key kernel at tiles 128 and 256.
    ("decode", 0, dict(kv=8192, splits=8)), ("key", 0, dict(kv=8192, splits=4)),
    ("key", 0, dict(kv=8192, splits=16, split_keys=2048)), ("decode", 0, dict(kv=8192, d=64, splits=1)),
    ("key", 0, dict(b=1, h=1, kv=1024, d=256, splits=1)), ("decode", 0, dict(kv=2048, d=256, splits=2)),
    ("decode", 0, dict(kv=8192, page=16, splits=1)),
    # Small pages, padded head dims and D 256: the same kernel at any size, past the
    # cache from half of it.
    ("decode", 0, dict(page=16, kv=16384)), ("decode", 128, dict(page=16, kv=16400)),
    ("decode", 128, dict(d=192, kv=65536)), ("decode", 128, dict(d=256, kv=65536)),
    ("key_groups", 128, dict(sq=8, page=16, kv=16400)),
    # Tile 32: row groups for whole blocks from 128 MiB on, cached loads.
    ("key", 0, dict(sq=8, d=32, kv=65472)), ("key_groups", 0, dict(sq=8, d=32, kv=65536)),
    ("decode", 0, dict(d=32, kv=131072)),
    # Heads that share 128-byte lines, and more than one query tile: never.
    ("decode", 0, dict(d=80, kv=65536)), ("key_groups", 0, dict(sq=8, d=96, kv=65536)),
    ("query_groups", 128, dict(sq=128, page=16, kv=32768, layout=0)),
    ("query_groups", 0, dict(sq=129, page=16, kv=32768, layout=0))])
def test_large_caches(name, stream, kwargs):
    _, info = launch(**kwargs)
    assert (info.name, info.stream_bytes) == (name, stream * MIB)


def test_a_shared_pool_is_not_counted_per_request():
    """64 requests that share 8192 rows: 32 MiB of K/V fit the cache, 2 GiB are read from it."""
    shape = _lib.Shape(64, 1, 8, 128, 8192, 128, 64, 0, _lib.DTYPE_BFLOAT16)
    plan = _lib.plan(shape, _lib.Request(0, -1, -1), DEVICE)
    info = _lib.launch_info(shape, plan)
    assert (info.name, info.stream_bytes) == ("key", 0)


@pytest.mark.parametrize("first,kwargs", [
    # Whole prompts, 1.5 to 8 items per CU.
    (1, dict(b=1, h=32, sq=4096, kv=4096)), (1, dict(b=8, h=32, sq=2048, kv=2048)),
    # Chunks of a long cache: two items per (b, h) re-read its K/V in the other order.
    (0, dict(b=8, h=32, sq=512, kv=8192)), (0, dict(b=8, h=32, sq=300, kv=8192)),
    (0, dict(b=8, h=32, sq=512, kv=8192, d=64)), (0, dict(b=16, h=32, sq=512, kv=2048)),
    # Little more than one item per CU, and not more than one; single tiles.
    (1, dict(b=9, h=16, sq=512, kv=8192)), (0, dict(b=8, h=16, sq=512, kv=8192)),
    (0, dict(b=12, h=16, sq=512, kv=8192)), (1, dict(b=12, h=16, sq=512, kv=8192, d=64)),
    (0, dict(b=9, h=32, sq=256, kv=2048)),
    # Half a long table: up to two and a half items per CU.
    (1, dict(b=5, h=8, sq=4096, kv=8192)), (0, dict(b=8, h=8, sq=4096, kv=8192)),
    # Not causal, another layout.
    (0, dict(b=1, h=32, sq=4096, kv=4096, causal=0)), (0, dict(b=1, h=32, sq=4096, kv=4096, d=256))])
def test_order_of_causal_items(first, kwargs):
    assert launch(**{"causal": 1, **kwargs})[1].longest_first == first


def test_device_cap_is_the_selected_kernels_residency():
    """One program per item of the single-token kernel, two per CU for length-balanced splits
    (whose items may not exist); one per CU of the double-stage key kernel."""
    assert launch(b=64, h=32, kv=64)[0].grid == 2048
    assert launch(b=64, h=32, kv=256, d=64)[0].grid == 2048
    assert launch(b=64, h=8, kv=256, splits=8, split_keys=64)[0].grid == 512
    assert launch(b=64, h=32, kv=64, page=6)[0].grid == 256  # the key kernel
    assert launch(b=64, h=32, kv=64, stages=2)[0].grid == 256  # asked for
    assert launch(b=64, h=32, kv=64, programs=0)[0].grid == 2048
    assert launch(b=64, h=32, kv=64, programs=300)[0].grid == 300


def test_half_tile_grids_keep_the_requested_cap():
    """The kernel's items are half the plan's tiles; the grid is counted in them."""
    half = dict(b=1, h=16, sq=1536, kv=1024)  # 96 tiles of 256 rows, 192 items
    for programs, grid in ((-1, 192), (0, 192), (300, 192), (192, 192), (100, 100), (96, 96), (7, 7)):
        plan, info = launch(**half, programs=programs)
        assert (info.name, info.rows_per_item, info.work_items) == ("half_tiles", 128, 192)
        assert plan.work_items == 96 and plan.grid == info.grid == grid
    # More items than the CUs: the device cap, but for causal plans.
    for items, grid, many in ((387, 256, dict(b=3, h=43, sq=257, kv=2048, d=64)),
                              (312, 312, dict(b=2, h=13, sq=1500, kv=1536, d=64, causal=1))):
        plan, info = launch(**many)
        assert (info.name, info.work_items, plan.grid) == ("half_tiles", items, grid)


@pytest.mark.parametrize("kwargs", [dict(b=1, h=16, sq=1536, kv=1024), dict(sq=4096), dict(), dict(sq=64)])
def test_a_grid_beyond_the_items_is_refused(kwargs):
    plan, info = launch(**kwargs, programs=0)
    assert plan.grid == info.work_items
    plan.grid += 1
    w = -(-kwargs.get("kv", 2048) // 64)
    b = kwargs.get("b", 2)
    shape = _lib.Shape(b, kwargs.get("sq", 1), kwargs.get("h", 8), 128, b * w * 64, w, 64, 0,
                       _lib.DTYPE_BFLOAT16)
    with pytest.raises(ValueError, match="does not match"):
        _lib.launch_info(shape, plan)


def test_a_plan_of_another_shape_is_refused():
    plan, _ = launch()
    other = _lib.Shape(3, 1, 8, 128, 4096, 32, 64, 0, _lib.DTYPE_BFLOAT16)
    with pytest.raises(ValueError, match="does not match"):
        _lib.launch_info(other, plan)


def _half_tiles_by_loop(b, sq, h, capacity, causal, dpad):
    """The rule's definition (half_tiles in fmha_api.hip), tile by tile."""
    def critical(rows, per_step, cost):
        q_tiles = -(-sq // rows)
        rounds = -(-(b * h * q_tiles) // 256)
        steps = lambda vis: -(-min(max(vis, 0), capacity) // (64 * per_step))  # noqa: E731
        path = rounds * steps(capacity)
        if causal:
            total = sum(steps(capacity - sq + min((t + 1) * rows, sq)) for t in range(q_tiles))
            path = max(total * b * h / 256, steps(capacity))
        return path * cost + 5.0 * rounds
    if b * h * -(-sq // 256) > 512:
        return False
    return critical(128, 2, 1.3 if dpad == 64 else 1.66) < 0.95 * critical(256, 1, 1.0)


@pytest.mark.parametrize("causal", [0, 1])
def test_half_tile_rule_over_seeded_shapes(causal):
    r = random.Random(31 + causal)
    taken = 0
    for _ in range(3000):
        b, h = r.choice((1, 2, 3, 8)), r.choice((1, 2, 5, 8, 16, 32))
        sq = r.choice((r.randint(1, 600), r.randint(1, 9000), 256 * r.randint(1, 20)))
        d, page = r.choice((48, 64, 96, 128)), r.choice((16, 64, 128, 272))
        kv = r.choice((r.randint(1, 3000), r.randint(1, 20000), sq))  # often below Sq
        _, info = launch(b=b, sq=sq, h=h, d=d, kv=kv, page=page, causal=causal, splits=1,
                         layout=_lib.LAYOUT_PREFILL)
        want = _half_tiles_by_loop(b, sq, h, -(-kv // page) * page, causal, 64 if d <= 64 else 128)
        assert info.name.startswith("half") == want, (b, sq, h, d, kv, page)
        taken += want
    assert 300 < taken < 2700
