"""Which kernel variant a planned call launches (CPU: the choice is host arithmetic)."""
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
           split_keys=0):
    width = -(-kv // page)
    shape = _lib.Shape(b, sq, h, d, b * width * page, width, page, causal, _lib.DTYPE_BFLOAT16)
    plan = _lib.plan(shape, _lib.Request(splits, programs, layout, split_keys), DEVICE)
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
    if not name.startswith("half"):
        assert (info.q_tiles, info.work_items, info.grid) == (plan.q_tiles, plan.work_items, plan.grid)


def test_a_plan_of_another_shape_is_refused():
    plan, _ = launch()
    other = _lib.Shape(3, 1, 8, 128, 4096, 32, 64, 0, _lib.DTYPE_BFLOAT16)
    with pytest.raises(ValueError, match="does not match"):
        _lib.launch_info(other, plan)
