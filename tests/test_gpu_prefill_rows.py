"""The prefill layout's per-instruction variants against the oracle: pages that a
64-key block straddles and head dims below their tile.

Where they can go wrong: caches that end inside an instruction's rows, page
sizes of one instruction's rows and off the powers of two, page ids outside
the pool, more blocks than one window of offsets holds (32 at head-dim tile
128, 64 at 64), several items per program (their output rows are deferred),
fp32 partials of a head dim below its tile, causal rows without a key. Rows
that no request reads hold NaN. The tolerance is the operator's (oracle
TOLERANCES: the input type's rounding of P and O).
"""
import pytest
import torch

from oracle import mha_oracle as O

gpu = pytest.mark.gpu


def _rows_kernel(d):
    return "prefill_groups" if d in (64, 128) else "prefill_padded"


def _check(b, sq, h, d, page, lengths, dtype, causal, outside=False, kernel=None, **plan):
    from fgw_amd.operators.mha.current import build_kernel
    width = -(-max(lengths) // page)
    q, k, v, table = O.make_inputs(("rows", b, sq, h, d, page, width), 5, dtype)
    lengths = torch.tensor(lengths, dtype=torch.int32)
    k, v = O.poison_unread(k, v, table, lengths, page)
    etable, ek, ev = table, k, v
    if outside:  # the oracle reads a page of zeros where the kernel's id is invalid
        table = table.clone()
        table[0, 1], table[-1, 0] = -1, k.shape[0] // page
        zeros = torch.zeros(page, h, d, dtype=dtype)
        ek, ev = torch.cat([k, zeros]), torch.cat([v, zeros])
        etable = table.clone()
        etable[0, 1] = etable[-1, 0] = k.shape[0] // page
    kern = build_kernel(b, sq, h, d, k.shape[0], width, page, causal,
                        "float16" if dtype == torch.float16 else "bfloat16", 0, layout="prefill",
                        **plan)
    if kernel:
        assert kern.launch_info.name == kernel
    got = kern(*[x.cuda() for x in (q, k, v, table, lengths)]).cpu()
    rtol, atol = O.TOLERANCES[dtype]
    torch.testing.assert_close(got, O.chunked_reference(q, ek, ev, etable, lengths, page, causal),
                               rtol=rtol, atol=atol)


@gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d,page,dtype", [
    (128, 4, torch.bfloat16), (128, 16, torch.float16), (128, 48, torch.bfloat16),
    (64, 8, torch.float16), (64, 32, torch.bfloat16), (96, 16, torch.bfloat16),
    (96, 64, torch.float16), (80, 12, torch.float16), (80, 128, torch.bfloat16),
    (128, 6, torch.bfloat16), (96, 5, torch.float16), (112, 16, torch.bfloat16)])
def test_ragged_pages_match_the_oracle(d, page, dtype, causal):
    lengths = [0, 1, 3, 63, 64, 65, 130, 257, 300]
    general = (d, page) in ((128, 6), (96, 5))  # pages that split a load instruction's rows
    for splits in (1, 2):  # (unsplit, some of these run on the half-tile kernel)
        _check(len(lengths), 257, 2, d, page, lengths, dtype, causal, num_splits=splits,
               kernel=None if splits == 1 else "prefill" if general else _rows_kernel(d))


@gpu
@pytest.mark.parametrize("d,page", [(128, 16), (64, 16), (96, 32)])
def test_more_blocks_than_a_window(d, page):
    keys = 8704 if d == 64 else 4500  # 68 blocks per split, 35 and 36
    _check(1, 300, 1, d, page, [keys], torch.bfloat16, False, num_splits=2, kernel=_rows_kernel(d))
    _check(2, 260, 1, d, page, [keys, 2111], torch.bfloat16, True, num_splits=2,
           kernel=_rows_kernel(d))


@gpu
@pytest.mark.parametrize("d,page", [(96, 64), (128, 16), (80, 16), (128, 48)])
def test_several_items_per_program(d, page):
    """At most 320 keys: an unsplit item is too short for the half-tile kernel."""
    for grid in (3, 8):
        for causal in (False, True):
            _check(2, 600, 3, d, page, [200, 288], torch.float16, causal, num_splits=1,
                   persistent_programs=grid, kernel=_rows_kernel(d))


@gpu
def test_several_items_per_program_head_dim_64():
    """531 query tiles: more than the half-tile kernel takes."""
    _check(1, 15000, 9, 64, 16, [250], torch.bfloat16, False, num_splits=1, persistent_programs=48,
           kernel="prefill_groups")


@gpu
@pytest.mark.parametrize("d,page", [(128, 16), (96, 64)])
def test_page_ids_outside_the_pool_read_as_zeros(d, page):
    _check(2, 200, 2, d, page, [320, 177], torch.bfloat16, False, outside=True, num_splits=1,
           kernel=_rows_kernel(d))


@gpu
@pytest.mark.parametrize("h,sq,lengths,first,plan", [
    (17, 2049, [2100, 2049], 1, dict(num_splits=1)),                  # 9 tiles x 34 (b, h)
    (17, 1030, [1030, 700], 1, dict(num_splits=2)),                   # Sq > len rows
    (17, 2049, [2100, 2049], 1, dict(num_splits=4, split_keys=640)),  # tiles of 1 to 4 splits
    (17, 2049, [2100, 2049], 1, dict(num_splits=1, persistent_programs=40)),
    (120, 300, [2100, 1000], 0, dict(num_splits=1)),                  # 2 tiles x 240
    (120, 300, [2100, 1000], 0, dict(num_splits=1, persistent_programs=50)),
])
def test_more_causal_items_than_cus(h, sq, lengths, first, plan):
    """Longest first or (b, h) after (b, h): every item is done once, whatever the plan and
    grid."""
    from fgw_amd.operators.mha.current import build_kernel
    b, d, page = 2, 64, 64
    width = -(-max(lengths) // page)
    q, k, v, table = O.make_inputs(("order", b, sq, h, d, page, width), 3, torch.float16)
    lengths = torch.tensor(lengths, dtype=torch.int32)
    kern = build_kernel(b, sq, h, d, k.shape[0], width, page, True, "float16", 0, layout="prefill",
                        **plan)
    assert kern.compute_work > 256 and kern.launch_info.name == "prefill"
    assert kern.launch_info.longest_first == first
    got = kern(*[x.cuda() for x in (q, k, v, table, lengths)]).cpu()
    rtol, atol = O.TOLERANCES[torch.float16]
    torch.testing.assert_close(got, O.chunked_reference(q, k, v, table, lengths, page, True),
                               rtol=rtol, atol=atol)
