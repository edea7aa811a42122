"""The single-token decode kernel (key layout, Sq = 1) against the oracle.

Where it can go wrong: caches that end inside a load instruction's rows, a step
or a wave's share; pages of one load instruction, of less than a step, and of
odd sizes (which take the general key kernel); head dims below their tile;
page ids outside the pool; more requests than one prefix scan; the fused and
the separate merge. Rows that no request reads hold NaN. The tolerance is the
operator's (oracle TOLERANCES: the input type's rounding of P and O).
"""
import pytest
import torch

from oracle import mha_oracle as O

gpu = pytest.mark.gpu


def _check(b, h, d, page, width, lengths, dtype, outside=False, kernel="decode", **plan):
    from fgw_amd.operators.mha.current import build_kernel
    case = ("decode", b, 1, h, d, page, width)
    q, k, v, table = O.make_inputs(case, 11, dtype)
    lengths = torch.tensor(lengths, dtype=torch.int32)
    k, v = O.poison_unread(k, v, table, lengths, page)
    expected_table, ek, ev = table, k, v
    if outside:  # the oracle reads a page of zeros where the kernel's id is invalid
        table = table.clone()
        table[0, 0], table[-1, -1] = -3, k.shape[0] // page + 5
        zeros = torch.zeros(page, h, d, dtype=dtype)
        ek, ev = torch.cat([k, zeros]), torch.cat([v, zeros])
        expected_table = table.clone()
        expected_table[0, 0] = expected_table[-1, -1] = k.shape[0] // page
    kern = build_kernel(b, 1, h, d, k.shape[0], width, page, False,
                        "float16" if dtype == torch.float16 else "bfloat16", 0, layout="key", **plan)
    assert kern.launch_info.name == kernel
    dev = [x.cuda() for x in (q, k, v, table, lengths)]
    expected = O.reference(q, ek, ev, expected_table, lengths, page, False)
    rtol, atol = O.TOLERANCES[dtype]
    for _ in range(2):  # the second call reuses the arrival counters
        torch.testing.assert_close(kern(*dev).cpu(), expected, rtol=rtol, atol=atol)
    return kern, dev


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,page", [(16, 16), (32, 48), (48, 64), (64, 8), (80, 16), (96, 48),
                                    (128, 4), (128, 16), (128, 128), (192, 2), (256, 16),
                                    (128, 6), (64, 5)])
def test_ragged_ends_match_the_oracle(d, page, dtype):
    width = -(-700 // page)
    ends = [0, 1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 127, 128, 129, 255, 257, 511, width * page]
    kernel = "key" if page in (5, 6) else "decode"
    _check(len(ends), 2, d, page, width, ends, dtype, num_splits=1, kernel=kernel)
    _check(len(ends), 2, d, page, width, ends, dtype, num_splits=4, kernel=kernel)


@gpu
@pytest.mark.parametrize("d,page,splits", [(128, 16, 1), (128, 128, 8), (64, 32, 2), (96, 16, 4)])
def test_page_ids_outside_the_pool_read_as_zeros(d, page, splits):
    width = 512 // page
    _check(3, 2, d, page, width, [512, 77, 512], torch.float16, outside=True, num_splits=splits)


@gpu
@pytest.mark.parametrize("splits,page", [(2, 16), (2, 32), (16, 32), (32, 32), (128, 32)])
def test_fused_and_separate_merge_agree(splits, page):
    # (Whole blocks in items of 2048 keys: the MFMA key kernel.)
    kern, dev = _check(2, 4, 128, page, 4096 // page, [4096, 1000], torch.bfloat16,
                       kernel="key" if (splits, page) == (2, 32) else "decode", num_splits=splits)
    parts, lse = kern.partial_kernel(*dev)
    assert torch.equal(kern.merge_kernel(parts, lse), kern(*dev))


@gpu
def test_length_balanced_over_more_requests_than_a_scan_takes():
    lengths = [(37 * i) % 513 for i in range(130)]
    _check(130, 2, 64, 16, 32, lengths, torch.bfloat16, num_splits=8, split_keys=96)
