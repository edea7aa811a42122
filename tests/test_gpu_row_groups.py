"""The row-group kernels of the key layout (Sq > 1) and the query layout against the oracle.

Where they can go wrong: caches that end inside an instruction's rows or a
block, pages of one instruction's rows and off the powers of two (odd sizes
take the per-key path), head dims below their tile, page ids outside the pool,
several query tiles, causal rows without a key, the single-stage kernel, K/V
large enough to be loaded non-temporally. Rows that no request reads hold
NaN. The tolerance is the operator's (oracle TOLERANCES: the input type's
rounding of P and O).
"""
import pytest
import torch

from oracle import mha_oracle as O

gpu = pytest.mark.gpu


def _check(b, sq, h, d, page, lengths, dtype, causal=False, outside=False, layout="key", kernel=None, **plan):
    from fgw_amd.operators.mha.current import build_kernel
    width = -(-max(lengths) // page)
    q, k, v, table = O.make_inputs(("groups", b, sq, h, d, page, width), 17, dtype)
    lengths = torch.tensor(lengths, dtype=torch.int32)
    k, v = O.poison_unread(k, v, table, lengths, page)
    etable, ek, ev = table, k, v
    if outside:  # the oracle reads a page of zeros where the kernel's id is invalid
        table = table.clone()
        table[0, 0], table[-1, 1] = -7, k.shape[0] // page
        zeros = torch.zeros(page, h, d, dtype=dtype)
        ek, ev = torch.cat([k, zeros]), torch.cat([v, zeros])
        etable = table.clone()
        etable[0, 0] = etable[-1, 1] = k.shape[0] // page
    kern = build_kernel(b, sq, h, d, k.shape[0], width, page, causal,
                        "float16" if dtype == torch.float16 else "bfloat16", 0, layout=layout, **plan)
    if kernel:
        assert kern.launch_info.name == kernel
    got = kern(*[x.cuda() for x in (q, k, v, table, lengths)]).cpu()
    rtol, atol = O.TOLERANCES[dtype]
    torch.testing.assert_close(got, O.chunked_reference(q, ek, ev, etable, lengths, page, causal),
                               rtol=rtol, atol=atol)


@gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d,page,dtype", [
    (16, 16, torch.bfloat16), (32, 48, torch.float16), (48, 8, torch.bfloat16),
    (64, 16, torch.float16), (80, 12, torch.bfloat16), (96, 64, torch.float16),
    (128, 4, torch.bfloat16), (128, 16, torch.float16), (128, 128, torch.bfloat16),
    (192, 2, torch.float16), (256, 16, torch.bfloat16), (128, 6, torch.float16)])
def test_ragged_ends_match_the_oracle(d, page, dtype, causal):
    lengths = [0, 1, 3, 16, 31, 32, 33, 127, 129, 255, 300, 520]
    # Whole blocks, and pages that split a load instruction's rows: the general kernel.
    kernel = "key" if (d, page) in ((128, 128), (128, 6)) else "key_groups"
    for sq, splits in ((2, 1), (17, 4), (40, 2)):
        _check(len(lengths), sq, 2, d, page, lengths, dtype, causal, num_splits=splits, kernel=kernel)


@gpu
@pytest.mark.parametrize("stages", [1, 2])
def test_both_stage_counts_and_ids_outside_the_pool(stages):
    for page, kernel in ((16, "key_groups"), (64, "key")):
        _check(3, 5, 2, 128, page, [700, 129, 1000], torch.bfloat16, num_splits=4, stages=stages,
               kernel=kernel)
        _check(2, 9, 2, 128, page, [256, 200], torch.float16, outside=True, num_splits=1,
               stages=stages, kernel=kernel)


@gpu
def test_length_balanced_and_non_temporal():
    _check(70, 2, 1, 64, 16, [(29 * i) % 400 for i in range(70)], torch.float16, num_splits=4,
           split_keys=128, kernel="key_groups")
    # 4 x 40 x 4096 x 8 x 64 bytes = 320 MiB of K/V, 272 MiB live; with pages of 16, 168 of 192.
    _check(40, 2, 8, 64, 128, [4096 - 31 * i for i in range(40)], torch.float16, num_splits=1,
           kernel="key_stream")
    _check(24, 2, 8, 64, 16, [4096 - 41 * i for i in range(24)], torch.float16, num_splits=1,
           kernel="key_groups")


@gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d,page,dtype", [
    (16, 16, torch.bfloat16), (32, 48, torch.float16), (48, 8, torch.bfloat16),
    (64, 32, torch.float16), (96, 64, torch.float16), (128, 16, torch.bfloat16),
    (192, 2, torch.bfloat16), (192, 64, torch.float16), (256, 16, torch.float16)])
def test_query_layout_ragged_ends(d, page, dtype, causal):
    lengths = [0, 1, 3, 63, 64, 65, 130, 257, 300, 520]
    for sq, splits in ((33, 1), (129, 2)):
        _check(len(lengths), sq, 2, d, page, lengths, dtype, causal, layout="query",
               num_splits=splits, kernel="query_groups")


@gpu
def test_query_layout_ids_outside_the_pool_and_several_items():
    _check(2, 150, 3, 256, 32, [400, 177], torch.bfloat16, outside=True, layout="query", num_splits=1,
           persistent_programs=4, kernel="query_groups")
    _check(2, 150, 3, 192, 64, [400, 177], torch.float16, outside=True, layout="query", num_splits=2,
           kernel="query_groups")
