"""The half-tile prefill kernel (128 query rows, key blocks shared out between two
wave groups) against the oracle.

Where it can go wrong: every number of key blocks (the groups end in different
phases; none, one, odd and even counts), caches that end inside a block or an
instruction's rows, partial query tiles, causal rows without a key, more blocks
than one window of offsets holds, pages that blocks straddle, head dims below
their tile, several items per program, more causal items than CUs. Rows that
no request reads hold NaN. The tolerance is the operator's (oracle TOLERANCES:
the input type's rounding of P and O).
"""
import pytest
import torch

from oracle import mha_oracle as O

gpu = pytest.mark.gpu


def _check(b, sq, h, d, page, lengths, dtype, causal, **plan):
    from fgw_amd.operators.mha.current import build_kernel
    width = -(-max(lengths) // page)
    q, k, v, table = O.make_inputs(("half", b, sq, h, d, page, width), 13, dtype)
    lengths = torch.tensor(lengths, dtype=torch.int32)
    k, v = O.poison_unread(k, v, table, lengths, page)
    kern = build_kernel(b, sq, h, d, k.shape[0], width, page, causal,
                        "float16" if dtype == torch.float16 else "bfloat16", 0, layout="prefill",
                        num_splits=1, **plan)
    assert kern.launch_info.name == ("half_tiles" if d in (64, 128) else "half_tiles_padded")
    got = kern(*[x.cuda() for x in (q, k, v, table, lengths)]).cpu()
    rtol, atol = O.TOLERANCES[dtype]
    torch.testing.assert_close(got, O.chunked_reference(q, k, v, table, lengths, page, causal),
                               rtol=rtol, atol=atol)


@gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d,page,dtype", [(64, 64, torch.bfloat16), (128, 128, torch.float16),
                                          (128, 16, torch.bfloat16), (96, 32, torch.float16),
                                          (48, 8, torch.bfloat16)])
def test_every_block_count(d, page, dtype, causal):
    lengths = [0] + [64 * n - (0, 1, 33)[n % 3] for n in range(1, 15)] + [1280]
    _check(len(lengths), 200, 2, d, page, lengths, dtype, causal)


@gpu
@pytest.mark.parametrize("sq", [129, 255, 256, 385])
def test_partial_query_tiles(sq):
    _check(2, sq, 3, 64, 32, [1024, 700], torch.bfloat16, True)
    _check(1, sq, 2, 128, 64, [1024], torch.float16, False)


@gpu
@pytest.mark.parametrize("d,page", [(64, 16), (128, 64)])
def test_more_blocks_than_a_window(d, page):
    _check(2, 260, 1, d, page, [8704, 4224], torch.bfloat16, False)


@gpu
def test_several_items_per_program_and_more_items_than_cus():
    _check(2, 900, 3, 64, 64, [960, 900], torch.float16, True, persistent_programs=5)
    _check(2, 1500, 13, 64, 64, [1536, 1500], torch.float16, True)
