"""The query layout's eight-wave kernel (head-dim tile 256) against the oracle.

Where it can go wrong: caches that end in the first or the second half of a key
block (the second set of waves then has no live key), no, one and two blocks,
odd and even counts, causal rows without a key, partial query tiles, splits,
several items per program, page ids outside the pool. Rows that no request
reads hold NaN. The tolerance is the operator's (oracle TOLERANCES: the input
type's rounding of P and O).
"""
import pytest
import torch

from tests.test_gpu_row_groups import _check

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("page,dtype", [(64, torch.bfloat16), (64, torch.float16),
                                        (128, torch.bfloat16), (256, torch.float16)])
def test_every_end_of_a_block(page, dtype, causal):
    lengths = [0, 1, 31, 32, 33, 63, 64, 65, 95, 97, 128, 130, 200, 257, 449, 640, 1000, 1536]
    for sq, splits in ((33, 1), (129, 1 if causal else 2), (300, 1)):
        _check(len(lengths), sq, 2, 256, page, lengths, dtype, causal, layout="query",
               num_splits=splits, kernel="query_eight_waves")


@gpu
def test_ids_outside_the_pool_and_several_items():
    _check(2, 300, 3, 256, 64, [1536, 777], torch.bfloat16, outside=True, layout="query",
           num_splits=1, persistent_programs=4, kernel="query_eight_waves")
    _check(2, 260, 3, 256, 64, [1920, 777], torch.float16, True, layout="query", num_splits=2,
           persistent_programs=5, kernel="query_eight_waves")
