"""Batches whose requests share a prefix: their tables name the same pages at the same
places. Calls too large for the last-level cache load K/V past it, except the
items of shared pages, which other requests read again (stream_kv in
fgw_amd/csrc/fmha_kernel.h). The outputs are checked against the oracle, and
the time of a shared batch against one of the same size with pages of its own:
the shared one reads an eighth or less from memory.
"""
import pytest
import torch

from oracle import mha_oracle as O

pytestmark = pytest.mark.gpu


def _kernel(b, sq, h, d, rows, width, page, dtype, kernel, **plan):
    from fgw_amd.operators.mha.current import build_kernel
    kern = build_kernel(b, sq, h, d, rows, width, page, False,
                        "float16" if dtype == torch.float16 else "bfloat16", 0, layout="key", **plan)
    info = kern.launch_info
    assert info.name == kernel and info.stream_bytes > 0
    return kern


@pytest.mark.parametrize("kernel,b,sq,h,d,page,width,dtype,plan", [
    ("key_stream", 33, 1, 16, 64, 64, 64, torch.bfloat16, dict(num_splits=1)),
    ("key_stream", 70, 3, 4, 128, 32, 64, torch.float16, dict(num_splits=2)),
    ("key_stream", 33, 2, 8, 128, 32, 64, torch.bfloat16, dict(num_splits=4, stages=1)),
    ("decode", 17, 1, 8, 128, 16, 256, torch.float16, dict(num_splits=1)),
    ("decode", 9, 1, 8, 256, 64, 64, torch.bfloat16, dict(num_splits=4)),
    ("key_groups", 17, 3, 16, 64, 16, 256, torch.bfloat16, dict(num_splits=2))])
def test_shared_prefixes_match_the_oracle(kernel, b, sq, h, d, page, width, dtype, plan):
    """The first half of the table is shared by the even requests; ragged ends."""
    capacity = width * page
    pages = b * width
    g = torch.Generator(device="cuda").manual_seed(b)
    q, k, v = (torch.randn(n, h, d, generator=g, device="cuda", dtype=dtype)
               for n in (b * sq, pages * page, pages * page))
    q = q.view(b, sq, h, d)
    table = torch.randperm(pages, generator=torch.Generator().manual_seed(3)).view(b, width)
    table[::2, :width // 2] = table[0, :width // 2]
    table = table.to(torch.int32).contiguous()
    lengths = torch.tensor([capacity - 7 * i for i in range(b)], dtype=torch.int32)
    kern = _kernel(b, sq, h, d, k.shape[0], width, page, dtype, kernel, **plan)
    got = kern(q, k, v, table.cuda(), lengths.cuda())
    rtol, atol = O.TOLERANCES[dtype]
    for i in (0, 1, 2, b - 1):  # one request at a time, on the CPU
        rows = (table[i].long()[:, None] * page + torch.arange(page)).flatten()
        one = torch.arange(width, dtype=torch.int32)[None]
        want = O.chunked_reference(q[i:i + 1].cpu(), k[rows.cuda()].cpu(), v[rows.cuda()].cpu(), one,
                                   lengths[i:i + 1], page, False)
        torch.testing.assert_close(got[i:i + 1].cpu(), want, rtol=rtol, atol=atol)


def _time(kern, inputs):
    for _ in range(3):
        kern(*inputs)
    best = float("inf")
    for _ in range(5):
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        kern(*inputs)
        start.record()
        for _ in range(10):
            kern(*inputs)
        end.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(end) / 10)
    return best


# Shared over own pages, cached loads on shared pages / non-temporal ones everywhere:
# 0.42 / 0.64 and 0.42 / 0.75; the bound lies between.
@pytest.mark.parametrize("kernel,b,sq,h,d,page,keys,bound", [
    ("key_stream", 32, 1, 8, 128, 64, 8192, 0.56),
    ("decode", 32, 1, 16, 64, 16, 8192, 0.59)])
def test_shared_pages_are_read_from_the_cache(kernel, b, sq, h, d, page, keys, bound):
    width = keys // page
    q = torch.randn(b, sq, h, d, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(b * keys, h, d, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    own = torch.randperm(b * width, device="cuda").view(b, width).to(torch.int32)
    shared = own[:1].repeat(b, 1)
    lengths = torch.full((b,), keys, dtype=torch.int32, device="cuda")
    kern = _kernel(b, sq, h, d, k.shape[0], width, page, torch.bfloat16, kernel)
    times = [_time(kern, (q, k, v, t, lengths)) for t in (shared, own)]
    print(f"shared {times[0] * 1e3:.1f} us, own pages {times[1] * 1e3:.1f} us", flush=True)
    assert times[0] < bound * times[1]
