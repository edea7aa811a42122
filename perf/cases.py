"""The workloads whose time is tracked: paged attention calls as a serving program makes them.

A case is one call of the operator: `entry` says how it is made.
  "kernel"  the launch callable of build_kernel, planned once per shape and kept,
            as a decode or prefill loop does (lengths stay on the device);
  "paged"   mha_paged_decode, the one-call public entry (it reads the lengths back,
            plans and launches on each call);
  "packed"  build_gather_attention: the live pages are copied to a dense cache,
            then attended to.
Sizes follow the repository's benchmark and test tables (B, Sq, H, D, page and
cache lengths there), and `draw` spreads over the same ranges. Inputs are
standard normal with shuffled pages, as in the benchmark; `q_std` 3 gives the
sharper softmax of trained heads.
"""
import torch

from fgw_amd.operators.mha import current
from fgw_amd.operators.mha.packed_cache import build_gather_attention

_DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16}
_MAX_PAIR_FLOPS = 2.0e11  # of a drawn case: under the largest listed prefill
_MAX_BYTES = 4.0e8        # of a drawn case: under the largest listed decode


def _case(name, entry, batch, sq, heads, dim, page, capacity, dtype, causal=False, ragged=False,
          q_std=1.0):
    case = dict(entry=entry, batch=batch, sq=sq, heads=heads, dim=dim, page=page,
                capacity=capacity, dtype=dtype, causal=causal, ragged=ragged, q_std=q_std)
    if name:
        case["name"] = name
    return case


def listed():
    bf, fp = "bfloat16", "float16"
    return [
        # The smallest call: one head, one token, a short cache. Latency alone.
        _case("decode_b1h1", "kernel", 1, 1, 1, 128, 128, 512, bf),
        # Short multi-token decode over a packed copy of a ragged cache (prefix packing).
        _case("packed_q16_d64", "packed", 4, 16, 8, 64, 64, 4096, fp, ragged=True),
        # A serving batch in mid-flight: ragged lengths, 16-token pages.
        _case("decode_ragged_page16", "kernel", 16, 1, 16, 128, 16, 4096, bf, ragged=True, q_std=3.0),
        # A full decode batch over many heads: the largest K/V read.
        _case("decode_batch_h32", "kernel", 8, 1, 32, 128, 64, 4096, fp),
        # Long-context decode (the benchmark's second headline).
        _case("decode_long", "kernel", 2, 1, 8, 128, 128, 32768, bf),
        # Verification of eight drafted tokens over ragged caches, through the one-call entry.
        _case("verify_q8", "paged", 4, 8, 16, 128, 32, 8192, bf, causal=True, ragged=True),
        # One chunk of a prompt against its cached prefix, 16-token pages.
        _case("chunk_q512_page16", "kernel", 1, 512, 32, 128, 16, 8192, bf, causal=True, q_std=3.0),
        # Prefill with head dim 96, odd query length and ragged caches, through the one-call entry.
        _case("ragged_q257_d96", "paged", 8, 257, 8, 96, 64, 1152, fp, ragged=True),
        # Prompt prefill, head dim 64.
        _case("causal_s4096_d64", "kernel", 1, 4096, 16, 64, 64, 4096, fp, causal=True, q_std=3.0),
        # Prompt chunk with the widest heads.
        _case("causal_q1024_d256", "kernel", 2, 1024, 8, 256, 256, 2048, bf, causal=True),
        # The benchmark's headline prefill and its long companion, the largest call.
        _case("prefill_q4096", "kernel", 2, 4096, 8, 128, 128, 2048, bf),
        _case("prefill_q32768", "kernel", 2, 32768, 8, 128, 128, 2048, bf),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    """A case of the listed ranges: odd sizes, every page size, head dims off the powers of two."""
    kind = rng.choice(("decode", "decode", "short", "chunk", "prefill", "packed"))
    dim = rng.choice((64, 64, 80, 96, 128, 128, 128, 128, 192, 256))
    page = rng.choice((16, 16, 32, 48, 64, 64, 128, 128, 256))
    dtype = rng.choice(("bfloat16", "bfloat16", "float16"))
    heads = rng.choice((1, 4, 8, 8, 12, 16, 32))
    ragged = rng.random() < 0.5
    causal = rng.random() < 0.5
    batch = _log_int(rng, 1, 64)
    if kind == "decode":
        sq, capacity, causal = 1, _log_int(rng, 128, 32768), False
    elif kind in ("short", "packed"):
        sq, capacity = rng.randint(2, 32), _log_int(rng, 128, 16384)
    elif kind == "chunk":
        sq, capacity, batch = _log_int(rng, 33, 1023), _log_int(rng, 256, 16384), _log_int(rng, 1, 8)
    else:
        sq, batch = _log_int(rng, 1024, 16384), _log_int(rng, 1, 4)
        capacity = sq if causal else _log_int(rng, 256, 8192)
    if causal:
        capacity = max(capacity, sq)
    capacity = -(-capacity // page) * page
    entry = "packed" if kind == "packed" else rng.choice(("kernel", "kernel", "paged"))
    case = _case(None, entry, batch, sq, heads, dim, page, capacity, dtype, causal, ragged,
                 rng.choice((1.0, 3.0)))
    while work(case)["flops"] > _MAX_PAIR_FLOPS or work(case)["bytes"] > _MAX_BYTES:
        if case["batch"] > 1:
            case["batch"] = case["batch"] // 2
        elif case["heads"] > 1:
            case["heads"] = case["heads"] // 2
        else:
            case["sq"] = max(1, case["sq"] // 2)
    return case


def _lengths(case):
    """Cache lengths before the seed orders them: full, or spread from a quarter of the
    capacity to all of it (with causal attention, never below the query length)."""
    b, cap = case["batch"], case["capacity"]
    if not case["ragged"]:
        return [cap] * b
    low = max(cap // 4, case["sq"] if case["causal"] else 1)
    return [low + (cap - low) * (2 * i + 1) // (2 * b) for i in range(b)]


def _width(case):
    return case["capacity"] // case["page"]


def _inputs(case, seed):
    """Q, K/V pool, block table, lengths on the GPU, and the lengths on the host."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    b, sq, h, d, page, width = (case[k] if k != "width" else _width(case)
                                for k in ("batch", "sq", "heads", "dim", "page", "width"))
    q = torch.randn(b, sq, h, d, generator=gen, device="cuda", dtype=dtype) * case["q_std"]
    k = torch.randn(b * width * page, h, d, generator=gen, device="cuda", dtype=dtype)
    v = torch.randn(b * width * page, h, d, generator=gen, device="cuda", dtype=dtype)
    table = torch.randperm(b * width, generator=gen, device="cuda").reshape(b, width).to(torch.int32)
    base = _lengths(case)
    order = torch.randperm(b, generator=torch.Generator().manual_seed(seed)).tolist()
    host = [base[i] for i in order]
    return q, k, v, table, torch.tensor(host, dtype=torch.int32, device="cuda"), host


def prepare(case, seed):
    q, k, v, table, lengths, host = _inputs(case, seed)
    state = dict(entry=case["entry"], inputs=(q, k, v, table, lengths), page=case["page"],
                 causal=case["causal"])
    if case["entry"] == "kernel":
        state["call"] = current.build_kernel(
            case["batch"], case["sq"], case["heads"], case["dim"], k.shape[0], _width(case),
            case["page"], case["causal"], case["dtype"], q.device.index,
            full_kv_cache=not case["ragged"])
    elif case["entry"] == "packed":
        shape = (case.get("name"), case["batch"], case["sq"], case["heads"], case["dim"],
                 case["page"], _width(case), host, case["causal"])
        state["call"], _ = build_gather_attention(shape, case["dtype"], state["inputs"], current,
                                                  None, q.device.index, check=False)
    return state


def run(state):
    if state["entry"] == "kernel":
        return state["call"](*state["inputs"])
    if state["entry"] == "packed":
        return state["call"]()
    return current.mha_paged_decode(*state["inputs"], state["page"], state["causal"])


def work(case):
    """Live K/V, Q, table and lengths read once and O written once; 4 D flops per visible pair."""
    b, sq, h, d = (case[k] for k in ("batch", "sq", "heads", "dim"))
    lengths = _lengths(case)
    if case["causal"]:
        pairs = sum(sum(range(max(0, n - sq + 1), n + 1)) if n < sq
                    else sq * (n - sq) + sq * (sq + 1) // 2 for n in lengths)
    else:
        pairs = sum(n * sq for n in lengths)
    return {"bytes": 2 * h * d * 2 * sum(lengths) + 2 * b * sq * h * d * 2 + 4 * b * _width(case) + 4 * b,
            "flops": 4 * h * d * pairs}


def tolerance(case):
    """P and O are rounded to the input type. Measured against 64 bits: 2.3e-3 (bf16) and
    2.9e-4 (fp16) at most over the listed cases; four times that."""
    if case["dtype"] == "bfloat16":
        return {"rel": 1.0e-2, "max": 0.06}
    return {"rel": 1.2e-3, "max": 8.0e-3}


def exact(case, seed):
    """Softmax attention in 64 bits over the live rows, laid out as the operator's output."""
    q, k, v, table, _, host = _inputs(case, seed)
    b, sq, h, d = q.shape
    out = torch.zeros(b, sq, h, d, dtype=torch.float64, device=q.device)
    for i in range(b):
        n = host[i]
        pos = torch.arange(n, device=q.device)
        rows = table[i, pos // case["page"]].long() * case["page"] + pos % case["page"]
        kk, vv = k[rows].double(), v[rows].double()
        chunk = max(1, min(sq, (1 << 26) // n))
        for j in range(h):
            for s in range(0, sq, chunk):
                e = min(sq, s + chunk)
                scores = (q[i, s:e, j].double() @ kk[:, j].T) * d ** -0.5
                if case["causal"]:
                    last = torch.arange(s, e, device=q.device) + (n - sq)
                    scores.masked_fill_(pos[None, :] > last[:, None], float("-inf"))
                out[i, s:e, j] = scores.softmax(-1).nan_to_num_(0.0) @ vv[:, j]
    return out
