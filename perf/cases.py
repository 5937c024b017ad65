"""The sorts that users of this library run, as measurable cases.

Inputs live where such a user has them: device-resident sorts, batches and
merges work on arenas in HBM (torch tensors here, handed over as pointers);
the Contest-shaped host entry and the server take host arrays.  Every size
and distribution is one of the repository's own workloads or test inputs,
over the range from the smallest served request to the 2 GiB sort.
"""
import ctypes
import importlib.util
import math
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _load():
    spec = importlib.util.spec_from_file_location(
        "ps5", os.path.join(ROOT, "parallel-string-sorting_amd", "ps5.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


ps5 = _load()

DIGITS, ACGT, ASCII = "digits", "acgt", "ascii"
LETTERS = {DIGITS: ps5.ALPHA_DIGITS, ACGT: ps5.ALPHA_ACGT, ASCII: ps5.ALPHA_ASCII94}
PAD = 16                    # NUL bytes behind the last string of an arena
CHUNK = 1 << 26             # elements made at a time where an index array is needed
REPEAT_LEN = 2048           # length of the text's repeated segments


def listed():
    return [
        # the smallest served request (10 KB of prefix-heavy strings), sorted alone: launches and round trips
        {"name": "sort_request_10kb", "op": "sort", "family": "prefixed", "strings": 167, "lcp": True},
        # one ordinary set of a batch workload, sorted alone by the contestant without LCPs
        {"name": "sort_set_acgt_no_lcp", "op": "sort", "family": "uniform", "strings": 40009, "lo": 4, "hi": 48,
         "alphabet": ACGT, "lcp": False},
        # the 10 MiB digits benchmark: a mid-sized latency-bound sort with LCPs
        {"name": "sort_10mb_digits", "op": "sort", "family": "uniform", "strings": 499331, "lo": 8, "hi": 32,
         "alphabet": DIGITS, "lcp": True},
        # every suffix of a DNA text with repeats (suffix mode of the test runner): overlapping, deep strings
        {"name": "sort_suffixes_4m", "op": "sort", "family": "suffixes", "strings": 4194301, "lcp": True},
        # 20 M reads of 100 bases with repeats: long shared prefixes and heavy equal keys
        {"name": "sort_windows_20m", "op": "sort", "family": "windows", "strings": 20000000, "width": 100, "lcp": True},
        # the 2 GiB random ASCII benchmark: the largest single sort
        {"name": "sort_2gb_ascii", "op": "sort", "family": "uniform", "strings": 64111915, "lo": 1, "hi": 64,
         "alphabet": ASCII, "lcp": True},
        # URL-like strings with LCPs and distinguishing characters (the LCP-cache contestant), 256 MB
        {"name": "cache_prefixed_256mb", "op": "cache", "family": "prefixed", "strings": 4400003},
        # many small independent sets in one pass
        {"name": "batch_512_small", "op": "batch", "sets": 512, "count_lo": 1000, "count_hi": 16000, "lo": 4,
         "hi": 48, "lcp": True},
        # uneven sets from 1 k to 2 M strings in one pass
        {"name": "batch_192_uneven", "op": "batch", "sets": 192, "count_lo": 1000, "count_hi": 2000000, "lo": 4,
         "hi": 48, "lcp": True},
        # eight sorted shards merged with their LCP arrays, the end of a sharded sort
        {"name": "merge_8_shards", "op": "merge", "family": "uniform", "strings": 16000003, "lo": 1, "hi": 64,
         "alphabet": ASCII, "shards": 8},
        # the host drop-in on the reference's random10 shape: pointers in, sorted pointers and LCPs out
        {"name": "host_random10_32mb", "op": "host", "strings": 1973789, "lo": 15, "hi": 17, "alphabet": DIGITS,
         "shuffled": False},
        # a burst of 16 requests from 10 KB to 4 MB through the server
        {"name": "serve_burst_16", "op": "serve", "requests": 16, "bytes_lo": 10000, "bytes_hi": 4000000},
    ]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    """One more case of the listed ranges: sizes log-uniform, so odd ones too."""
    op = rng.choice(["sort", "sort", "sort", "sort", "cache", "batch", "merge", "host", "serve"])
    if op == "batch":
        sets = rng.randint(16, 192) if rng.random() < 0.5 else rng.randint(193, 512)
        hi = 2000000 if sets <= 192 else 16000
        lo = rng.choice([4, 8])
        return {"op": op, "sets": sets, "count_lo": 1000, "count_hi": _log_int(rng, 4000, hi), "lo": lo,
                "hi": rng.randint(lo + 8, 48), "lcp": rng.random() < 0.75}
    if op == "serve":
        return {"op": op, "requests": rng.randint(4, 16), "bytes_lo": 10000, "bytes_hi": _log_int(rng, 40000, 4000000)}
    if op == "host":
        return {"op": op, "strings": _log_int(rng, 1000, 1973789), "lo": 15, "hi": 17,
                "alphabet": rng.choice([DIGITS, ACGT, ASCII]), "shuffled": rng.random() < 0.25}
    if op == "cache":
        return {"op": op, "family": "prefixed", "strings": _log_int(rng, 1000, 4400003)}
    lens = {DIGITS: (8, 32), ACGT: (4, 48), ASCII: (1, 64)}
    alphabet = rng.choice([DIGITS, ACGT, ASCII])
    if op == "merge":
        return {"op": op, "family": "uniform", "strings": _log_int(rng, 100000, 16000003), "lo": lens[alphabet][0],
                "hi": lens[alphabet][1], "alphabet": alphabet, "shards": rng.randint(2, 8)}
    family = rng.choice(["uniform", "uniform", "prefixed", "windows", "suffixes"])
    case = {"op": op, "family": family, "lcp": rng.random() < 0.75}
    if family == "uniform":
        case.update(strings=_log_int(rng, 160, 64111915), lo=lens[alphabet][0], hi=lens[alphabet][1],
                    alphabet=alphabet)
    elif family == "prefixed":
        case.update(strings=_log_int(rng, 160, 4400003))
    elif family == "windows":
        case.update(strings=_log_int(rng, 10000, 20000000), width=rng.randint(50, 100))
    else:
        case.update(strings=_log_int(rng, 10000, 4194301))
    return case


# ------------------------------------------------------------------ inputs

def _letters(gen, n, alphabet):
    """n characters of an alphabet, i.i.d."""
    if alphabet == ASCII:
        return torch.randint(33, 127, (n,), generator=gen, device="cuda", dtype=torch.uint8)
    if alphabet == DIGITS:
        return torch.randint(48, 58, (n,), generator=gen, device="cuda", dtype=torch.uint8)
    lut = torch.tensor(list(ps5.ALPHA_ACGT), dtype=torch.uint8, device="cuda")
    out = torch.empty(n, dtype=torch.uint8, device="cuda")
    for b in range(0, n, CHUNK):
        e = min(n, b + CHUNK)
        out[b:e] = lut[torch.randint(0, 4, (e - b,), generator=gen, device="cuda")]
    return out


def _laid_out(lens):
    """start and end offsets of strings of these lengths, laid out in order with a NUL behind each"""
    ends = torch.cumsum(lens + 1, 0)
    return ends - (lens + 1), ends


def _u32(t):
    """int64 values below 2^32 as the same bits in int32"""
    return t.to(torch.int32) if int(t[-1]) < 2**31 else torch.where(t >= 2**31, t - 2**32, t).to(torch.int32)


def _uniform(gen, case):
    lens = torch.randint(case["lo"], case["hi"] + 1, (case["strings"],), generator=gen, device="cuda")
    starts, ends = _laid_out(lens)
    used = int(ends[-1])
    arena = torch.zeros(used + PAD, dtype=torch.uint8, device="cuda")
    arena[:used] = _letters(gen, used, case["alphabet"])
    arena[ends - 1] = 0
    return arena, _u32(starts)


def _prefixed(gen, case, nprefix=1000, zipf=1.1):
    """one of 1000 prefixes of 8..40 characters by Zipf rank, then 10..60 random characters"""
    n = case["strings"]
    plen = torch.randint(8, 41, (nprefix,), generator=gen, device="cuda")
    prefix = _letters(gen, nprefix * 40, ASCII).view(nprefix, 40)
    weight = torch.arange(1, nprefix + 1, device="cuda", dtype=torch.float64) ** -zipf
    ranks = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) * weight.sum()
    rank = torch.searchsorted(torch.cumsum(weight, 0), ranks).clamp_(max=nprefix - 1)
    starts, ends = _laid_out(plen[rank] + torch.randint(10, 61, (n,), generator=gen, device="cuda"))
    used = int(ends[-1])
    arena = torch.zeros(used + PAD, dtype=torch.uint8, device="cuda")
    arena[:used] = _letters(gen, used, ASCII)
    arena[ends - 1] = 0
    column = torch.arange(40, device="cuda")
    for b in range(0, n, CHUNK // 40):
        r, s = rank[b:b + CHUNK // 40], starts[b:b + CHUNK // 40]
        inside = column[None, :] < plen[r][:, None]
        arena[(s[:, None] + column[None, :])[inside]] = prefix[r][inside]
    return arena, _u32(starts)


def _text(gen, n):
    """i.i.d. ACGT; 5% of its 2 kb blocks are copies of ten segments"""
    text = _letters(gen, n, ACGT)
    blocks = n // REPEAT_LEN
    copies = int(0.05 * blocks)
    if copies:
        segment = _letters(gen, 10 * REPEAT_LEN, ACGT).view(10, REPEAT_LEN)
        at = torch.randperm(blocks, generator=gen, device="cuda")[:copies]
        text[:blocks * REPEAT_LEN].view(blocks, REPEAT_LEN)[at] = segment[
            torch.randint(0, 10, (copies,), generator=gen, device="cuda")]
    return text


def _windows(gen, case):
    n, width = case["strings"], case["width"]
    text = _text(gen, max(1 << 16, int(26.8 * n)))
    at = torch.randint(0, text.numel() - width + 1, (n,), generator=gen, device="cuda")
    arena = torch.zeros(n * (width + 1) + PAD, dtype=torch.uint8, device="cuda")
    rows = arena[:n * (width + 1)].view(n, width + 1)
    column = torch.arange(width, device="cuda")
    for b in range(0, n, CHUNK // width):
        rows[b:b + CHUNK // width, :width] = text[at[b:b + CHUNK // width, None] + column[None, :]]
    return arena, _u32(torch.arange(n, device="cuda") * (width + 1))


def _suffixes(gen, case):
    n = case["strings"]
    arena = torch.zeros(n + PAD, dtype=torch.uint8, device="cuda")
    arena[:n] = _text(gen, n)
    return arena, torch.arange(n, device="cuda", dtype=torch.int32)


FAMILIES = {"uniform": _uniform, "prefixed": _prefixed, "windows": _windows, "suffixes": _suffixes}


def _set_counts(case):
    """log-uniform set sizes at the quantiles of their range, large and small ones mixed"""
    k = case["sets"]
    counts = [int(case["count_lo"] * (case["count_hi"] / case["count_lo"]) ** ((i + 0.5) / k)) for i in range(k)]
    return [counts[int(i)] for i in np.random.RandomState(7).permutation(k)]


def _request_strings(case):
    """strings per request: log-uniform at the quantiles of the range of bytes, 60 bytes each on average"""
    k = case["requests"]
    sizes = [int(case["bytes_lo"] * (case["bytes_hi"] / case["bytes_lo"]) ** (i / (k - 1))) for i in range(k)]
    return [sizes[int(i)] // 60 for i in np.random.RandomState(7).permutation(k)]


def _request(seed, n):
    arena, offs = ps5.gen_prefixed(seed, 68 * n + 1000)
    end = int(offs[n])
    return np.concatenate([arena[:end], np.zeros(PAD, np.uint8)]), offs[:n].copy()


class _Tensor:
    """a torch tensor where the binding takes a device buffer"""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def _out(n, dtype=torch.int32):
    return _Tensor(torch.zeros(n, dtype=dtype, device="cuda"))


_held = {}                  # the sort context and the server a program creates once and keeps


def _context(n):
    if "context" not in _held:
        _held["context"] = ps5.Context(torch.cuda.current_device())
    ps5._check(ps5.load().ps5_ctx_reserve(_held["context"].h, n), "ps5_ctx_reserve")
    return _held["context"]


def _server():
    if "server" not in _held:
        _held["server"] = ps5.Server(torch.cuda.current_device(), hbm_budget=8 << 30, slots=4,
                                     max_batch_strings=1 << 20)
    return _held["server"]


def prepare(case, seed):
    op = case["op"]
    if op == "host":
        # host strings in one arena, in order (as read from a file) or through shuffled pointers
        n = case["strings"]
        cap = n * (case["hi"] + 1)
        arena, offs = ps5.gen_uniform(seed, cap, case["lo"], case["hi"], LETTERS[case["alphabet"]])
        strings = (offs[:n].astype(np.uint64) + np.uint64(arena.ctypes.data))
        if case["shuffled"]:
            strings = strings[np.random.RandomState(seed % 2**32).permutation(n)]
        return {"op": op, "arena": arena, "n": n, "strings": np.ascontiguousarray(strings),
                "sorted": np.zeros(n, np.uint64), "lcp": np.zeros(n, np.uint64)}
    if op == "serve":
        requests = [_request(seed * 1000 + i, n) for i, n in enumerate(_request_strings(case))]
        return {"op": op, "requests": requests, "server": _server()}
    gen = torch.Generator("cuda")
    gen.manual_seed(seed)
    if op == "batch":
        counts = _set_counts(case)
        first = np.concatenate([[0], np.cumsum(np.array(counts, np.uint64))]).astype(np.uint64)
        n = int(first[-1])
        lens = torch.randint(case["lo"], case["hi"] + 1, (n,), generator=gen, device="cuda")
        starts, ends = _laid_out(lens)
        edge = [0] + ends[torch.from_numpy(first[1:].astype(np.int64)).cuda() - 1].tolist()
        arena = torch.zeros(edge[-1] + PAD, dtype=torch.uint8, device="cuda")
        for k in range(len(counts)):
            arena[edge[k]:edge[k + 1]] = _letters(gen, edge[k + 1] - edge[k], (ACGT, DIGITS, ASCII)[k % 3])
        arena[ends - 1] = 0
        state = {"op": op, "ctx": _context(n), "arena": _Tensor(arena), "offs": _Tensor(starts), "first": first,
                 "perm": _out(n), "lcp": _out(n) if case["lcp"] else None}
        torch.cuda.synchronize()
        return state
    arena, offs = FAMILIES[case["family"]](gen, case)
    n = case["strings"]
    state = {"op": op, "n": n, "ctx": _context(n), "arena": _Tensor(arena), "offs": _Tensor(offs), "perm": _out(n),
             "lcp": _out(n) if case.get("lcp", True) else None}
    torch.cuda.synchronize()
    if op == "cache":
        state["cache"] = _out(n, torch.uint8)
    if op == "merge":
        # the shards are contiguous ranges, each sorted on its own; indices are global
        bounds = [n * k // case["shards"] for k in range(case["shards"] + 1)]
        idx, lcp = _out(n), _out(n)
        for b, e in zip(bounds[:-1], bounds[1:]):
            state["ctx"].sort_device(state["arena"], arena.numel(), _Tensor(offs[b:e]), e - b,
                                     _Tensor(idx.tensor[b:e]), _Tensor(lcp.tensor[b:e]))
            idx.tensor[b:e] += b
        state.update(first=np.array(bounds, np.uint64), idx=idx, run_lcp=lcp)
    torch.cuda.synchronize()
    return state


def run(state):
    op = state["op"]
    if op == "host":
        at = state["strings"].ctypes.data
        ps5._check(ps5.load().ps5_sort_strings(ctypes.c_void_p(at), state["n"],
                                               ctypes.c_void_p(state["lcp"].ctypes.data),
                                               ctypes.c_void_p(state["sorted"].ctypes.data)), "ps5_sort_strings")
        # addresses differ from process to process: offsets into the arena are the result
        return state["sorted"] - np.uint64(state["arena"].ctypes.data), state["lcp"]
    if op == "serve":
        server = state["server"]
        ids = [server.submit(arena, offs) for arena, offs in state["requests"]]
        return [server.wait(i)[:2] for i in ids]
    ctx, arena, offs, perm, lcp = (state[k] for k in ("ctx", "arena", "offs", "perm", "lcp"))
    size = arena.tensor.numel()
    if op == "batch":
        ctx.sort_batch_device(arena, size, offs, state["first"], perm, lcp)
    elif op == "merge":
        ctx.merge_device(arena, size, offs, state["first"], state["idx"], state["run_lcp"], perm, lcp)
    else:
        ctx.sort_device(arena, size, offs, state["n"], perm, lcp)
    if op == "cache":
        ctx.dist_chars_device(arena, size, offs, state["n"], perm, lcp, state["cache"])
        return perm.tensor, lcp.tensor, state["cache"].tensor
    return (perm.tensor,) if lcp is None else (perm.tensor, lcp.tensor)


def work(case):
    """Arena and offsets read once, permutation and LCPs (and what else comes back) written once."""
    op = case["op"]
    if op == "serve":
        return {"bytes": sum(_request_strings(case)) * (60 + 4 + 8), "flops": 0}
    if op == "batch":
        n = sum(_set_counts(case))
        return {"bytes": n * ((case["lo"] + case["hi"]) / 2 + 1 + 8 + 4 + (4 if case["lcp"] else 0)), "flops": 0}
    n = case["strings"]
    family = case.get("family", "uniform")
    chars = {"prefixed": 60.0, "suffixes": 1.0, "windows": case.get("width", 0) + 1.0}.get(family)
    if chars is None:
        chars = (case["lo"] + case["hi"]) / 2 + 1
    each = {"host": 8 + 8 + 8, "merge": 4 + 8 + 8, "cache": 4 + 9}.get(op, 4 + (8 if case.get("lcp") else 4))
    return {"bytes": n * (chars + each), "flops": 0}
