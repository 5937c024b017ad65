"""GPU tests of single paths of the sort, each at the sizes where it can go
wrong, bit-exact against the oracle."""
import ctypes

import numpy as np
import pytest

from strsets import pack, random_strings

pytestmark = pytest.mark.gpu


def check(ctx, oracle, arena, offs, with_lcp=True):
    perm, lcp = ctx.sort(arena, offs, with_lcp=with_lcp)
    r, msg = oracle.verify(arena, offs, perm, lcp) if with_lcp else oracle.verify(arena, offs, perm)
    assert r == 0, msg


@pytest.mark.parametrize("syncs", [1, 2, 3])
def test_new_context_ignores_recycled_sequence_words(ps5, oracle, syncs):
    """a context created after another one's pinned memory was returned sorts
    from its own staged counters, whatever number the memory still holds"""
    small = pack(random_strings(5000, 0, 12, b"abcdefgh", 11))
    large = pack(random_strings(60000, 0, 40, b"ab", 12))
    first = ps5.Context(0)
    first.set_planning(1)
    for _ in range(syncs):
        first.sort(*small)
    first.close()
    second = ps5.Context(0)
    try:
        check(second, oracle, *large)
    finally:
        second.close()


def packed_case(sigma, n, seed, hi=60, rare=None):
    """(arena, offs) of n strings over sigma characters drawn from the whole
    byte range, many sharing 8 characters and more; `rare` puts a character
    outside that alphabet at that place of one string"""
    rng = np.random.default_rng(seed)
    alpha = np.sort(rng.choice(np.arange(1, 255), sigma, replace=False)).astype(np.uint8)
    lens = rng.integers(0, hi, n)
    chars = alpha[rng.integers(0, sigma, (n, hi))]
    stems = alpha[rng.integers(0, sigma, (40, 24))][rng.integers(0, 40, n)]
    keep = np.arange(24)[None, :] < rng.integers(0, 25, n)[:, None]
    chars[:, :24] = np.where(keep, stems, chars[:, :24])
    if rare is not None:
        i = int(rng.integers(0, n))
        lens[i] = hi - 1
        chars[i, rare] = 255
    ends = np.cumsum(lens + 1)
    offs = (ends - lens - 1).astype(np.uint32)
    arena = np.zeros(int(ends[-1]) + 16, np.uint8)
    inside = np.arange(hi)[None, :] < lens[:, None]
    arena[(offs[:, None].astype(np.int64) + np.arange(hi)[None, :])[inside]] = chars[inside]
    return arena, offs


def concatenated(sets):
    """one arena, uint64 offsets and set boundaries of several (arena, offs)"""
    base = np.cumsum([0] + [len(a) for a, _ in sets])
    arena = np.concatenate([a for a, _ in sets])
    offs = np.concatenate([o.astype(np.uint64) + np.uint64(b) for (_, o), b in zip(sets, base)])
    return arena, offs, np.cumsum([0] + [len(o) for _, o in sets]).astype(np.uint64)


@pytest.mark.parametrize("sigma", [1, 2, 4, 7, 8, 15, 16, 31, 32])
@pytest.mark.parametrize("n", [2049, 30011, 1050003])
def test_packed_roots(ctx, oracle, sigma, n):
    """every code width (3, 4, 5 bits and none) at the edges of its alphabet"""
    check(ctx, oracle, *packed_case(sigma, n, 100 * sigma + n))


@pytest.mark.parametrize("at", [0, 7, 20, 21, 40])
def test_packed_root_meets_an_unknown_character(ctx, oracle, at):
    """one string holds a character the samples do not show: in the packed
    key (the sort starts over) or behind it (it stands)"""
    check(ctx, oracle, *packed_case(4, 1060000, at, rare=at))
    check(ctx, oracle, *packed_case(4, 1060000, 7 + at, rare=at), with_lcp=False)


@pytest.mark.parametrize("planning", [0, 1])
def test_packed_batch_of_mixed_alphabets(ps5, oracle, planning):
    """sets of one batch choose their own key formats; one of them meets an
    unknown character, and small sets stay unpacked"""
    sets = [packed_case(4, 9000, 1), packed_case(12, 5000, 2), packed_case(40, 7000, 3), packed_case(2, 700, 4), pack([b""]),
            packed_case(20, 6000, 5), packed_case(4, 1060000, 6)]
    for rare in (None, 5):
        if rare is not None:
            sets[-1] = packed_case(4, 1060000, 6, rare=rare)
        arena, offs, first = concatenated(sets)
        c = ps5.Context(0)
        try:
            c.set_planning(planning)
            perm, lcp = c.sort_batch(arena, offs, first)
        finally:
            c.close()
        for k in range(len(sets)):
            b, e = int(first[k]), int(first[k + 1])
            r, msg = oracle.verify(arena, offs[b:e].astype(np.uint32), perm[b:e], lcp[b:e])
            assert r == 0, (k, msg)


@pytest.mark.parametrize("n", [2049, 4095, 4096, 4097, 6145, 65537, 262143, 262145, 600011])
@pytest.mark.parametrize("kind", ["spread", "sorted", "heavy"])
def test_partition_edges(ctx, oracle, n, kind):
    """chunk and group remainders; buckets that lie in few chunks (sorted
    input) and in all of them (heavy duplicates)"""
    rng = np.random.default_rng(n)
    hi = 24
    lens = rng.integers(0, hi, n) if kind != "heavy" else rng.integers(0, 3, n)
    chars = rng.integers(33, 127, (n, hi)).astype(np.uint8)
    if kind == "sorted":
        chars[:, :4] = np.sort(rng.integers(33, 127, (n, 4)).astype(np.uint8).view(">u4").ravel()).view(np.uint8).reshape(n, 4)
    ends = np.cumsum(lens + 1)
    offs = (ends - lens - 1).astype(np.uint32)
    arena = np.zeros(int(ends[-1]) + 16, np.uint8)
    inside = np.arange(hi)[None, :] < lens[:, None]
    arena[(offs[:, None].astype(np.int64) + np.arange(hi)[None, :])[inside]] = chars[inside]
    check(ctx, oracle, arena, offs)
    check(ctx, oracle, arena, offs, with_lcp=False)


@pytest.mark.parametrize("planning", [0, 1])
@pytest.mark.parametrize("tuning", [(64, 2, 4), (64, 3, 2), (256, 10, 32)])
def test_many_levels_and_rounds(ps5, oracle, planning, tuning):
    """rounds of three levels and more reuse the buffers and run tables their
    earlier leaves lie in, and later rounds start from the permutation"""
    c = ps5.Context(0)
    try:
        c.set_planning(planning)
        c.set_tuning(*tuning)
        for sigma, n, seed in ((3, 300007, 1), (60, 150001, 2), (2, 70001, 3)):
            check(c, oracle, *packed_case(sigma, n, seed, hi=40))
    finally:
        c.close()


@pytest.mark.parametrize("planning", [0, 1])
@pytest.mark.parametrize("shared", [0, 7, 8, 15, 63, 64, 65, 200])
def test_runs_with_long_common_prefixes(ps5, oracle, shared, planning):
    """equal-key runs that share `shared` characters past their key, some
    strings ending inside them, some identical"""
    rng = np.random.default_rng(shared)
    strs = []
    for g in range(3):
        stem = bytes([65 + g]) * 8 + rng.integers(97, 123, shared).astype(np.uint8).tobytes()
        for _ in range(6000):
            kind = rng.integers(0, 20)
            tail = rng.integers(97, 123, rng.integers(0, 12)).astype(np.uint8).tobytes()
            if kind == 0 and shared:
                strs.append(stem[:8 + rng.integers(0, shared + 1)])
            elif kind == 1:
                strs.append(stem)
            else:
                strs.append(stem + tail)
        if g == 2:      # one run that shares all of it
            strs = [s if not s.startswith(b"C") else stem + s[len(stem):] for s in strs]
    order = rng.permutation(len(strs))
    c = ps5.Context(0)
    try:
        c.set_planning(planning)
        check(c, oracle, *pack([strs[i] for i in order]))
    finally:
        c.close()


@pytest.mark.parametrize("leaf_keys", [3, 8])
@pytest.mark.parametrize("groups", [
    {40: 3, 2048: 1}, {64: 9, 65: 1}, {256: 2, 257: 2, 512: 2, 513: 2, 1024: 2, 1025: 2},
    {20: 200, 700: 9, 5000: 2}, {200: 700, 400: 700, 900: 700}, {100: 2500, 30: 17, 1500: 3}])
def test_leaves_of_all_kinds_together(ps5, oracle, groups, leaf_keys):
    """leaves of every kind, few of each in one launch, many in their own
    kernels; every fourth group repeats one string, so that it is one run"""
    rng = np.random.default_rng(len(groups) + sum(groups))
    strs = []
    for size, count in groups.items():
        for g in range(count):
            stem = rng.integers(97, 123, 6).astype(np.uint8).tobytes()
            if g % 4 == 3:
                strs += [stem] * size
            else:
                tails = rng.integers(97, 123, (size, 12)).astype(np.uint8)
                cut = rng.integers(0, 13, size)
                strs += [stem + t[:k].tobytes() for t, k in zip(tails, cut)]
    order = rng.permutation(len(strs))
    c = ps5.Context(0)
    try:
        c.set_shape(leaf_keys=leaf_keys)
        arena, offs = pack([strs[i] for i in order])
        check(c, oracle, arena, offs)
        check(c, oracle, arena, offs, with_lcp=False)
    finally:
        c.close()


@pytest.mark.parametrize("bytes_each, count", [(2000, 9), ((1 << 20) - 8, 24), (1 << 20, 3), ((1 << 20) + 1, 3)])
def test_served_requests_staged_and_direct(ps5, oracle, bytes_each, count):
    """requests at the size where they are no longer packed together, in
    batches that need more staging memory than a slot has, beside empty ones
    and ones without LCPs"""
    reqs = [ps5.gen_uniform(900 + i, bytes_each, 3, 40, ps5.ALPHA_ASCII94) for i in range(count)]
    reqs.insert(1, (np.zeros(16, np.uint8), np.zeros(0, np.uint32)))
    reqs.insert(2, (np.zeros(16, np.uint8), np.zeros(1, np.uint32)))
    srv = ps5.Server(0, hbm_budget=4 << 30, slots=2, max_batch_strings=16 << 20)
    try:
        ids = [srv.submit(a, o, with_lcp=i % 3 != 2) for i, (a, o) in enumerate(reqs)]
        out = [srv.wait(i) for i in ids]
    finally:
        srv.close()
    for i, ((a, o), (p, l, _)) in enumerate(zip(reqs, out)):
        if len(o):
            assert oracle.verify(a, o, p, l)[0] == 0 if i % 3 != 2 else oracle.verify(a, o, p)[0] == 0


@pytest.mark.parametrize("sizes", [(1, 1), (1023, 1), (1024, 1024), (1, 3000), (4095, 4097, 2), (20000, 7, 0, 20001),
                                   (9000,) * 9])
@pytest.mark.parametrize("kind", ["ascii", "equal", "deep"])
def test_merge_tile_edges(ps5, ctx, oracle, sizes, kind):
    """tile remainders, runs much shorter than others, empty runs; runs whose
    strings are all equal or differ past their first 8 characters only"""
    rng = np.random.default_rng(sum(sizes) + len(kind))
    n = sum(sizes)
    stem = {"ascii": b"", "equal": b"same", "deep": b"a-common-prefix-"}[kind]
    strs = [stem if kind == "equal" else stem + rng.integers(97, 105, rng.integers(0, 9)).astype(np.uint8).tobytes()
            for _ in range(n)]
    arena, offs = pack(strs)
    bounds = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    idx, lcp = np.zeros(n, np.uint32), np.zeros(n, np.uint32)
    for b, e in zip(bounds[:-1].astype(int), bounds[1:].astype(int)):
        if e > b:
            p, l = oracle.brute_sort(arena, offs[b:e])
            idx[b:e] = p + b
            lcp[b:e] = l
    mi, ml = ctx.merge(arena, offs, bounds, idx, lcp)
    r, msg = oracle.verify(arena, offs, mi, ml)
    assert r == 0, msg


@pytest.mark.parametrize("n", [2, 64, 65, 255, 256, 257, 512, 513, 1025, 2048])
@pytest.mark.parametrize("with_lcp", [True, False])
def test_sorts_of_one_block(ps5, ctx, oracle, n, with_lcp):
    """a sort that is one block of each size class, with deep common prefixes"""
    strs = [b"http://host%d/" % (i % 3) + s for i, s in enumerate(random_strings(n, 0, 30, b"ab/", n))]
    check(ctx, oracle, *pack(strs), with_lcp=with_lcp)


def mix64(z):
    """the sampler's hash (uint64 arrays)"""
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def unlucky_sets(nsets, m, samples, seed):
    """sets of m strings of which the root level's samples show the smallest
    ones only: all others, half of them in groups that share 8 characters and
    more, end in one bucket; every other sampled string starts alike"""
    rng = np.random.default_rng(seed)
    n, width = nsets * m, 20
    rows = np.zeros((n, width), np.uint8)
    rows[:, :width - 1] = rng.integers(98, 123, (n, width - 1))
    for s in range(nsets):
        b = s * m
        stems = rng.integers(98, 123, (40, 8)).astype(np.uint8)
        rows[b:b + m // 2, :8] = stems[rng.integers(0, 40, m // 2)]
        rows[b:b + m] = rows[b + rng.permutation(m)]
        h = mix64(np.uint64(0x5EED5EED) ^ (np.uint64(b) << np.uint64(21)) ^ np.arange(samples, dtype=np.uint64))
        at = b + ((h >> np.uint64(32)) * np.uint64(m) >> np.uint64(32)).astype(np.int64)
        rows[at, 0] = 97
        rows[at[::2], :8] = 97
    cut = rng.integers(0, 10, n)      # strings of 10 to 19 characters
    rows[np.arange(width)[None, :] >= width - 1 - cut[:, None]] = 0
    arena = np.concatenate([rows.reshape(-1), np.zeros(16, np.uint8)])
    return arena, np.arange(n, dtype=np.uint64) * np.uint64(width), np.arange(nsets + 1, dtype=np.uint64) * np.uint64(m)


def test_host_finishes_a_round_with_a_chained_level(ps5, oracle, monkeypatch):
    """one level planned on the device leaves 4 M strings and more in large
    segments: the host's next level chains the one after it, while leaves of
    both earlier levels are listed, each of which is finished once"""
    nsets, m, leaf_target, oversample = 112, 45000, 64, 2
    samples = 1023 * oversample       # 2^10 buckets, the depth that 45000 / 64 asks for
    arena, offs, first = unlucky_sets(nsets, m, samples, 5)
    stats = {}
    for chain in ("1", "0"):
        monkeypatch.setenv("PS5_CHAIN_LEVELS", chain)
        c = ps5.Context(0)
        try:
            c.set_planning(1)
            c.set_tuning(leaf_target, 10, oversample)
            perm, lcp = c.sort_batch(arena, offs, first)
            stats[chain] = c.work_stats()
        finally:
            c.close()
        for k in range(nsets):
            b, e = int(first[k]), int(first[k + 1])
            r, msg = oracle.verify(arena, offs[b:e].astype(np.uint32), perm[b:e], lcp[b:e])
            assert r == 0, (chain, k, msg)
    # (the host chains a level where it finds, without chaining, none left)
    assert stats["1"]["levels"] == stats["0"]["levels"] + 1, stats


@pytest.mark.parametrize("known, others, as_sigma", [
    (4, 1, 5), (4, 3, 7), (4, 4, 8), (7, 1, 8), (4, 11, 15), (4, 12, 16), (15, 1, 16), (20, 11, 31), (4, 28, 32), (31, 1, 32), (4, 200, 204)])
def test_packed_root_with_a_wider_alphabet(ctx, oracle, known, others, as_sigma):
    """characters outside the samples' alphabet, each in one string only: the
    sort starts over with the alphabet of all, and is split as if the samples
    had shown it (plain keys from 32 characters on)"""
    n, hi = 1060000, 60
    arena, offs = packed_case(known, n, 17 * known + others, hi=hi)
    rng = np.random.default_rng(others)
    used = np.unique(arena)
    unused = np.setdiff1d(np.arange(1, 256), used).astype(np.uint8)
    offs64 = offs.astype(np.int64)
    long = np.flatnonzero(np.diff(np.append(offs64, arena.size - 16)) > 12)
    at = offs64[rng.choice(long, others, replace=False)] + rng.integers(0, 9, others)
    arena[at] = rng.choice(unused, others, replace=False)
    check(ctx, oracle, arena, offs)
    rounds = ctx.work_stats()["rounds"]
    check(ctx, oracle, arena, offs, with_lcp=False)
    # the same strings' shape where every character is frequent
    common, common_offs = packed_case(as_sigma, n, 17 * known + others, hi=hi)
    ctx.sort(common, common_offs)
    assert rounds == ctx.work_stats()["rounds"], ctx.work_stats()


def device_bytes_free():
    """free memory of the current device, asked of the HIP runtime that the library uses"""
    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def reserve_and_sort(ps5, oracle, n):
    """device bytes that a context takes when it reserves room for n strings,
    and in the first sort after that"""
    arena, offs = pack(random_strings(30000, 0, 40, b"abc", 4))
    m = len(offs)
    bufs = [ps5.DeviceBuffer(arena.size)] + [ps5.DeviceBuffer(4 * m) for _ in range(3)]
    da, do, dp, dl = bufs
    c = ps5.Context(0)
    try:
        da.upload(arena)
        do.upload(offs)
        # (what the runtime takes for these kernels on these streams: the same
        # sort in the static scratch)
        ps5._check(ps5.load().ps5_sort_device_noalloc(c.h, da.ptr, int(arena.size), do.ptr, m, dp.ptr, dl.ptr), "noalloc")
        free = [device_bytes_free()]
        ps5._check(ps5.load().ps5_ctx_reserve(c.h, n), "ps5_ctx_reserve")
        free.append(device_bytes_free())
        c.sort_device(da, int(arena.size), do, m, dp, dl)
        free.append(device_bytes_free())
        r, msg = oracle.verify(arena, offs, dp.download(np.uint32, m), dl.download(np.uint32, m))
        assert r == 0, msg
        return free[0] - free[1], free[1] - free[2]
    finally:
        c.close()
        for b in bufs:
            b.free()


def test_work_buffers_of_a_large_context(ps5, oracle):
    """a context for 40 M strings takes 86 bytes a string (and what the
    allocator rounds up to): splitters and depths take room for what a level
    can have, not for every string and segment"""
    n, slack = 40_000_000, 64 << 20
    reserved, first = reserve_and_sort(ps5, oracle, n)
    assert reserved + first <= 86 * n + slack, (reserved + first) / n


def test_reserved_context_allocates_nothing(ps5, oracle):
    """the first sort after ps5_ctx_reserve finds every work buffer there"""
    reserved, first = reserve_and_sort(ps5, oracle, 3_000_000)
    assert reserved > 0 and first == 0, (reserved, first)


@pytest.mark.parametrize("n", [200_000, 1 << 20, 5_000_000, 20_000_000])
def test_work_bytes_are_what_a_context_holds(ps5, oracle, n):
    """the bytes that a server charges for work buffers are those that
    contexts allocate, up to what the allocator rounds up to"""
    work_bytes = ps5.load()._ZN3ps510work_bytesEm
    work_bytes.restype, work_bytes.argtypes = ctypes.c_uint64, [ctypes.c_uint64]
    reserved, first = reserve_and_sort(ps5, oracle, n)
    assert work_bytes(n) - (1 << 20) <= reserved + first <= work_bytes(n) + (64 << 20)


@pytest.mark.parametrize("planning", [0, 1])
@pytest.mark.parametrize("target, oversample", [(64, 2), (64, 32), (1024, 32)])
def test_runs_of_every_length_continue(ps5, oracle, planning, target, oversample):
    """blocks with more short runs of equal keys than they finish themselves
    (the rest are tiny leaves of the next round, whose depth is their own),
    between runs at the edge of a tiny leaf and of a block"""
    rng = np.random.default_rng(target + oversample)
    strs = []
    for g, size in enumerate([2] * 3000 + [3] * 900 + [63, 64, 65, 66] * 20 + [2047, 2048, 2049, 5000]):
        stem = b"%c%07d" % (97 + g % 5, g // 5)
        tails = rng.integers(97, 100, (size, 20)).astype(np.uint8)
        strs += [stem + t[:k].tobytes() for t, k in zip(tails, rng.integers(0, 21, size))]
    order = rng.permutation(len(strs))
    c = ps5.Context(0)
    try:
        c.set_planning(planning)
        c.set_tuning(target, 10, oversample)
        check(c, oracle, *pack([strs[i] for i in order]))
    finally:
        c.close()


def test_rows_of_many_runs(ps5, oracle):
    """67 M strings in chunks of 2048: buckets of 32861 runs, more than 64 of
    them to each sampled one where a chunk or an equal-key leaf is mapped, and
    longer rows than a tree, a block or a leaf looks at in LDS"""
    n, width, chunk = 67_300_000, 12, 2048
    assert -(-n // chunk) > 64 * 512
    rng = np.random.default_rng(9)
    rows = rng.integers(48, 89, (n, width), dtype=np.uint8)
    stems = rng.integers(48, 89, (500, 8), dtype=np.uint8)
    rows[:n // 4, :8] = stems[rng.integers(0, 500, n // 4)]
    rows[n // 4:, 5] = 0                     # strings of up to 5 characters
    rows[:n // 4, width - 1] = 0             # and of 8 to 11
    cut = rng.integers(0, 4, n, dtype=np.uint8)
    for k in range(1, 4):
        rows[:n // 4, width - 1 - k][cut[:n // 4] >= k] = 0
        rows[n // 4:, 5 - k][cut[n // 4:] >= k] = 0
    rows = rows.reshape(-1)
    arena = np.concatenate([rows, np.zeros(16, np.uint8)])
    del rows
    order = np.arange(n, dtype=np.uint32).reshape(100, -1).T.reshape(-1)     # (both kinds in every chunk)
    offs = order * np.uint32(width)
    c = ps5.Context(0)
    try:
        c.set_shape(chunk, chunk, 512, 8)
        check(c, oracle, arena, offs)
    finally:
        c.close()


@pytest.mark.parametrize("sigma, stem, tail, rare, packed", [
    (4, 16, 4, 0, True), (7, 16, 4, 0, True), (15, 11, 4, 0, True), (31, 8, 3, 0, True), (32, 8, 3, 0, False),
    (4, 16, 4, 1, True), (4, 16, 4, 3, True), (7, 11, 4, 8, True), (15, 8, 3, 16, True), (31, 8, 3, 1, False), (4, 16, 4, 28, False)])
def test_roots_pack_their_keys(ctx, oracle, sigma, stem, tail, rare, packed):
    """strings that a packed key of their alphabet holds whole are sorted in
    one round, in plain keys (which groups of them share) in more; so too when
    `rare` characters are in one string each, where the samples miss them"""
    n = 1_060_000
    rng = np.random.default_rng(sigma + rare)
    chars = np.sort(rng.choice(np.arange(1, 256), sigma + rare, replace=False)).astype(np.uint8)
    chars = rng.permutation(chars)
    alpha = chars[:sigma]
    width = stem + tail + 1
    rows = np.zeros((n, width), np.uint8)
    rows[:, :stem] = alpha[rng.integers(0, sigma, (300, stem))][rng.integers(0, 300, n)]
    rows[:, stem:-1] = alpha[rng.integers(0, sigma, (n, tail))]
    rows[rng.choice(n, rare, replace=False), rng.integers(0, width - 1, rare)] = chars[sigma:]
    arena = np.concatenate([rows.reshape(-1), np.zeros(16, np.uint8)])
    offs = (np.arange(n, dtype=np.uint32) * np.uint32(width))
    check(ctx, oracle, arena, offs)
    rounds = ctx.work_stats()["rounds"]
    assert (rounds == 1) == packed, rounds


def test_noalloc_sort_starts_over(ps5, ctx, oracle):
    """the largest allocation-free sort packs its keys and meets a character
    that its samples do not show"""
    n = int(ps5.load().ps5_noalloc_max_strings())
    arena, offs = packed_case(4, n, 8, rare=5)
    bufs = [ps5.DeviceBuffer(arena.size)] + [ps5.DeviceBuffer(4 * n) for _ in range(3)]
    da, do, dp, dl = bufs
    try:
        da.upload(arena)
        do.upload(offs)
        ps5._check(ps5.load().ps5_sort_device_noalloc(ctx.h, da.ptr, int(arena.size), do.ptr, n, dp.ptr, dl.ptr), "noalloc")
        r, msg = oracle.verify(arena, offs, dp.download(np.uint32, n), dl.download(np.uint32, n))
        assert r == 0, msg
    finally:
        for b in bufs:
            b.free()


def sorted_runs(ctx, ps5, arena, offs, bounds):
    """(idx, lcp) of contiguous ranges sorted on their own"""
    idx, lcp = np.zeros(len(offs), np.uint32), np.zeros(len(offs), np.uint32)
    for b, e in zip(bounds[:-1].astype(int), bounds[1:].astype(int)):
        if e > b:
            p, l = ctx.sort(arena, offs[b:e])
            idx[b:e] = p + np.uint32(b)
            lcp[b:e] = l
    return idx, lcp


@pytest.mark.parametrize("n, runs", [(60_000, 3), (8_400_000, 2), (8_400_000, 5), (33_600_000, 2), (33_600_000, 7)])
@pytest.mark.parametrize("alphabet, lo, hi", [(b"ACGT", 4, 24), (b"ab", 0, 14), (bytes(range(33, 127)), 1, 20)])
def test_merges_of_every_size_class(ps5, ctx, oracle, n, runs, alphabet, lo, hi):
    """rounds whose tiles are searched by eight lanes, four and one; strings
    that their first 8 characters decide and that they do not, identical ones"""
    if n > 10_000_000 and hi > 20:
        n, lo, hi = 33_600_000, 4, 14
    arena, offs = ps5.gen_uniform(n + runs, n * (hi + 1), lo, hi, alphabet)
    offs = offs[:n]
    rng = np.random.default_rng(runs)
    bounds = np.concatenate([[0], np.sort(rng.integers(0, n, runs - 1)), [n]]).astype(np.uint64)
    idx, lcp = sorted_runs(ctx, ps5, arena, offs, bounds)
    mi, ml = ctx.merge(arena, offs, bounds, idx, lcp)
    r, msg = oracle.verify(arena, offs, mi, ml)
    assert r == 0, msg


@pytest.mark.parametrize("n", [785_407, 785_408, 786_433])
@pytest.mark.parametrize("runs", [2, 6])
def test_merges_where_threads_begin_to_search_in_pairs(ps5, ctx, oracle, n, runs):
    """rounds of 767, 768 and 769 tiles of strings with long common prefixes,
    some identical"""
    rng = np.random.default_rng(n)
    stems = [b"http://%d/" % i * (1 + i % 4) for i in range(40)]
    pool = [stems[i % 40] + s for i, s in enumerate(random_strings(6000, 0, 9, b"ab", 3))]
    arena, where = pack(pool)
    offs = where[rng.integers(0, len(pool), n)]
    bounds = np.concatenate([[0], np.sort(rng.integers(0, n, runs - 1)), [n]]).astype(np.uint64)
    idx, lcp = sorted_runs(ctx, ps5, arena, offs, bounds)
    mi, ml = ctx.merge(arena, offs, bounds, idx, lcp)
    r, msg = oracle.verify(arena, offs, mi, ml)
    assert r == 0, msg


@pytest.mark.parametrize("planning, rounds", [(1, 0), (0, 2)])
@pytest.mark.parametrize("n", [2049, 4097, 30011, 65536, 131071, 131072, 131073, 133121])
def test_small_levels_planned_on_the_device(ps5, oracle, n, planning, rounds):
    """single roots whose run tables k_children writes, roots of one group of
    chunks that have longer ones, and roots of two groups; the same strings in
    several sets"""
    rng = np.random.default_rng(n)
    strs = random_strings(n, 0, 14, b"abcdefgh", n)
    arena, offs = pack(strs)
    first = np.concatenate([[0], np.sort(rng.integers(0, n, 2)), [n]]).astype(np.uint64)
    c = ps5.Context(0)
    try:
        c.set_planning(planning)
        c.set_graph_rounds(rounds)
        check(c, oracle, arena, offs)
        c.set_tuning(64, 10, 4)
        check(c, oracle, arena, offs)
        perm, lcp = c.sort_batch(arena, offs.astype(np.uint64), first)
    finally:
        c.close()
    for b, e in zip(first[:-1].astype(int), first[1:].astype(int)):
        if e > b:
            r, msg = oracle.verify(arena, offs[b:e], perm[b:e], lcp[b:e])
            assert r == 0, msg
