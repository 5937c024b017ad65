"""Host-side failure handling of the serving loop (no GPU needed): a server
none of whose slots can start completes every request with an error instead
of leaving its waiter blocked, and malformed requests are rejected at submit,
before they could share a batch.  The slots here ask for a device index that
does not exist, so the same failure is forced on any machine."""
import ctypes

import numpy as np
import pytest

from strsets import pack

NO_SUCH_DEVICE = 4096


@pytest.mark.timeout(120)
def test_server_without_slots_fails_requests(ps5):
    srv = ps5.Server(NO_SUCH_DEVICE, hbm_budget=1 << 30, slots=3)
    try:
        arena, offs = pack([b"b", b"a", b"c"])
        ids = [srv.submit(arena, offs) for _ in range(4)]
        for rid in ids:
            with pytest.raises(ps5.Ps5Error) as e:
                srv.wait(rid)
            assert "no serving slot could start" in str(e.value)
        h = srv.health()
        assert h["live_slots"] == 0 and h["failed"] == 4
        # a request submitted after the slots failed fails at once as well
        rid = srv.submit(arena, offs)
        with pytest.raises(ps5.Ps5Error):
            srv.wait(rid)
    finally:
        srv.close()


@pytest.mark.timeout(120)
def test_server_rejects_malformed_requests(ps5):
    srv = ps5.Server(NO_SUCH_DEVICE, hbm_budget=1 << 30, slots=1)
    try:
        arena, offs = pack([b"xy", b"z"])
        bad = offs.copy()
        bad[1] = arena.size          # an offset outside the arena
        with pytest.raises(ps5.Ps5Error, match="outside the arena"):
            srv.submit(arena, bad)
        unterminated = np.frombuffer(b"xy\0zz", np.uint8).copy()
        with pytest.raises(ps5.Ps5Error, match="last byte must be a NUL"):
            srv.submit(unterminated, np.array([0, 3], np.uint32))
        # rejected requests take no id: the first valid one gets id 1, after
        # which a fault can no longer be planted in it
        srv.inject_fault(2)
        rid = srv.submit(arena, offs)
        assert rid == 1
        with pytest.raises(ps5.Ps5Error, match="already submitted"):
            srv.inject_fault(1)
    finally:
        srv.close()


@pytest.mark.parametrize("n", [1, 100, 5000, 1 << 20, 3_000_000, 1 << 28])
def test_server_charges_what_a_request_holds(ps5, n):
    """a request's share of the budget: characters, offsets of both widths,
    results and the work buffers of a context for its strings"""
    lib = ps5.load()
    work_bytes, request_bytes = lib._ZN3ps510work_bytesEm, lib._ZN3ps513request_bytesEmm
    for f, k in ((work_bytes, 1), (request_bytes, 2)):
        f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_uint64] * k
    per_string = 24 + 8 + 42 if n > 1 << 20 else 24 + 8 + 42 + 5 * 4
    assert work_bytes(n) >= per_string * n
    chars = 60 * n
    assert chars + 20 * n + work_bytes(n) - work_bytes(0) <= request_bytes(chars, n) <= chars + 20 * n + work_bytes(n) + 8192
    # requests batched together are charged no less than one context for all of them
    assert 16 * request_bytes(chars, n) >= 16 * (chars + 20 * n) + work_bytes(16 * n) - work_bytes(0)
