"""Counts read through a thread's pinned word (jaxsplat_count_begin / _wait): a read
that its thread abandons, and what becomes of the word when the thread ends."""

import ctypes
import threading

import pytest

from jaxsplat_amd import _lib
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _stream(s):
    return ctypes.c_void_p(s.cuda_stream)


def _begin(count, s):
    ticket = ctypes.c_uint64()
    _lib.check(_lib.lib().jaxsplat_count_begin(H.P(count), ctypes.byref(ticket), _stream(s)))
    return ticket


def _wait(count, ticket, s):
    value = ctypes.c_int32(-1)
    _lib.check(_lib.lib().jaxsplat_count_wait(H.P(count), ticket, ctypes.byref(value), _stream(s)))
    return value.value


def _counts(*values):
    t = H.torch()
    c = [t.tensor([v], dtype=t.int32, device="cuda") for v in values]
    t.cuda.synchronize()
    return c


def _work(ms):
    """A function that queues about ms milliseconds of products."""
    t = H.torch()
    a = t.randn(4096, 4096, device="cuda")
    out = t.empty_like(a)
    ev = [t.cuda.Event(enable_timing=True) for _ in range(2)]
    for _ in range(2):
        ev[0].record()
        for _ in range(10):
            t.mm(a, a, out=out)
        ev[1].record()
        t.cuda.synchronize()
    reps = int(ms / (ev[0].elapsed_time(ev[1]) / 10)) + 1

    def queue():
        for _ in range(reps):
            t.mm(a, a, out=out)

    return queue


def test_thread_ends_before_its_count_is_stored():
    """Threads that begin a read behind 30 ms of work and end: the next threads
    (which get their words) and this one read their own counts, before and after the
    late stores."""
    t = H.torch()
    queue = _work(30)
    late, mine, theirs = _counts(111, 7, 8)
    slow, idle = t.cuda.Stream(), t.cuda.Stream()
    assert _wait(mine, _begin(mine, idle), idle) == 7
    got = []

    def abandon():
        _begin(late, slow)

    def read():
        for _ in range(3):
            got.append(_wait(theirs, _begin(theirs, idle), idle))

    def run(f):
        th = threading.Thread(target=f)
        th.start()
        th.join()

    with t.cuda.stream(slow):
        queue()
    for _ in range(3):
        run(abandon)
        run(read)
    assert not slow.query(), "the late stores came too early for this test"
    slow.synchronize()
    run(read)
    assert got == [8] * 12
    assert _wait(mine, _begin(mine, idle), idle) == 7


@pytest.mark.parametrize("ms", [0, 4, 30])
def test_wait_does_not_wait_for_what_is_behind(ms):
    """A count behind `ms` of work and before 300 ms more arrives while that runs."""
    t = H.torch()
    before, behind = _work(ms), _work(300)
    (count,) = _counts(12345)
    s = t.cuda.Stream()
    with t.cuda.stream(s):
        before()
        ticket = _begin(count, s)
        behind()
    assert _wait(count, ticket, s) == 12345
    assert not s.query(), "the work behind the count has ended"
    s.synchronize()


def test_late_store_of_an_abandoned_read():
    """A read abandoned behind 20 ms of work stores over the count of the next one,
    which is then copied; the abandoned ticket is refused, before and after."""
    t, L = H.torch(), _lib.lib()
    queue = _work(20)
    first, second = _counts(111, 222)
    slow, idle = t.cuda.Stream(), t.cuda.Stream()
    value = ctypes.c_int32(-1)

    def refused():
        return L.jaxsplat_count_wait(H.P(first), abandoned, ctypes.byref(value),
                                     _stream(slow)) == _lib.ERR_INVALID and value.value == -1

    with t.cuda.stream(slow):
        queue()
        abandoned = _begin(first, slow)
    ticket = _begin(second, idle)
    assert refused()
    idle.synchronize()
    assert not slow.query(), "the late store came too early for this test"
    slow.synchronize()                  # now the word holds the abandoned read's count
    assert _wait(second, ticket, idle) == 222
    assert refused()
    assert _wait(first, _begin(first, idle), idle) == 111
