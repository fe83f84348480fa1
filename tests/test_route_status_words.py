"""Host side of the routing status words: a check that ends while its word is
in flight gives it up without waiting for the pool's lock."""

import ctypes
import threading

from placemoe_amd import kernels


def _pool():
    words = kernels._StatusWords()
    view = (ctypes.c_int32 * words.BLOCK)()
    words._blocks.append((None, ctypes.addressof(view), view))
    words._free = [0, 1, 2]
    return words, view


def test_a_check_that_ends_does_not_wait_for_the_lock():
    words, _ = _pool()
    with words._lock:  # a garbage collection inside lease() runs on this thread
        t = threading.Thread(target=words.orphan, args=(2,), daemon=True)
        t.start()
        t.join(10)
        assert not t.is_alive()
    assert list(words._orphans) == [2]


def test_orphans_come_back_once_written():
    words, view = _pool()
    (a, address), (b, _), (c, _) = words.lease(), words.lease(), words.lease()
    assert {a, b, c} == {0, 1, 2} and address == ctypes.addressof(view) + 4 * a
    words.orphan(a)
    words.orphan(b)
    view[b] = 0  # its kernel has run, a's has not
    assert words.lease()[0] == b and list(words._orphans) == [a]
    assert view[b] == words.PENDING
