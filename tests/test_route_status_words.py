"""Host side of the routing status words: a check that ends while its word is
in flight gives it up without waiting for the pool's lock."""

import contextlib
import ctypes
import subprocess
import sys
import threading
from pathlib import Path

import pytest
import torch

from placemoe_amd import _capi, kernels

ROOT = Path(__file__).resolve().parents[1]


def _pool():
    words = kernels._StatusWords()
    view = (ctypes.c_int32 * words.BLOCK)()
    words._blocks.append((None, ctypes.addressof(view), view))
    words._free = [0, 1, 2]
    return words, view


def _devices(monkeypatch, capturing):
    """torch.cuda of a host whose device 0 is current; the streams of the
    devices in ``capturing`` are being captured."""
    current = [0]

    @contextlib.contextmanager
    def device(d):
        current.append(torch.device(d).index)
        yield
        current.pop()

    monkeypatch.setattr(torch.cuda, "current_device", lambda: current[-1])
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: current[-1] in capturing)


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


def test_checks_pending_at_interpreter_exit_end_quietly():
    """A serving process ends with its last forward's check unread."""
    code = """
from placemoe_amd import experts, kernels
for word in range(3):
    check = kernels.RouteCheck()
    check._word = word  # in flight
    experts._PENDING_CHECKS.append(check)
"""
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert out.returncode == 0 and "Exception ignored" not in out.stderr, out.stderr


def test_waiting_uses_no_stream(monkeypatch):
    """A wait ends when the word lands; the stream of the launch, which its
    owner may have destroyed since, is not touched."""
    words, view = _pool()
    monkeypatch.setattr(kernels, "_STATUS_WORDS", words)
    _devices(monkeypatch, capturing=())
    for name in ("ExternalStream", "default_stream", "synchronize"):
        monkeypatch.setattr(torch.cuda, name, lambda *a, **k: pytest.fail("waits on a stream or the device"))
    for status in (0, 1):
        check = kernels.RouteCheck()
        check._word, _ = words.lease()
        check._device = torch.device("cuda", 0)
        kernel = threading.Timer(0.1, view.__setitem__, (check._word, status))
        kernel.start()
        assert check.failed() == bool(status)
        kernel.join()
    assert sorted(words._free) == [0, 1, 2]


def test_waiting_raises_what_ended_the_device(monkeypatch):
    words, _ = _pool()
    monkeypatch.setattr(kernels, "_STATUS_WORDS", words)
    _devices(monkeypatch, capturing=())

    class Dead:
        def query(self):
            raise RuntimeError("device error")

    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: Dead())
    check = kernels.RouteCheck()
    check._word, _ = words.lease()
    check._device = torch.device("cuda", 0)
    with pytest.raises(RuntimeError, match="device error"):
        check.failed()


@pytest.mark.parametrize("capturing", [0, 1])
@pytest.mark.parametrize("launch", [0, 1])
def test_capture_is_asked_of_the_launch_device(monkeypatch, launch, capturing):
    """A routing captured on its own device leases no word (every replay would
    write to it); one beside another device's capture does."""
    words, _ = _pool()
    monkeypatch.setattr(kernels, "_STATUS_WORDS", words)
    _devices(monkeypatch, capturing=(capturing,))
    check = kernels.RouteCheck()
    address = check.arm(torch.device("cuda", launch))
    assert (address is None) == check.checked == (launch == capturing)
    assert len(words._free) == (3 if launch == capturing else 2)


@pytest.mark.parametrize("written,settles", [(False, True), (True, True), (False, False)])
def test_a_failed_launch_gives_its_word_back(monkeypatch, written, settles):
    """The scan may have been launched before the launch that failed: the word
    comes back once the device has settled, and not before."""
    words, view = _pool()
    monkeypatch.setattr(kernels, "_STATUS_WORDS", words)
    _devices(monkeypatch, capturing=())
    monkeypatch.setattr(kernels, "_check_dev", lambda *t: torch.device("cpu"))
    monkeypatch.setattr(kernels, "_stream", lambda device: 0)
    leased = []

    def fails(name, *args):
        leased.extend(set(range(3)) - set(words._free))
        raise _capi.PmxError(name, _capi.PMX_ERR_HIP)

    def synchronize(device):
        if not settles:
            raise RuntimeError("device error")
        if written:
            view[leased[0]] = 0

    monkeypatch.setattr(_capi, "call", fails)
    monkeypatch.setattr(torch.cuda, "synchronize", synchronize)
    check = kernels.RouteCheck()
    with pytest.raises(_capi.PmxError):
        kernels.route(torch.zeros((4, 2), dtype=torch.int64), 3, check=check)
    assert len(leased) == 1
    assert sorted(words._free) == ([0, 1, 2] if settles else sorted({0, 1, 2} - set(leased)))
    assert (check._word is None) == settles
