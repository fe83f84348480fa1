"""The routing status that the kernel stores to pinned host memory: it lands
without a synchronisation by the caller, for every routing form; words come
back only after their kernel has written them; a captured routing holds none
and replays with the eager result."""

import gc
import time

import pytest
import torch

from placemoe_amd import kernels

pytestmark = pytest.mark.gpu


def _words_out():
    w = kernels._STATUS_WORDS
    with w._lock:
        w._collect_orphans()
        return len(w._blocks) * w.BLOCK - len(w._free)


@pytest.mark.parametrize("T,K,C", [(0, 2, 5), (8, 2, 5), (5000, 8, 160), (300, 4, 2000), (200, 2, 9000)],
                         ids=["empty", "one_block", "three_kernels", "many_copies", "global_table"])
@pytest.mark.parametrize("bad", [False, True])
def test_status_lands_without_a_synchronisation(cuda, T, K, C, bad):
    if T == 0 and bad:
        pytest.skip("no ids")
    sel = torch.randint(0, C, (T, K), device=cuda)
    if bad:
        sel[-1, -1] = C
    check = kernels.RouteCheck()
    kernels.route(sel, C, check=check)
    end = time.time() + 20
    while not check.ready() and time.time() < end:
        time.sleep(0.001)
    assert check.ready(), "the status did not reach the host"
    assert check.failed() == bad


def _spin(seconds):
    """Keep the current stream busy; the event that follows."""
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    cycles = 10_000_000
    torch.cuda._sleep(cycles)
    a.record()
    torch.cuda._sleep(cycles)
    b.record()
    torch.cuda.synchronize()
    torch.cuda._sleep(int(cycles * seconds * 1e3 / a.elapsed_time(b)))
    done = torch.cuda.Event()
    done.record()
    return done


def test_words_in_flight_are_not_reused(cuda):
    sel = torch.randint(0, 4, (16, 2), device=cuda)
    torch.cuda.synchronize()
    gc.collect()
    before = _words_out()
    spin = _spin(2.0)
    held = [kernels.RouteCheck() for _ in range(50)]
    for c in held:
        kernels.route(sel, 4, check=c)
    words = {c._word for c in held}
    assert len(words) == 50
    dropped = held[:20]
    del held[:20], dropped, c
    gc.collect()
    out = _words_out()  # 30 held, 20 whose checks are gone while their kernels wait
    more = [kernels.RouteCheck() for _ in range(10)]
    for m in more:
        kernels.route(sel, 4, check=m)
    again = words & {m._word for m in more}
    assert not spin.query(), "the spin ended before the words were counted"
    assert out == before + 50 and not again
    torch.cuda.synchronize()
    assert all(c.ready() and not c.failed() for c in held + more)
    assert _words_out() == before


def test_refused_arguments_give_the_word_back(cuda):
    before = _words_out()
    check = kernels.RouteCheck()
    with pytest.raises(ValueError):
        kernels.route(torch.zeros((4, 2), dtype=torch.int64, device=cuda), 1 << 25, check=check)
    assert _words_out() == before


def test_captured_routing_replays(cuda):
    sel = torch.randint(0, 7, (64, 2), device=cuda)
    kernels.route(sel, 7, check=kernels.RouteCheck())
    torch.cuda.synchronize()
    graph, check = torch.cuda.CUDAGraph(), kernels.RouteCheck()
    with torch.cuda.graph(graph):
        r = kernels.route(sel, 7, check=check)
    assert check.checked and check.ready() and check._word is None
    for seed in range(3):
        sel.copy_(torch.randint(0, 7, (64, 2), generator=torch.Generator().manual_seed(seed)))
        graph.replay()
        torch.cuda.synchronize()
        want = kernels.route(sel, 7)
        assert torch.equal(r.pos, want.pos) and torch.equal(r.offsets, want.offsets)
