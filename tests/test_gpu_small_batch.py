"""Small batches take one-launch forms of the routing and of the top-1
permute; at the edges of their ranges (and one past them, where the general
kernels run) both must give what the oracle gives, bit for bit: the routing
against the CPU oracle's stable sort, the permute against the scatter it
stands for, including rows that no token names."""

import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from placemoe_amd import kernels
from tests.helpers import assert_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,C", [(1, 1, 1), (1, 8, 160), (63, 1, 2), (8191, 1, 64), (1024, 8, 896), (1024, 8, 897),
                                   (1025, 8, 160), (4096, 2, 3), (8192, 1, 1), (8193, 1, 5), (513, 4, 300)])
@pytest.mark.parametrize("mapped", [True, False])
def test_routing(cuda, T, K, C, mapped):
    rng = np.random.default_rng(T * 31 + C)
    S, E = (3, C + 7) if mapped else (1, C)
    # few distinct experts in places, so that one segment of 64 holds many equal copies
    sel = np.where(rng.random((T, K)) < 0.5, rng.integers(0, E, (T, K)), rng.integers(0, min(E, 2), (T, K)))
    M = rng.integers(0, C, (S, E)) if mapped else np.arange(C).reshape(1, C)
    src = rng.integers(0, S, T)
    dev = lambda a: torch.as_tensor(a, dtype=torch.int64, device=cuda)
    r = kernels.route(dev(sel), C, mapping=dev(M) if mapped else None, sources=dev(src) if mapped else None)
    phys, counts, offsets, pos = O.route(M, src, sel, C)
    assert kernels.route_status(r) == 0
    for name, got, want in (("phys", r.phys, phys), ("counts", r.counts, counts), ("offsets", r.offsets, offsets),
                            ("pos", r.pos, pos)):
        assert_exact(got, want, name)


@pytest.mark.parametrize("bad", [0, 63, 64, 1000, 4095])
def test_routing_flags_an_invalid_id_anywhere(cuda, bad):
    sel = torch.zeros((1024, 4), dtype=torch.int64, device=cuda)
    sel.view(-1)[bad] = 99
    r = kernels.route(sel, 5)
    assert kernels.route_status(r) == 1
    assert int(r.phys.view(-1)[bad]) == 4 and int(r.counts.sum()) == 4096  # clamped and counted


@pytest.mark.parametrize("T", [1, 2, 300, 1024, 1025])
@pytest.mark.parametrize("H", [8, 1024, 7168])
def test_top1_permute_with_unnamed_rows(cuda, T, H):
    gen = torch.Generator(device=cuda).manual_seed(T + H)
    x = torch.randn((T, H), generator=gen, device=cuda).to(torch.bfloat16)
    w = torch.rand((T, 1), generator=gen, device=cuda).to(torch.bfloat16)
    pos = torch.randperm(T, generator=gen, device=cuda).to(torch.int32)
    dropped = torch.zeros(T, dtype=torch.bool, device=cuda)
    dropped[::5] = T > 1
    pos[dropped] = T + 4  # names no row
    xp, src, row_w = kernels.moe_scatter_src(x, pos.view(T, 1), w)
    token = torch.arange(T, device=cuda)[~dropped]
    row = pos[~dropped].long()
    want = torch.zeros_like(x)
    want[row] = x[token]
    named = torch.full((T,), -1, dtype=torch.int32, device=cuda)
    named[row] = token.to(torch.int32)
    assert torch.equal(xp, want) and torch.equal(src, named)
    assert torch.equal(row_w.view(-1)[row], w.view(-1)[token])
