"""GPU expert-parallel payloads (pmx_ep_dispatch_payload,
pmx_ep_combine_aggregate) against the CPU oracle: bit-exact integer
payloads and row copies, the reference's aggregation known answer, and the
dispatch + experts + combine round trip across ranks simulated on one GPU."""

import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from placemoe_amd import _capi
from placemoe_amd import ep_payload as EP
from placemoe_amd import kernels
from placemoe_amd.workloads import make_workload
from tests.helpers import assert_bf16_close
from tests.test_ep_payload import simulate_ep

pytestmark = pytest.mark.gpu


def _check_payload(cuda, hidden, phys, w, num_slots, R):
    got = EP.build_local_payload(hidden.to(cuda), torch.as_tensor(phys).to(cuda), w.to(cuda), num_slots, R,
                                 physical_experts=torch.as_tensor(phys).to(cuda))
    ref = O.build_local_payload(hidden, np.asarray(phys), w, num_slots, R)
    send_hidden, send_meta, send_w, utok, usplits, asplits, ranks = got
    assert usplits == ref["unique_send_splits"]
    assert asplits == ref["assignment_send_splits"]
    np.testing.assert_array_equal(send_meta.cpu().numpy(), ref["send_meta"])
    np.testing.assert_array_equal(utok.cpu().numpy(), ref["unique_tokens"])
    np.testing.assert_array_equal(ranks.cpu().numpy(), ref["target_ranks"])
    assert torch.equal(send_hidden.cpu(), ref["send_hidden"])
    assert torch.equal(send_w.cpu(), ref["send_weights"])


@pytest.mark.parametrize("seed,T,K,R,L,H", [(0, 7, 2, 2, 3, 8), (1, 300, 4, 4, 2, 64), (2, 129, 8, 3, 5, 40),
                                            (3, 50, 1, 4, 1, 16), (4, 1000, 32, 8, 4, 24)])
def test_payload_matches_oracle(cuda, seed, T, K, R, L, H):
    print(f"payload seed={seed} T={T} K={K} R={R} L={L} H={H}", flush=True)
    g = torch.Generator().manual_seed(seed)
    phys = torch.randint(0, R * L, (T, K), generator=g).numpy()
    hidden = torch.randn(T, H, generator=g).to(torch.bfloat16)
    w = torch.rand(T, K, generator=g).to(torch.bfloat16)
    _check_payload(cuda, hidden, phys, w, R * L, R)


def test_payload_at_qwen3_routing(cuda):
    """The config-2 routing (160 copies over 8 ranks of 20 slots), full size."""
    wl = make_workload("qwen3", weights=False)
    phys = O.map_logical_to_physical(wl.mapping.numpy(), wl.sources.numpy(), wl.selected.numpy())
    _check_payload(cuda, wl.hidden, phys, wl.routing_weights, wl.C, 8)


def test_payload_empty_and_bad_slot(cuda):
    got = EP.build_local_payload(torch.zeros((0, 8), dtype=torch.bfloat16, device=cuda),
                                 torch.zeros((0, 2), dtype=torch.long, device=cuda),
                                 torch.zeros((0, 2), dtype=torch.bfloat16, device=cuda), 4, 2)
    assert got[4] == [0, 0] and got[5] == [0, 0] and got[0].shape == (0, 8)
    with pytest.raises(ValueError, match="outside"):
        EP.build_local_payload(torch.zeros((1, 8), dtype=torch.bfloat16, device=cuda),
                               torch.tensor([[0, 9]], device=cuda), torch.ones((1, 2), dtype=torch.bfloat16,
                                                                                 device=cuda), 4, 2)


def test_aggregate_reference_known_answer(cuda):
    weighted = torch.tensor([[1.0], [2.0]], device=cuda)
    combined, splits = EP.aggregate_weighted_outputs(weighted, torch.tensor([3, 0], device=cuda), [1, 1],
                                                     key_stride=4)
    assert splits == [1, 1]
    torch.testing.assert_close(combined.cpu(), weighted.cpu())


@pytest.mark.parametrize("seed,N,H,R", [(0, 1, 8, 1), (1, 500, 64, 4), (2, 3000, 2048, 8)])
def test_combine_aggregate_matches_oracle(cuda, seed, N, H, R):
    g = torch.Generator().manual_seed(seed)
    splits = torch.multinomial(torch.ones(R), N, replacement=True, generator=g).bincount(minlength=R).tolist()
    # tokens ascending within each source rank, with repeats (several local experts per token)
    tokens = np.concatenate([np.sort(torch.randint(0, max(1, n // 2), (n,), generator=g).numpy()) for n in splits])
    y = torch.randn(N, H, generator=g).to(torch.bfloat16)
    pos = torch.randperm(N, generator=g)
    w = torch.rand(N, generator=g).to(torch.bfloat16)
    ranks = torch.repeat_interleave(torch.arange(R), torch.as_tensor(splits))
    got, gsplits = EP.combine_aggregate(y.to(cuda), pos.to(cuda), w.to(cuda), ranks.to(cuda),
                                        torch.as_tensor(tokens).to(cuda), R)
    weighted = (y[pos].float() * w.float()[:, None]).to(torch.bfloat16)
    ref, rsplits = O.aggregate_weighted_outputs(weighted, tokens, splits)
    assert gsplits == rsplits
    assert_bf16_close(got.cpu(), ref)


@pytest.mark.parametrize("seed,R,L,T,K,H", [(0, 2, 2, 16, 2, 32), (1, 4, 3, 24, 4, 64), (2, 8, 2, 12, 8, 16)])
def test_round_trip_across_simulated_ranks(cuda, seed, R, L, T, K, H):
    g = torch.Generator().manual_seed(seed)
    W = (torch.randn(R * L, H, H, generator=g) * 0.1).to(torch.bfloat16)
    hid = [torch.randn(T, H, generator=g).to(torch.bfloat16) for _ in range(R)]
    phys = [torch.randint(0, R * L, (T, K), generator=g).numpy() for _ in range(R)]
    w = [torch.rand(T, K, generator=g).to(torch.bfloat16) for _ in range(R)]

    def gpu_payload(hidden, ph, wt, num_slots, ranks):
        sh, meta, sw, utok, us, asp, tr = EP.build_local_payload(hidden, torch.as_tensor(ph).to(cuda), wt,
                                                                  num_slots, ranks,
                                                                  physical_experts=torch.as_tensor(ph).to(cuda))
        return {"send_hidden": sh, "send_meta": meta.cpu().numpy(), "send_weights": sw, "unique_tokens": utok.cpu(),
                "unique_send_splits": us, "assignment_send_splits": asp}

    def gpu_aggregate(weighted, tokens, splits, stride):
        return EP.aggregate_weighted_outputs(weighted, torch.as_tensor(tokens).to(cuda), splits, stride)

    outs = simulate_ep([h.to(cuda) for h in hid], phys, [x.to(cuda) for x in w], W.to(cuda), R, L,
                       payload=gpu_payload, aggregate=gpu_aggregate)
    for r in range(R):
        eager = torch.zeros(T, H, dtype=torch.float64)
        for t in range(T):
            for k in range(K):
                eager[t] += w[r][t, k].double() * (hid[r][t].double() @ W[phys[r][t, k]].double().t())
        assert_bf16_close(outs[r].cpu().to(torch.bfloat16), eager.float())


# Segments of whole tokens (64 // K of them), chunks of four segments, more
# than 1024 chunks, one rank, and more ranks than LDS counters (4096).
@pytest.mark.parametrize("T,K,R,L", [(1, 1, 1, 1), (63, 1, 3, 2), (257, 1, 2, 1), (36, 7, 4, 3), (37, 7, 4, 3),
                                     (9, 22, 5, 4), (8, 32, 2, 9), (40001, 7, 8, 2), (90, 6, 4096, 1),
                                     (90, 6, 4097, 1), (700, 3, 5000, 2)])
def test_payload_at_segment_and_chunk_edges(cuda, T, K, R, L):
    print(f"payload T={T} K={K} R={R} L={L}", flush=True)
    g = torch.Generator().manual_seed(T + K)
    phys = torch.randint(0, R * L, (T, K), generator=g)
    phys[::3] = phys[::3] % max(1, R * L // 3)  # several assignments of a token on one rank
    phys[1::5] = R * L - 1  # ... and all of them
    hidden = torch.randn(T, 8, generator=g).to(torch.bfloat16)
    w = torch.rand(T, K, generator=g).to(torch.bfloat16)
    _check_payload(cuda, hidden, phys.numpy(), w, R * L, R)


# Runs past 64 rows, odd ones, and rows around the 64 and 256 chunks of a pass.
@pytest.mark.parametrize("H", [8, 504, 520, 2040, 2048, 2056, 4104])
def test_combine_aggregate_run_lengths(cuda, H):
    g = torch.Generator().manual_seed(H)
    lengths = [1, 2, 3, 63, 64, 65, 1, 128, 129, 200, 5]
    tokens = np.repeat(np.arange(len(lengths)), lengths)
    N = len(tokens)
    splits = [int(sum(lengths[:4])), 0, int(sum(lengths[4:]))]
    y = torch.randn(N, H, generator=g).to(torch.bfloat16)
    pos = torch.randperm(N, generator=g)
    w = torch.rand(N, generator=g).to(torch.bfloat16)
    ranks = torch.repeat_interleave(torch.arange(3), torch.as_tensor(splits))
    got, gsplits = EP.combine_aggregate(y.to(cuda), pos.to(cuda), w.to(cuda), ranks.to(cuda),
                                        torch.as_tensor(tokens).to(cuda), 3)
    weighted = (y[pos].float() * w.float()[:, None]).to(torch.bfloat16)
    ref, rsplits = O.aggregate_weighted_outputs(weighted, tokens, splits)
    assert gsplits == rsplits
    assert_bf16_close(got.cpu(), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,R", [(1, 1), (1000, 3), (5000, 5000)])
def test_combine_aggregate_of_either_index_type(cuda, N, R, dtype):
    g = torch.Generator(device=cuda).manual_seed(N)
    ranks = torch.sort(torch.randint(0, R, (N,), generator=g, device=cuda)).values
    tokens = torch.arange(N, device=cuda) // 3
    y = torch.randn((N, 72), generator=g, device=cuda).to(dtype)
    pos, w = torch.randperm(N, generator=g, device=cuda), torch.rand((N,), generator=g, device=cuda).to(dtype)
    got, splits = EP.combine_aggregate(y, pos, w, ranks, tokens, R)
    ref, ref_splits = EP.combine_aggregate(y, pos.int(), w, ranks.int(), tokens.int(), R)
    mixed, mixed_splits = EP.combine_aggregate(y, pos, w, ranks.int(), tokens, R)
    assert splits == ref_splits == mixed_splits and torch.equal(got, ref) and torch.equal(got, mixed)


def test_payload_of_int32_slots_through_the_c_entry(cuda):
    T, K, R, L, H = 300, 6, 4, 5, 16
    g = torch.Generator(device=cuda).manual_seed(2)
    phys = torch.randint(0, R * L, (T, K), generator=g, device=cuda)
    hidden = torch.randn((T, H), generator=g, device=cuda).to(torch.bfloat16)
    w = torch.rand((T, K), generator=g, device=cuda).to(torch.bfloat16)
    want = EP.build_local_payload(hidden, phys, w, R * L, R)
    A = T * K
    i32 = lambda *s: torch.zeros(s, dtype=torch.int32, device=cuda)
    p32, ac, ao, uc, uo = phys.int(), i32(R), i32(R + 1), i32(R), i32(R + 1)
    sh, sw = torch.zeros((A, H), dtype=torch.bfloat16, device=cuda), torch.zeros(A, dtype=torch.bfloat16, device=cuda)
    ut, meta, tr, status = i32(A), i32(A, 3), i32(A), i32(1)
    ws = torch.empty(_capi.load().pmx_ep_payload_workspace_bytes(A, R), dtype=torch.uint8, device=cuda)
    _capi.call("pmx_ep_dispatch_payload", *(t.data_ptr() for t in (p32, hidden, w)), T, K, H, R, L,
               *(t.data_ptr() for t in (ac, ao, uc, uo, sh, ut, meta, sw, tr, status, ws)), ws.numel(),
               torch.cuda.current_stream(cuda).cuda_stream)
    U = int(uo[-1])
    assert uc.tolist() == want[4] and ac.tolist() == want[5] and int(ao[-1]) == A and U == sum(want[4])
    assert torch.equal(sh[:U], want[0]) and torch.equal(meta, want[1]) and torch.equal(sw[:, None], want[2])
    assert torch.equal(ut[:U].long(), want[3]) and torch.equal(tr.view(T, K).long(), want[6])
