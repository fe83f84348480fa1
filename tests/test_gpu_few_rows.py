"""The few-rows grouped GEMM (64- and 128-row tiles) against the 256-row
kernels and fp32 products.

Calls whose copies hold few rows on average go to another kernel than the
rest; the build ``libplacemoe_amd_w8.so`` keeps the 256-row kernels for every
call.  Both must agree within the bf16 bar over every form the rule accepts:
copies that end on and next to the tile edges (64, 128), empty copies, one
copy, as many as the kernel takes (1024) and one more (which goes to the other
kernels), averages past the kernels' lines, K off the 64-deep K-tile, columns off the 256-wide tile, split fc1
weights whose split is (and is not) a whole number of K-tiles, and top-1 row
maps with targets outside the output.
"""

import numpy as np
import pytest
import torch

from placemoe_amd import _capi, build, kernels
from tests.helpers import assert_bf16_close
from tests.test_gpu_gemm_random_layouts import check_every_kind

pytestmark = pytest.mark.gpu

EDGES = [1, 0, 15, 16, 17, 63, 64, 65, 0, 2, 127, 128, 129, 31, 33, 5]


def _off(counts):
    off = np.zeros(len(counts) + 1, dtype=np.int64)
    np.cumsum(counts, out=off[1:])
    return off


def _sparse(G, seed):
    c = np.zeros(G, dtype=np.int64)
    rng = np.random.default_rng(seed)
    c[rng.choice(G, 20, replace=False)] = rng.integers(1, 150, 20)
    c[0], c[-1] = 3, 66
    return c


CASES = {
    "tiny": ([3, 0, 1, 7, 0, 9], 512, 192),
    "edges": (EDGES, 576, 264),
    "edges128": ([128, 127, 129, 60, 200, 100], 320, 136),
    "edges128_tile": ([128, 127, 129, 60, 200, 100], 320, 192),
    "edges128_below": ([128, 127, 129, 60, 100, 90], 320, 136),
    "edges128_k_tail": ([128, 127, 129, 60, 100, 90], 200, 264),
    "edges32": ([129, 1, 0, 64, 2, 3, 17, 40], 576, 192),
    "wide": ([1 + i % 29 for i in range(80)] + [0, 63, 64, 65, 128], 1096, 776),
    "k_tail": (EDGES, 200, 72),
    "one_copy": ([37], 1024, 640),
    "one_k_tile": ([5, 70, 0, 12], 64, 64),
    "below_one_k_tile": ([5, 70, 0, 12], 40, 24),
    "g1024": (_sparse(1024, 1), 128, 72),
    "g1025": (_sparse(1025, 2), 128, 72),
}


@pytest.mark.parametrize("name", list(CASES))
def test_every_kind_against_fp32(cuda, name):
    counts, H, I = CASES[name]
    print(f"few rows {name}: G={len(counts)} rows={int(np.sum(counts))} H={H} I={I}", flush=True)
    check_every_kind(cuda, _off(counts), H, I, 21, name)


def _outputs(cuda, counts, H, I, dtype):
    off = _off(counts)
    G, A = len(counts), int(off[-1])
    offd = torch.as_tensor(off, dtype=torch.int32, device=cuda)
    gen = torch.Generator(device=cuda).manual_seed(4)

    def rn(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device=cuda) * scale).to(dtype)

    x, dy = rn(A, H), rn(A, H)
    w1, w2 = rn(G, 2 * I, H, scale=0.05), rn(G, H, I, scale=0.05)
    perm = torch.randperm(A, generator=gen, device=cuda).to(torch.int32)
    perm[::7] = A + 3  # targets outside the output are dropped
    perm[3::11] = -1
    rw = (0.05 + 0.95 * torch.rand((A,), generator=gen, device=cuda)).to(dtype)
    gate, up = w1[:, :I].contiguous(), w1[:, I:].contiguous()
    gu, act = kernels.gemm_fc1_swiglu(x, gate, up, I * H, offd, G, I)
    keep = perm[(perm >= 0) & (perm < A)].long()
    y, out = kernels.group_gemm_nt_combine_top1(act, w2, offd, perm, rw)
    dg1 = kernels.gemm_fc2_dgrad_swiglu(dy, w2, gu, offd)
    return {"gu": gu, "act": act, "y": y, "out": out[keep], "dg1": dg1, "dact": kernels.group_gemm_nn(dy, w2, offd),
            "dxp": kernels.group_gemm_nn(dg1, gate, offd, b_second=up),
            "dx": kernels.group_gemm_nn_unpermute_top1(dg1, w1, offd, perm)[keep]}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("name", list(CASES))
def test_same_as_the_256_row_kernels(cuda, name, dtype):
    variant = build.variant_path("w8")
    assert variant.exists(), f"{variant} is not built (python -m placemoe_amd.build)"
    counts, H, I = CASES[name]
    print(f"few rows against 256-row kernels, {name} {dtype}", flush=True)
    got = _outputs(cuda, counts, H, I, dtype)
    with _capi.using(variant):
        ref = _outputs(cuda, counts, H, I, dtype)
    torch.cuda.synchronize()
    for k in ref:
        assert_bf16_close(got[k], ref[k], name=f"{name} {k}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("counts,H,I", [([3, 0, 65, 129], 576, 264), ([300, 1, 0, 257], 512, 192),
                                        ([1300, 0, 700], 256, 320), ([300, 40], 200, 72)],
                         ids=["few", "mid", "large", "k_tail"])
def test_fc1_with_row_weights_is_fc1_then_weight_rows(cuda, counts, H, I, dtype):
    """Bit for bit, on each kernel that fc1 runs on, and the backward that
    recomputes the activations against the one that reads them."""
    off = _off(counts)
    G, A = len(counts), int(off[-1])
    offd = torch.as_tensor(off, dtype=torch.int32, device=cuda)
    gen = torch.Generator(device=cuda).manual_seed(9)
    rn = lambda *s: torch.randn(s, generator=gen, device=cuda).to(dtype)
    x, w1, row_w, d = rn(A, H), rn(G, 2 * I, H) * 0.05, rn(A), rn(A, I)
    up = w1.view(-1)[I * H:]
    gu, act = kernels.gemm_fc1_swiglu(x, w1, up, 2 * I * H, offd, G, I)
    gu2, act_w = kernels.gemm_fc1_swiglu(x, w1, up, 2 * I * H, offd, G, I, row_w=row_w)
    assert torch.equal(gu, gu2) and torch.equal(act_w, kernels.weight_rows(act, row_w))
    src = torch.randperm(A, generator=gen, device=cuda).to(torch.int32)
    for got, want in zip(kernels.swiglu_bwd_weighted(d, gu, None, row_w, src, A),
                         kernels.swiglu_bwd_weighted(d, gu, act, row_w, src, A)):
        assert torch.equal(got, want)


WGRAD_CASES = [([1, 0, 31, 32, 33, 63, 64, 65, 0, 129], 264, 136), ([0, 0, 0, 5], 8, 1024),
               ([0, 0, 0, 300, 0, 0, 0], 400, 72), ([3, 190] + [1] * 7, 1160, 1032), ([128, 0, 0], 128, 128),
               ([200, 0, 56, 0, 0, 0], 400, 72), ([90, 0] * 10, 136, 200), ([48], 128, 256)]
WGRAD_PAST_THE_LINE = [([128], 128, 128), ([200, 0, 56], 400, 72), ([90] * 20, 136, 200)]  # the 256-row kernels


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("counts,M,N", WGRAD_CASES + WGRAD_PAST_THE_LINE)
def test_weight_gradient(cuda, counts, M, N, split, dtype):
    """Few rows per copy: against fp32 products and the 256-row kernels; empty
    copies are zero, rows past the last copy (NaN here) reach nothing."""
    off = _off(counts)
    G, A = len(counts), int(off[-1])
    offd = torch.as_tensor(off, dtype=torch.int32, device=cuda)
    gen = torch.Generator(device=cuda).manual_seed(M + N)
    a = torch.randn((A + 70, M), generator=gen, device=cuda).to(dtype)
    b = torch.randn((A + 70, N), generator=gen, device=cuda).to(dtype)
    a[A:] = float("nan")
    b[A:] = float("nan")
    run = lambda: kernels.group_gemm_tn(a, b, offd, split=M // 2 if split else None)
    got = run()
    with _capi.using(build.variant_path("w8")):
        ref = run()
    got, ref = (torch.cat(t, 1) if split else t for t in (got, ref))
    assert_bf16_close(got, ref, name="against the 256-row kernel")
    for g, n in enumerate(counts):
        s = int(off[g])
        want = a[s:s + n].float().t() @ b[s:s + n].float() if n else torch.zeros((M, N), device=cuda)
        assert_bf16_close(got[g], want, name=f"copy {g} ({n} rows)")


def _all_kinds(x, dy, w1, w2, counts):
    off = _off(counts)
    G, I = len(counts), w2.shape[2]
    offd = torch.as_tensor(off, dtype=torch.int32, device=x.device)
    up = w1.view(-1)[I * x.shape[1]:]
    gu, act = kernels.gemm_fc1_swiglu(x, w1, up, 2 * I * x.shape[1], offd, G, I)
    dg1 = kernels.gemm_fc2_dgrad_swiglu(dy, w2, gu, offd)
    return {"gu": gu, "act": act, "y": kernels.group_gemm_nt(act, w2, offd), "dg1": dg1,
            "dx": kernels.group_gemm_nn(dg1, w1, offd)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_bits_depend_on_neither_the_copy_nor_the_batch(cuda, dtype):
    """Replicas of one expert give a row the same bits whichever slot serves
    it, and so do calls with few and with many rows per copy: the placement and
    the batch a token comes in are not to be seen in its result."""
    G, H, I, n = 23, 1024, 384, 20
    gen = torch.Generator(device=cuda).manual_seed(12)
    rn = lambda *s: torch.randn(s, generator=gen, device=cuda).to(dtype)
    w1, w2 = (rn(1, 2 * I, H) * 0.03).repeat(G, 1, 1), (rn(1, H, I) * 0.05).repeat(G, 1, 1)
    x0, dy0 = rn(n, H), rn(n, H)
    want = {}
    for extra in (0, 30, 80, 300, 700):  # 20 .. 720 rows per copy: every kernel the kinds run on
        print(f"few rows, same bits: {dtype} {n + extra} rows per copy", flush=True)
        x = torch.cat([t for _ in range(G) for t in (x0, rn(extra, H))])
        dy = torch.cat([t for _ in range(G) for t in (dy0, rn(extra, H))])
        for k, t in _all_kinds(x, dy, w1, w2, [n + extra] * G).items():
            t = t.view(G, n + extra, -1)[:, :n]
            assert torch.equal(t, t[:1].expand_as(t)), f"{k}, {n + extra} rows: the slot changes the bits"
            assert torch.equal(t[0], want.setdefault(k, t[0].clone())), f"{k}: {n + extra} rows per copy change the bits"
