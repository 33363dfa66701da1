"""The persistent kernel's large-batch form (more than 1024 routes, 256 tokens or 512 local experts;
MXFP4, MXFP8 and FP8F128 activations) against the plain form: a token's output does not depend on the tokens beside
it, so y of one large call equals, bit for bit, y of the same tokens in calls small enough for the
plain form. Its dispatch table against the oracle's, and the recv stats against the counts."""
import os
import re

import numpy as np
import pytest
import torch

from oracle import moe
from tests.gpu_common import need_gpu

ROOT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hopper_megamoe_basedondeepgemm_amd", "csrc")


def test_route_to_token_multiply_is_exact_at_the_large_batch_limit():
    """div_small at the large-batch form's route limit: every route and top-k the host accepts."""
    n = int(re.search(r"FUSED_BIG_ROUTES\s*=\s*(\d+)", open(os.path.join(ROOT, "dgm_fused.hpp")).read()).group(1))
    r = np.arange(n, dtype=np.uint64)
    for d in range(1, 17):
        m = np.uint64((2 ** 20 + d - 1) // d)
        assert (r * m < 2 ** 32).all() and ((r * m) >> np.uint64(20) == r // np.uint64(d)).all(), d


def _weights(dgm, E, H, I, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for n, k in ((2 * I, H), (H, I)):
        out.append((torch.randint(0, 256, (E, n, k // 2), generator=g, device="cuda", dtype=torch.uint8),
                    torch.randint(118, 121, (E, n, k // 32), generator=g, device="cuda", dtype=torch.uint8)))
    return dgm.transform_mxfp4_weights_for_mega_moe_fused(*out)


def _routing(kind, rng, M, E, topk):
    if kind == "random":
        idx = np.argsort(rng.random((M, E)), axis=1)[:, :topk]
    elif kind == "one":           # every token on the same experts
        idx = np.tile(np.arange(topk)[::-1], (M, 1))
    else:                         # most on expert 0, some tokens unrouted, some slots empty
        idx = np.argsort(rng.random((M, E)), axis=1)[:, :topk]
        idx[rng.random(M) < 0.7, 0] = 0
        for t in range(M):        # distinct experts within a token
            row = idx[t]
            for s in range(1, topk):
                if row[s] in row[:s]:
                    row[s] = -1
        idx[rng.random(M) < 0.1] = -1
    return idx.astype(np.int64), rng.random((M, topk)).astype(np.float32)


def _call(dgm, x, idx, w, l1, l2, fmt, cap, E, topk, H, I, ep, rank, split=False):
    m = x.size(0)
    buf = dgm.get_fused_symm_buffer_for_mega_moe(None, E, cap, topk, H, I, act_format=fmt, ep_size=ep, ep_rank=rank)
    dgm.mega._cast_into(buf, x, fmt)
    buf.topk_idx[:m].copy_(torch.from_numpy(idx))
    buf.topk_weights[:m].copy_(torch.from_numpy(w))
    y = torch.full((m, H), 7.0, dtype=torch.bfloat16, device="cuda")
    stats = torch.zeros(E // ep, dtype=torch.int32, device="cuda")
    for _ in range(2):            # (the second call uses the other counter set)
        dgm.mega._fused(y, l1, l2, buf, stats, 10.0, split=split)
    torch.cuda.synchronize()
    assert buf.kernel_error() == 0
    return y, stats, buf


CASES = [  # M, topk, E, ep, H, I, routing
    (129, 8, 16, 1, 512, 256, "random"),        # just beyond 1024 routes
    (257, 3, 24, 2, 512, 256, "uneven"),        # just beyond 256 tokens, one of two ranks
    (512, 8, 512, 1, 512, 256, "random"),       # 4096 routes over 512 local experts
    (511, 8, 8, 1, 1024, 512, "one"),           # every expert with 32 slabs, the last ragged
    (4096, 1, 4, 1, 512, 256, "uneven"),        # most routes on one expert
    (300, 8, 384, 8, 3072, 1280, "random"),     # one of eight ranks, the full width
]


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8", "fp8f128"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_large_batch_equals_small_calls(case, fmt):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    M, topk, E, ep, H, I, kind = case
    print(f"large batch {case} {fmt}", flush=True)
    rank, local = ep // 2, E // ep
    rng = np.random.default_rng(M + topk)
    l1, l2 = _weights(dgm, local, H, I, M)
    x = torch.randn((M, H), generator=torch.Generator(device="cuda").manual_seed(M), device="cuda").bfloat16()
    idx, w = _routing(kind, rng, M, E, topk)
    args = (l1, l2, fmt, M, E, topk, H, I, ep, rank)
    y, stats, buf = _call(dgm, x, idx, w, *args)
    assert dgm.mega.fused_last_form(buf) == 4
    counts, active, offs, routes = moe.dispatch(idx, rank * local, local)
    for got, want in zip(buf.pool_table(), (counts, active, offs, routes)):
        np.testing.assert_array_equal(got.numpy(), want)
    np.testing.assert_array_equal(stats.cpu().numpy(), 2 * counts)
    step = min(256, 1024 // topk) // 2
    for t in range(0, M, step):
        n = min(step, M - t)
        ys, _, bs = _call(dgm, x[t:t + n], idx[t:t + n], w[t:t + n], l1, l2, fmt, n, E, topk, H, I, ep, rank)
        assert dgm.mega.fused_last_form(bs) == 0
        assert torch.equal(ys.view(torch.int16), y[t:t + n].view(torch.int16)), t


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("split", [False, True])
def test_many_local_experts_equal_the_routed_ones(fmt, split):
    """1000 local experts (few tokens, top-k left to the layer call): the same y as a layer that
    holds only the routed experts, renumbered."""
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    M, topk, E, H, I = 7, 8, 1000, 512, 256
    print(f"1000 local experts {fmt} split={split}", flush=True)
    l1, l2 = _weights(dgm, E, H, I, 5)
    g = torch.Generator(device="cuda").manual_seed(6)
    x = torch.randn((M, H), generator=g, device="cuda").bfloat16()
    rw = (torch.randn((E, H), generator=g, device="cuda") / 20).bfloat16()
    buf = dgm.get_fused_symm_buffer_for_mega_moe(None, E, M, topk, H, I, act_format=fmt)
    dgm.fable_router_quant_topk_frontend(x, rw, buf, select_in_mega=True)
    y = torch.full((M, H), 7.0, dtype=torch.bfloat16, device="cuda")
    stats = torch.zeros(E, dtype=torch.int32, device="cuda")
    dgm.mega._fused(y, l1, l2, buf, stats, 10.0, split=split)
    torch.cuda.synchronize()
    assert buf.kernel_error() == 0 and dgm.mega.fused_last_form(buf) == 4
    idx = buf.topk_idx[:M].cpu().numpy()
    counts, active, offs, routes = moe.dispatch(idx, 0, E)
    for got, want in zip(buf.pool_table(), (counts, active, offs, routes)):
        np.testing.assert_array_equal(got.numpy(), want)
    np.testing.assert_array_equal(stats.cpu().numpy(), counts)
    act = torch.from_numpy(active).cuda()
    sub = [tuple(t[act].contiguous() if t is not None else None for t in l) for l in (l1, l2)]
    ys, _, bs = _call(dgm, x, np.searchsorted(active, idx), buf.topk_weights[:M].cpu().numpy(), sub[0], sub[1], fmt, M,
                      len(active), topk, H, I, 1, 0)
    assert dgm.mega.fused_last_form(bs) == 0
    assert torch.equal(ys.view(torch.int16), y.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8", "fp8f128"])
def test_split_launches_equal_one_launch(fmt):
    """The plain form as L1, L2 and combine launches: y of the one launch bit for bit, with a token
    of one local route (written by L2 itself in the one launch), unrouted tokens and ragged slabs."""
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    M, topk, E, ep, H, I = 90, 4, 16, 2, 1024, 512
    print(f"split launches {fmt}", flush=True)
    rng = np.random.default_rng(9)
    l1, l2 = _weights(dgm, E // ep, H, I, 8)
    x = torch.randn((M, H), generator=torch.Generator(device="cuda").manual_seed(9), device="cuda").bfloat16()
    idx, w = _routing("uneven", rng, M, E, topk)
    outs = [_call(dgm, x, idx, w, l1, l2, fmt, M, E, topk, H, I, ep, 0, split=sp)[:2] for sp in (False, True)]
    assert torch.equal(outs[0][0].view(torch.int16), outs[1][0].view(torch.int16))
    assert torch.equal(outs[0][1], outs[1][1])
