"""Per-call options on the calls that run as several launches (the split API, and MXFP4 / MXFP8 /
FP8F128 calls beyond the one-launch limits)."""
import numpy as np
import pytest
import torch

from tests.gpu_common import need_gpu
from tests.test_gpu_large_batch import _routing, _weights

pytestmark = pytest.mark.gpu

H, I, TOPK, E = 512, 256, 8, 64


def _filled(dgm, fmt, M, seed=21):
    l1, l2 = _weights(dgm, E, H, I, seed)
    x = torch.randn((M, H), generator=torch.Generator(device="cuda").manual_seed(M), device="cuda").bfloat16()
    idx, w = _routing("random", np.random.default_rng(M), M, E, TOPK)
    buf = dgm.get_fused_symm_buffer_for_mega_moe(None, E, M, TOPK, H, I, act_format=fmt)
    dgm.mega._cast_into(buf, x, fmt)
    buf.topk_idx[:M].copy_(torch.from_numpy(idx))
    buf.topk_weights[:M].copy_(torch.from_numpy(w))
    return l1, l2, buf


def _call(dgm, l1, l2, buf, M, split=True, **kw):
    y = torch.full((M, H), 7.0, dtype=torch.bfloat16, device="cuda")
    stats = torch.zeros(E, dtype=torch.int32, device="cuda")
    dgm.mega._fused(y, l1, l2, buf, stats, 10.0, split=split, **kw)
    torch.cuda.synchronize()
    assert buf.kernel_error() == 0 and buf.host_error() == 0
    return y.view(torch.int16), stats


@pytest.mark.parametrize("M,split", [(20, True), (300, False)])
@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8", "fp8f128"])
def test_cooperative_option_same_results(fmt, M, split):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"cooperative option fmt={fmt} M={M} split={split}", flush=True)
    l1, l2, buf = _filled(dgm, fmt, M)
    out = []
    for coop in (False, True):
        buf.cooperative = coop
        out.append(_call(dgm, l1, l2, buf, M, split))
    for u, v in zip(*out):
        assert torch.equal(u, v)


@pytest.mark.parametrize("fmt,M,split", [("mxfp8", 20, True), ("mxfp8", 300, False), ("qoq", 20, True)])
def test_phase_stamps_of_both_launches(fmt, M, split):
    """The L1 launch stamps the first rows and the L2 launch as many behind them, each in phase order
    within the launch, L2's launch entered once every workgroup of L1's was done; y does not
    change, and a stamp array that ends inside either launch's rows is not written past."""
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"stamps of both launches fmt={fmt} M={M} split={split}", flush=True)
    if fmt == "qoq":
        from tests.test_gpu_qoq import make_qoq_weights
        _, _, buf = _filled(dgm, "mxfp8", M)
        idx, w = buf.topk_idx.clone(), buf.topk_weights.clone()
        (l1, l2), kw = make_qoq_weights(E, H, I, 22)[0], {"fmt": "qoq"}
        buf = dgm.get_fused_symm_buffer_for_mega_moe(None, E, M, TOPK, H, I, act_format=fmt)
        x = torch.randn((M, H), generator=torch.Generator(device="cuda").manual_seed(M), device="cuda").bfloat16()
        dgm.mega._cast_into(buf, x, fmt)
        buf.topk_idx.copy_(idx)
        buf.topk_weights.copy_(w)
    else:
        l1, l2, buf = _filled(dgm, fmt, M)
        kw = {}
    y0, s0 = _call(dgm, l1, l2, buf, M, split, **kw)
    st = torch.zeros((2048, 8), dtype=torch.int64, device="cuda")
    y1, s1 = _call(dgm, l1, l2, buf, M, split, phase_stamps=st, **kw)
    assert torch.equal(y0, y1) and torch.equal(s0, s1)
    G = dgm.mega.fused_workgroups(buf)
    a = st.cpu().numpy()
    assert 0 < 2 * G < 2048 and (a[2 * G:] == 0).all()
    one, two = a[:G], a[G:2 * G]
    for r in (one, two):
        assert (r[:, 0] > 0).all() and (r[:, 1] >= r[:, 0]).all() and (r[:, 2] >= r[:, 1]).all()
        assert (r[:, 4] >= r[:, 2]).all() and (r[:, 5] >= r[:, 4]).all()
        assert (r[:, 6] + r[:, 7] <= r[:, 5] - r[:, 0]).all()
    assert two[:, 0].min() >= one[:, 2].max()
    assert (one[:, 6] > 0).any() and (two[:, 6:] == 0).all()          # (L1 K loops run in the first alone)
    for n in (G + G // 2, G // 2):
        part = torch.zeros((2 * G, 8), dtype=torch.int64, device="cuda")
        y2, _ = _call(dgm, l1, l2, buf, M, split, phase_stamps=part[:n], **kw)
        p = part.cpu().numpy()
        assert torch.equal(y0, y2) and (p[:n, 0] > 0).all() and (p[n:] == 0).all()


@pytest.mark.parametrize("flags", ["raw", "raw and forced-balanced"])
@pytest.mark.parametrize("M", [5, 12])          # within and beyond the in-kernel selection's tokens
@pytest.mark.parametrize("fmt,split", [("mxfp4", True), ("mxfp8", True), ("fp8f128", True), ("mxfp8", False)])
def test_raw_weights_selected_by_the_layer_call(fmt, split, M, flags):
    """DGM_FE_RAW_WEIGHTS with the top-k left to the layer call: the routing and y of the same top-k
    selected beforehand."""
    need_gpu()
    import ctypes
    import hopper_megamoe_basedondeepgemm_amd as dgm
    from hopper_megamoe_basedondeepgemm_amd import _lib
    print(f"raw weights fmt={fmt} split={split} M={M} {flags}", flush=True)
    bits = _lib.FE_RAW_WEIGHTS | (_lib.FE_FORCE_BALANCED if "forced" in flags else 0)
    l1, l2, buf = _filled(dgm, fmt, M)
    logits = torch.randn((M, E), generator=torch.Generator(device="cuda").manual_seed(31), device="cuda").bfloat16()
    out = []
    for left in (0, _lib.FE_SELECT_IN_MEGA):
        _lib.check(_lib.load().dgm_router_logits_topk_launch(
            _lib.ptr(logits), M, E, TOPK, bits | left, 0, _lib.ptr(buf.buffer), ctypes.byref(buf.layout), _lib.stream()))
        buf._fe_select = (bits, 0) if left else None
        y, stats = _call(dgm, l1, l2, buf, M, split)
        out.append((y, stats, buf.topk_idx.clone(), buf.topk_weights.clone()))
    for u, v in zip(*out):
        assert torch.equal(u, v)
    if "forced" not in flags:
        assert torch.equal(out[1][3], logits.float().sort(dim=1, descending=True).values[:, :TOPK])


@pytest.mark.parametrize("fmt,M", [("mxfp8", 20), ("fp8f128", 300)])
def test_graph_replays(fmt, M):
    """A captured split call replayed with other routings, eager calls and a one-launch call between the
    replays: every replay gives the eager result bit for bit."""
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"graph replays fmt={fmt} M={M}", flush=True)
    l1, l2, buf = _filled(dgm, fmt, M)
    weights = [buf.topk_weights.clone() * f for f in (1.0, 0.5, 2.0)]
    refs = []
    for w in weights:
        buf.topk_weights.copy_(w)
        refs.append(_call(dgm, l1, l2, buf, M))
    y = torch.empty((M, H), dtype=torch.bfloat16, device="cuda")
    stats = torch.zeros(E, dtype=torch.int32, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dgm.mega._fused(y, l1, l2, buf, stats, 10.0, split=True)
    for i in (0, 1, 2, 1):
        buf.topk_weights.copy_(weights[i])
        y.fill_(7.0)
        stats.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), refs[i][0]) and torch.equal(stats, refs[i][1]), i
        for split in (True, False):
            for u, v in zip(_call(dgm, l1, l2, buf, M, split), refs[i]):
                assert torch.equal(u, v), i
