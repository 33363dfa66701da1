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
