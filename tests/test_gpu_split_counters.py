"""The MXFP4 / MXFP8 / FP8F128 calls that run as several launches (the split API, and calls beyond the
one-launch limits) keep nothing in the buffer between calls: counters of any content give the y and
the recv stats of a cleared buffer, bit for bit, and leave the counters as the one-launch layer needs
them."""
import numpy as np
import pytest
import torch

from tests.gpu_common import need_gpu
from tests.test_gpu_large_batch import _routing, _weights

pytestmark = pytest.mark.gpu

H, I, TOPK, E = 1024, 512, 8, 256     # (about 2000 L1 units: more than two per workgroup, so some are claimed)


@pytest.mark.parametrize("M", [100, 300])          # split API; beyond 256 tokens and 1024 routes
@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8", "fp8f128"])
def test_counters_of_any_content(fmt, M):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"counters of any content fmt={fmt} M={M}", flush=True)
    l1, l2 = _weights(dgm, E, H, I, 11)
    x = torch.randn((M, H), generator=torch.Generator(device="cuda").manual_seed(M), device="cuda").bfloat16()
    idx, w = _routing("random", np.random.default_rng(M), M, E, TOPK)
    buf = dgm.get_fused_symm_buffer_for_mega_moe(None, E, M, TOPK, H, I, act_format=fmt)
    dgm.mega._cast_into(buf, x, fmt)
    buf.topk_idx[:M].copy_(torch.from_numpy(idx))
    buf.topk_weights[:M].copy_(torch.from_numpy(w))
    L = buf.layout
    counters = buf.buffer[L.counters:L.total_bytes].view(torch.int32)

    def call(split, m=M):
        y = torch.full((m, H), 7.0, dtype=torch.bfloat16, device="cuda")
        stats = torch.zeros(E, dtype=torch.int32, device="cuda")
        buf.l2_acts.view(torch.uint8).zero_()
        buf.combine_partials.zero_()
        dgm.mega._fused(y, l1, l2, buf, stats, 10.0, split=split)
        torch.cuda.synchronize()
        assert buf.kernel_error() == 0 and buf.host_error() == 0
        return y.view(torch.int16), stats

    ref = call(True)
    one = call(False, 64)
    gen = torch.Generator(device="cuda").manual_seed(12)
    for fill in (1 << 20, 3, -1, 0x7FFFFFFF, None):
        header = counters[:16].clone()
        if fill is None:
            counters.random_(-(1 << 31), 1 << 31, generator=gen)
        else:
            counters.fill_(fill)
        counters[1:16] = header[1:]                # (the error words: the caller's)
        for got, want in zip(call(True), ref):
            assert torch.equal(got, want), fill
        for got, want in zip(call(False, 64), one):
            assert torch.equal(got, want), fill
