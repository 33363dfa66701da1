"""The frontend's matrix-core router tiles (beyond 64 tokens, where they are enough) against its one-wave
rows (below 64 tokens), and beyond 64 tokens the rows of eight tokens where tiles are few: fp32 logits, top-k keys and activation bytes bit for bit, with ragged token and expert
tiles, every hidden size, zero rows, subnormal and huge values, infinities and NaN; and the logits
of the finite rows against the oracle's fixed order."""
import numpy as np
import pytest
import torch

from oracle import moe
from tests.gpu_common import need_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,E,H,act", [(112, 384, 3072, "mxfp8"), (129, 48, 512, "mxfp4"), (143, 8, 1024, "qoq"),
                                       (160, 1000, 512, "nvfp4"), (200, 72, 2048, "fp8f128"), (131, 20, 4096, "mxfp8"),
                                       (65, 200, 4096, "mxfp4"), (65, 8, 512, "mxfp8"), (111, 150, 3072, "fp8f128"),
                                       # (few tiles: rows of eight tokens, the last ragged)
                                       (70, 48, 2048, "mxfp4"), (101, 20, 3072, "mxfp8")])
def test_router_tiles_equal_router_rows(M, E, H, act):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    from hopper_megamoe_basedondeepgemm_amd import _lib
    print(f"router tiles M={M} E={E} H={H} {act}", flush=True)
    g = torch.Generator().manual_seed(M + E)
    x = torch.randn((M, H), generator=g)
    x[3] = 0.0
    x[5] *= 2.0 ** -130            # subnormal bf16 values and products
    x[6] *= 2.0 ** 100
    x[7, 11] = float("inf")
    x[8, 12] = float("-inf")
    x[8, 13] = float("inf")
    x[M - 1, H - 1] = float("nan")
    x = x.bfloat16()
    w = torch.randn((E, H), generator=g) * 0.05
    w[1] *= 2.0 ** -100
    w = w.bfloat16()
    w[0] = 0.0

    def front(rows):
        b = dgm.get_fused_symm_buffer_for_mega_moe(None, E, rows.size(0), 8, H, 256, act_format=act)
        dgm.fable_router_quant_topk_frontend(rows, w.cuda(), b, select_in_mega=False, zero_row_unrouted=True)
        torch.cuda.synchronize()
        n = rows.size(0)
        return [t.view(torch.uint8).view(n, -1).cpu() for t in (b.logits[:n], b.fe_keys[:n], b.x[:n], b.x_sf[:n])]

    xc = x.cuda()
    big = front(xc)
    small = [torch.cat(p) for p in zip(*(front(xc[t:t + 50]) for t in range(0, M, 50)))]
    for name, u, v in zip(("logits", "keys", "codes", "scales"), big, small):
        assert torch.equal(u, v), name
    assert (big[1][3] == 0).all()            # a zero row's keys
    rows = [0, 1, 64, M - 2]                 # (not row 5: the oracle rounds its subnormal products)
    ref = moe.router_logits_f32(x[rows].float().numpy(), w.float().numpy())
    np.testing.assert_array_equal(big[0][rows].view(torch.float32).numpy().view(np.uint32), ref.view(np.uint32))
    # the same without the cast rows beside the router's (the split API's router_input)
    b = dgm.get_fused_symm_buffer_for_mega_moe(None, E, M, 8, H, 256, act_format=act)
    _lib.check(_lib.load().dgm_router_topk_launch(
        _lib.ptr(xc), _lib.ptr(w.cuda()), M, H, E, 8, _lib.ACT_FORMATS[act], _lib.FE_NO_CAST, 0, _lib.ptr(b.buffer),
        __import__("ctypes").byref(b.layout), _lib.stream()))
    torch.cuda.synchronize()
    assert torch.equal(b.logits.view(torch.uint8).view(M, -1).cpu(), big[0]) and not b.x.view(torch.uint8).any()
    # one stamp row per workgroup: the router tiles, then the cast
    dgm.fable_router_quant_topk_frontend(xc, w.cuda(), b, stamps=1)
    st = dgm.fable_frontend_stamps(b, E).cpu()
    n = dgm.fable_frontend_router_ctas(M, E, H)
    assert st.shape[0] > n and (st[:n, 3] > 0).all() and (st[:n, 5] == 0).all() and (st[n:, 5] > 0).all()
