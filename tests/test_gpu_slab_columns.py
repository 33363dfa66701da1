"""The activation slab's columns: a token's output does not depend on the tokens beside it, so y of M
tokens on the same expert (slabs of M, or of 16 and the rest, columns) equals, bit for bit, y of each
token alone. Every format, every column count of a slab, the first counts of a second and third."""
import pytest
import torch

from tests.gpu_common import need_gpu

pytestmark = pytest.mark.gpu


def _weights(dgm, fmt, E, H, I):
    g = torch.Generator(device="cuda").manual_seed(H)
    out = []
    for n, k in ((2 * I, H), (H, I)):
        u8 = lambda lo, hi, shape: torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)
        packed = u8(0, 256, (E, n, k // 2))
        if fmt == "qoq":
            s1 = (torch.rand((E, n), generator=g, device="cuda") * 2e-4 + 5e-4).bfloat16().float()
            out.append((packed, u8(1, 16, (E, n, k // 128)), u8(0, 16, (E, n, k // 128)), s1))
        elif fmt == "nvfp4":
            out.append((packed, u8(0x10, 0x20, (E, n, k // 16))))
        else:
            out.append((packed, u8(118, 121, (E, n, k // 32))))
    return {"qoq": dgm.transform_qoq_weights_for_mega_moe_fused,
            "nvfp4": dgm.transform_nvfp4_weights_for_mega_moe_fused}.get(
                fmt, dgm.transform_mxfp4_weights_for_mega_moe_fused)(*out)


@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8", "fp8f128", "qoq", "nvfp4"])
@pytest.mark.parametrize("H,I,counts", [(512, 256, tuple(range(1, 19)) + (31, 33)), (1024, 512, (3, 7)),
                                        (3072, 1280, (1, 2, 3, 5, 11, 16, 17))])
def test_columns_are_independent(fmt, H, I, counts):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"slab columns {fmt} H={H} I={I}", flush=True)
    E = 3
    l1, l2 = _weights(dgm, fmt, E, H, I)
    x = torch.randn((max(counts), H), generator=torch.Generator(device="cuda").manual_seed(I), device="cuda").bfloat16()

    def call(rows):
        m = rows.size(0)
        b = dgm.get_fused_symm_buffer_for_mega_moe(None, E, m, 2, H, I, act_format=fmt)
        dgm.mega._cast_into(b, rows, fmt)
        b.topk_idx[:m] = torch.tensor([2, 0], device="cuda")
        b.topk_weights[:m] = torch.tensor([0.625, 0.375], device="cuda")
        y = torch.full((m, H), 7.0, dtype=torch.bfloat16, device="cuda")
        dgm.mega._fused(y, l1, l2, b, None, 10.0, fmt=fmt)
        torch.cuda.synchronize()
        assert b.kernel_error() == 0
        return y.view(torch.int16)

    alone = torch.cat([call(x[t:t + 1]) for t in range(x.size(0))])
    assert alone.view(torch.bfloat16).float().abs().max() > 0 and torch.isfinite(alone.view(torch.bfloat16).float()).all()
    for m in counts:
        assert torch.equal(call(x[:m]), alone[:m]), m
