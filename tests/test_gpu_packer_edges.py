"""The weight packers at the values where their scales and codes turn, bit-exact against the
oracle for bf16, fp16 and fp32 sources: group maxima at and one step beside every power of two
times 6 (MXFP4's ceil(log2) edge), elements on, just below and just above every E2M1 midpoint of
their scale, signed zeros, rows of zeros, tiny and large magnitudes; row lengths that leave partial
waves; QoQ rows beyond the register-held length and from an unaligned source."""
import numpy as np
import pytest
import torch

from oracle import packers as pk
from tests.gpu_common import need_gpu

pytestmark = pytest.mark.gpu
MIDS = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)


def _edge_rows(dtype, K, group):
    """Rows of K values: per group a maximum near 6 * 2^e and elements around the midpoints."""
    g = torch.Generator().manual_seed(K + group)
    lo, hi = (-12, 10) if dtype == torch.float16 else (-90, 90)
    rows = []
    for e in range(lo, hi, 3 if dtype == torch.float16 else 7):
        for step in (-1, 0, 1):
            top = torch.tensor(6.0 * 2.0 ** e).to(dtype)
            top = (top.view(torch.int32 if dtype == torch.float32 else torch.int16) + step).view(dtype)
            v = torch.randn(K, generator=g) * 2.0 ** e * 2
            for i in range(K):
                m = MIDS[i % 7] * 2.0 ** (e + (i // 7) % 2)
                if i % 3 == 0:
                    t = torch.tensor(m).to(dtype)
                    t = (t.view(torch.int32 if dtype == torch.float32 else torch.int16) + (i // 3) % 3 - 1).view(dtype)
                    v[i] = float(t) * (-1 if i % 2 else 1)
            v[::11] = -0.0
            v = v.clamp(-float(top), float(top))
            v[::group] = float(top)
            rows.append(v)
    rows.append(torch.zeros(K))
    rows.append(torch.randn(K, generator=g) * 2.0 ** (-14 if dtype == torch.float16 else -120))
    return torch.stack(rows).to(dtype)


def _np(t):
    return t.float().numpy()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("K", [96, 544])
def test_mxfp4_and_nvfp4_edges(dtype, K):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"packer edges {dtype} K={K}", flush=True)
    w = _edge_rows(dtype, K, 16)
    for fn, ref in ((dgm.quantization_mxfp4_fused.quantize_to_mxfp4, pk.quantize_to_mxfp4_fused),
                    (dgm.quantization_mxfp4.quantize_to_mxfp4, pk.quantize_to_mxfp4_split),
                    (dgm.quantization_nvfp4.quantize_to_nvfp4, pk.quantize_to_nvfp4)):
        got, want = fn(w.cuda()), ref(_np(w))
        for u, v in zip(got, want):
            np.testing.assert_array_equal(u.cpu().numpy(), v)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("K,unaligned", [(128, False), (1664, False), (4096, False), (4224, False), (640, True)])
def test_qoq_edges(dtype, K, unaligned):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"QoQ edges {dtype} K={K} unaligned={unaligned}", flush=True)
    g = torch.Generator().manual_seed(K)
    w = torch.randn((19, K), generator=g) * 0.02
    w[1] = 0.0
    w[2, :128] = 0.0
    w[3] = (torch.arange(K) % 241 - 120).float() * 0.5            # quotients on half integers
    w[4] = torch.randint(-16, 17, (K,), generator=g).float() / 4
    w[5].abs_()
    w[6] *= 2.0 ** (-6 if dtype == torch.float16 else -110)        # s1 at its floor / divisions
    w[7] *= 2.0 ** (15 if dtype == torch.float16 else 104)
    w[8, 5] = 3.0
    w = w.to(dtype)
    src = w.cuda()
    if unaligned:
        flat = torch.empty(w.numel() + 1, dtype=dtype, device="cuda")
        src = flat[1:].view(w.shape)
        src.copy_(w.cuda())
        assert src.data_ptr() % 16
    for u, v in zip(dgm.quantization_qoq_fused.quantize_to_qoq(src), pk.quantize_to_qoq(_np(w)[None])):
        np.testing.assert_array_equal(u.cpu().numpy().reshape(v.shape), v)
    for u, v in zip(dgm.quantization_mxfp4.quantize_to_qoq_int4(src[None]), pk.quantize_to_qoq_int4(_np(w)[None])):
        np.testing.assert_array_equal(u.cpu().numpy().reshape(v.shape), v)


def test_qoq_transform_refuses_wide_meta():
    """z or s2 beyond a nibble raises, from the fused tuple and from the int4 plane."""
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    w = [torch.randn((2, n, k), device="cuda").bfloat16() for n, k in ((64, 256), (128, 128))]
    q = [dgm.quantization_qoq_fused.quantize_to_qoq(x) for x in w]
    i4 = [dgm.quantization_mxfp4.quantize_to_qoq_int4(x) for x in w]
    dgm.transform_qoq_weights_for_mega_moe_fused(*q)
    dgm.transform_qoq_int4_weights_for_mega_moe_sm90(*i4)
    for k in (1, 2):
        bad = [t.clone() for t in q[1]]
        bad[k][1, 127, 0] = 16
        with pytest.raises(ValueError, match="out of range"):
            dgm.transform_qoq_weights_for_mega_moe_fused(q[0], tuple(bad))
    for shift in (0, 8):
        bad = (i4[0][0], (i4[0][1] & ~(0xFF << shift)) | (200 << shift))
        with pytest.raises(ValueError, match="out of range"):
            dgm.transform_qoq_int4_weights_for_mega_moe_sm90(bad, i4[1])


@pytest.mark.parametrize("offset", [0, 4])
def test_nvfp4_transform_at_any_alignment(offset):
    """The layout transform from a source 4 bytes off its 16-byte alignment equals the aligned one."""
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    E, N, K = 2, 64, 384
    g = torch.Generator(device="cuda").manual_seed(3)
    packed = torch.randint(0, 256, (E, N, K // 2), generator=g, device="cuda", dtype=torch.uint8)
    sc = torch.randint(0, 120, (E, N, K // 16), generator=g, device="cuda", dtype=torch.uint8)
    flat = torch.empty(packed.numel() + offset, dtype=torch.uint8, device="cuda")
    src = flat[offset:].view(packed.shape)
    src.copy_(packed)
    for order in ("marlin", "low_first"):
        v, s = dgm.mega._transform_nvfp4_one(src, sc, True, order)
        rv, rs = pk.nvfp4_to_tile(packed.cpu().numpy(), sc.cpu().numpy(), order, 1)
        np.testing.assert_array_equal(v.cpu().numpy().reshape(rv.shape), rv)
        np.testing.assert_array_equal(s.cpu().numpy().reshape(rs.shape), rs)
