"""The L1 -> L2 intermediate of MXFP4, MXFP8 and FP8F128 calls (one launch, split, large batch) against
the oracle's rules, code by code and scale by scale, of every pool row.

The inputs make the L1 products exact: integer activations, E2M1 weights times 2^-9 .. 2^-7, so every
partial sum is a multiple of 2^-10 below 2^14 and fits fp32 in any order. What is left to rounding is
the activation function (fast_math=False: expf, one division, three products: at most eight roundings of
2^-24, far below EPS), so a code or scale must be the oracle's of a value within EPS of the exact one."""
import numpy as np
import pytest
import torch

from oracle import numerics as nu
from oracle import packers as pk
from oracle import moe
from tests.gpu_common import need_gpu
from tests.test_gpu_large_batch import _routing

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -20
TOPK = 4


def _inputs(fmt, rng, M, H):
    """Activation values [M, H], exact in the format."""
    vals = np.array([0, 1, 2, 3, 4, 6]) if fmt == "mxfp4" else np.arange(9)
    return (rng.choice(vals, (M, H)) * rng.choice([-1, 1], (M, H))).astype(np.float32)


def _exact_act(x, packed, scale, w, I, fmt):
    """Expert activations of rows x with routing weights w, in 64 bits (gate and up as the kernel has
    them: exact, rounded to bf16 but for FP8F128)."""
    h = x.astype(np.float64) @ pk.dequantize_mxfp4_marlin(packed, scale).astype(np.float64).T
    assert np.abs(h * 1024 - np.rint(h * 1024)).max() == 0 and np.abs(h).max() < 2 ** 14
    if fmt != "fp8f128":
        h = nu.round_bf16(h.astype(np.float32)).astype(np.float64)
    g, u = np.minimum(h[:, :I], 10.0), np.clip(h[:, I:], -10.0, 10.0)
    return g / (1.0 + np.exp(-g)) * u * w[:, None].astype(np.float64)


def _scale_exp(amax, fmt):
    amax = amax.astype(np.float32)
    if fmt == "mxfp4":
        return np.log2(nu.ceil_to_ue8m0(np.maximum(amax, np.float32(1e-30)) / np.float32(6.0))).astype(int)
    if fmt == "mxfp8":
        return nu.ceil_log2_f32(np.maximum(amax, np.float32(1e-30)) / np.float32(448.0)).astype(int)
    return nu.ceil_log2_f32(np.maximum(amax / np.float32(448.0), moe.FLT_TINY)).astype(int)


@pytest.mark.parametrize("M,mode", [(40, "one launch"), (40, "split"), (300, "large batch")])
@pytest.mark.parametrize("E,H,I", [(16, 512, 256), (8, 3072, 1280)])
@pytest.mark.parametrize("fmt", ["mxfp4", "mxfp8", "fp8f128"])
def test_intermediate_codes_and_scales(fmt, E, H, I, M, mode):
    need_gpu()
    import hopper_megamoe_basedondeepgemm_amd as dgm
    print(f"intermediate fmt={fmt} E={E} H={H} I={I} M={M} {mode}", flush=True)
    rng = np.random.default_rng(M + H)
    q = [(rng.integers(0, 256, (E, n, k // 2), dtype=np.uint8), rng.integers(118, 121, (E, n, k // 32), dtype=np.uint8))
         for n, k in ((2 * I, H), (H, I))]
    l1, l2 = dgm.transform_mxfp4_weights_for_mega_moe_fused(*[tuple(torch.from_numpy(a).cuda() for a in m) for m in q])
    x = _inputs(fmt, rng, M, H)
    idx, w = _routing("uneven", rng, M, E, TOPK)
    buf = dgm.get_fused_symm_buffer_for_mega_moe(None, E, M, TOPK, H, I, act_format=fmt)
    if fmt == "fp8f128":
        buf.x[:M].copy_(torch.from_numpy(x).to(torch.float8_e4m3fn))
        buf.x_sf[:M].fill_(1.0)
    else:
        np.testing.assert_array_equal(moe.quant_act(x, fmt)[2], x)
        dgm.mega._cast_into(buf, torch.from_numpy(x).bfloat16().cuda(), fmt)
    buf.topk_idx[:M].copy_(torch.from_numpy(idx))
    buf.topk_weights[:M].copy_(torch.from_numpy(w))
    y = torch.empty((M, H), dtype=torch.bfloat16, device="cuda")
    dgm.mega._fused(y, l1, l2, buf, None, 10.0, split=mode == "split", fast_math=False)
    torch.cuda.synchronize()
    assert buf.kernel_error() == 0 and dgm.mega.fused_last_form(buf) == (4 if mode == "large batch" else 0)
    counts, active, offs, routes = moe.dispatch(idx, 0, E)
    n = int(counts.sum())
    codes = buf.l2_acts[:n].view(torch.uint8).cpu().numpy()
    if fmt == "mxfp4":
        codes = np.stack([codes & 15, codes >> 4], axis=-1).reshape(n, I)
    sf = buf.l2_acts_sf[:n].view(torch.uint8).view(n, -1)[:, :I // 32].cpu().numpy().astype(int) - 127
    a = np.concatenate([_exact_act(x[routes[o:p] // TOPK], q[0][0][e], q[0][1][e], w.reshape(-1)[routes[o:p]], I, fmt)
                        for e, o, p in zip(active, offs[:-1], offs[1:])])
    group = 64 if fmt == "fp8f128" else 32
    amax = np.abs(a).reshape(n, -1, group).max(axis=-1).repeat(group // 32, axis=1)
    assert (sf >= _scale_exp(amax * (1 - EPS), fmt)).all() and (sf <= _scale_exp(amax * (1 + EPS), fmt)).all()
    bits = 7 if fmt == "mxfp4" else 127
    mag = lambda v: ((nu.e2m1_code_ties_down if fmt == "mxfp4" else nu.e4m3_encode)(v.astype(np.float32)) & bits).astype(int)
    v = np.abs(a) / np.exp2(sf).repeat(32, axis=1)
    got = (codes & bits).astype(int)
    assert (got >= mag(v * (1 - EPS))).all() and (got <= mag(v * (1 + EPS))).all()
    assert (got != mag(v)).mean() < 1e-4          # (values on a rounding boundary)
    some = got > 0
    assert ((codes[some] > bits) == (a[some] < 0)).all()
