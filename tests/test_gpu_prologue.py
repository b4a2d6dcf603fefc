"""Fused RMSNorm + RoPE + INT8 prologue on the GPU: bit-exact against the oracle (norm_rope, then the
per-block quantizer), and the fused Wan self-attention against the unfused path."""

import numpy as np
import pytest
import torch

from tests.gpu_util import log, require_gpu
from tests.inputs import bf16_bits, cosine

pytestmark = pytest.mark.gpu
LOG2E = 1.44269504


def _inputs(B, L, H, D, seed):
    g = torch.Generator().manual_seed(seed)
    xq = (torch.randn((B, L, H * D), generator=g) * 2).to(torch.bfloat16)
    xk = (torch.randn((B, L, H * D), generator=g) * 2 + 0.3).to(torch.bfloat16)
    xv = torch.randn((B, L, H * D), generator=g).to(torch.bfloat16)
    wq = (1 + 0.1 * torch.randn((H * D,), generator=g)).to(torch.bfloat16)
    wk = (1 + 0.1 * torch.randn((H * D,), generator=g)).to(torch.bfloat16)
    ang = torch.rand((L, 1, D // 2), generator=g, dtype=torch.float64) * 6.3  # the reference's fp64 freqs
    return xq, xk, xv, wq, wk, ang.cos(), ang.sin()


@pytest.mark.parametrize("B,L,H", [(1, 300, 2), (2, 777, 3)])
def test_prologue_bit_exact(oracle, B, L, H):
    dev = require_gpu()
    from telefuser_amd.prologue import norm_rope_quant_qk

    D = 128
    xq, xk, xv, wq, wk, fc, fs = _inputs(B, L, H, D, seed=L)
    log(f"prologue B={B} L={L} H={H}")
    q8, qs, k8, ks, km = norm_rope_quant_qk(*(t.to(dev) for t in (xq, xk, wq, wk, fc, fs)), num_heads=H)
    torch.cuda.synchronize()
    cs, sn = fc.reshape(L, -1).float().numpy(), fs.reshape(L, -1).float().numpy()
    qn = oracle.norm_rope(bf16_bits(xq), bf16_bits(wq), cs, sn, D).reshape(B, L, H, D)
    kn = oracle.norm_rope(bf16_bits(xk), bf16_bits(wk), cs, sn, D).reshape(B, L, H, D)
    kmb = km.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    # the smoothing vector: the mean of the rotated K, to one bf16 rounding of the fp64 mean
    km_ref = oracle.bf16_bits_to_f32(oracle.k_mean_bits(kn))
    assert np.abs(oracle.bf16_bits_to_f32(kmb) - km_ref).max() <= np.abs(km_ref).max() * 2 ** -8
    oq8, oqs = oracle.quant_per_block_int8(qn, sm_scale=D ** -0.5 * LOG2E, blk=128)
    ok8, oks = oracle.quant_per_block_int8(kn, km_bits=kmb, blk=64)
    assert np.array_equal(qs.cpu().numpy(), oqs) and np.array_equal(q8.cpu().numpy(), oq8)
    assert np.array_equal(ks.cpu().numpy(), oks) and np.array_equal(k8.cpu().numpy(), ok8)


def test_fused_wan_self_attention_matches_unfused(oracle):
    dev = require_gpu()
    from telefuser_amd import sageattn2 as sa
    from telefuser_amd.prologue import wan_self_attention

    B, L, H, D = 1, 1000, 2, 128
    xq, xk, xv, wq, wk, fc, fs = _inputs(B, L, H, D, seed=5)
    o = wan_self_attention(*(t.to(dev) for t in (xq, xk, xv, wq, wk, fc, fs)), num_heads=H)
    # the unfused route: norm and rope materialised (oracle), then the drop-in sage call
    cs, sn = fc.reshape(L, -1).float().numpy(), fs.reshape(L, -1).float().numpy()
    to_t = lambda bits: torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).reshape(B, L, H, D)
    qn = to_t(oracle.norm_rope(bf16_bits(xq), bf16_bits(wq), cs, sn, D))
    kn = to_t(oracle.norm_rope(bf16_bits(xk), bf16_bits(wk), cs, sn, D))
    vn = xv.reshape(B, L, H, D)
    o2 = sa.sageattn_qk_int8_pv_fp8_cuda(qn.to(dev), kn.to(dev), vn.to(dev), tensor_layout="NHD",
                                         qk_quant_gran="per_block", pv_accum_dtype="fp32+fp32")
    torch.cuda.synchronize()
    truth = oracle.attn_fp64(bf16_bits(qn), bf16_bits(kn), bf16_bits(vn), D ** -0.5)
    a, b = o.float().cpu().numpy().reshape(B, L, H, D), o2.float().cpu().numpy()
    log(f"fused vs unfused cos={cosine(a, b):.7f} fused vs truth cos={cosine(a, truth):.6f}")
    assert cosine(a, b) >= 0.99999
    assert cosine(a, truth) >= 0.999


@pytest.mark.parametrize("B,L,H,D,dtype,variant,smooth_k", [
    (1, 1, 1, 64, torch.bfloat16, "cuda", True),        # one row, less than a wave of chunks
    (2, 129, 5, 128, torch.float16, "triton", True),    # a row past a 128-row block
    (1, 64, 12, 64, torch.bfloat16, "cuda", True),
    (1, 257, 6, 128, torch.bfloat16, "triton", False),
    (1, 200, 12, 128, torch.float16, "cuda", True),     # the widest row of the one-pass statistics
    (1, 70, 13, 128, torch.bfloat16, "cuda", True),     # wider: separate statistics
    (2, 1100, 8, 64, torch.bfloat16, "cuda", True),     # one chunk per lane, the last one full
])
@pytest.mark.parametrize("strided", [False, True])
def test_prologue_shapes(B, L, H, D, dtype, variant, smooth_k, strided):
    """norm + rope + INT8 over row widths, block edges, types, roundings and strided rows, against the same arithmetic
    in torch (fp32 products, the fused multiply-add through float64) quantized by the plain quantizer."""
    dev = require_gpu()
    from telefuser_amd import sageattn2 as sa
    from telefuser_amd.prologue import norm_rope_quant_qk, row_rstd

    g = torch.Generator().manual_seed(L + H)
    n = H * D
    x = (torch.randn((2, B, L, n + 64), generator=g) * 2 + 0.3).to(dtype).to(dev)
    xq, xk = (t[..., :n] if strided else t[..., :n].contiguous() for t in x)
    wq, wk = ((1 + 0.1 * torch.randn(n, generator=g)).to(dtype).to(dev) for _ in range(2))
    ang = torch.rand((L, 1, D // 2), generator=g, dtype=torch.float64).to(dev) * 6.3
    fc, fs = ang.cos().float(), ang.sin().float()
    log(f"prologue shapes B={B} L={L} H={H} D={D} {dtype} {variant} strided={strided}")
    q8, qs, k8, ks, km = norm_rope_quant_qk(xq, xk, wq, wk, fc, fs, H, smooth_k=smooth_k, variant=variant)

    def rotated(t, w):
        r = row_rstd(t, 1e-6)
        var = (t.double().square().sum(-1) / n).float()
        assert torch.equal(r, 1.0 / (var + 1e-6).sqrt())
        y = ((t.float() * r[..., None]) * w.float()).to(dtype).float().view(B, L, H, D // 2, 2)
        y1, y2 = y[..., 0], y[..., 1]
        c, s = fc.view(1, L, 1, -1), fs.view(1, L, 1, -1)
        fma = lambda a, b, c_: (a.double() * b.double() + c_.double()).float().to(dtype)
        return torch.stack((fma(-y2, s, y1 * c), fma(y1, s, y2 * c)), -1).view(B, L, H, D)

    qn, kn = rotated(xq, wq), rotated(xk, wk)
    if smooth_k:
        ref = kn.double().mean(1)
        assert float((km.double() - ref).abs().max()) <= float(ref.abs().max()) * 2 ** -8
    else:
        assert km is None
    want = sa.per_block_int8(qn, kn, km, sm_scale=D ** -0.5, tensor_layout="NHD", variant=variant)
    for name, a, b in zip(("q_int8", "q_scale", "k_int8", "k_scale"), (q8, qs, k8, ks), want):
        if dtype == torch.float16 and a.dtype == torch.int8:
            # an fp32 product on its way to fp16 is rounded once on the GPU (v_fma_mixlo_f16) and twice here, which
            # differs where the fp32 rounding makes a tie: about 2^-13 of the values, by an fp16 ulp (2^-11 of the
            # value), and of those the ~1 in 16 whose code (up to 127) lies that near a rounding edge
            d = (a.int() - b.int()).abs()
            assert int(d.max()) <= 1 and int((d > 0).sum()) <= 1 + a.numel() * 2.0 ** -15, name
        else:
            assert torch.equal(a, b), name
