"""The weight-streaming kernel on row-major operands (at most 64 activation rows): ends of tiles, of 256-K blocks and of the
waves' shares of K, every number of K steps in the last block, scale bytes beyond K that are NaN, and the one-row kernels
and the general ones beside it.  Tolerance: that of test_gemm_gpu.py, |y - ref| <= 2^-8 |ref| + 1e-5 sum |dq(x)||dq(w)|."""
import pytest
import torch

from oracle import fpq_oracle as O

pytestmark = pytest.mark.gpu


def _codes(rows, k, gen):
    return torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, generator=gen)


def _scales(rows, k, fmt, gen, stride):
    group, low, high = (32, 118, 134) if fmt == "mxfp4" else (16, 0x18, 0x60)
    out = torch.full((rows, stride), 0xFF, dtype=torch.uint8)   # (beyond K: NaN in both formats)
    out[:, :k // group] = torch.randint(low, high, (rows, k // group), dtype=torch.uint8, generator=gen)
    return out


@pytest.mark.parametrize("fmt", ["mxfp4", "nvfp4"])
@pytest.mark.parametrize("m,n,k", [
    (1, 40, 544), (2, 33, 576), (16, 31, 608), (17, 32, 640), (31, 70, 672), (32, 96, 704), (33, 65, 736), (64, 64, 768),
    (17, 24, 32), (40, 264, 96), (3, 264, 1792), (33, 40, 2080), (5, 72, 2304), (64, 130, 2528), (48, 264, 4352),
    (1, 264, 2048), (1, 1040, 8192), (1, 40, 8448), (16, 8, 512), (8, 40, 480),
])
@pytest.mark.parametrize("pad", [0, 1])
def test_row_major_few_rows(fmt, m, n, k, pad):
    import capi
    gen = torch.Generator().manual_seed(m * 7919 + n * 31 + k)
    groups = k // (32 if fmt == "mxfp4" else 16)
    stride = (groups + 3) // 4 * 4 + (4 if pad else 0)
    if k % 2048 == 0 and pad:
        stride = groups + 1   # (an odd stride: the general kernels)
    xq, wq = _codes(m, k, gen), _codes(n, k, gen)
    xs, ws = _scales(m, k, fmt, gen, stride), _scales(n, k, fmt, gen, stride)
    bias = torch.randn(n, generator=gen).to(torch.bfloat16) if pad else None
    y = capi.gemm(xq, xs, wq, ws, 0.01, fmt, bias)
    ref, mag = O.gemm_ref(xq, xs[:, :groups].contiguous(), wq, ws[:, :groups].contiguous(), 0.01, fmt)
    tol = 2.0 ** -8 * ref.abs() + 1e-5 * mag
    if bias is not None:   # added after the rounding to bf16: one rounding more
        ref = ref + bias.double()
        tol = tol + 2.0 ** -8 * ref.abs()
    err = (y.double() - ref).abs()
    assert (err <= tol).all(), f"{fmt} {m}x{n}x{k}: worst excess {float((err - tol).max())}"


def test_negative_e4m3_scales_keep_their_sign():
    import capi
    gen = torch.Generator().manual_seed(5)
    m, n, k = 20, 48, 800
    xq, wq = _codes(m, k, gen), _codes(n, k, gen)
    xs, ws = (_scales(r, k, "nvfp4", gen, 52) for r in (m, n))
    ws[::2, :] |= 0x80
    pos = capi.gemm(xq, xs, wq, ws & 0x7F, 0.01, "nvfp4")
    y = capi.gemm(xq, xs, wq, ws, 0.01, "nvfp4")
    assert torch.equal(y[:, ::2], -pos[:, ::2]) and torch.equal(y[:, 1::2], pos[:, 1::2])


@pytest.mark.parametrize("m,n,k", [(1, 48, 2048), (2, 48, 2048), (1, 1100, 4096), (1, 33, 8192), (1, 48, 480), (64, 48, 2048)])
def test_signed_e4m3_scales_match_the_oracle(m, n, k):
    """Up to 64 rows every kernel, the one-row ones too, takes a scale byte's sign."""
    import capi
    gen = torch.Generator().manual_seed(m + n + k)
    xq, wq = _codes(m, k, gen), _codes(n, k, gen)
    xs, ws = (_scales(r, k, "nvfp4", gen, k // 16) for r in (m, n))
    xs, ws = (s ^ (0x80 * torch.randint(0, 2, s.shape, dtype=torch.uint8, generator=gen)) for s in (xs, ws))
    y = capi.gemm(xq, xs, wq, ws, 0.01, "nvfp4")
    ref, mag = O.gemm_ref(xq, xs, wq, ws, 0.01, "nvfp4")
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * mag).all()
