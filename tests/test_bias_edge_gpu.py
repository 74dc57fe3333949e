"""The bias on the last row and column of tiles, where the epilogue fetches it with clamped columns: bf16(bf16(alpha * sum)
+ bias) of the product without a bias, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv", (False, True))
@pytest.mark.parametrize("offset", (0, 1))   # the bias 8-byte aligned, or not
@pytest.mark.parametrize("m,n", [(1, 33), (40, 31), (130, 257), (333, 8640), (333, 8643), (1100, 2049), (1100, 2052), (4100, 8198)])
def test_bias_on_edge_tiles(m, n, offset, nv):
    from fp_quant import _engine
    lib, k = _engine.lib(), 256
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    rand = lambda low, high, size: torch.randint(low, high, (size,), generator=gen, device="cuda", dtype=torch.uint8)
    scales = lambda rows: (rand(40, 72, lib.fpq_packed_scales_bytes_nv(rows, k)) if nv
                           else rand(124, 130, lib.fpq_packed_scales_bytes(rows, k)))
    xq, wq = (rand(0, 256, lib.fpq_packed_codes_bytes(r, k)) for r in (m, n))
    xs, ws = scales(m), scales(n)
    alpha = torch.full((1,), 0.01, device="cuda")
    bias = (torch.randn(n + offset, generator=gen, device="cuda") * 3).to(torch.bfloat16)[offset:]
    entry = lib.fpq_gemm_nvf4_packed if nv else lib.fpq_gemm_mxf4_packed
    plain, got = (torch.empty(m, n, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    stream = torch.cuda.current_stream().cuda_stream
    for b, y in ((None, plain), (bias.data_ptr(), got)):
        assert entry(xq.data_ptr(), xs.data_ptr(), wq.data_ptr(), ws.data_ptr(), alpha.data_ptr(), b, y.data_ptr(), m, n, k,
                     stream) == 0
    assert torch.equal(got.view(torch.int16), (plain + bias).view(torch.int16))
