"""MXFP4 with several weight tiles per workgroup of the weight-streaming kernel, K step by K step, against the oracle: two,
three and four weight tiles and up to three activation tiles in one round of the CUs; row slabs of two weight tiles by two,
three and four; every number of 256-K blocks that a wave's loop takes on a way of its own (none to six); an odd last weight
tile, groups of weight tiles that are no multiple of eight, a short last slab, N that ends inside a tile."""
import pytest
import torch

from oracle import fpq_oracle as O
import capi
from conftest import needs_packed
from test_few_rows_gpu import check_same_bits_as_two_kernels
from test_norm_rows_gpu import check_bits
from test_packed_gpu import pack_by_definition

pytestmark = [pytest.mark.gpu, needs_packed]

# 256 CUs: 257 to 512, 768, 1024 weight tiles of 32 are two, three, four per workgroup
ROWS = [(m, n, k) for m, n in ((5, 8200), (32, 16384), (33, 8296), (64, 16390), (96, 8264), (80, 16384),
                               (31, 16448), (64, 24576), (3, 24584), (40, 32768)) for k in (256, 1280, 2304, 3328, 4352, 6144)]
ROWS += [(16, 15360, 2048), (24, 32760, 4096), (24, 26000, 2048), (7, 24570, 4096)]   # one again, where that fills its rounds
FEW_ROWS = [(1, 256, 16392), (3, 768, 24584), (2, 2304, 16456), (1, 5120, 32768), (1, 256, 24680), (4, 4096, 16456),
            (1, 4096, 20488), (2, 5120, 16456)]
SLABS = [(129, 4104, 1024), (250, 4096, 1536), (463, 2200, 1280), (333, 4096, 1024), (160, 8192, 2048), (161, 8000, 1024),
         (700, 2048, 1280), (512, 4096, 8192), (257, 8100, 8448), (250, 8100, 8448), (400, 4000, 9984),
         (1100, 690, 1024), (200, 5390, 1024), (500, 2680, 1280), (600, 3190, 8192)]   # (the XCDs' rows of workgroups)


@pytest.mark.parametrize("m,n,k", ROWS + SLABS)
def test_against_the_oracle(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    xq = torch.randint(0, 256, (m, k // 2), dtype=torch.uint8, generator=g)
    wq = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, generator=g)
    xs = torch.randint(118, 134, (m, k // 32), dtype=torch.uint8, generator=g)
    ws = torch.randint(118, 134, (n, k // 32), dtype=torch.uint8, generator=g)
    xp, xsp = pack_by_definition(xq, xs, k)
    wp, wsp = pack_by_definition(wq, ws, k)
    bias = torch.randn(n, generator=g).to(torch.bfloat16) if k % 512 else None
    residual = torch.randn(m, n, generator=g).to(torch.bfloat16) if k % 512 and m % 2 else None
    y = capi.gemm_packed(xp, xsp, wp, wsp, m, n, k, 0.111328125, bias=bias, residual=residual)
    ref, mag = O.gemm_ref(xq, xs, wq, ws, 0.111328125, "mxfp4")
    want = ref.to(torch.bfloat16)
    big = want.double().abs()
    for add in (bias, residual):
        if add is not None:
            want = want + add
            big = torch.maximum(big, want.double().abs())
    # 2^-8 for each rounding to bf16 (up to three, of values no larger than `big`), twice that where a sum next to a tie
    # rounds the other way; 1e-5 of the sum of magnitudes for fp32 sums in another order
    tol = 2.0 ** -8 * 2 * (1 + (bias is not None) + (residual is not None)) * big + 1e-5 * mag + 1e-6
    assert ((y.double() - want.double()).abs() <= tol).all()


# A row's sums are those of a few rows by themselves wherever both are slabs (K in four parts, in one order)
@pytest.mark.parametrize("m,n,k", [(512, 2048, 768), (1000, 1000, 768), (256, 2790, 512), (256, 4090, 768),
                                   (24577, 32, 1024), (32740, 24, 1280)])
def test_bits_of_fewer_rows(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    xq, wq = (torch.randint(0, 256, (r, k // 2), dtype=torch.uint8, generator=g) for r in (m, n))
    xs, ws = (torch.randint(118, 134, (r, k // 32), dtype=torch.uint8, generator=g) for r in (m, n))
    w = pack_by_definition(wq, ws, k)
    few = capi.gemm_packed(*pack_by_definition(xq[:m // 4], xs[:m // 4], k), *w, m // 4, n, k, 0.111328125)
    assert torch.equal(capi.gemm_packed(*pack_by_definition(xq, xs, k), *w, m, n, k, 0.111328125)[:m // 4], few)


# 513 to 1024 weight tiles: two per workgroup that quantizes its rows itself or, where that does not pay, one: the bits of the
# two kernels.  One block per wave and up, in one pass and in two (4 x 4096)
@pytest.mark.parametrize("init,g", [("hadamard", 32), ("hadamard", 128), ("identity", 64)])
def test_few_rows(init, g):
    check_same_bits_as_two_kernels("mxfp4", init, g, False, FEW_ROWS)


@pytest.mark.parametrize("m,k,ns", [(1, 768, (16640,)), (4, 2048, (8448, 8192)), (2, 3328, (24832,)), (1, 4096, (14336, 14336)),
                                    (1, 768, (24832,)), (4, 2048, (16640, 8448)), (2, 4096, (16640,)), (1, 6144, (20480,))])
def test_few_rows_with_a_norm(m, k, ns):
    check_bits(0, m, k, ns, 0, 128, m % 2)
