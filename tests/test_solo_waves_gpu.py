"""64 x 128 workgroup tiles of eight waves that multiply an eighth of K each: the oracle's values, bias and residual
included, and the same bits on every repetition.  NVFP4 from eight 256-K blocks on (one per wave; two for some and one for
the others; an odd number), MXFP4 where row slabs of the weight-streaming kernel fall behind (a long K with a short last slab or
with many slabs; the other MXFP4 shapes here are such slabs); rows and columns cut off inside the last tile."""
import pytest
import torch

from oracle import fpq_oracle as O
import capi
from test_packed_gpu import pack_by_definition
from test_tile_split_gpu import _operands
from test_tile_split_gpu import test_two_groups_per_workgroup_match_the_oracle as _matches_the_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(300, 4096, 3328), (257, 2750, 2304), (333, 2760, 7936), (129, 4100, 2048), (129, 8192, 3840),
                                   (511, 4090, 2560), (385, 2100, 4864), (512, 4096, 14336)])
def test_nvfp4_matches_the_oracle(m, n, k):
    _matches_the_oracle(m, n, k)


@pytest.mark.parametrize("m,n,k", [(129, 8190, 8192), (300, 4100, 8448), (512, 4096, 14336), (511, 2500, 10240), (1025, 1025, 8192),
                                   (257, 4000, 9984),
                                   # eight waves: 1 to 64 rows in the last slab, numbers of blocks that eight do and do not
                                   # divide; five slabs; six and seven that are no eights of groups of weight tiles; 14; 27 of 96 rows
                                   (385, 4090, 8448), (416, 4096, 10496), (448, 4000, 12544), (320, 5110, 12288), (600, 3190, 14592),
                                   (760, 2680, 8192), (833, 2300, 9984), (1700, 1020, 10240), (2500, 500, 8448)])
def test_mxfp4_matches_the_oracle(m, n, k):
    xq, _, wq, _, bias, res, g = _operands(m, n, k, m + n + k)
    xs = torch.randint(120, 131, (m, k // 32), dtype=torch.uint8, generator=g)
    ws = torch.randint(120, 131, (n, k // 32), dtype=torch.uint8, generator=g)
    wp, wsp = pack_by_definition(wq, ws, k)
    xp, xsp = pack_by_definition(xq, xs, k)
    alpha = 2.0 ** -8
    y = capi.gemm_packed_splitk(xp, xsp, wp, wsp, m, n, k, alpha, bias=bias, residual=res)
    ri = torch.cat([torch.tensor([0, 127, 128, m - 1]), torch.randperm(m, generator=g)[:40]]).unique()
    ci = torch.cat([torch.tensor([0, 63, 64, 127, 128, n - 1]), torch.randperm(n, generator=g)[:160]]).unique()
    ref, mag = O.gemm_ref(xq[ri], xs[ri], wq[ci], ws[ci], alpha, "mxfp4")
    want = (ref.to(torch.bfloat16) + bias[ci]) + res[ri][:, ci]
    got = y[ri][:, ci]
    tol = 2.0 ** -7 * torch.maximum(want.double().abs(), ref.abs()) + 2.0 ** -7 * res[ri][:, ci].double().abs() + 1e-5 * mag + 1e-6
    assert ((got.double() - want.double()).abs() <= tol).all()
    for _ in range(3):   # the parts are added in a fixed order
        again = capi.gemm_packed_splitk(xp, xsp, wp, wsp, m, n, k, alpha, bias=bias, residual=res)
        assert torch.equal(again.view(torch.int16), y.view(torch.int16))
