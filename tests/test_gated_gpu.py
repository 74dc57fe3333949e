"""Gate and up projections whose GEMM forms, rotates and quantizes bf16(silu(gate)) * up in its epilogue: every byte as
from the GEMM into gate and up and the SiLU*up quantizer behind it (which the oracle checks), on every tile shape, at the
ends of row tiles, with every rotation, and with gates and products in every range: zero, below and above the lookup
table's, infinite, NaN, and groups outside the range of the two-operation division.  (Not compared: the codes of elements
that are NaN once rotated, and rotation blocks of finite products that come within a factor of three of the largest float.)"""
import ctypes

import pytest
import torch

from oracle import fpq_oracle as O
from tests.conftest import needs_packed

pytestmark = pytest.mark.gpu


def _operands(rows, k, nv, low, high, gen):
    from fp_quant import _engine
    lib = _engine.lib()
    codes = torch.randint(0, 256, (lib.fpq_packed_codes_bytes(rows, k),), dtype=torch.uint8, generator=gen)
    size = (lib.fpq_packed_scales_bytes_nv if nv else lib.fpq_packed_scales_bytes)(rows, k)
    return codes.cuda(), torch.randint(low, high, (size,), dtype=torch.uint8, generator=gen).cuda()


# (600: 256 x 128 tiles in both formats; 4096 x 2048: NVFP4's 256 x 256; 8300 x 256: two tiles of weights)
@pytest.mark.parametrize("nv", [0, 1])
@pytest.mark.parametrize("m,channels,k,rot,g,wide", [
    (600, 4096, 256, 0, 128, 0), (641, 4096, 768, 0, 64, 0), (1001, 2304, 512, 0, 32, 1), (4096, 2048, 256, 0, 16, 0),
    (3969, 2048, 1024, 0, 128, 1), (8300, 256, 512, 1, 32, 0), (527, 4352, 512, 0, 128, 1),
    (1001, 2304, 512, 1, 32, 1),
])
def test_gated_bytes(nv, m, channels, k, rot, g, wide):
    from fp_quant import _engine
    from fp_quant.module import hip_ops
    lib = _engine.lib()
    gen = torch.Generator().manual_seed(m + channels + k)
    low, high = (0x20, 0x58) if nv else (119, 127)
    x, w = _operands(m, k, nv, low, high, gen), _operands(2 * channels, k, nv, low, high, gen)
    if wide:   # a base scale for each row: gates from zero to infinity (NVFP4: to 10^5)
        rt, per = (m + 31) // 32, 8 if nv else 4
        base = torch.randint(0, 0x78 if nv else 248, (rt, 1, 64, 1), dtype=torch.uint8, generator=gen)
        x = x[0], (base + torch.randint(0, 7, (rt, k // 256, 64, per), dtype=torch.uint8, generator=gen)).flatten().cuda()
    else:
        x[1][:64] = 0 if nv else 20   # the first rows' products: zeros or tiny
    alpha = torch.tensor([1e-3 if nv else 0.02], device="cuda")
    gs = torch.tensor([12.5], device="cuda")
    norm = float(torch.tensor(g ** -0.5, dtype=torch.bfloat16)) if rot == 0 else 1.0
    stream = torch.cuda.current_stream().cuda_stream
    gate, up, product = (torch.empty(m, channels, dtype=torch.bfloat16, device="cuda") for _ in range(3))

    def outputs():
        size = (lib.fpq_packed_scales_bytes_nv if nv else lib.fpq_packed_scales_bytes)(m, channels)
        return (torch.full((lib.fpq_packed_codes_bytes(m, channels),), 0xA5, dtype=torch.uint8, device="cuda"),
                torch.full((size,), 0xA5, dtype=torch.uint8, device="cuda"))
    want, got = outputs(), outputs()
    operands = [t.data_ptr() for t in (*x, *w, alpha)]
    assert lib.fpq_gemm_packed_gated_takes(nv, m, channels, k) == 1
    multi = lib.fpq_gemm_nvf4_packed_multi if nv else lib.fpq_gemm_mxf4_packed_multi
    ys, ns = (ctypes.c_void_p * 2)(gate.data_ptr(), up.data_ptr()), (ctypes.c_int64 * 2)(channels, channels)
    _engine.check(multi(*operands, None, ys, ns, 2, m, k, stream), "multi")
    args = (gate.data_ptr(), channels, up.data_ptr(), channels, m, channels, rot, g, norm)
    if nv:
        st = lib.fpq_silu_mul_quantize_nv_packed(*args, gs.data_ptr(), product.data_ptr(), *(t.data_ptr() for t in want), 0, stream)
    else:
        st = lib.fpq_silu_mul_quantize_mx_packed(*args, product.data_ptr(), *(t.data_ptr() for t in want), 0, stream)
    _engine.check(st, "silu")
    _engine.check(lib.fpq_gemm_packed_gated(nv, *operands, m, channels, k, rot, g, norm, gs.data_ptr() if nv else None,
                                            *(t.data_ptr() for t in got), 0, stream), "gated")
    torch.cuda.synchronize()
    if wide and not nv:
        assert torch.isinf(gate).any() and (gate.float().abs() < 1e-5).any()
    # By rotation blocks.  Left out: those whose finite sums may overflow on the way in one order of additions and not in
    # another.  What comes out of the rotation as NaN (whose code takes its sign, or is zero where its wave takes the slow
    # division) has no code to compare; everything else has.
    per = max(g, 32)
    blocks = product.cpu().double().view(m, channels // per, per)
    finite = blocks.isfinite().all(-1)
    compared = ~finite | (blocks.abs().sum(-1) < 1e38)
    turned = blocks if rot == 1 else (blocks.view(m, -1, g) @ O.hadamard_matrix(g).double()).view_as(blocks)
    assert compared.any() and (wide or compared.all() and finite.all())
    (wc, ws_), (gc, gs_) = ([t.cpu().view(m, channels // per, -1) for t in hip_ops.unpack_fp4(*o, m, channels, bool(nv))]
                            for o in (want, got))
    assert torch.equal(gs_[compared], ws_[compared])
    known = ~turned.isnan() & compared.unsqueeze(-1)
    gn, wn = (torch.stack((c & 15, c >> 4), -1).view_as(turned) for c in (gc, wc))
    assert torch.equal(gn[known], wn[known])
    quiet = compared & finite
    if quiet.all():   # the padding too
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_refusals():
    from fp_quant import _engine
    lib = _engine.lib()
    t = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    p = t.data_ptr()

    def call(m=600, channels=4096, k=256, rot=0, g=128, policy=0, codes=p):
        return lib.fpq_gemm_packed_gated(0, p, p, p, p, p, m, channels, k, rot, g, 0.1, None, codes, p, policy, None)
    assert call(m=64) == _engine.E_UNSUPPORTED and not lib.fpq_gemm_packed_gated_takes(0, 64, 4096, 256)
    assert call(channels=4128) == call(rot=2) == call(g=256) == call(policy=1) == _engine.E_UNSUPPORTED
    assert call(k=100) == -2 and call(m=-1) == -2 and call(codes=None) == -1 and call(codes=p + 8) == -4 and call(m=0) == 0


# More than 16384 channels: a single row tile is large tiles to the tile kernels, but up to 96 rows (MXFP4: 64) the GEMM that
# would be replaced streams its weights, in another order of sums.
@pytest.mark.parametrize("nv,m,channels,taken", [
    (0, 1, 20480, 0), (0, 64, 16640, 0), (0, 65, 16640, 1), (0, 97, 16640, 1), (0, 128, 16640, 1),
    (1, 1, 20480, 0), (1, 64, 16640, 0), (1, 65, 16640, 0), (1, 96, 20480, 0), (1, 97, 16640, 1), (1, 128, 16640, 1),
])
def test_few_rows_of_many_channels(nv, m, channels, taken):
    from fp_quant import _engine
    lib = _engine.lib()
    assert lib.fpq_gemm_packed_gated_takes(nv, m, channels, 512) == taken
    if taken:
        return test_gated_bytes(nv, m, channels, 512, 0, 128, 0)
    p = torch.zeros(1 << 10, dtype=torch.uint8, device="cuda").data_ptr()   # (nothing is launched)
    assert lib.fpq_gemm_packed_gated(nv, p, p, p, p, p, m, channels, 512, 0, 128, 0.1, p, p, p, 0, None) == _engine.E_UNSUPPORTED


@pytest.mark.parametrize("nv,m,channels", [(0, 129, 8448), (0, 97, 16640), (0, 130, 16640), (1, 129, 8448)])
def test_long_inner_dimension(nv, m, channels):
    """K = 8192: MXFP4 at most one workgroup per CU (a ring of eight units), and more."""
    test_gated_bytes(nv, m, channels, 8192, 0, 128, 0)


@needs_packed
@pytest.mark.parametrize("fmt,g,m", [("mxfp4", 128, 1037), ("mxfp4", 32, 2048), ("nvfp4", 16, 1037)])
def test_fused_block_runs_the_gated_gemm(fmt, g, m, monkeypatch):
    """A block of enough rows takes it on its second call (the first makes the plans), with the bits of the separate
    kernels; a weight that is written to is noticed; replays of a recorded call give the same."""
    from perf.cases import Block
    from fp_quant.utils import fuse, fuse_producers
    block = Block(dict(fmt=fmt, g=g, hidden=512, kv=256, inter=2048), torch.Generator(device="cuda").manual_seed(3))
    assert fuse_producers(block)
    x = torch.randn(1, m, 512, device="cuda", dtype=torch.bfloat16)
    native, taken = fuse._native(), []

    class Counts:
        def __getattr__(self, name):
            def call(*args):
                out = getattr(native, name)(*args)
                if name == "gated_mlp" and out is not None:
                    taken.append(name)
                return out
            return call

    class Apart(Counts):
        gated_mlp = staticmethod(lambda *args: None)

    def run(how):
        monkeypatch.setattr(fuse, "_native_module", how())
        return block(x)

    with torch.no_grad():
        run(Counts)
        for change in (lambda: None, lambda: block.mlp.up_proj.qweight.bitwise_xor_(7),
                       lambda: block.mlp.down_proj.scales.add_(1)):
            change()
            for _ in range(2):   # (the group, then its plan are made anew)
                run(Counts)
            taken.clear()
            got = run(Counts)
            assert taken == ["gated_mlp"]
            assert torch.equal(got, run(Apart))
        run(Counts)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = run(Counts)
        for seed in range(3):
            x.normal_(generator=torch.Generator(device="cuda").manual_seed(seed))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, run(Apart))
