"""RMSNorm joined to the projections that read it: fpq_norm_rows_multi (the norm of at most four rows inside the GEMM) gives
the bits of the norm's own kernel and the GEMM behind it, for rows that are finite and rows that are not; and a fused block
whose projections take the norm gives the bits of one that runs its norms, and runs them where somebody looks."""
import ctypes

import pytest
import torch

from tests.conftest import SINGLE_WEIGHT_COPY, needs_packed

pytestmark = pytest.mark.gpu


def check_bits(nv, m, k, ns, kind, g, bias):
    from fp_quant import _engine
    lib = _engine.lib()
    if not nv and g == 16:
        g = 32
    gen = torch.Generator().manual_seed(7 * m + k)
    x = torch.randn(m, k, generator=gen) * torch.logspace(-2, 2, m).view(-1, 1)
    x[:, ::57] *= 30
    n = sum(ns)
    wn = (1 + 0.1 * torch.randn(k, generator=gen)).bfloat16().cuda()
    scales_bytes = lib.fpq_packed_scales_bytes_nv if nv else lib.fpq_packed_scales_bytes
    wq = torch.randint(0, 256, (lib.fpq_packed_codes_bytes(n, k),), dtype=torch.uint8, generator=gen).cuda()
    low, high = (0x20, 0x58) if nv else (119, 127)
    ws = torch.randint(low, high, (scales_bytes(n, k),), dtype=torch.uint8, generator=gen).cuda()
    alpha, gs = torch.tensor([1e-2], device="cuda"), torch.tensor([12.5], device="cuda")
    b = torch.randn(n, generator=gen).bfloat16().cuda() if bias else None
    norm = float(torch.tensor(g ** -0.5, dtype=torch.bfloat16)) if kind == 0 else 1.0
    stream = torch.cuda.current_stream().cuda_stream
    c_ns = (ctypes.c_int64 * len(ns))(*ns)

    def outputs():
        ys = [torch.full((m, width), 7.0, dtype=torch.bfloat16, device="cuda") for width in ns]
        return ys, (ctypes.c_void_p * len(ns))(*(y.data_ptr() for y in ys))

    tail = (wq.data_ptr(), ws.data_ptr(), alpha.data_ptr(), None if b is None else b.data_ptr())
    for special in (None, 0.0, float("inf"), float("nan"), 1e38):
        if special is not None:
            x[0, 3] = special
            if special == 0.0:
                x[0] = 0.0
        xd = x.bfloat16().cuda()
        codes = torch.zeros(lib.fpq_packed_codes_bytes(m, k), dtype=torch.uint8, device="cuda")
        sc = torch.zeros(scales_bytes(m, k), dtype=torch.uint8, device="cuda")
        head = (xd.data_ptr(), k, wn.data_ptr(), m, k, 1e-5, kind, g, norm)
        outs = (None, None, codes.data_ptr(), sc.data_ptr(), 0, stream)
        _engine.check(lib.fpq_rmsnorm_rows_quantize_nv_packed(*head, gs.data_ptr(), *outs) if nv
                      else lib.fpq_rmsnorm_rows_quantize_mx_packed(*head, *outs), "norm")
        want, ptrs = outputs()
        multi = lib.fpq_gemm_nvf4_packed_multi if nv else lib.fpq_gemm_mxf4_packed_multi
        _engine.check(multi(codes.data_ptr(), sc.data_ptr(), *tail, ptrs, c_ns, len(ns), m, k, stream), "multi")
        got, ptrs = outputs()
        st = lib.fpq_norm_rows_multi(nv, xd.data_ptr(), wn.data_ptr(), 1e-5, m, k, kind, g, norm, gs.data_ptr() if nv else None,
                                     *tail, ptrs, c_ns, len(ns), 0, stream)
        if m * -(-k // 1024) * 8 > 64:   # more 32-element chunks than a wave holds
            assert st == _engine.E_UNSUPPORTED
            return
        _engine.check(st, "norm_rows_multi")
        for a, c in zip(got, want):
            assert torch.equal(a.view(torch.int16), c.view(torch.int16)), special


# (256, 512, 768: waves without a block; 4 x 2048 and 1 x 8192: as many chunks as a wave holds; 5120: blocks that the waves
# do not share evenly; 14336 columns: the GEMM's variant for many workgroups; 3 x 5120, 1 x 16384: refused)
@pytest.mark.parametrize("nv", [0, 1])
@pytest.mark.parametrize("m,k,ns,kind,g,bias", [
    (1, 256, (256,), 0, 128, 0), (4, 512, (256, 512), 0, 64, 1), (3, 768, (256, 256, 256), 0, 32, 0),
    (4, 2048, (512, 256), 1, 32, 1), (1, 4096, (4096, 1024, 1024), 0, 128, 0), (2, 4096, (14336,), 0, 16, 0),
    (2, 4096, (4096, 256), 0, 128, 1), (1, 8192, (512,), 0, 64, 0), (1, 5120, (1024, 256), 0, 128, 0), (3, 5120, (256,), 0, 64, 0), (1, 16384, (256,), 0, 128, 0),
])
def test_bits(nv, m, k, ns, kind, g, bias):
    check_bits(nv, m, k, ns, kind, g, bias)


def test_refusals():
    from fp_quant import _engine
    lib = _engine.lib()
    p = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda").data_ptr()

    def call(m=1, k=256, n=256, x=p, g=32, kind=0, policy=0, nv=0, y=p):
        return lib.fpq_norm_rows_multi(nv, x, p, 1e-5, m, k, kind, g, 0.1, None, p, p, p, None, (ctypes.c_void_p * 1)(y),
                                       (ctypes.c_int64 * 1)(n), 1, policy, None)
    assert call(m=5) == call(kind=_engine.ROT_GSR) == call(policy=1) == _engine.E_UNSUPPORTED
    assert call(k=128) == call(n=100) == -2 and call(x=None) == call(nv=1) == -1 and call(x=p + 2) == call(y=p + 8) == -4
    assert call(m=0) == 0


# (n: one weight tile, and on both sides of NVFP4's four tiles per CU)
@pytest.mark.parametrize("nv", [0, 1])
@pytest.mark.parametrize("m,k,n", [(1, 8192, 256), (1, 8448, 256), (2, 4096, 256), (2, 4352, 256), (3, 2048, 256), (3, 2304, 256),
                                   (4, 2048, 256), (4, 2304, 256), (4, 256, 256), (1, 384, 256), (5, 256, 256),
                                   (1, 1024, 32768), (1, 1024, 33024), (4, 1024, 33024)])
def test_rule_offers_what_the_kernel_takes(nv, m, k, n):
    from types import SimpleNamespace
    from fp_quant import FPQuantDtype, _engine
    from fp_quant.utils.fuse import _norm_bounds
    buffer = torch.zeros(48 << 20, dtype=torch.uint8, device="cuda")
    p = buffer.data_ptr()
    st = _engine.lib().fpq_norm_rows_multi(nv, p, p, 1e-5, m, k, 0, 32, 0.1, p, p, p, p, None, (ctypes.c_void_p * 1)(p + (32 << 20)),
                                           (ctypes.c_int64 * 1)(n), 1, 0, None)
    config = SimpleNamespace(forward_dtype=FPQuantDtype.NVFP4 if nv else FPQuantDtype.MXFP4)
    few, many = _norm_bounds([SimpleNamespace(in_features=k, out_features=n // 2, config=config, qweight=buffer,
                                              forward_hadamard_matrix=torch.eye(32, device="cuda").bfloat16())] * 2)
    assert (m * k <= few) == (st == 0) and few <= 4 * k < 64 * k <= many


@needs_packed
@pytest.mark.parametrize("fmt,g,init", [("mxfp4", 128, "hadamard"), ("nvfp4", 16, "identity"), ("mxfp4", 64, "gsr")])
@pytest.mark.parametrize("k,rows", [(2048, (1, 4, 5, 64, 65)), (8448, (1, 64, 65, 640, 641)), (16384, (1, 512, 513)), (1152, (1, 64, 65))])
def test_rule_offers_what_the_call_takes(fmt, g, init, k, rows):
    from fp_quant.utils import fuse
    from perf.cases import BlockRMSNorm, _linear
    if SINGLE_WEIGHT_COPY and k % 256 != 0:
        pytest.skip("ragged weights that are held in the packed layout only are no group")
    gen = torch.Generator(device="cuda").manual_seed(k)
    layers = tuple(_linear(dict(fmt=fmt, g=g, init=init), k, 256, False, gen) for _ in range(2))
    norm = BlockRMSNorm(k, gen)
    assert fuse.fuse_rmsnorm(norm, layers[0])
    group = fuse._weight_group(layers, create=True)
    few, many = fuse._norm_bounds(layers)
    with torch.no_grad():
        for m in rows:
            x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
            want = fuse._native_group(group, layers, norm(x))   # (the first makes the plans)
            outs = fuse._native_group(group, layers, x, norm)
            assert want is not None and (outs is None or all(torch.equal(a, b) for a, b in zip(outs, want)))
            assert (outs is not None) == (m * k <= few or m * k > many), m


@needs_packed
@pytest.mark.parametrize("fmt,g", [("mxfp4", 128), ("nvfp4", 16)])
@pytest.mark.parametrize("m,kv", [(1, 256), (4, 512), (65, 256), (600, 512), (2, 128), (70, 128)])
def test_block_bits(fmt, g, m, kv, monkeypatch):
    import fp_quant.utils.fuse as fuse
    from fp_quant.module import eager
    from perf.cases import Block
    block = Block(dict(fmt=fmt, g=g, hidden=512, kv=kv, inter=768), torch.Generator(device="cuda").manual_seed(m))
    assert fuse.fuse_producers(block)
    x = torch.randn(1, m, 512, device="cuda", dtype=torch.bfloat16)

    def run():
        cache = []
        with torch.no_grad():
            return [block(x, cache=cache), *cache[0]]
    run()
    joined = []
    hands_on = fuse._hands_on
    monkeypatch.setattr(fuse, "_hands_on", lambda *a: joined.append(hands_on(*a)) or joined[-1])
    got = run()
    assert joined == [True, True]
    monkeypatch.setattr(fuse, "_hands_on", lambda *a: False)
    eager._shared_activations.clear()
    for a, b in zip(got, run()):
        assert torch.equal(a, b)
    # somebody looks at a norm's output, or at what the readers are given: the norm runs, and they see it
    monkeypatch.setattr(fuse, "_hands_on", hands_on)
    seen = []
    handles = [block.input_layernorm.register_forward_hook(lambda mod, args, out: seen.append(out.clone())),
               block.mlp.register_forward_pre_hook(lambda mod, args: seen.append(args[0].clone()))]
    for a, b in zip(got, run()):
        assert torch.equal(a, b)
    want = block.input_layernorm._fpq_unfused_forward(x)
    assert len(seen) == 2 and (seen[0].float() - want.float()).norm() <= 1e-3 * want.float().norm()
    for handle in handles:
        handle.remove()
    block.post_attention_layernorm.forward = block.post_attention_layernorm._fpq_unfused_forward   # (another's patch)
    assert not hands_on(block.post_attention_layernorm, block.mlp) and hands_on(block.input_layernorm, block.self_attn)
