"""fpq_linear_rows (a few rows quantized by the GEMM itself) gives the bits of the quantizer and the GEMM it replaces:
one and two passes, blocks that some waves do not have, padded K, N that ends inside a tile, K split across workgroups,
groups that leave the fast division's range."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import fp_quant
    from fp_quant import _engine
    from fp_quant.module import eager, hip_ops, host
    from fp_quant.module import linear as linear_module

SHAPES = [(1, 256, 32), (3, 512, 72), (16, 1024, 40), (1, 4224, 520), (2, 640, 264), (4, 4096, 96), (2, 14336, 64),
          (1, 12800, 8224)]


def _layer(fmt, init, g, k, n, bias):
    dtype = fp_quant.FPQuantDtype.MXFP4 if fmt == "mxfp4" else fp_quant.FPQuantDtype.NVFP4
    cfg = fp_quant.FPQuantConfig(forward_dtype=dtype, forward_method="abs_max", backward_dtype=fp_quant.FPQuantDtype.BF16,
                                 hadamard_group_size=g, transform_init=init)
    gen = torch.Generator(device="cuda").manual_seed(k + n + g)
    layer = fp_quant.FPQuantLinear(k, n, cfg, bias=bias, device="cuda", dtype=torch.bfloat16)
    layer.weight.data = torch.randn(n, k, generator=gen, device="cuda", dtype=torch.bfloat16)
    if bias:
        layer.bias.data = torch.randn(n, generator=gen, device="cuda", dtype=torch.bfloat16)
    layer.pre_forward()
    return layer


def check_same_bits_as_two_kernels(fmt, init, g, silu, shapes):
    lib, nv = _engine.lib(), fmt == "nvfp4"
    for m, k, n in shapes:
        if k % g:
            continue
        layer = _layer(fmt, init, g, k, n, bias=m == 3)
        wp, wsp = hip_ops.packed_weight(layer.qweight, layer.scales, nv)
        alpha = eager.linear_alpha(layer.weight_global_scale, layer.act_global_scale)
        gs = eager.as_f32_scalar(layer.act_global_scale)
        kind, norm = hip_ops.classify_rotation(layer.forward_hadamard_matrix)
        x = torch.randn(m, k, device="cuda") * 4
        x[:, :32] = 0
        x[:, 64:96] *= 1e-34
        x[:, 128:160] *= 1e32
        x[-1, 197], x[0, 227] = float("nan"), float("inf")
        x = x.to(torch.bfloat16)
        up = torch.randn(m, k, device="cuda", dtype=torch.bfloat16) if silu else None
        res = torch.randn(m, n, device="cuda", dtype=torch.bfloat16)
        need = hip_ops.splitk_need(n, k, nv)
        ws = torch.zeros(need, dtype=torch.uint8, device="cuda") if need else None
        tail = (ws.data_ptr() if need else None, need, hip_ops._current_stream(0))
        bias = layer.bias.data_ptr() if layer.bias is not None else None
        a, b = hip_ops.quantize_mx_packed(x, layer.forward_hadamard_matrix) if not (nv or silu) else (
            torch.empty(lib.fpq_packed_codes_bytes(m, k), dtype=torch.uint8, device="cuda"),
            torch.empty((lib.fpq_packed_scales_bytes_nv if nv else lib.fpq_packed_scales_bytes)(m, k), dtype=torch.uint8,
                        device="cuda"))
        out = (a.data_ptr(), b.data_ptr(), 0, tail[2])
        if silu:
            head = (x.data_ptr(), k, up.data_ptr(), k, m, k, kind, g, norm)
            st = (lib.fpq_silu_mul_quantize_nv_packed(*head, gs.data_ptr(), None, *out) if nv
                  else lib.fpq_silu_mul_quantize_mx_packed(*head, None, *out))
            assert st == 0
        elif nv:
            assert lib.fpq_quantize_nv_packed_padded(x.data_ptr(), m, k, kind, g, norm, gs.data_ptr(), *out) == 0
        y, y2 = (torch.full((m, n), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(2))
        gemm = lib.fpq_gemm_nvf4_packed_splitk if nv else lib.fpq_gemm_mxf4_packed_splitk
        assert gemm(a.data_ptr(), b.data_ptr(), wp.data_ptr(), wsp.data_ptr(), alpha.data_ptr(), bias, res.data_ptr(),
                    y.data_ptr(), m, n, hip_ops.padded_k(k), *tail) == 0
        a2, b2 = torch.zeros_like(a), torch.zeros_like(b)
        st = lib.fpq_linear_rows(int(nv), x.data_ptr(), up.data_ptr() if silu else None, m, k, kind, g, norm, gs.data_ptr(),
                                 wp.data_ptr(), wsp.data_ptr(), alpha.data_ptr(), bias, res.data_ptr(), y2.data_ptr(), n,
                                 a2.data_ptr(), b2.data_ptr(), *tail[:2], 0, tail[2])
        # chunks of the wave with the most, with the whole of K in one workgroup (a split leaves fewer): one pass of 64, or,
        # but for SiLU*up, two
        if m * -(-(-(-k // 256)) // 4) * 8 > (64 if silu else 128) and st == _engine.E_UNSUPPORTED:
            continue
        assert st == 0, (m, k, n)
        assert torch.equal(y.view(torch.int16), y2.view(torch.int16)), (m, k, n)
        for p, q in zip(hip_ops.unpack_fp4(a, b, m, k, nv), hip_ops.unpack_fp4(a2, b2, m, k, nv)):
            assert torch.equal(p, q), (m, k, n)
        if need:
            assert not ws[:16384].any()   # the counters are back at zero


@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("fmt,init,g", [("mxfp4", "hadamard", 32), ("mxfp4", "hadamard", 64), ("mxfp4", "hadamard", 128),
                                        ("mxfp4", "identity", 32), ("nvfp4", "hadamard", 16), ("nvfp4", "hadamard", 128),
                                        ("nvfp4", "identity", 64)])
def test_same_bits_as_two_kernels(fmt, init, g, silu):
    check_same_bits_as_two_kernels(fmt, init, g, silu, SHAPES)


def test_refused_calls():
    lib = _engine.lib()
    layer = _layer("mxfp4", "hadamard", 128, 4096, 64, False)
    wp, wsp = hip_ops.packed_weight(layer.qweight, layer.scales)
    alpha = eager.linear_alpha(layer.weight_global_scale, layer.act_global_scale)
    x = torch.randn(64, 4096, device="cuda", dtype=torch.bfloat16)
    y = torch.zeros(64, 64, device="cuda", dtype=torch.bfloat16)

    def call(m=1, k=4096, kind=0, g=128, policy=0, at=0, w=wp.data_ptr()):
        return lib.fpq_linear_rows(0, x.data_ptr() + at, None, m, k, kind, g, 0.1, None, w, wsp.data_ptr(), alpha.data_ptr(),
                                   None, None, y.data_ptr(), 64, None, None, None, 0, policy, hip_ops._current_stream(0))

    assert call(m=5) == call(m=64) == call(kind=2) == call(kind=3) == call(policy=1) == call(at=2) == _engine.E_UNSUPPORTED
    assert call(g=24) == call(g=256) == _engine.E_UNSUPPORTED
    for bad in (call(m=0), call(k=0), call(k=40), call(k=-1), call(w=None), call(w=wp.data_ptr() + 1)):
        assert bad < 0 and bad != _engine.E_UNSUPPORTED
    torch.cuda.synchronize()
    assert not y.any()


@pytest.mark.parametrize("fmt,g", [("mxfp4", 128), ("nvfp4", 16)])
@pytest.mark.parametrize("k,n", [(4096, 256), (14336, 256)])
def test_layer_under_capture(fmt, g, k, n):
    """Replays of a captured layer follow new inputs; eager calls in between give the same bits."""
    layer = _layer(fmt, "hadamard", g, k, n, True)
    x = torch.randn(1, 1, k, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        layer(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layer(x)
        for i in range(4):
            x.copy_(torch.randn(1, 1, k, device="cuda", dtype=torch.bfloat16))
            want = layer(x.clone())
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want)
            saved, linear_module._native = linear_module._native, None
            assert torch.equal(layer(x.clone()), want)
            linear_module._native = saved
