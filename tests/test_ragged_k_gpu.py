"""Inner dimensions that are a multiple of 32 but not of 256: the packed operands are padded to whole 256-K blocks with
zero codes and scale bytes, and the packed kernels multiply them."""
import pytest
import torch

import fp_quant
from fp_quant import _engine
from fp_quant.module import eager, hip_ops
from oracle import fpq_oracle as O
from tests import capi
from tests.conftest import SINGLE_WEIGHT_COPY, make_student_t, needs_packed
from tests.test_packed_gpu import pack_by_definition, pack_nv_by_definition

pytestmark = pytest.mark.gpu


def _padded_pack(codes, scales, k, nv):
    kp = (k + 255) // 256 * 256
    group = 16 if nv else 32
    codes = torch.nn.functional.pad(codes, (0, (kp - k) // 2))
    scales = torch.nn.functional.pad(scales[:, : k // group], (0, (kp - k) // group))
    return (pack_nv_by_definition if nv else pack_by_definition)(codes, scales, kp)


def _quantize_padded(x, kind, rot, g, gs):
    lib = _engine.lib()
    rows, cols = x.shape
    xd = x.cuda()
    scales = lib.fpq_packed_scales_bytes_nv if kind == "nv" else lib.fpq_packed_scales_bytes
    pc = torch.full((lib.fpq_packed_codes_bytes(rows, cols),), 0xCD, dtype=torch.uint8, device="cuda")
    ps = torch.full((scales(rows, cols),), 0xCD, dtype=torch.uint8, device="cuda")
    norm = float(torch.tensor(g ** -0.5, dtype=torch.bfloat16))
    st = torch.cuda.current_stream().cuda_stream
    if kind == "nv":
        gsd = torch.tensor([gs], dtype=torch.float32, device="cuda")
        rc = lib.fpq_quantize_nv_packed_padded(xd.data_ptr(), rows, cols, capi.ROT[rot], g, norm, gsd.data_ptr(),
                                               pc.data_ptr(), ps.data_ptr(), 0, st)
    else:
        rc = lib.fpq_quantize_mx_packed_padded(xd.data_ptr(), rows, cols, int(kind == "quest"), capi.ROT[rot], g, norm,
                                               pc.data_ptr(), ps.data_ptr(), 0, st)
    _engine.check(rc, "padded")
    torch.cuda.synchronize()
    return pc.cpu(), ps.cpu()


# generic kernel (up to 64 rows) and tile kernel; a row shorter than a block, one chunk and all but one chunk of the last
@pytest.mark.parametrize("kind", ["mx", "quest", "nv"])
@pytest.mark.parametrize("rot,g", [("hadamard", 128), ("hadamard", 32), ("identity", 32), ("gsr", 32)])
@pytest.mark.parametrize("rows,cols", [(1, 384), (33, 128), (65, 384), (70, 3200), (131, 896)])
def test_padded_quantizers_bit_exact(kind, rot, g, rows, cols):
    x = make_student_t(rows, cols, seed=rows + g) * 2
    if rows > 4:
        x[3] *= 2.0 ** -120
        x[4] = 0.0
    okind = {"hadamard": O.ROT_HADAMARD, "identity": O.ROT_IDENTITY, "gsr": O.ROT_GSR}[rot]
    norm = float(O.hadamard_matrix(g)[0, 0])
    gs = 777.0
    if kind == "mx":
        c, s, _ = O.quantize_mx(x, okind, g, norm)
    elif kind == "quest":
        c, s = O.quantize_mx_quest(x, okind, g, norm)[:2]
    else:
        c, s, _ = O.quantize_nv(x, gs, okind, g, norm)
    want = _padded_pack(c, s, cols, kind == "nv")
    got = _quantize_padded(x, kind, rot, g, gs)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("nv", [False, True])
@pytest.mark.parametrize("rows,k", [(5, 32), (33, 288), (64, 480), (40, 3200)])
def test_pack_and_unpack(nv, rows, k):
    gen = torch.Generator().manual_seed(k)
    group = 16 if nv else 32
    codes = torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, generator=gen).cuda()
    scales = torch.randint(1, 120, (rows, k // group), dtype=torch.uint8, generator=gen).cuda()
    pc, ps = (hip_ops.pack_nvf4 if nv else hip_ops.pack_mxf4)(codes, scales, rows, k)
    want = _padded_pack(codes.cpu(), scales.cpu(), k, nv)
    assert torch.equal(pc.cpu(), want[0]) and torch.equal(ps.cpu(), want[1])
    back = hip_ops.unpack_fp4(pc, ps, rows, k, nv)
    assert torch.equal(back[0], codes) and torch.equal(back[1], scales)


# the weight-streaming kernel, its row slabs and the tile kernels; gsr 64 beyond 64 rows is quantized row-major and re-tiled
@needs_packed
@pytest.mark.parametrize("fmt,method,init,g", [("mxfp4", "abs_max", "hadamard", 128), ("mxfp4", "quest", "hadamard", 64),
                                               ("nvfp4", "abs_max", "hadamard", 16), ("mxfp4", "abs_max", "gsr", 64)])
@pytest.mark.parametrize("m,k,n", [(1, 384, 200), (48, 3200, 96), (90, 896, 520), (300, 640, 1056)])
def test_layer_matches_the_oracle(fmt, method, init, g, m, k, n):
    cfg = fp_quant.FPQuantConfig(forward_dtype=fp_quant.FPQuantDtype(fmt), forward_method=method,
                                 backward_dtype=fp_quant.FPQuantDtype.BF16, hadamard_group_size=g, transform_init=init)
    torch.manual_seed(m + k)
    layer = fp_quant.FPQuantLinear(k, n, cfg, bias=True, device="cuda", dtype=torch.bfloat16)
    layer.weight.data.normal_(0, 0.02)
    layer.bias.data.normal_()
    layer.pre_forward()
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        y = layer(x)
    assert (getattr(layer.qweight, "_fpq_packed", None) is None) == SINGLE_WEIGHT_COPY
    okind = O.ROT_GSR if init == "gsr" else O.ROT_HADAMARD
    norm = float(O.hadamard_matrix(g)[0, 0])
    if fmt == "nvfp4":
        xc, xs, _ = O.quantize_nv(x.cpu(), 3.0, okind, g, norm)
    elif method == "quest":
        xc, xs = O.quantize_mx_quest(x.cpu(), okind, g, norm)[:2]
    else:
        xc, xs, _ = O.quantize_mx(x.cpu(), okind, g, norm)
    alpha = float((1.0 / (layer.weight_global_scale * layer.act_global_scale)).float())
    ref, mag = O.gemm_ref(xc, xs, layer.qweight.cpu(), layer.scales.cpu(), alpha, fmt)
    bias = layer.bias.detach().cpu()
    # the GEMM's bound (one bf16 rounding and fp32 sums), then the bias' bf16 addition: one more rounding of the result
    want = ref + bias.double()
    tol = 2.0 ** -8 * ref.abs() + 1e-5 * mag + 2.0 ** -8 * want.abs() + 1e-6
    assert ((y.cpu().double() - want).abs() <= tol).all()


# (K = 512: a whole number of blocks)
@needs_packed
@pytest.mark.parametrize("fmt,g", [("mxfp4", 128), ("nvfp4", 16)])
@pytest.mark.parametrize("k", [640, 512])
def test_packed_weights_made_inside_a_capture_stay_there(fmt, g, k, monkeypatch):
    """A layer whose first call is recorded into a graph: what the recording packs is not there before a replay, so
    calls outside the graph pack for themselves; replays follow the row-major weight."""
    monkeypatch.setattr(eager, "SHARE_ACT_QUANT", False)   # (NVFP4 reads the activation scale on the host to share)
    cfg = fp_quant.FPQuantConfig(forward_dtype=fp_quant.FPQuantDtype(fmt), forward_method="abs_max",
                                 backward_dtype=fp_quant.FPQuantDtype.BF16, hadamard_group_size=g)

    def layer(seed):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        out = fp_quant.FPQuantLinear(k, 288, cfg, bias=False, device="cuda", dtype=torch.bfloat16)
        out.weight.data = torch.randn(288, k, generator=gen, device="cuda", dtype=torch.bfloat16)
        out.pre_forward()
        return out

    captured, x = layer(1), torch.randn(4, k, device="cuda", dtype=torch.bfloat16)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad():
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            y = captured(x)
        want = layer(1)(x)
        assert torch.equal(captured(x), want)
        for seed in (1, 2, 2):
            if captured.qweight.dim() == 2:
                captured.qweight.copy_(layer(seed).qweight)
                captured.scales.copy_(layer(seed).scales)
                want = layer(seed)(x)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want) and torch.equal(captured(x), want)


@needs_packed
@pytest.mark.parametrize("fmt,g", [("mxfp4", 128), ("nvfp4", 16)])
def test_ragged_weights_are_held_once_where_asked_for(fmt, g, monkeypatch):
    """FPQ_SINGLE_WEIGHT_COPY=1: a weight that cannot be held in the packed layout only gets no packed copy next to it,
    in layers, fused blocks' groups and operators; its results are those of the row-major kernels."""
    monkeypatch.setenv("FPQ_SINGLE_WEIGHT_COPY", "1")
    monkeypatch.setattr(eager, "SHARE_ACT_QUANT", False)
    nv = fmt == "nvfp4"
    layers = []
    for i in range(2):
        cfg = fp_quant.FPQuantConfig(forward_dtype=fp_quant.FPQuantDtype(fmt), forward_method="abs_max",
                                     backward_dtype=fp_quant.FPQuantDtype.BF16, hadamard_group_size=g)
        gen = torch.Generator(device="cuda").manual_seed(i)
        layers.append(fp_quant.FPQuantLinear(640, 96, cfg, bias=False, device="cuda", dtype=torch.bfloat16))
        layers[-1].weight.data = torch.randn(96, 640, generator=gen, device="cuda", dtype=torch.bfloat16)
        layers[-1].pre_forward()
    assert eager.weight_group([(l.qweight, l.scales, None, 640) for l in layers], True, nv) is None
    layer = layers[0]
    alpha = (1.0 / (layer.weight_global_scale * layer.act_global_scale)).float()
    for rows in (1, 70, 300):
        x = torch.randn(rows, 640, device="cuda", dtype=torch.bfloat16)
        with torch.no_grad():
            y = layer(x)
            if nv:
                codes, scales = hip_ops.fused_quantize_nv_op(x, layer.forward_hadamard_matrix, layer.act_global_scale.float())
                op = hip_ops.matmul_nvf4_bf16_tn_op
            else:
                codes, scales, _ = hip_ops.fused_quantize_mx_op(x, layer.forward_hadamard_matrix, "abs_max", False)
                op = hip_ops.matmul_mxf4_bf16_tn_op
            out = op(codes, layer.qweight, scales, layer.scales, alpha)
            monkeypatch.setenv("FPQ_PACKED_WEIGHTS", "0")
            want = op(codes, layer.qweight, scales, layer.scales, alpha)
            monkeypatch.delenv("FPQ_PACKED_WEIGHTS")
        assert torch.equal(y, want) and torch.equal(out, want)
        assert not hasattr(layer.qweight, "_fpq_packed") and layer.qweight.dim() == 2
