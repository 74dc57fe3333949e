"""The native host path (csrc/fpq_host.cpp) gives the Python path's bits on every form of call that it accepts, declines
the others, and notices every change of what its plans were made from."""
import copy
import io
import threading

import pytest
import torch

from tests.conftest import SINGLE_WEIGHT_COPY, needs_packed, needs_row_major_parameters

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import fp_quant
    from fp_quant.module import eager, hip_ops, host
    from fp_quant.module import linear as linear_module


class _Declines:
    def __getattr__(self, name):
        return lambda *args: None


class _Counts:
    def __init__(self):
        self.answered = []

    def __getattr__(self, name):
        def call(*args):
            out = getattr(host.native, name)(*args)
            if out is not None and out is not False:
                self.answered.append(name)
            return out
        return call


@pytest.fixture
def native(monkeypatch):
    counts = _Counts()
    monkeypatch.setattr(linear_module, "_native", counts)
    return counts


def _python(layer, x, residual=None):
    """The layer's result through the Python path, without a shared quantization."""
    saved, linear_module._native = linear_module._native, _Declines()
    share, eager.SHARE_ACT_QUANT = eager.SHARE_ACT_QUANT, False
    try:
        layer.__dict__["_fpq_residual"] = residual
        return layer(x)
    finally:
        linear_module._native, eager.SHARE_ACT_QUANT = saved, share


def _layer(fmt="mxfp4", method="abs_max", init="hadamard", g=128, k=512, n=288, bias=False, seed=0):
    dtype = fp_quant.FPQuantDtype.MXFP4 if fmt == "mxfp4" else fp_quant.FPQuantDtype.NVFP4
    cfg = fp_quant.FPQuantConfig(forward_dtype=dtype, forward_method=method, backward_dtype=fp_quant.FPQuantDtype.BF16,
                                 hadamard_group_size=g, transform_init=init)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    layer = fp_quant.FPQuantLinear(k, n, cfg, bias=bias, device="cuda", dtype=torch.bfloat16)
    layer.weight.data = torch.randn(n, k, generator=gen, device="cuda", dtype=torch.bfloat16)
    if bias:
        layer.bias.data = torch.randn(n, generator=gen, device="cuda", dtype=torch.bfloat16)
    layer.pre_forward()
    return layer


FORMS = [("mxfp4", "abs_max", "hadamard", 128), ("mxfp4", "quest", "hadamard", 32), ("mxfp4", "abs_max", "identity", 64),
         ("mxfp4", "abs_max", "gsr", 128), ("mxfp4", "quest", "gsr", 128), ("mxfp4", "abs_max", "general", 64),
         ("nvfp4", "abs_max", "hadamard", 16), ("nvfp4", "abs_max", "gsr", 128), ("nvfp4", "abs_max", "general", 32)]


# (K = 640 stays on the row-major weight where weights are held once: nothing for native code)
@needs_packed
@pytest.mark.parametrize("fmt,method,init,g", FORMS)
@pytest.mark.parametrize("k", [512] if SINGLE_WEIGHT_COPY else [512, 640])
def test_linear_forms(fmt, method, init, g, k, native):
    general = init == "general"
    layer = _layer(fmt, method, "hadamard" if general else init, g, k, bias=True)
    if general:
        q, _ = torch.linalg.qr(torch.randn(g, g, generator=torch.Generator().manual_seed(1)))
        layer.forward_hadamard_matrix = torch.nn.Buffer(q.to(torch.bfloat16).contiguous().cuda())
    shapes = [(1, k), (33, k), (2, 3, k), (1, 1, 5, k), (130, k)]
    with torch.no_grad():
        layer(torch.randn(2, k, device="cuda", dtype=torch.bfloat16))   # the plans are made here
        for i, shape in enumerate(shapes):
            x = torch.randn(shape, device="cuda", dtype=torch.bfloat16)
            res = torch.randn(*shape[:-1], 288, device="cuda", dtype=torch.bfloat16)
            native.answered.clear()
            got = layer(x)
            assert native.answered == ["linear"] and layer._fpq_residual is None
            assert torch.equal(got, _python(layer, x)) and torch.equal(layer(x), got)   # (the second: shared)
            layer._fpq_residual = res
            assert torch.equal(layer(x), _python(layer, x, res)) and layer._fpq_residual is None


@needs_packed
def test_declined_calls(native, monkeypatch):
    layer = _layer(bias=True)
    x = torch.randn(6, 512, device="cuda", dtype=torch.bfloat16)
    layer(x)
    strided = torch.randn(512, 6, device="cuda", dtype=torch.bfloat16).t()
    for call in (x.float(), strided):
        native.answered.clear()
        assert torch.equal(layer(call), _python(layer, call)) and not native.answered
    native.answered.clear()
    xg = x.clone().requires_grad_()
    assert layer(xg).requires_grad and not native.answered
    with pytest.raises(Exception):
        layer(x[:, :256].contiguous())
    assert layer(x[:0]).shape == (0, 288)
    with torch.inference_mode():
        xi = x * 1.0
        assert torch.equal(layer(xi), _python(layer, x)) and native.answered == ["linear"]
        assert not eager._shared_activations or eager._shared_activations[0].ref() is not xi
    native.answered.clear()
    monkeypatch.setenv("FPQ_PACKED_WEIGHTS", "0")
    assert torch.equal(layer(x), _python(layer, x))
    assert native.answered == (["linear"] if layer.weights_packed_only else [])


@needs_packed
@needs_row_major_parameters   # (another layer's are loaded)
def test_plans_notice_changes(native):
    layer = _layer("nvfp4", g=16, k=512)
    x = torch.randn(40, 512, device="cuda", dtype=torch.bfloat16)
    layer(x), layer(x)
    other = _layer("nvfp4", g=16, k=512, seed=3)

    def check():
        want = _python(layer, x)
        for _ in range(3):
            assert torch.equal(layer(x), want)
        assert native.answered and native.answered[-1] == "linear"
        native.answered.clear()

    check()
    with torch.no_grad():
        layer.qweight.copy_(other.qweight)
        check()
        layer.scales.data = other.scales.data.clone()
        check()
        layer.act_global_scale.fill_(5.0)
        check()
        layer.weight_global_scale.fill_(20.0)
        check()
        layer.forward_hadamard_matrix.copy_(torch.eye(16))
        check()
        layer.bias = torch.nn.Parameter(torch.randn(288, device="cuda", dtype=torch.bfloat16))
        check()
        x.mul_(-2.0)
        check()
        layer.load_state_dict({**layer.state_dict(), "qweight": other.qweight.flip(0).contiguous()})
        check()
    assert layer.release_row_major()
    check()
    layer.restore_row_major()
    check()
    twin = copy.deepcopy(layer)
    assert torch.equal(twin(x), layer(x)) and torch.equal(twin(x), layer(x))
    buf = io.BytesIO()
    torch.save(layer, buf)
    buf.seek(0)
    loaded = torch.load(buf, weights_only=False)   # (written above)
    assert torch.equal(loaded(x), layer(x))


@needs_packed
@pytest.mark.parametrize("fmt,g", [("mxfp4", 64), ("nvfp4", 16)])
def test_streams_and_threads(fmt, g, native):
    """One layer that splits K (a workspace per stream) called from threads with a stream each."""
    layer = _layer(fmt, g=g, k=14336, n=512)
    xs = [torch.randn(8, 14336, device="cuda", dtype=torch.bfloat16) for _ in range(4)]
    want = [_python(layer, x) for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream), torch.no_grad():
            for _ in range(20):
                if not torch.equal(layer(xs[i]), want[i]):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad and "linear" in native.answered


@needs_packed
def test_source_of_a_shared_quantization_dies(native):
    layer = _layer()
    x = torch.randn(6, 512, device="cuda", dtype=torch.bfloat16)
    layer(x)
    y = torch.randn(6, 512, device="cuda", dtype=torch.bfloat16)
    native.answered.clear()
    layer(y)
    assert native.answered == ["linear"] and eager._shared_activations[0].ref() is y
    del y
    assert 0 not in eager._shared_activations


@pytest.mark.parametrize("fmt,m,n,k", [("mxfp4", 1, 72, 512), ("mxfp4", 47, 264, 288), ("mxfp4", 48, 264, 288),
                                       ("mxfp4", 200, 256, 512), ("nvfp4", 1, 72, 512), ("nvfp4", 64, 264, 288),
                                       ("nvfp4", 65, 264, 288), ("nvfp4", 200, 256, 512)])
def test_operators(fmt, m, n, k):
    """Operators called plainly and through the dispatcher (torch.ops): the same tensors; native code takes the plain calls."""
    mx = fmt == "mxfp4"
    w = torch.randn(n, k, device="cuda", dtype=torch.bfloat16)
    x = torch.randn(m, k, device="cuda", dtype=torch.bfloat16)
    gs = torch.full((1,), 3.0, device="cuda")
    alpha = torch.full((1,), 0.3, device="cuda")
    bias = torch.randn(n, device="cuda", dtype=torch.bfloat16)
    ops = torch.ops.fp_quant
    h = linear_module.get_hadamard_matrix(32, torch.bfloat16, torch.device("cuda"))

    def same(a, b):
        assert len(a) == len(b)
        for p, q in zip(a, b):
            assert (p is None and q is None) or (p.dtype == q.dtype and p.shape == q.shape
                                                 and torch.equal(p.view(torch.uint8), q.view(torch.uint8)))

    name = "mxf4" if mx else "nvf4"
    for _ in range(2):   # (the first call classifies the rotation and packs the weight)
        if mx:
            for method in ("abs_max", "quest"):
                same(hip_ops.fused_quantize_mx_op(x, h, method, False), ops.fused_quantize_mx_op(x, h, method, False))
            (qx, sx, _), (qw, sw, _) = (ops.fused_quantize_mx_op(t, h, "abs_max", False) for t in (x, w))
        else:
            same(hip_ops.fused_quantize_nv_op(x, h, gs), ops.fused_quantize_nv_op(x, h, gs))
            x3 = x.view(1, m, k)
            same(hip_ops.fused_quantize_nv_op(x3, h, gs), ops.fused_quantize_nv_op(x3, h, gs))
            (qx, sx), (qw, sw) = (ops.fused_quantize_nv_op(t, h, gs) for t in (x, w))
    for _ in range(2):
        same([getattr(hip_ops, f"matmul_{name}_bf16_tn_op")(qx, qw, sx, sw, alpha)],
             [getattr(ops, f"matmul_{name}_bf16_tn_op")(qx, qw, sx, sw, alpha)])
        same([getattr(hip_ops, f"matmul_{name}_bf16_tn_bias_op")(qx[None], qw, sx, sw, alpha, bias)],
             [getattr(ops, f"matmul_{name}_bf16_tn_bias_op")(qx[None], qw, sx, sw, alpha, bias)])
    native = host.native
    assert (native.quantize_mx(x, h, "abs_max", False) if mx else native.quantize_nv(x, h, gs)) is not None
    matmul = native.matmul_mx if mx else native.matmul_nv
    assert matmul(qx, qw, sx, sw, alpha) is not None and matmul(qx[None], qw, sx, sw, alpha, bias) is not None
    with pytest.raises(ValueError):
        getattr(hip_ops, f"matmul_{name}_bf16_tn_op")(qx, qw[:, : k // 4], sx, sw, alpha)
    with pytest.raises(ValueError):
        (hip_ops.fused_quantize_mx_op(x.float(), h, "abs_max", False) if mx else
         hip_ops.fused_quantize_nv_op(x.float(), h, gs))


@needs_packed
@pytest.mark.parametrize("fmt,g,kv", [("mxfp4", 64, 256), ("nvfp4", 64, 256), ("mxfp4", 64, 128)])
def test_fused_block_after_a_weight_changes(fmt, g, kv, monkeypatch):
    """The grouped projections of a fused block: a member that is written to, and a rotation that is replaced.  Native code
    answers every norm, group (but for widths that are no multiples of 256) and MLP, and the output projection."""
    from perf.cases import Block
    from fp_quant.utils import fuse_producers
    gen = torch.Generator(device="cuda").manual_seed(5)
    case = dict(fmt=fmt, g=g, hidden=512, kv=kv, inter=768)
    block = Block(case, gen)
    assert fuse_producers(block)
    x = torch.randn(1, 5, 512, device="cuda", dtype=torch.bfloat16)

    def run(native_path):
        saved = fuse._native_module, linear_module._native
        if not native_path:
            fuse._native_module = linear_module._native = _Declines()
            eager._shared_activations.clear()
        try:
            cache = []
            return [block(x, cache=cache), *cache[0]]
        finally:
            fuse._native_module, linear_module._native = saved

    import fp_quant.utils.fuse as fuse

    counts = _Counts()
    monkeypatch.setattr(fuse, "_native_module", counts)
    monkeypatch.setattr(linear_module, "_native", counts)

    def check():
        run(True)
        counts.answered.clear()
        got = run(True)
        # (such widths are column ranges of one matrix: the output projection's input is strided too)
        assert counts.answered == ["rmsnorm", *(["group", "linear"] if kv % 256 == 0 else []), "rmsnorm", "group", "gated_down"]
        for a, b in zip(got, run(False)):
            assert torch.equal(a, b)

    with torch.no_grad():
        check()
        block.self_attn.v_proj.qweight.bitwise_xor_(7)
        check()
        block.mlp.up_proj.scales.add_(1)
        check()
        block.mlp.down_proj.qweight.bitwise_xor_(3)
        check()
        for layer in (block.self_attn.q_proj, block.self_attn.k_proj, block.self_attn.v_proj):
            layer.forward_hadamard_matrix.copy_(linear_module.get_identity_matrix(64, torch.bfloat16, x.device))
        check()
        block.self_attn.q_proj.weight_global_scale.mul_(2)
        check()
        block.input_layernorm.weight.mul_(0.5)
        check()


def test_operators_are_recorded_by_a_jit_trace():
    x, other = (torch.randn(64, 512, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    layer = _layer("nvfp4", g=16, k=512)
    h, scale = layer.forward_hadamard_matrix, layer.act_global_scale.float()

    def quantize(v):
        return hip_ops.fused_quantize_nv_op(v, h, scale)

    quantize(x)
    traced = torch.jit.trace(quantize, (x,), check_trace=False)
    for got, want in zip(traced(other), quantize(other)):
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))


@needs_packed
def test_group_of_a_rewritten_weight_is_not_rebuilt_inside_a_capture():
    """A member written to, then the block recorded: calls outside the graph find no half-made group, and later ones
    rebuild it."""
    from perf.cases import Block
    from fp_quant.utils import fuse_producers
    gen = torch.Generator(device="cuda").manual_seed(6)
    block = Block(dict(fmt="mxfp4", g=64, hidden=512, kv=256, inter=768), gen)
    assert fuse_producers(block)
    x = torch.randn(1, 5, 512, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        block(x), block(x)
        block.self_attn.k_proj.qweight.bitwise_xor_(7)
        block.mlp.gate_proj.qweight.bitwise_xor_(5)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            cache = []
            outs = [block(x, cache=cache), *cache[0]]
        assert block.self_attn._fpq_weight_group is not None and block.mlp._fpq_weight_group is not None
        for i in range(3):
            cache = []
            want = [block(x, cache=cache), *cache[0]]
            if i:   # (the first call comes before any replay)
                graph.replay()
                torch.cuda.synchronize()
                for a, b in zip(outs, want):
                    assert torch.equal(a, b)
        assert block.self_attn._fpq_weight_group.key == tuple(
            eager._member_key(l.qweight, l.scales, l.bias)
            for l in (block.self_attn.q_proj, block.self_attn.k_proj, block.self_attn.v_proj))
    twin = copy.deepcopy(block.self_attn.k_proj)
    assert torch.equal(twin(x), block.self_attn.k_proj(x))


@needs_packed
@pytest.mark.parametrize("kv,fmt,g", [(128, "mxfp4", 64), (384, "mxfp4", 128), (128, "nvfp4", 16)])
def test_a_group_that_native_code_cannot_serve_is_asked_about_once(kv, fmt, g, monkeypatch):
    """Projections whose widths are no multiple of 256 share one output matrix, which only the Python path lays out."""
    from perf.cases import Block
    from fp_quant.utils import fuse_producers
    block = Block(dict(fmt=fmt, g=g, hidden=512, kv=kv, inter=768), torch.Generator(device="cuda").manual_seed(7))
    assert fuse_producers(block)
    learned, learn = [], host.learn_group
    monkeypatch.setattr(host, "learn_group", lambda group, layers: (learned.append(group), learn(group, layers)))
    x = torch.randn(1, 5, 512, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        block(x)
        for _ in range(4):
            block(x)
        qkv = block.self_attn._fpq_weight_group
        assert qkv is not None and sum(g is qkv for g in learned) <= 1
        block.self_attn.k_proj.qweight.bitwise_xor_(7)   # (another group now)
        for _ in range(4):
            block(x)
        assert len(learned) <= 4


def test_weights_that_cannot_be_in_a_plan_are_not_asked_about(native, monkeypatch):
    """Layers built under inference mode: native code declines at once, and nobody tries to make a plan."""
    from perf.cases import Block
    from fp_quant.utils import fuse_producers
    tried = []
    for name in ("learn_linear", "learn_quant", "learn_group"):
        monkeypatch.setattr(host, name, lambda *args, name=name: tried.append(name))
    with torch.inference_mode():
        for fmt, g in (("mxfp4", 128), ("nvfp4", 16)):
            layer = _layer(fmt, g=g, bias=True)
            for x in (torch.randn(6, 512, device="cuda", dtype=torch.bfloat16), torch.randn(6, 512).cuda().bfloat16()):
                assert torch.equal(layer(x), _python(layer, x))
            block = Block(dict(fmt=fmt, g=g, hidden=512, kv=256, inter=768), torch.Generator(device="cuda").manual_seed(8))
            assert fuse_producers(block)
            for _ in range(2):
                block(torch.randn(1, 5, 512, device="cuda", dtype=torch.bfloat16))
    assert not tried and not native.answered


@needs_packed
def test_a_layer_whose_plan_is_refused_gets_a_marker(native, monkeypatch):
    layer = _layer()
    x = torch.randn(6, 512, device="cuda", dtype=torch.bfloat16)
    alpha, learned, learn = host.linear_alpha, [], host.learn_linear
    monkeypatch.setattr(host, "linear_alpha", lambda *args: alpha(*args).expand(2))   # (no scalar: no plan takes it)
    monkeypatch.setattr(host, "learn_linear", lambda layer: (learned.append(layer), learn(layer)))
    for _ in range(4):
        assert torch.equal(layer(x), _python(layer, x))
    assert len(learned) == 1 and not native.answered


def test_calls_that_stay_on_the_row_major_weight_are_not_asked_about():
    """Fewer rows than FPQ_PACKED_MIN_ROWS, or FPQ_PACKED_WEIGHTS=0: nobody tries to make a plan."""
    import os
    import subprocess
    import sys
    code = """
import sys
sys.path[:0] = ["fp-quant_amd", "."]
import torch
from tests.test_host_path_gpu import _layer, host
from perf.cases import Block
from fp_quant.utils import fuse_producers
tried, learn = [], host.learn_linear
host.learn_linear = lambda layer: (tried.append(layer), learn(layer))
layer = _layer()
block = Block(dict(fmt="mxfp4", g=64, hidden=512, kv=256, inter=768), torch.Generator(device="cuda").manual_seed(7))
assert fuse_producers(block)
with torch.no_grad():
    for m in (4, 4, 4):
        layer(torch.randn(m, 512, device="cuda", dtype=torch.bfloat16))
        block(torch.randn(1, m, 512, device="cuda", dtype=torch.bfloat16))
    assert not tried, len(tried)
    if len(sys.argv) > 1:   # (rows that run on packed weights: planned after all)
        x = torch.randn(40, 512, device="cuda", dtype=torch.bfloat16)
        ys = [layer(x) for _ in range(4)]
        assert tried and all(torch.equal(y, ys[0]) for y in ys) and host.native.linear_plan_current(layer)
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    for env, args in (({"FPQ_PACKED_MIN_ROWS": "32"}, ["rows"]), ({"FPQ_PACKED_WEIGHTS": "0"}, [])):
        base = {k: v for k, v in os.environ.items() if k not in ("FPQ_PACKED_WEIGHTS", "FPQ_SINGLE_WEIGHT_COPY")}
        r = subprocess.run([sys.executable, "-c", code, *args], cwd=root, env={**base, **env}, capture_output=True,
                           text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
