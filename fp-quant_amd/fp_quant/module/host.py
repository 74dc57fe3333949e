"""Plans of the native host path (csrc/fpq_host.cpp): what the Python path of eager.py works out once per layer,
handed to native code that repeats the call without the interpreter.  A plan hangs on the tensor it describes
(`_fpq_qplan` on a rotation, `_fpq_plan` on a layer's codes, `plan` of a WeightGroup), names the tensors it was made
from, and is compared with them on every call.  Plans are made outside tracing and captures, by the first call that
could have used them; a layer or group that the native path cannot serve gets a marker, so that it is not asked again.
(Native code declines by itself where a tensor cannot be in a plan: inference tensors, tensor subclasses.)"""
import torch

from .. import _engine
from . import eager, hip_ops
from .eager import as_f32_scalar, cached_on, linear_alpha

native = eager._host


def _plain(*tensors) -> bool:
    return all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda and not t.is_inference() for t in tensors)


def learnable() -> bool:
    return (native is not None and not torch.compiler.is_compiling()
            and not torch.cuda.is_current_stream_capturing())


def learn_quant(h, act_global_scale, nvfp4: bool) -> None:
    """The QuantPlan of the rotation `h` with this activation scale."""
    if not _plain(h, act_global_scale) or native.quant_plan_current(h, act_global_scale, nvfp4):
        return
    kind, norm = hip_ops.classify_rotation(hip_ops.as_bf16(h))
    g = h.shape[0]
    rot = (kind, norm, g) if kind != _engine.ROT_GENERAL else (kind, id(h), hip_ops._version(h))
    if h.dtype != torch.bfloat16 or not h.is_contiguous():
        kind = -1    # (a marker: called on a converted copy)
    gs = gs_host = None
    if nvfp4 and kind >= 0:
        gs = as_f32_scalar(act_global_scale)
        if eager.SHARE_ACT_QUANT:
            gs_host = cached_on(act_global_scale, "_fpq_host",
                                (hip_ops._version(act_global_scale), act_global_scale.data_ptr()),
                                lambda: float(act_global_scale))
    plan = native.quant_plan(h, act_global_scale, nvfp4, kind, norm, g, gs, rot, gs_host)
    h._fpq_qplan = plan or native.quant_plan(h, act_global_scale, nvfp4, -1, norm, g, None, rot, None)


def learn_linear(layer) -> None:
    """The plans of an FPQuantLinear, and what they hold: its packed weight, alpha, fp32 activation scale."""
    q, s, h = layer.qweight, layer.scales, layer.forward_hadamard_matrix
    wgs, ags, bias = layer.weight_global_scale, layer.act_global_scale, layer.bias
    nvfp4 = layer.config.forward_dtype == hip_ops.FPQuantDtype.NVFP4
    if not _plain(q, s, h, wgs, ags) or (bias is not None and not _plain(bias)):
        return
    learn_quant(h, ags, nvfp4)
    if native.linear_plan_current(layer):
        return
    n, k = layer.out_features, layer.in_features
    packed_only = hip_ops.is_packed_only(q)
    packed = getattr(q, "_fpq_packed", None)
    usable = (q.dtype == torch.uint8 and s.dtype == torch.uint8 and q.is_contiguous() and s.is_contiguous()
              and hip_ops.packable_k(k)
              and (bias is None or (bias.dtype == torch.bfloat16 and bias.is_contiguous() and bias.numel() == n)))
    if usable and packed_only:
        usable = hip_ops.weight_rows(q, k) == n
    elif usable:
        usable = q.shape == (n, k // 2)
        if usable and not hip_ops.packed_weight_ready(q, s, nvfp4):
            if not hip_ops.packed_weights_enabled() or (not nvfp4 and hip_ops.PACKED_LINEAR_MIN_M > 1):
                return    # (the layer may get its packed copy later)
            with hip_ops.on_device(q.device):
                hip_ops.packed_weight(q, s, nvfp4)
            packed = q._fpq_packed
    alpha = linear_alpha(wgs, ags)
    need = hip_ops.splitk_need(n, k, nvfp4) if usable else 0
    args = (q, s, wgs, ags, bias, alpha, None if packed_only else packed, n, k, need,
            hip_ops.SPLIT_K_MAX_ROWS if nvfp4 else hip_ops.SPLIT_K_ROWS,
            hip_ops.NV_PACKED_LINEAR_MIN_M if nvfp4 else hip_ops.PACKED_LINEAR_MIN_M, nvfp4, packed_only)
    q._fpq_plan = native.linear_plan(*args, usable) or native.linear_plan(*args, False)


def learn_group(group, layers) -> None:
    """The GroupPlan of a WeightGroup that holds `layers`."""
    first = layers[0]
    wgs, ags, h = first.weight_global_scale, first.act_global_scale, first.forward_hadamard_matrix
    if (not _plain(wgs, ags, h) or len(layers) != len(group.splits)
            or group.key != tuple(eager._member_key(l.qweight, l.scales, l.bias) for l in layers)):
        return    # (written to since the group was built: the Python path builds it anew)
    learn_quant(h, ags, group.nvfp4)
    alpha = linear_alpha(wgs, ags)
    key = (group.key, hip_ops._version(wgs), wgs.data_ptr(), hip_ops._version(ags), ags.data_ptr(), id(alpha))
    if group.plan_key == key:
        return
    group.plan = None
    members = tuple(t for l in layers for t in (l.qweight, l.scales, l.bias))
    if len(layers) <= 4 and _plain(*(t for t in members if t is not None)):
        # (a matrix of its own per layer needs whole 256-column tiles)
        args = (members, tuple(group.splits), wgs, ags, alpha, group.wp, group.wsp, group.bias, group.k, group.nvfp4)
        group.plan = (native.group_plan(*args, all(n % 256 == 0 for n in group.splits))
                      or native.group_plan(*args, False))
    group.plan_key = key
