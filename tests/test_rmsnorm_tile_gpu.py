"""RMSNorm, rotation and quantization of many rows in one pass (fpq_rmsnorm_tile_quantize_*_packed): the row statistic,
the normalised tensor and the packed codes and scales of the oracle, bit for bit."""
import pytest
import torch

from oracle import fpq_oracle as O
from tests import capi
from tests.conftest import make_student_t, needs_packed
from tests.test_ragged_k_gpu import _padded_pack

pytestmark = pytest.mark.gpu


# one row tile and its neighbours, a last row tile with a part of a workgroup's four rows; one 256-column block, rows
# that end inside a wave's last octet or inside a 256-K block, and both sides of the 4096 and 8192 columns at which a lane holds more octets
@pytest.mark.parametrize("fmt,rot,g", [("mxfp4", "hadamard", 128), ("mxfp4", "hadamard", 32), ("mxfp4", "identity", 32),
                                       ("nvfp4", "hadamard", 16), ("nvfp4", "hadamard", 128)])
@pytest.mark.parametrize("rows,cols", [(1, 256), (65, 768), (98, 4096), (35, 4352), (34, 8192), (5, 8448), (33, 16384), (70, 384), (37, 896)])
def test_rmsnorm_of_many_rows_in_one_pass_bit_exact(fmt, rot, g, rows, cols):
    x = make_student_t(rows, cols, seed=rows + g) * 2
    gen = torch.Generator().manual_seed(cols)
    w = (1 + 0.3 * torch.randn(cols, generator=gen)).to(torch.bfloat16)
    if rows > 4:
        w[64:96] = 0.0                    # zero groups
        x[3] *= 2.0 ** -60
        x[4] = 0.0                        # an all-zero row: 1 / sqrt(eps)
        w[128:160] *= 2.0 ** -110         # scales outside the range of the two-operation division
    want_v = O.rmsnorm(x, w, 1e-5)
    okind = O.ROT_HADAMARD if rot == "hadamard" else O.ROT_IDENTITY
    norm = float(O.hadamard_matrix(g)[0, 0])
    gs = None if fmt == "mxfp4" else 777.0
    if fmt == "mxfp4":
        wc, ws, _ = O.quantize_mx(want_v, okind, g, norm)
    else:
        wc, ws, _ = O.quantize_nv(want_v, gs, okind, g, norm)
    want_c, want_s = _padded_pack(wc, ws, cols, fmt == "nvfp4")
    ld = cols + 64 if rows in (5, 33, 98) else None
    pc, ps, out, inv = capi.rmsnorm_rows_quantize_packed(x, w, g=g, rot=rot, ld=ld, global_scale=gs, entry="tile")
    assert torch.equal(inv, O.row_inv_rms(x, 1e-5))
    assert torch.equal(out.view(torch.int16), want_v.view(torch.int16))
    assert torch.equal(pc, want_c) and torch.equal(ps, want_s)
    pc2, ps2, none, none2 = capi.rmsnorm_rows_quantize_packed(x, w, g=g, rot=rot, want_out=False, want_inv=False,
                                                              global_scale=gs, entry="tile")
    assert none is None and none2 is None and torch.equal(pc2, want_c) and torch.equal(ps2, want_s)


# both sides of every line: 64 and 640 rows, 8192 columns, 2^23 elements, a row that is no whole number of blocks
@needs_packed
@pytest.mark.parametrize("fmt,g", [("mxfp4", 128), ("nvfp4", 16)])
@pytest.mark.parametrize("rows,cols,two", [(64, 8448, False), (65, 8192, False), (65, 8448, True), (65, 8480, False),
                                           (512, 16384, True), (513, 16384, False), (640, 8448, True), (641, 8448, False)])
def test_wide_rows_take_the_statistic_in_a_launch_of_its_own(fmt, g, rows, cols, two, monkeypatch):
    """The fused norm where its rows are wide and few: two launches, the tile kernel's bits."""
    from fp_quant import _engine
    from fp_quant.module import eager, hip_ops, linear
    nv, cols = fmt == "nvfp4", cols + 96 if cols % g else cols
    x = (make_student_t(rows, cols, seed=rows) * 2).cuda()
    w = torch.randn(cols, device="cuda").to(torch.bfloat16)
    h = linear.get_hadamard_matrix(g, torch.bfloat16, x.device)
    gs = torch.full((1,), 3.0, device="cuda")
    lib, calls = _engine.lib(), []
    entry = lib.fpq_row_inv_rms
    monkeypatch.setattr(lib, "fpq_row_inv_rms", lambda *args: (calls.append(args), entry(*args))[1])
    y = eager.rmsnorm_quantize(x, w, 1e-5, h, gs, nv)
    if not hip_ops.packable_k(cols):   # (weights held once: the row-major forms)
        return
    assert len(calls) == two
    _, norm = hip_ops.classify_rotation(h)
    pc = torch.empty(lib.fpq_packed_codes_bytes(rows, cols), dtype=torch.uint8, device="cuda")
    ps = torch.empty((lib.fpq_packed_scales_bytes_nv if nv else lib.fpq_packed_scales_bytes)(rows, cols), dtype=torch.uint8,
                     device="cuda")
    out = torch.empty_like(x)
    head = (x.data_ptr(), cols, w.data_ptr(), rows, cols, 1e-5, _engine.ROT_HADAMARD, g, norm)
    tail = (None, out.data_ptr(), pc.data_ptr(), ps.data_ptr(), 0, hip_ops._current_stream(0))
    _engine.check(lib.fpq_rmsnorm_tile_quantize_nv_packed(*head, gs.data_ptr(), *tail) if nv
                  else lib.fpq_rmsnorm_tile_quantize_mx_packed(*head, *tail), "tile")
    qa = eager._shared_activations[0]
    assert torch.equal(y, out) and qa.ref() is y
    for a, b in zip(qa.packed(), (pc, ps)):
        assert torch.equal(a, b)
