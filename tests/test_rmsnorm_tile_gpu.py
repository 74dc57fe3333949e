"""RMSNorm, rotation and quantization of many rows in one pass (fpq_rmsnorm_tile_quantize_*_packed): the row statistic,
the normalised tensor and the packed codes and scales of the oracle, bit for bit."""
import pytest
import torch

from oracle import fpq_oracle as O
from tests import capi
from tests.conftest import make_student_t
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
