"""SiLU*up quantization of more than 64 rows into the packed layout: every bf16 gate value goes through the activation
lookup (the table's busy part, the small magnitudes beside it, the large ones, infinities and NaN), against the oracle."""
import pytest
import torch

from fp_quant.module import hip_ops
from oracle import fpq_oracle as O
from tests import capi
from tests.test_ragged_k_gpu import _padded_pack

pytestmark = pytest.mark.gpu


def test_every_gate_value():
    gate = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).reshape(256, 256)
    gate = gate[torch.randperm(256, generator=torch.Generator().manual_seed(1))].contiguous()
    up = torch.ones(256, 256, dtype=torch.bfloat16)
    pc, ps, out = capi.fused_quantize_packed("silu_mul", gate, up, g=128)
    want = O.silu_mul(gate, up)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(out), nan)
    assert torch.equal(out.view(torch.int16)[~nan], want.view(torch.int16)[~nan])
    # and the codes and scales of every 128-wide block that is finite and overflows nowhere
    quiet = torch.where(torch.isfinite(want) & (want.abs() < 1e36), want, torch.zeros_like(want))
    clean = (quiet == want).view(256, 2, 128).all(-1)
    assert clean.sum() > 100
    c, s, _ = O.quantize_mx(quiet, O.ROT_HADAMARD, 128, float(O.hadamard_matrix(128)[0, 0]))
    codes, scales = (t.cpu() for t in hip_ops.unpack_fp4(pc.cuda(), ps.cuda(), 256, 256))
    assert torch.equal(codes.view(256, 2, 64)[clean], c.view(256, 2, 64)[clean])
    assert torch.equal(scales.view(256, 2, 4)[clean], s[:256, :8].reshape(256, 2, 4)[clean])


# eight rows a wave, the last row tile with part of them; one 256-column block per row, several, and
# a part of one (20 rows: the generic kernel)
@pytest.mark.parametrize("gs,g", [(None, 128), (None, 32), (777.0, 16), (777.0, 128)])
@pytest.mark.parametrize("rows,cols", [(65, 256), (97, 768), (300, 2304), (70, 384), (20, 896)])
def test_packed_codes_bit_exact(gs, g, rows, cols):
    gen = torch.Generator().manual_seed(rows + g)
    gate = (torch.randn(rows, cols, generator=gen) * 2).to(torch.bfloat16)
    up = torch.randn(rows, cols, generator=gen).to(torch.bfloat16)
    gate[3] = 0.0
    gate[5, ::7] *= 2.0 ** -16
    up[7] *= 2.0 ** -110                  # scales outside the range of the two-operation division
    want_v = O.silu_mul(gate, up)
    norm = float(O.hadamard_matrix(g)[0, 0])
    if gs is None:
        c, s, _ = O.quantize_mx(want_v, O.ROT_HADAMARD, g, norm)
    else:
        c, s, _ = O.quantize_nv(want_v, gs, O.ROT_HADAMARD, g, norm)
    want = _padded_pack(c, s, cols, gs is not None)
    pc, ps, out = capi.fused_quantize_packed("silu_mul", gate, up, g=g, ld_a=cols + 64, ld_b=2 * cols, global_scale=gs)
    assert torch.equal(out.view(torch.int16), want_v.view(torch.int16))
    assert torch.equal(pc, want[0]) and torch.equal(ps, want[1])
