"""The any-shape kernels at the edges of their tiles, against float64 with the same rounding points.

Bounds: eps is one unit in the last place of the I/O type (relative); an operand rounded to the I/O
type may fall on the neighbouring value, so a product over it may differ by eps times its absolute
sum, and the result is rounded once more.
"""

import pytest
import torch

import triangleops_amd as tops  # noqa: F401

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0**-7, torch.float16: 2.0**-10, torch.float32: 2.0**-18}
TYPES = [torch.bfloat16, torch.float16, torch.float32]


def _rnd(g, dtype, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, dtype=torch.float64) * scale).to(dtype)


def _within(out, ref, bound, name):
    d = (out.double().cpu() - ref).abs()
    worst = (d / bound).max().item()
    assert worst <= 1.0, f"{name}: {worst:.2f} of the bound, max |d| {d.max().item():.2e}"


# tokens: one, one short of and past a 32- and a 64-token tile, past the one-tile-per-CU rule
# (32 * 256 tokens) and past the 64-token rule (64 * 8 * 256 tokens)
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("M,Cin,HD,Cout", [(1, 64, 64, 64), (31, 384, 384, 384), (65, 33, 40, 7), (8225, 96, 72, 100),
                                           (8225, 24, 24, 24), (131137, 32, 32, 32), (33, 512, 512, 130)])
@pytest.mark.parametrize("extras", [False, True])
def test_gate_any_shape(device, dtype, M, Cin, HD, Cout, extras):
    """extras: LayerNorm of the gate input, both biases, a residual, and rows of o and of the gate input
    that are column slices of wider tensors (odd strides: element-wise loads)."""
    from triangleops_amd.triangle_attn.kernel import _gate_out_generic

    g = torch.Generator().manual_seed(M + Cin)
    pad = 3 if extras else 0
    o, gin = _rnd(g, dtype, M, 1, HD + pad), _rnd(g, dtype, M, 1, Cin + pad)
    wg, wo = _rnd(g, dtype, HD, Cin, scale=Cin**-0.5), _rnd(g, dtype, Cout, HD, scale=HD**-0.5)
    bg, bo, res, w_ln, b_ln = (_rnd(g, dtype, *s) if extras else None for s in
                               ((HD,), (Cout,), (M, 1, Cout), (Cin,), (Cin,)))
    dev = [t if t is None else t.to(device) for t in (o, gin, wg, bg, wo, bo, res, w_ln, b_ln)]
    out = _gate_out_generic(dev[0][..., :HD], dev[1][..., :Cin], dev[2], dev[3], dev[4], dev[5],
                            ln=(dev[7], dev[8], 1e-5) if extras else None, residual=dev[6])
    od, gd = o[..., :HD].double(), gin[..., :Cin].double()
    slack = 0.0
    if extras:
        gd = torch.nn.functional.layer_norm(gd, (Cin,), w_ln.double(), b_ln.double(), 1e-5).to(dtype).double()
        slack = gd.abs() @ wg.double().T.abs() / 4  # the sigmoid's slope
    z = gd @ wg.double().T + (bg.double() if extras else 0.0)
    y = (od * torch.sigmoid(z)).to(dtype).double()
    ref = y @ wo.double().T + (bo.double() if extras else 0.0)
    ysum = (y.abs() + od.abs() * slack) @ wo.double().T.abs()
    bound = EPS[dtype] * (ref.abs() + ysum + 1e-3)
    if extras:
        ref = res.double() + ref
        bound = bound + EPS[dtype] * ref.abs()
    _within(out, ref, bound, f"gate {dtype} {M} {Cin} {HD} {Cout}")
