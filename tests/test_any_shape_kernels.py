"""The any-shape kernels at the edges of their tiles, against float64 with the same rounding points.

Bounds: with 16-bit I/O, EPS is one unit in the last place of the type (relative): an operand rounded to
it may fall on the neighbouring value, so a product over it may differ by EPS times its absolute sum, and
the result is rounded once more.  Nothing is rounded in fp32 but the sums: each addition is off by up to
2^-24 of its partial sum, and EPS, 2^-18, is the worst element with 64 of them all to one side, over sums of
up to 1100 products.  Over all elements such errors have no common sign: the 2-norm of what an fp32 result
is off by stays within one unit in the last place, 2^-23, of that of the absolute sums (the largest here is
2/3 of it, in the attention, and 0.3 of it elsewhere).
"""

import pytest
import torch

import triangleops_amd as tops  # noqa: F401

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0**-7, torch.float16: 2.0**-10, torch.float32: 2.0**-18}
TYPES = [torch.bfloat16, torch.float16, torch.float32]


def _rnd(g, dtype, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, dtype=torch.float64) * scale).to(dtype)


def _within(out, ref, bound, name, eps=EPS[torch.float32]):
    """Every element within `bound`; fp32 results also in the 2-norm, where bound / eps is the absolute sums."""
    d = (out.double().cpu() - ref).abs()
    worst = (d / bound).max().item()
    assert worst <= 1.0, f"{name}: {worst:.2f} of the bound, max |d| {d.max().item():.2e}"
    if out.dtype == torch.float32:
        norm = (d.norm() / bound.norm()).item() * eps
        assert norm <= 2.0**-23, f"{name}: 2-norm {norm * 2**23:.2f} units in the last place of the absolute sums"


# tokens: one, one short of and past a 32-token tile and past two, past the one-tile-per-CU rule
# (32 * 256 tokens), and thousands of blocks
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("M,Cin,HD,Cout", [(1, 64, 64, 64), (31, 384, 384, 384), (65, 33, 40, 7), (8225, 96, 72, 100),
                                           (8225, 24, 24, 24), (131137, 32, 32, 32), (33, 512, 512, 130),
                                           (33, 387, 390, 384)])
@pytest.mark.parametrize("extras", ["", "bias", "ln"])
def test_gate_any_shape(device, dtype, M, Cin, HD, Cout, extras):
    """bias: both biases and a residual; ln: also LayerNorm of the gate input, and rows of o and of the
    gate input that are column slices of wider tensors (odd strides: element-wise loads).  Few tokens with
    wide rows and no LayerNorm run as two launches."""
    from triangleops_amd.triangle_attn.kernel import _gate_out_generic

    g = torch.Generator().manual_seed(M + Cin)
    pad = 3 if extras == "ln" else 0
    o, gin = _rnd(g, dtype, M, 1, HD + pad), _rnd(g, dtype, M, 1, Cin + pad)
    wg, wo = _rnd(g, dtype, HD, Cin, scale=Cin**-0.5), _rnd(g, dtype, Cout, HD, scale=HD**-0.5)
    bg, bo, res, w_ln, b_ln = (_rnd(g, dtype, *s) if extras else None for s in
                               ((HD,), (Cout,), (M, 1, Cout), (Cin,), (Cin,)))
    dev = [t if t is None else t.to(device) for t in (o, gin, wg, bg, wo, bo, res, w_ln, b_ln)]
    out = _gate_out_generic(dev[0][..., :HD], dev[1][..., :Cin], dev[2], dev[3], dev[4], dev[5],
                            ln=(dev[7], dev[8], 1e-5) if extras == "ln" else None, residual=dev[6])
    od, gd = o[..., :HD].double(), gin[..., :Cin].double()
    slack = 0.0
    if extras == "ln":
        gd = torch.nn.functional.layer_norm(gd, (Cin,), w_ln.double(), b_ln.double(), 1e-5).to(dtype).double()
        slack = (gd.abs() + 1e-2) @ wg.double().T.abs() / 4  # the sigmoid's slope; see size below for small values
    z = gd @ wg.double().T + (bg.double() if extras else 0.0)
    y = (od * torch.sigmoid(z)).to(dtype).double()
    ref = y @ wo.double().T + (bo.double() if extras else 0.0)
    ysum = (y.abs() + od.abs() * slack) @ wo.double().T.abs()
    bound = EPS[dtype] * (ref.abs() + ysum + 1e-3)
    if extras:
        ref = res.double() + ref
        bound = bound + EPS[dtype] * ref.abs()
    _within(out, ref, bound, f"gate {dtype} {M} {Cin} {HD} {Cout}")


# few tokens with wide rows, the two launches' 16-byte and element-wise forms: rows that are column slices of
# wider tensors, a residual and a destination with strides of their own (a transposed view's, odd, in place)
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("M,Cin,HD,Cout", [(33, 384, 384, 384), (70, 400, 392, 500), (33, 387, 390, 386)])
@pytest.mark.parametrize("pad", [0, 3, 8])
def test_gate_few_tokens_strided(device, dtype, M, Cin, HD, Cout, pad):
    from triangleops_amd import _native
    from triangleops_amd._common.dtype import any_shape_dtype_code
    from triangleops_amd.triangle_attn.kernel import gate_out_forward

    assert _native.gate_generic_workspace_bytes(M, 1, Cin, HD, Cout, 0, any_shape_dtype_code(dtype)) > 0
    g = torch.Generator().manual_seed(M + pad)
    o, gin, res = (_rnd(g, dtype, M, 1, c + pad) for c in (HD, Cin, Cout))
    wg, wo, bg, bo = (_rnd(g, dtype, *s) for s in ((HD, Cin), (Cout, HD), (HD,), (Cout,)))
    wg, wo = wg * Cin**-0.5, wo * HD**-0.5
    od, gd, rd, *w = (t.to(device) for t in (o, gin, res, wg, bg, wo, bo))
    big = torch.full((M, 3, Cout + 2 * pad), 7.0, device=device, dtype=dtype)
    dst = big[:, 1:2, pad:pad + Cout]
    out = gate_out_forward(od[..., :HD], gd[..., :Cin], *w, residual=rd[..., :Cout], out=dst)
    assert out.data_ptr() == dst.data_ptr()
    y = (o[..., :HD].double() * torch.sigmoid(gin[..., :Cin].double() @ wg.double().T + bg.double())).to(dtype).double()
    ref = y @ wo.double().T + bo.double()
    bound = EPS[dtype] * (ref.abs() + y.abs() @ wo.double().T.abs() + 1e-3)
    ref = res[..., :Cout].double() + ref
    _within(out, ref, bound + EPS[dtype] * ref.abs(), f"{dtype} {M} {Cin} {HD} {Cout} {pad}")
    rest = torch.ones_like(big, dtype=torch.bool)
    rest[:, 1:2, pad:pad + Cout] = False
    assert (big[rest] == 7.0).all()
    alone = gate_out_forward(od[..., :HD], gd[..., :Cin], *w, residual=rd[..., :Cout])
    inplace = rd.clone()[..., :Cout]
    gate_out_forward(od[..., :HD], gd[..., :Cin], *w, residual=inplace, out=inplace)
    assert torch.equal(alone, out) and torch.equal(inplace, alone)


# one launch and two; weights of another dtype, or transposed: the launcher makes copies
@pytest.mark.parametrize("C", [96, 128, 384])
@pytest.mark.parametrize("form", ["fp32", "transposed"])
def test_gate_converted_weights_bitwise(device, C, form):
    """Weights that the launcher has to convert give the bits of the same weights converted beforehand."""
    from triangleops_amd.triangle_attn.kernel import gate_out_forward

    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(C)
    o, gin, res = (_rnd(g, dtype, 33, 1, C).to(device) for _ in range(3))
    w = [_rnd(g, dtype, *s).to(device) for s in ((C, C), (C,), (C, C), (C,))]
    other = [t.float() for t in w] if form == "fp32" else [t.t().contiguous().t() if t.dim() == 2 else t for t in w]
    assert torch.equal(gate_out_forward(o, gin, *other), gate_out_forward(o, gin, *w))
    assert torch.equal(gate_out_forward(o, gin, *other, residual=res.float()),
                       gate_out_forward(o, gin, *w, residual=res))


# grids of one token, one short of and past a 32-token tile, a few thousand blocks;
# head widths of every store width, C of one and several k batches and with a tail
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("N,C,H,D", [(1, 64, 2, 64), (6, 24, 3, 24), (9, 40, 5, 10), (13, 33, 2, 12), (21, 200, 9, 16),
                                     (33, 1024, 4, 64), (130, 128, 4, 32)])
@pytest.mark.parametrize("ln", [False, True])
def test_tri_prep_any_shape(device, dtype, N, C, H, D, ln):
    """LN(x), Q / K / V and the pair bias of a transposed view (ln) or of a channel slice."""
    from triangleops_amd.triangle_attn.kernel import generic_prep_forward

    g = torch.Generator().manual_seed(N + C)
    x = _rnd(g, dtype, N, N, C).transpose(0, 1) if ln else _rnd(g, dtype, N, N, C + 1)[..., :C]
    w, wz = _rnd(g, dtype, H, 3, D, C, scale=C**-0.5), _rnd(g, dtype, H, C, scale=C**-0.5)
    w_ln, b_ln, bz = _rnd(g, dtype, C), _rnd(g, dtype, C), _rnd(g, torch.float32, H)
    xd = x.to(device) if not ln else x.transpose(0, 1).contiguous().to(device).transpose(0, 1)
    out = generic_prep_forward(xd, w_ln.to(device), b_ln.to(device), w.to(device), wz.to(device), bz.to(device),
                               apply_ln=ln)
    xn = x.double()
    size = xn.abs()  # of what an element is summed from: x and the mean, the scaled result and the bias may cancel
    if ln:
        mean, std = xn.mean(-1, keepdim=True), (xn.var(-1, correction=0, keepdim=True) + 1e-5).sqrt()
        size = (xn.abs() + mean.abs()) / std * w_ln.double().abs() + b_ln.double().abs()
        xn = torch.nn.functional.layer_norm(xn, (C,), w_ln.double(), b_ln.double(), 1e-5)
    xr = xn.to(dtype).double()
    _within(out[0], xr, EPS[dtype] * xr.abs() + EPS[torch.float32] * size, "xln")
    for i, name in enumerate("qkv"):
        wi = w[:, i].double().reshape(H * D, C)
        ref = (xr @ wi.T).view(N, N, H, D)
        bound = EPS[dtype] * (ref.abs() + (xr.abs() @ wi.abs().T).view(N, N, H, D) + 1e-3)
        _within(out[1 + i], ref, bound, name)
    ref = (xn @ wz.double().T + bz.double()).permute(2, 0, 1)
    bound = EPS[torch.float32] * ((xn.abs() @ wz.double().abs().T).permute(2, 0, 1) + 1.0)
    _within(out[4], ref, bound, "bias")


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("M,C,H,D", [(1, 8, 1, 8), (31, 384, 16, 24), (33, 30, 3, 10), (65, 512, 2, 64), (64, 520, 3, 20),
                                     (40, 1100, 5, 16), (1000, 40, 16, 24), (1000, 1100, 16, 24)])
def test_apb_qkv_any_shape(device, dtype, M, C, H, D):
    """Q / K / V for few tokens (the k range split over a block's waves) and for more (rows staged 512
    channels at a time), odd channel counts and head widths."""
    from triangleops_amd import _native
    from triangleops_amd._common.dtype import any_shape_dtype_code

    g = torch.Generator().manual_seed(M + C)
    x, w = _rnd(g, dtype, M, C), _rnd(g, dtype, H, 3, D, C, scale=C**-0.5)
    xd, wd, z = x.to(device), w.to(device), torch.zeros(M, M, 8, device=device, dtype=dtype)
    wc, bc = torch.zeros(H, 8, device=device), torch.zeros(H, device=device)
    out = torch.empty(3, M, H * D, device=device, dtype=dtype)  # rows of odd sizes: misaligned k and v
    bias = torch.empty(H, M, M, device=device)
    _native.call("tops_apb_generic_prep", xd.data_ptr(), wd.data_ptr(), z.data_ptr(), M * 8, 8, wc.data_ptr(),
                 bc.data_ptr(), *(o.data_ptr() for o in out), bias.data_ptr(), M, C, 8, H, D, 1e-5,
                 any_shape_dtype_code(dtype), _native.stream_of(xd))
    for i, name in enumerate("qkv"):
        wi = w[:, i].double().reshape(H * D, C)
        ref = x.double() @ wi.T
        _within(out[i], ref, EPS[dtype] * (ref.abs() + x.double().abs() @ wi.abs().T + 1e-3), name)


# key chunks and query tiles of 32: one, one less one, one, one more, several; D at and below 16, 32 and 64, with
# and without 16-byte rows; few query tiles (keys split over the waves) and many
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("N,H,D", [(1, 2, 32), (31, 3, 24), (32, 2, 64), (33, 1, 10), (129, 4, 32), (70, 9, 40),
                                   (100, 8, 64), (160, 4, 6), (65, 4, 16), (100, 4, 8)])
@pytest.mark.parametrize("mask", ["none", "random", "rows", "inf"])
def test_attention_any_shape(device, dtype, N, H, D, mask):
    """Triangle attention (a random pair mask; whole rows masked) and attention over one row (mask
    "inf": masked keys -inf, some chunks wholly masked)."""
    from triangleops_amd import _native
    from triangleops_amd._common.dtype import any_shape_dtype_code
    from triangleops_amd.triangle_attn.kernel import generic_attention

    g = torch.Generator().manual_seed(N + D)
    R = 1 if mask == "inf" else N
    q, k, v = (_rnd(g, dtype, R, N, H, D) for _ in range(3))
    bias = _rnd(g, torch.float32, H, N, N)
    scale = D**-0.5
    m = None
    if mask != "none":
        m = torch.rand(R, N, generator=g) < 0.8
        m[:, : min(40, N // 2)] = False
        m[:, N - 1] = True
        if mask == "rows":
            m[::3] = False
    dev = [t.to(device) for t in (q, k, v, bias)]
    md = None if m is None else m.to(device)
    out = torch.empty(R, N, H * D, device=device, dtype=dtype)
    if mask == "inf":
        _native.call("tops_apb_generic_attention", *(t.data_ptr() for t in dev), md.view(torch.int8).data_ptr(),
                     out.data_ptr(), N, H, D, scale, any_shape_dtype_code(dtype), _native.stream_of(out))
    else:
        generic_attention(*dev, out, scale=scale, mask=md)
    s = torch.einsum("iqhd,ikhd->ihqk", q.double(), k.double()) * scale + bias.double()
    if m is not None:
        s = s.masked_fill(~m[:, None, None, :], float("-inf")) if mask == "inf" else \
            (s + torch.where(m, 0.0, -1e9)[:, None, None, :]).float().double()  # the fp32 add rounds to 64s
    p = torch.softmax(s, -1)
    ref = torch.einsum("ihqk,ikhd->iqhd", p, v.double()).reshape(R, N, H * D)
    size = torch.einsum("ihqk,ikhd->iqhd", p, v.double().abs()).reshape(R, N, H * D)
    # fp32 scores of a few units are off by some 2^-22, the weights relatively so; one rounding of the result
    _within(out, ref, 0.5 * EPS[dtype] * ref.abs() + EPS[torch.float32] * size + 1e-7, f"{dtype} {N} {H} {D} {mask}")


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("N,D", [(400, 16), (391, 10), (400, 40)])
def test_attention_one_row_many_heads(device, dtype, N, D):
    """One row of queries whose 64 heads are tiles enough to leave the keys unsplit, some chunks wholly masked."""
    test_attention_any_shape(device, dtype, N, 64, D, "inf")


# keys split over the waves (H = 2) and not (H = 8); one and two 32-channel tiles
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("N,H,D", [(40, 2, 24), (40, 8, 24), (40, 2, 64), (40, 8, 64)])
def test_attention_weights_keep_fp32(device, dtype, N, H, D):
    """The weights count with fp32's 24 bits, large and small ones alike.  Scores come from the bias alone.

    Rows of even i: V of the first keys is chosen so that the weighted sum cancels to a few units of fp32, each
    key taking off what the I/O type's rounding left of the ones before.  A weight exp(s - max) with |s| <= 1.4 is
    off by one unit of exp2 and less than one of its argument's, 2 * 2^-23, and the sums of 4 terms round to less
    than that again: 2^-21 of the absolute sum, plus the rounding of the result.
    Rows of odd i: all of an output is one large V under a weight of about e^-18 (a unit of the argument is
    2^-20 there, and there are two of them)."""
    from triangleops_amd.triangle_attn.kernel import generic_attention

    g = torch.Generator().manual_seed(N + D)
    b = torch.rand(H, N, generator=g) * 1.4 - 1.4
    b[:, 0] = 0.0
    b[:, 6:] = -18.0 - torch.rand(H, N - 6, generator=g)
    w = torch.exp(b.double())
    v = torch.zeros(N, N, H, D, dtype=dtype)
    acc = torch.zeros(N, H, D, dtype=torch.float64)
    steps = {torch.bfloat16: 4, torch.float16: 3, torch.float32: 2}[dtype]
    for k in range(steps):
        vk = torch.rand(N, H, D, generator=g, dtype=torch.float64) + 1.0 if k == 0 else -acc / w[None, :, k, None]
        v[:, k] = vk.to(dtype)
        acc += w[None, :, k, None] * v[:, k].double()
    v[1::2] = 0.0
    for d in range(D):
        v[1::2, 6 + d % (N - 6), :, d] = 6e4
    q, k = torch.zeros(N, N, H, D, dtype=dtype), _rnd(g, dtype, N, N, H, D)
    bias = b[:, None, :].expand(H, N, N).contiguous()
    out = torch.empty(N, N, H * D, device=device, dtype=dtype)
    generic_attention(*(t.to(device) for t in (q, k, v, bias)), out)
    p = w / w.sum(-1, keepdim=True)
    ref = torch.einsum("hk,ikhd->ihd", p, v.double()).reshape(N, 1, H * D)
    size = torch.einsum("hk,ikhd->ihd", p, v.double().abs()).reshape(N, 1, H * D)
    ulp = torch.tensor([2.0**-21, 2.0**-18], dtype=torch.float64).repeat(N // 2)[:, None, None]
    bound = 0.5 * EPS[dtype] * ref.abs() + ulp * size
    _within(out, ref.expand(out.shape), bound.expand(out.shape), f"{dtype} {H} {D}", eps=2.0**-21)


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("H,D", [(2, 32), (8, 32), (2, 64), (8, 64)])
def test_attention_infinities_in_v(device, dtype, H, D):
    """An infinity or a NaN of V reaches its own channel and no other, as in a plain sum of products."""
    from triangleops_amd.triangle_attn.kernel import generic_attention

    N, inf = 70, float("inf")
    g = torch.Generator().manual_seed(D)
    q, k, v = (_rnd(g, dtype, N, N, H, D) for _ in range(3))
    bias = _rnd(g, torch.float32, H, N, N)
    v[3, 0, :, 1], v[3, 69, :, 5], v[3, 40, :, 9] = inf, -inf, float("nan")
    v[5, 31, :, 0], v[5, 32, :, 0], v[5, 33, 1, 17] = inf, -inf, inf
    out = torch.empty(N, N, H * D, device=device, dtype=dtype)
    generic_attention(*(t.to(device) for t in (q, k, v, bias)), out, scale=D**-0.5)
    s = torch.einsum("iqhd,ikhd->ihqk", q.double(), k.double()) * D**-0.5 + bias.double()
    vf = v.double().nan_to_num(0.0, 0.0, 0.0)
    p = torch.softmax(s, -1)
    ref = torch.einsum("ihqk,ikhd->iqhd", p, vf) + (v.double() - vf).sum(1)[:, None]
    size = torch.einsum("ihqk,ikhd->iqhd", p, vf.abs())
    ref, size = ref.reshape(out.shape), size.reshape(out.shape)
    got, ok = out.double().cpu(), ref.isfinite()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[ref.isinf()], ref[ref.isinf()])
    bound = 0.5 * EPS[dtype] * ref.abs() + EPS[torch.float32] * size + 1e-7
    _within(got[ok], ref[ok], bound[ok], f"{dtype} {H} {D}")


# pairs: one, below and past a 16-pair step, several steps per wave; C_z of every chunk count with tails;
# one, exactly 16 and more heads
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("M,Cz,H", [(1, 128, 4), (3, 8, 1), (5, 33, 17), (40, 64, 16), (67, 250, 3), (260, 128, 16),
                                    (33, 256, 5), (20, 300, 2)])
@pytest.mark.parametrize("offset", [0.0, 30.0])
def test_apb_bias_any_shape(device, dtype, M, Cz, H, offset):
    """The pair bias LN(z) . Wc + Bc of a Z slice with odd strides (offset 0) or of contiguous Z whose
    values share an offset (the statistics must not cancel)."""
    from triangleops_amd import _native
    from triangleops_amd._common.dtype import any_shape_dtype_code

    g = torch.Generator().manual_seed(M + Cz)
    z = (_rnd(g, torch.float64, M, M, Cz + (1 if offset == 0 else 0)) + offset).to(dtype)
    zd = z.to(device)[..., :Cz]
    z = z[..., :Cz].double()
    wc, bc = _rnd(g, torch.float32, H, Cz, scale=Cz**-0.5), _rnd(g, torch.float32, H)
    wd, bd = wc.to(device), bc.to(device)
    x, w = torch.zeros(M, 8, device=device, dtype=dtype), torch.zeros(H, 3, 8, 8, device=device, dtype=dtype)
    scratch, out = torch.empty(3, M, H * 8, device=device, dtype=dtype), torch.empty(H, M, M, device=device)
    _native.call("tops_apb_generic_prep", x.data_ptr(), w.data_ptr(), zd.data_ptr(), zd.stride(0), zd.stride(1),
                 wd.data_ptr(), bd.data_ptr(), *(t.data_ptr() for t in scratch), out.data_ptr(), M, 8, Cz, H, 8, 1e-5,
                 any_shape_dtype_code(dtype), _native.stream_of(x))
    mean, std = z.mean(-1, keepdim=True), (z.var(-1, correction=0, keepdim=True) + 1e-5).sqrt()
    ref = ((z - mean) / std @ wc.double().T + bc.double()).permute(2, 0, 1)
    size = ((z.abs() + mean.abs()) / std @ wc.double().abs().T + bc.double().abs()).permute(2, 0, 1)
    _within(out, ref, EPS[torch.float32] * size, f"bias {dtype} {M} {Cz} {H}")


# one and several 64-token tiles per row with every kind of tail; C of one k-step, with tails, of one
# and several weight batches, wider than the 64-token tile fits; few and many 32-feature chunks
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("B,L,C", [(1, 1, 8), (2, 33, 64), (1, 64, 96), (1, 65, 33), (1, 100, 256), (1, 20, 500),
                                   (1, 200, 32)])
@pytest.mark.parametrize("transpose", [False, True])
def test_tmu_phases_any_shape(device, dtype, B, L, C, transpose):
    """Input phase (masked, padded columns zero) and output phase (with a residual when transpose)."""
    from triangleops_amd.triangle_mul.kernel import input_phase, output_phase

    g = torch.Generator().manual_seed(L + C)
    x, res = _rnd(g, dtype, B, L, L, C), _rnd(g, dtype, B, L, L, C)
    mask = torch.rand(B, L, L, generator=g) < 0.8
    ld = (L + 63) // 64 * 64
    y = _rnd(g, dtype, C, B, L, ld)
    y[..., L:] = float("nan")  # never part of a result
    (wp, wg), (bp, bg) = (_rnd(g, dtype, 2, 2 * C, C, scale=C**-0.5), _rnd(g, torch.float32, 2, 2 * C))

    def norm(t):
        t = t.double()
        return torch.nn.functional.layer_norm(t, (C,), eps=1e-5).to(dtype).double()

    def gated(a, b, n):
        w, v = wp[:n].double(), wg[:n].double()
        p, s = a @ w.T + bp[:n].double(), torch.sigmoid(b @ v.T + bg[:n].double())
        # rounding of the normalised operands (some 2e-2 of them close to a rounding step of x - mean)
        slack = (a.abs() + 1e-2) @ w.T.abs() * s + p.abs() * s * (1 - s) * ((b.abs() + 1e-2) @ v.T.abs())
        return p * s, EPS[dtype] * ((p * s).abs() + slack + 1e-3)

    sums = torch.zeros(2 * C, device=device)
    dev = [t.to(device) for t in (x, mask, wp, wg, bp, bg, y, res)]
    ab = input_phase(dev[0], dev[1], dev[2], dev[3], sums, sums, dev[4], dev[5], 1e-5, transpose=transpose, ld=ld)
    ref, bound = gated(norm(x), norm(x), 2 * C)
    ref = ref * mask[..., None]
    if transpose:
        ref, bound = ref.transpose(1, 2), bound.transpose(1, 2)
    assert ab.shape == (2 * C, B, L, ld) and not ab[..., L:].any()
    _within(ab[..., :L], ref.permute(3, 0, 1, 2), bound.permute(3, 0, 1, 2), f"input phase {dtype} {L} {C}")

    out = output_phase(dev[6], dev[0], dev[2][:C], dev[3][:C], sums[:C], sums[:C], dev[4][:C], dev[5][:C], 1e-5, ldy=ld,
                       residual=dev[7] if transpose else None)
    ref, bound = gated(norm(y[..., :L].permute(1, 2, 3, 0)), norm(x), C)
    if transpose:
        ref = res.double() + ref
        bound = bound + EPS[dtype] * ref.abs()
    _within(out, ref, bound, f"output phase {dtype} {L} {C}")


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("L,C", [(33, 64), (70, 100), (5, 500)])
@pytest.mark.parametrize("transpose", [False, True])
def test_tmu_padding_zero_beside_nan(device, dtype, L, C, transpose):
    """Columns [L, ld) are zero where the last token of a row is NaN, and only its own row's values are NaN."""
    from triangleops_amd.triangle_mul.kernel import input_phase

    g = torch.Generator().manual_seed(L)
    x = _rnd(g, dtype, 1, L, L, C)
    x[0, 2, L - 1], x[0, L - 1, 3, 0] = float("nan"), float("inf")
    (wp, wg), c = _rnd(g, dtype, 2, C, C), torch.zeros(C, device=device)
    ab = input_phase(x.to(device), None, wp.to(device), wg.to(device), c, c, c, c, 1e-5, transpose=transpose,
                     ld=(L + 63) // 64 * 64)
    assert not ab[..., L:].any()
    bad = torch.zeros(1, L, L, dtype=torch.bool, device=device)
    bad[0, 2, L - 1] = bad[0, L - 1, 3] = True
    assert torch.equal(ab[..., :L].isnan(), (bad.transpose(1, 2) if transpose else bad).expand(C, 1, L, L))
