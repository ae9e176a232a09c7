"""Timed calls of the three pair-representation ops and of the block that composes them.

Each case is one call as an inference program makes it: the weights are folded once by
`precompute`, the activations and masks are on the GPU, and one pass is one `forward` (or one
whole `pairformer_block`).  Inputs follow the benchmark's distributions: activations N(0, 1),
weights N(0, 1 / fan_in), LayerNorm gamma = 1 + 0.1 N(0, 1), beta = 0.1 N(0, 1), every tensor
rounded once to the I/O type.  Masks mark padding (the last tenth of rows and columns of the pair
grid, the last twentieth of the tokens) or are drawn at random.
"""

from __future__ import annotations

import math

import torch

import triangleops_amd as tops
from triangleops_amd import pairformer

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _tmu(n, *, c=128, batch=1, dtype="bf16", direction="outgoing", mask="pad"):
    return {"op": "tmu", "n": n, "c": c, "batch": batch, "dtype": dtype, "direction": direction, "mask": mask}


def _tri(n, *, c=128, h=4, d=32, dtype="bf16", ending=False, mask="pad"):
    return {"op": "tri", "n": n, "c": c, "h": h, "d": d, "dtype": dtype, "ending": ending, "mask": mask}


def _apb(n, *, c=128, cz=128, h=4, d=32, dtype="bf16", qknorm=False, mask="pad"):
    return {"op": "apb", "n": n, "c": c, "cz": cz, "h": h, "d": d, "dtype": dtype, "qknorm": qknorm, "mask": mask}


def _block(n, *, dtype="bf16", mask="pad"):
    return {"op": "block", "n": n, "c": 128, "h": 4, "d": 32, "dtype": dtype, "mask": mask}


def listed():
    cases = {
        # a short chain (peptide, small domain): three launches of a few microseconds each
        "tmu_out_bf16_128": _tmu(128, mask="none"),
        # a sequence length as it comes, no multiple of any tile, in half precision
        "tmu_in_fp16_389": _tmu(389, dtype="fp16", direction="incoming"),
        # the long-crop call that the benchmark's headline number is quoted on
        "tmu_out_bf16_1024": _tmu(1024),
        # single-precision inference (checking a checkpoint, numerically delicate inputs)
        "tmu_out_fp32_256": _tmu(256, dtype="fp32"),
        # the narrower pair representation of a template stack
        "tmu_in_bf16_c64_512": _tmu(512, c=64, direction="incoming"),
        # an ordinary training-crop size of the starting node
        "tri_start_bf16_256": _tri(256),
        # the longest sequences, ending node: the N^3 attention regime on a transposed grid
        "tri_end_bf16_2048": _tri(2048, ending=True),
        # single precision again, on the attention op, with a ragged size
        "tri_start_fp32_200": _tri(200, dtype="fp32"),
        # the single representation's attention on a short chain: launch and latency bound
        "apb_bf16_128": _apb(128),
        # the same on the longest sequences: one read of the pair representation
        "apb_bf16_2048": _apb(2048),
        # a wide single representation with many narrow heads, ragged token count
        "apb_bf16_h16_600": _apb(600, c=384, h=16, d=24),
        # a whole block (four pair updates with residuals, then the single update), ragged size
        "block_bf16_500": _block(500),
    }
    return [{"name": name, **case} for name, case in cases.items()]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the ranges above: any op, I/O type, direction and mask, ragged sizes."""
    op = rng.choices(("tmu", "tri", "apb", "block"), (4, 4, 4, 1))[0]
    dtype = rng.choices(("bf16", "fp16", "fp32"), (6, 2, 2))[0]
    mask = rng.choice(("none", "pad", "pad", "random"))
    default_shape = rng.random() < 0.7
    slow = dtype == "fp32" or not default_shape  # sizes kept smaller where a call takes longer
    if op == "tmu":
        c = 128 if default_shape else rng.choice((32, 64, 64, 96, 192, 256))
        batch = rng.choice((1, 1, 1, 2))
        return _tmu(_size(rng, 96, 448 if slow else 1024), c=c, batch=batch, dtype=dtype, mask=mask,
                    direction=rng.choice(("outgoing", "incoming")))
    if op == "tri":
        c, h, d = (128, 4, 32) if default_shape else rng.choice(((64, 4, 16), (64, 4, 16), (128, 8, 16), (96, 3, 24),
                                                                 (64, 2, 64)))
        return _tri(_size(rng, 96, 320 if slow else 1400), c=c, h=h, d=d, dtype=dtype, mask=mask,
                    ending=rng.random() < 0.5)
    if op == "apb":
        c, cz, h, d = (128, 128, 4, 32) if default_shape else rng.choice(((384, 128, 16, 24), (384, 128, 16, 24),
                                                                          (128, 128, 8, 16), (96, 64, 3, 24),
                                                                          (64, 32, 2, 64)))
        return _apb(_size(rng, 96, 800 if slow else 2048), c=c, cz=cz, h=h, d=d, dtype=dtype, mask=mask,
                    qknorm=rng.random() < 0.25)
    return _block(_size(rng, 96, 640), dtype=rng.choice(("bf16", "bf16", "fp16")), mask=mask)


# ---------------------------------------------------------------------------------------------- inputs
class _Draw:
    """N(0, 1) tensors from one seed, made on the GPU, rounded to the I/O type."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def __call__(self, *shape, scale=1.0, base=0.0):
        t = torch.randn(*shape, generator=self.g, device="cuda")
        return t.mul_(scale).add_(base).to(self.dtype)

    def mask(self, kind, shape):
        if kind == "none":
            return None
        if kind == "random":
            return torch.rand(*shape, generator=self.g, device="cuda") < 0.85
        n = shape[-1]
        if len(shape) == 1:
            return torch.arange(n, device="cuda") < n - n // 20
        valid = torch.arange(n, device="cuda") < n - n // 10
        return (valid[:, None] & valid[None, :]).expand(shape).contiguous()


def _tmu_weights(rnd, c):
    s = c**-0.5
    return {
        "norm_in_weight": rnd(c, scale=0.1, base=1.0),
        "norm_in_bias": rnd(c, scale=0.1),
        "p_in_weight": rnd(2 * c, c, scale=s),
        "g_in_weight": rnd(2 * c, c, scale=s),
        "norm_out_weight": rnd(c, scale=0.1, base=1.0),
        "norm_out_bias": rnd(c, scale=0.1),
        "p_out_weight": rnd(c, c, scale=s),
        "g_out_weight": rnd(c, c, scale=s),
    }


def _tri_weights(rnd, c, h, d):
    s, hd = c**-0.5, h * d
    return {
        "W_ln": rnd(c, scale=0.1, base=1.0),
        "B_ln": rnd(c, scale=0.1),
        "WQ": rnd(c, hd, scale=s),
        "WK": rnd(c, hd, scale=s),
        "WV": rnd(c, hd, scale=s),
        "W_proj_z": rnd(c, h, scale=s),
        "B_proj_z": rnd(h, scale=0.1),
        "W_proj_g": rnd(hd, c, scale=s),
        "W_proj_o": rnd(c, hd, scale=hd**-0.5),
    }


def _apb_weights(rnd, c, cz, h, d, qknorm):
    s, hd = c**-0.5, h * d
    w = {
        "WQ": rnd(c, hd, scale=s),
        "WK": rnd(c, hd, scale=s),
        "WV": rnd(c, hd, scale=s),
        "W_ln": rnd(cz, scale=0.1, base=1.0),
        "B_ln": rnd(cz, scale=0.1),
        "W_proj_z": rnd(cz, h, scale=cz**-0.5),
        "B_proj_z": rnd(h, scale=0.1),
        "W_proj_g": rnd(hd, c, scale=s),
        "W_proj_o": rnd(c, hd, scale=hd**-0.5),
    }
    if qknorm:
        w["b_q"] = rnd(hd, scale=0.5)
        for k in ("q", "k"):
            w["qkn_w_" + k] = rnd(hd, scale=0.2, base=1.0)
            w["qkn_b_" + k] = rnd(hd, scale=0.2)
    else:
        w["B_proj_g"] = rnd(hd, scale=0.1)
        w["B_proj_o"] = rnd(c, scale=0.1)
    return w


def _inputs(case, seed):
    """Everything the call reads, on the GPU, from the seed alone."""
    op, n, c = case["op"], case["n"], case["c"]
    rnd = _Draw(seed, DTYPES[case["dtype"]])
    if op == "tmu":
        b = case["batch"]
        return {"x": rnd(b, n, n, c), "mask": rnd.mask(case["mask"], (b, n, n)), "w": _tmu_weights(rnd, c)}
    h, d = case["h"], case["d"]
    if op == "tri":
        return {"x": rnd(n, n, c), "mask": rnd.mask(case["mask"], (n, n)), "w": _tri_weights(rnd, c, h, d)}
    if op == "apb":
        cz = case["cz"]
        return {"s": rnd(n, c), "z": rnd(n, n, cz), "mask": rnd.mask(case["mask"], (n,)),
                "w": _apb_weights(rnd, c, cz, h, d, case["qknorm"])}
    return {
        "z": rnd(n, n, c),
        "s": rnd(n, c),
        "pair_mask": rnd.mask(case["mask"], (n, n)),
        "single_mask": rnd.mask(case["mask"], (n,)),
        "tmu_out": _tmu_weights(rnd, c),
        "tmu_in": _tmu_weights(rnd, c),
        "tri_start": _tri_weights(rnd, c, h, d),
        "tri_end": _tri_weights(rnd, c, h, d),
        "apb": _apb_weights(rnd, c, c, h, d, False),
    }


def prepare(case, seed):
    """The activations, masks and folded weights that a program holds before the call."""
    t = _inputs(case, seed)
    t["case"] = case
    op = case["op"]
    if op == "tmu":
        t["pre"] = tops.triangle_mul.precompute(**t.pop("w"))
    elif op == "tri":
        w = t.pop("w")
        t["proj"] = {"W_proj_g": w.pop("W_proj_g"), "B_proj_g": None, "W_proj_o": w.pop("W_proj_o"), "B_proj_o": None}
        t["pre"] = tops.triangle_attn.precompute(**w, H=case["h"], D=case["d"])
        if case["ending"]:
            t["x"] = t["x"].transpose(0, 1)
            t["mask"] = None if t["mask"] is None else t["mask"].T
    elif op == "apb":
        w = t.pop("w")
        names = ("WQ", "WK", "WV", "W_ln", "B_ln", "W_proj_z", "B_proj_z")
        t["pre"] = tops.attn_pair_bias.precompute(**{k: w.pop(k) for k in names}, H=case["h"], D=case["d"])
        t["proj"] = w
    else:
        weights = [t.pop(k) for k in ("tmu_out", "tmu_in", "tri_start", "tri_end", "apb")]
        t["pre"] = pairformer.precompute(*weights, H=case["h"], D=case["d"])
    return t


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "tmu":
        return tops.triangle_mul.forward(state["x"], state["pre"], direction=case["direction"], mask=state["mask"])
    if op == "tri":
        return tops.triangle_attn.forward(state["x"], state["pre"], mask=state["mask"], scale=case["d"] ** -0.5,
                                          **state["proj"])
    if op == "apb":
        if case["qknorm"]:
            return tops.attn_pair_bias.forward_qknorm(state["s"], state["z"], state["pre"], key_mask=state["mask"],
                                                      scale=case["d"] ** -0.5, **state["proj"])
        return tops.attn_pair_bias.forward(state["s"], state["z"], state["pre"], mask=state["mask"],
                                           scale=case["d"] ** -0.5, **state["proj"])
    return pairformer.pairformer_block(state["z"], state["s"], state["pre"], pair_mask=state["pair_mask"],
                                       single_mask=state["single_mask"])


# ---------------------------------------------------------------------------------------------- work
def _valid(case, n, frac):
    """Tokens of an axis that are not padding (a random mask leaves every token something to do)."""
    return n - n // frac if case["mask"] == "pad" else n


def _tmu_flops(case, n, c, batch):
    v = _valid(case, n, 10)
    return batch * (2 * c * v**3 + 12 * n * n * c * c)


def _tri_flops(case, n, c, h, d):
    v = _valid(case, n, 10)
    return 4 * v * n * v * h * d + 2 * n * n * c * (5 * h * d + h)


def _apb_flops(case, n, c, cz, h, d):
    v = _valid(case, n, 20)
    return 4 * n * v * h * d + 2 * n * v * cz * h + 10 * n * c * h * d


def work(case):
    """Bytes: each activation read once, each result written once.  Flops: the projections over every
    token, the products over what the mask leaves."""
    op, n, c = case["op"], case["n"], case["c"]
    es = 4 if case["dtype"] == "fp32" else 2
    has_mask = 0 if case["mask"] == "none" else 1
    if op == "tmu":
        b = case["batch"]
        return {"bytes": b * n * n * (2 * c * es + has_mask), "flops": _tmu_flops(case, n, c, b)}
    h, d = case["h"], case["d"]
    if op == "tri":
        return {"bytes": n * n * (2 * c * es + has_mask), "flops": _tri_flops(case, n, c, h, d)}
    if op == "apb":
        v = _valid(case, n, 20)
        return {"bytes": n * v * case["cz"] * es + 2 * n * c * es, "flops": _apb_flops(case, n, c, case["cz"], h, d)}
    flops = 2 * _tmu_flops(case, n, c, 1) + 2 * _tri_flops(case, n, c, h, d) + _apb_flops(case, n, c, c, h, d)
    return {"bytes": 2 * (n * n + n) * c * es + (n * n + n) * has_mask, "flops": flops}


# Four times the largest distances from 64 bits over the listed cases and forty drawn ones (2-norm;
# single elements): bf16 5.4e-3 and 6.5e-2, fp16 6.7e-4 and 6.4e-3, fp32 5.2e-7 and 4.8e-6, and for
# the single representation's attention 3.9e-3 and 2.1e-2, 5.0e-4 and 2.7e-3, 4.6e-7 and 2.3e-6.
_PAIR_TOLERANCE = {"bf16": (2.2e-2, 0.26), "fp16": (2.7e-3, 0.026), "fp32": (2.1e-6, 2e-5)}
_SINGLE_TOLERANCE = {"bf16": (1.6e-2, 0.085), "fp16": (2e-3, 0.011), "fp32": (1.9e-6, 1e-5)}


def tolerance(case):
    rel, largest = (_SINGLE_TOLERANCE if case["op"] == "apb" else _PAIR_TOLERANCE)[case["dtype"]]
    return {"rel": rel, "max": largest}


# ---------------------------------------------------------------------------------------------- 64 bits
def _norm(x, w, b, eps=1e-5):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w + b


def _tmu_exact(x, mask, w, direction):
    """x (L, L, C) in 64 bits."""
    xn = _norm(x, w["norm_in_weight"], w["norm_in_bias"])
    ab = torch.sigmoid(xn @ w["g_in_weight"].T) * (xn @ w["p_in_weight"].T)
    if mask is not None:
        ab = ab * mask[..., None]
    if direction == "incoming":
        ab = ab.transpose(0, 1)
    a, b = ab.permute(2, 0, 1).contiguous().chunk(2)
    y = torch.bmm(a, b.transpose(1, 2).contiguous()).permute(1, 2, 0)
    gate = torch.sigmoid(xn @ w["g_out_weight"].T)
    return gate * (_norm(y, w["norm_out_weight"], w["norm_out_bias"]) @ w["p_out_weight"].T)


def _tri_exact(x, mask, w, h, d):
    """x (N, N, C) in 64 bits, some rows at a time."""
    n = x.shape[0]
    xn = _norm(x, w["W_ln"], w["B_ln"])
    bias = (xn @ w["W_proj_z"] + w["B_proj_z"]).permute(2, 0, 1)
    out = torch.empty(n, n, w["W_proj_o"].shape[0], device=x.device, dtype=x.dtype)
    rows = max(1, (1 << 28) // (h * n * n))
    for i in range(0, n, rows):
        r = xn[i:i + rows]
        q, k, v = ((r @ w[name]).view(-1, n, h, d).transpose(1, 2) for name in ("WQ", "WK", "WV"))
        sc = torch.matmul(q * d**-0.5, k.transpose(2, 3).contiguous()).add_(bias)
        if mask is not None:
            sc.masked_fill_(~mask[i:i + rows, None, None, :], -1e9)
        o = torch.matmul(torch.softmax(sc, -1), v.contiguous()).transpose(1, 2).reshape(-1, n, h * d)
        out[i:i + rows] = (o * torch.sigmoid(r @ w["W_proj_g"].T)) @ w["W_proj_o"].T
    return out


def _apb_exact(s, z, mask, w, h, d):
    """s (M, C), z (M, M, Cz) in 64 bits."""
    m = s.shape[0]
    bias = (_norm(z, w["W_ln"], w["B_ln"]) @ w["W_proj_z"] + w["B_proj_z"]).permute(2, 0, 1)
    q, k, v = s @ w["WQ"], s @ w["WK"], s @ w["WV"]
    if "b_q" in w:
        q = _norm(q + w["b_q"], w["qkn_w_q"], w["qkn_b_q"])
        k = _norm(k, w["qkn_w_k"], w["qkn_b_k"])
    q, k, v = (t.view(m, h, d).transpose(0, 1) for t in (q, k, v))
    sc = torch.matmul(q * d**-0.5, k.transpose(1, 2).contiguous()) + bias
    if mask is not None:
        sc.masked_fill_(~mask, float("-inf"))
    o = torch.matmul(torch.softmax(sc, -1), v.contiguous()).transpose(0, 1).reshape(m, h * d)
    gate = s @ w["W_proj_g"].T + w.get("B_proj_g", 0.0)
    return (o * torch.sigmoid(gate)) @ w["W_proj_o"].T + w.get("B_proj_o", 0.0)


def _double(t):
    if isinstance(t, dict):
        return {k: _double(v) for k, v in t.items()}
    return t.double() if torch.is_tensor(t) and t.dtype != torch.bool else t


def exact(case, seed):
    """What `run` returns for these inputs, in 64 bits."""
    t = _double(_inputs(case, seed))
    op = case["op"]
    if op == "tmu":
        return torch.stack([_tmu_exact(x, None if t["mask"] is None else t["mask"][i], t["w"], case["direction"])
                            for i, x in enumerate(t["x"])])
    h, d = case["h"], case["d"]
    if op == "tri":
        if not case["ending"]:
            return _tri_exact(t["x"], t["mask"], t["w"], h, d)
        mask = None if t["mask"] is None else t["mask"].T
        return _tri_exact(t["x"].transpose(0, 1), mask, t["w"], h, d)
    if op == "apb":
        return _apb_exact(t["s"], t["z"], t["mask"], t["w"], h, d)
    z, mask = t["z"], t["pair_mask"]
    z = z + _tmu_exact(z, mask, t["tmu_out"], "outgoing")
    z = z + _tmu_exact(z, mask, t["tmu_in"], "incoming")
    z = z + _tri_exact(z, mask, t["tri_start"], h, d)
    zt = z.transpose(0, 1)
    z = (zt + _tri_exact(zt, None if mask is None else mask.T, t["tri_end"], h, d)).transpose(0, 1)
    return z, t["s"] + _apb_exact(t["s"], z, t["single_mask"], t["apb"], h, d)
