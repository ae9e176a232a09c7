"""attention_pair_bias at few tokens: every block shape of the one-step kernel against the oracle."""

import pytest
import torch
from _inputs import TOL_COS, TOL_MAX_ABS, apb_inputs, apb_qkn_inputs, compare, to_dev

import triangleops_amd as tops
from oracle import reference as ref

pytestmark = pytest.mark.gpu

CALL = ("X", "WQ", "WK", "WV", "Z", "W_ln", "B_ln", "W_proj_z", "B_proj_z", "W_proj_g", "B_proj_g", "W_proj_o", "B_proj_o",
        "H", "D")


# blocks of 4 (up to M = 128 or so), 8, 16 and 32 queries, the last size that has one and the first that
# does not; M at and around the edges of the query and key tiles
@pytest.mark.parametrize("M", [1, 3, 32, 33, 127, 181, 256, 257, 300, 385, 512, 513])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mask", ["none", "random", "tiles"])
def test_apb_few_tokens(device, M, dtype, mask):
    """mask "tiles": whole 32-key steps without a valid key."""
    inp = apb_inputs(M, seed=M, mask="none" if mask == "tiles" else mask, biases=True, dtype=dtype)
    if mask == "tiles":
        inp["mask"] = (torch.arange(M) // 32) % 2 == ((M - 1) // 32) % 2
    elif mask == "random":
        inp["mask"][M - 1] = True
    d = to_dev(inp, device)
    out = tops.attention_pair_bias(*(d[k] for k in CALL), scale=d["scale"], mask=d["mask"])
    expect = ref.attention_pair_bias(*(inp[k] for k in CALL), scale=inp["scale"], eps=1e-5, mask=inp["mask"])
    diff, cos = compare(out, expect)
    assert diff <= TOL_MAX_ABS[dtype] and cos >= TOL_COS, f"M={M}: max|d|={diff:.3e} cos={cos:.6f}"


@pytest.mark.parametrize("M", [33, 200, 300, 400])
def test_apb_few_tokens_from_x_and_from_qkv_bitwise(device, M):
    """The kernel's own projections and given Q / K / V (the pre-pass's) leave the same bits."""
    from triangleops_amd.attn_pair_bias.kernel import apb_forward, apb_forward_qkv, apb_qkn_prep

    inp = to_dev(apb_inputs(M, seed=M, mask="random", biases=True), device)
    pre = tops.attn_pair_bias.precompute(*(inp[k] for k in ("WQ", "WK", "WV", "W_ln", "B_ln", "W_proj_z", "B_proj_z")),
                                         inp["H"], inp["D"])
    args = (inp["Z"], pre["W_combined"], pre["sum_W_combined"], pre["B_const"])
    a, b = torch.empty(M, 128, device=device, dtype=torch.bfloat16), torch.empty(M, 128, device=device,
                                                                                 dtype=torch.bfloat16)
    apb_forward(inp["X"], pre["W_QKV"], *args, a, scale=inp["scale"], mask=inp["mask"], wqkv_hm=pre["wqkv_hm"])
    q, k, v = apb_qkn_prep(inp["X"], pre["wqkv_hm"], qscale=inp["scale"])
    apb_forward_qkv(q, k, v, *args, b, mask=inp["mask"])
    assert torch.equal(a, b)


# every block shape; remainders of the query and key tiles
@pytest.mark.parametrize("M", [33, 100, 127, 181, 200, 300, 400, 512])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mask", ["none", "random"])
def test_apb_few_tokens_bits_of_the_general_kernel(device, M, dtype, mask):
    """The few-token kernel leaves the bits of the pre-pass and the general kernel: the same tokens at the head of
    the first size that has no such form, where the keys are split into steps of 32 as well and the tokens added
    are masked keys (their steps end with an empty sum)."""
    from triangleops_amd import _native
    from triangleops_amd.attn_pair_bias.kernel import apb_forward

    big = next(n for n in range(M, 2049) if not _native.apb_single_launch(n, 4, 32))
    inp = apb_inputs(big, seed=M, mask="random", biases=True, dtype=dtype)
    inp["mask"][M - 1] = True
    inp["mask"][M:] = False
    if mask == "none":
        inp["mask"][:M] = True
    d = to_dev(inp, device)
    pre = tops.attn_pair_bias.precompute(*(d[k] for k in ("WQ", "WK", "WV", "W_ln", "B_ln", "W_proj_z", "B_proj_z")),
                                         d["H"], d["D"])
    outs = []
    for n in (M, big):
        assert _native.apb_single_launch(n, 4, 32) == (n == M)
        out = torch.empty(n, 128, device=device, dtype=dtype)
        apb_forward(d["X"][:n], pre["W_QKV"], d["Z"][:n, :n].contiguous(), pre["W_combined"], pre["sum_W_combined"],
                    pre["B_const"], out, scale=d["scale"], mask=d["mask"][:n], wqkv_hm=pre["wqkv_hm"])
        outs.append(out[:M])
    assert torch.equal(*outs)


@pytest.mark.parametrize("M", [40, 300])
def test_apb_few_tokens_qknorm(device, M):
    inp = apb_qkn_inputs(M, seed=M, mask="random")
    out = tops.attn_pair_bias.attention_pair_bias_qknorm(**to_dev(inp, device))
    expect = ref.attention_pair_bias_qknorm(**inp)
    diff, cos = compare(out, expect)
    assert diff <= TOL_MAX_ABS[torch.bfloat16] and cos >= TOL_COS, f"M={M}: max|d|={diff:.3e} cos={cos:.6f}"
