"""SiLU of the wide tiled kernels (wide.hip) at every value a 16-bit gate can take: the class (finite,
infinite, NaN), the exact value rounded to the activation type, and no more misrounded outputs than
the weight-streaming kernels have; and the bits of the terms that the down projection weighs. One
expert; each token carries one gate pattern.

The finite gates: x[t] = (pattern_t, 1, 0, ...), W1 row i = (1, 0, ...), W3 row i = (0, u_i, 0, ...),
W2 = identity: output h is round(silu(pattern_t) * u_h), with no sum of more than one non-zero
product. Infinite gates come from an overflowing product (an infinite x would meet the zeros of the
other rows as inf * 0)."""
import numpy as np
import pytest
import torch

from ae_amd import _lib
from ae_amd.layers import stack_fused_moe, tiled_min_tokens

pytestmark = pytest.mark.gpu
DEV = "cuda"
H = I = 128
# bits below the leading one; smallest normal exponent
FORM = {torch.bfloat16: (7, -126), torch.float16: (10, -14)}


def _layer(x, w1, w3, w2, wide, w=None):
    T = x.shape[0]
    pool = torch.cat([w1.reshape(-1), w3.reshape(-1), w2.reshape(-1)]).to(x.dtype).view(1, -1)
    ids = torch.zeros((T, 1), dtype=torch.int32, device=DEV)
    w = torch.ones((T, 1), device=DEV) if w is None else w
    slots = torch.zeros((1,), dtype=torch.int64, device=DEV)
    logits = torch.zeros((T, 1), dtype=x.dtype, device=DEV)
    code = _lib.SMX_BF16 if x.dtype == torch.bfloat16 else _lib.SMX_F16
    with tiled_min_tokens(0 if wide else 1 << 62):
        plan = _lib.plan_info(T, H, I, 1, 1, code)
        assert (plan["wide_pairs"] > 0, plan["splits"]) == (wide, 1)
        y = stack_fused_moe(x.clone(), pool, slots, logits, w, ids, False, inplace=False)
    torch.cuda.synchronize()
    return y


def _finite_gates(dtype):
    p = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype)
    p = p[torch.isfinite(p.float())].to(DEV)
    u = (0.5 + torch.arange(I, device=DEV) / (2.0 * I)).to(dtype)  # exact in both types
    x = torch.zeros((p.numel(), H), dtype=dtype, device=DEV)
    x[:, 0], x[:, 1] = p, 1.0
    w1 = torch.zeros((I, H), device=DEV)
    w1[:, 0] = 1.0
    w3 = torch.zeros((I, H), device=DEV)
    w3[:, 1] = u.float()
    return p, u, x, w1, w3, torch.eye(H, I, device=DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_finite_gate(dtype):
    p, u, x, w1, w3, w2 = _finite_gates(dtype)
    y = _layer(x, w1, w3, w2, True)
    assert torch.isfinite(y.float()).all(), int((~torch.isfinite(y.float())).any(1).sum())
    ys = _layer(x, w1, w3, w2, False)
    g = p.double()
    exact = (g / (1.0 + torch.exp(-g)))[:, None] * u.double()
    # half a unit of the type for its rounding; the fp32 value before it is within 2^-21 of the
    # exact one (under two units of 2^-23 of SiLU, half a unit of the product), 2^-10 of a unit of
    # fp16. Results below the smallest normal number are only bounded by it: they may be flushed.
    # Where 1 + e^-g overflows (g < -88.72) the result is -0 for an exact value above -2.8e-37.
    bits, emin = FORM[dtype]
    unit = torch.exp2(torch.floor(torch.log2(exact.abs().clamp_min(2.0 ** emin))) - bits)
    err, errs = (y.double() - exact).abs(), (ys.double() - exact).abs()
    over = (g < -88.72)[:, None].expand_as(err)
    small = (exact.abs() < 2.0 ** emin) & ~over
    rest = ~small & ~over
    assert (err <= (0.5 + 2.0 ** -9) * unit)[rest].all(), (err / unit)[rest].max().item()
    assert (err <= 2.0 ** emin)[small].all()
    assert (y[over] == 0).all() and (exact[over] >= -2.8e-37).all()
    # outputs that are not the nearest value of the type (about the fp32 error in units of the
    # type: one in 10^4 to 10^5); another SiLU of the same error misrounds others, as many
    wrong, wrongs = (int((q > 0.5 * unit)[rest].sum()) for q in (err, errs))
    print(f"misrounded of {int(rest.sum())}: wide {wrong}, streaming {wrongs}")
    assert wrong <= 1.1 * wrongs + 3 * wrongs ** 0.5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_weighted_terms(dtype):
    """One K split: the down kernel weighs and rounds its sums itself, as the combine does
    elsewhere: in fp16 rounded once from the exact product, in bf16 from the fp32 product."""
    p, _, x, w1, w3, w2 = _finite_gates(dtype)
    g = torch.Generator(device=DEV).manual_seed(5)
    w = torch.rand((p.numel(), 1), generator=g, device=DEV) + 0.25
    act = _layer(x, w1, w3, w2, True)  # weight 1: the sums themselves
    y = _layer(x, w1, w3, w2, True, w)
    if dtype == torch.float16:
        prod = act.cpu().double().numpy() * w.cpu().double().numpy()
        with np.errstate(over="ignore"):  # weights above 1 overflow the largest gates
            want = torch.from_numpy(prod.astype(np.float16)).to(DEV)
    else:
        want = (act.float() * w).to(dtype)
    assert torch.equal(y, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinite_and_nan_gates(dtype):
    big = 2.0 ** (100 if dtype == torch.bfloat16 else 15)
    T = 384
    x = torch.zeros((T, H), dtype=dtype, device=DEV)
    x[0::3, 0], x[1::3, 0], x[2::3, 0] = big, -big, float("nan")
    x[:, 1] = 1.0
    w1 = torch.zeros((I, H), device=DEV)
    w1[0, 0] = big
    w3 = torch.zeros((I, H), device=DEV)
    w3[0, 1] = 1.0
    w2 = torch.zeros((H, I), device=DEV)
    w2[:, 0] = 1.0
    for wide in (True, False):
        y = _layer(x, w1, w3, w2, wide).float()
        assert torch.isposinf(y[0::3]).all(), wide  # silu(inf) = inf
        assert torch.isnan(y[1::3]).all(), wide     # -inf / (1 + inf)
        assert torch.isnan(y[2::3]).all(), wide
