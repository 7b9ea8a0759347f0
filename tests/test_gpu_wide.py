"""GPU parity of the wide tiled kernels (wide.hip: 256 tokens x 256 weight rows, 16-bit types, from
128 expected tokens per active expert) against the oracle, at the sizes where they can go wrong:
token counts around the quarters of a tile (64) and around one and two tiles, experts without
tokens, more pairs of ranges than one wave looks at in one round, several blocks of ranges
of one expert, H of half a down tile and of one and a half, K walks of two steps, a shared
expert over several token groups, and routings with dropped assignments."""
import numpy as np
import pytest
import torch

from oracle import moe_ref as ref
from ae_amd import _lib
from ae_amd.layers import (fused_moe_forward, fused_moe_shared_forward, stack_fused_moe,
                           stack_fused_moe_shared, tiled_min_tokens)
from ae_amd.layers._torch import ptr, stream_of
from tests.helpers import (TOL, TORCH_TO_ORACLE, f32_of, make_pool, max_rel_err, nan_buffers,
                           to_oracle)

pytestmark = pytest.mark.gpu
DEV = "cuda"
DCODE = {torch.float16: _lib.SMX_F16, torch.bfloat16: _lib.SMX_BF16}


def _stack(counts, H, I, dtype, seed, unmapped=(), splits=1):
    """Every token picks one expert (k = 1): expert e gets counts[e] tokens, in a shuffled order."""
    E, T = len(counts), sum(counts)
    g = torch.Generator(device=DEV).manual_seed(seed)
    ids = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(counts, device=DEV))
    ids = ids[torch.randperm(T, generator=g, device=DEV)].to(torch.int32).view(T, 1)
    x = torch.randn((T, H), generator=g, device=DEV).to(dtype)
    w = torch.rand((T, 1), generator=g, device=DEV) + 0.5
    pool, slots = make_pool(E, H, I, dtype, num_slots=E + 2, seed=seed + 1)
    for e in unmapped:
        slots[e] = -1
    logits = torch.zeros((T, E), dtype=dtype, device=DEV)
    with tiled_min_tokens(0):
        plan = _lib.plan_info(T, H, I, E, 1, DCODE[dtype])
        assert plan["wide_pairs"] > 0 and plan["splits"] == splits
        y = stack_fused_moe(x.clone(), pool, slots, logits, w, ids, False, inplace=False)
    with tiled_min_tokens(1 << 62):
        ys = stack_fused_moe(x.clone(), pool, slots, logits, w, ids, False, inplace=False)
    torch.cuda.synchronize()
    assert torch.isfinite(y.float()).all()
    # another order of the K sums than the streaming kernels: both lie within TOL of the exact value
    assert max_rel_err(f32_of(y), f32_of(ys)) <= 2 * TOL[dtype]
    y_ref = ref.stack_fused_moe(to_oracle(x), to_oracle(pool), slots.cpu().numpy(), w.cpu().numpy(),
                                ids.cpu().numpy(), TORCH_TO_ORACLE[dtype])
    assert max_rel_err(f32_of(y), y_ref) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,H,I", [
    ([1, 511], 128, 128),                       # a one-token tile; two full tiles; two-step walks
    ([63, 64, 65, 320], 256, 256),
    ([127, 128, 129, 191, 192, 193], 384, 128),  # one and a half down tiles
    ([255, 256, 257, 0, 384, 385], 256, 384),
    ([2049, 0, 1], 128, 256),                   # nine tiles of one expert: three blocks
    ([200] * 70, 128, 128),                     # 140 ranges, 70 pairs
])
def test_wide_token_counts(dtype, counts, H, I):
    _stack(counts, H, I, dtype, seed=sum(counts) + H)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,H,I,splits", [
    ([2049, 0, 1], 128, 640, 5),
    ([63, 64, 65, 320], 256, 1024, 8),
    ([127, 128, 129, 191, 192, 193], 384, 1152, 9),
])
def test_wide_partials(dtype, counts, H, I, splits):
    """Walks of more than 6 steps: K splits, whose fp32 partials the combine adds."""
    _stack(counts, H, I, dtype, seed=sum(counts) + I, splits=splits)


@pytest.mark.parametrize("I,splits", [(256, 1), (1024, 8)])
def test_wide_dropped_assignments(I, splits):
    _stack([300, 150, 257, 129], 256, I, torch.bfloat16, seed=7, unmapped=(1,), splits=splits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("I,splits", [(128, 1), (1024, 4)])
@pytest.mark.parametrize("Is", [0, 384])
def test_wide_dropped_picks_of_a_token(dtype, I, splits, Is):
    """Tokens with some and with all of their three picks dropped (an unmapped expert, ids outside the
    experts), on an output of NaN and a workspace of 0xFF bytes: a row of terms or partials that the
    down kernel did not write is not added."""
    T, H, E, k = 700, 256, 6, 3
    r = np.random.default_rng(I + Is)
    ids = np.argsort(r.random((T, E)), axis=1)[:, :k].astype(np.int32)
    ids[r.random((T, k)) < 0.1] = -1
    ids[::7] = [2, -1, E]  # expert 2 is unmapped: nothing is left of these
    w = (r.random((T, k)) + 0.2).astype(np.float32)
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn((T, H), generator=g, device=DEV).to(dtype)
    page = (torch.randn((3 * Is * H,), generator=g, device=DEV) * 0.02).to(dtype) if Is else None
    sgate = torch.randn((T, 1), generator=g, device=DEV).to(dtype) if Is else None
    pool, slots = make_pool(E, H, I, dtype, num_slots=E + 2, seed=E)
    slots[2] = -1
    with tiled_min_tokens(0):
        plan = _lib.plan_info(T, H, I, E, k, DCODE[dtype], Is)
        assert plan["wide_pairs"] > 0 and plan["splits"] == splits
        nbytes = _lib.lib().smx_moe_shared_workspace_size(T, H, I, E, k, Is, DCODE[dtype])
        out, ws = nan_buffers(x, nbytes)
        y = stack_fused_moe_shared(x, pool, slots, torch.from_numpy(w).to(DEV), torch.from_numpy(ids).to(DEV),
                                   page, sgate, 1.0, inplace=False, out=out, workspace=ws)
    torch.cuda.synchronize()
    assert torch.isfinite(y.float()).all()
    y_ref = ref.stack_fused_moe_shared(to_oracle(x), to_oracle(pool), slots.cpu().numpy(), w, ids,
                                       TORCH_TO_ORACLE[dtype], shared_page=None if page is None else to_oracle(page),
                                       shared_gate_logits=None if sgate is None else f32_of(sgate))
    assert max_rel_err(f32_of(y), y_ref) <= TOL[dtype]
    if not Is:
        assert (y[::7] == 0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,Is", [(257, 640), (1100, 128)])
def test_wide_shared_expert(dtype, T, Is):
    H, I, E, k = 256, 128, 4, 2
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn((T, H), generator=g, device=DEV).to(dtype)
    logits = (torch.randn((T, E), generator=g, device=DEV) * 2.0).to(dtype)
    sgate = (torch.randn((T, 1), generator=g, device=DEV) * 2.0).to(dtype)
    page = (torch.randn((3 * Is * H,), generator=g, device=DEV) * 0.02).to(dtype)
    pool, slots = make_pool(E, H, I, dtype, num_slots=E + 2, seed=E + 1)
    with tiled_min_tokens(0):
        assert _lib.plan_info(T, H, I, E, k, DCODE[dtype], Is)["wide_pairs"] > 0
        y = fused_moe_shared_forward(x.clone(), logits, pool, slots, k, True, page, sgate, 1.0, inplace=False)
    torch.cuda.synchronize()
    y_ref, _, _ = ref.fused_moe_shared_forward(
        to_oracle(x), f32_of(logits), to_oracle(pool), slots.cpu().numpy(), k, True, TORCH_TO_ORACLE[dtype],
        shared_page=to_oracle(page), shared_gate_logits=f32_of(sgate), routed_scaling_factor=1.0)
    assert max_rel_err(f32_of(y), y_ref) <= TOL[dtype]


@pytest.mark.parametrize("I", [128, 1024])
def test_wide_allocation_free_entry_gives_the_same_bits(I):
    T, H, E, k = 700, 256, 4, 2
    dtype = torch.float16
    g = torch.Generator(device=DEV).manual_seed(I)
    x = torch.randn((T, H), generator=g, device=DEV).to(dtype)
    logits = (torch.randn((T, E), generator=g, device=DEV) * 2.0).to(dtype)
    pool, slots = make_pool(E, H, I, dtype, num_slots=E + 1, seed=3)
    y2 = torch.full_like(x, float("nan"))
    w = torch.empty((T, k), dtype=torch.float32, device=DEV)
    ids = torch.empty((T, k), dtype=torch.int32, device=DEV)
    with tiled_min_tokens(0):
        assert _lib.plan_info(T, H, I, E, k, _lib.SMX_F16)["wide_pairs"] > 0
        y = fused_moe_forward(x.clone(), logits, pool, slots, k, True, inplace=False)
        _lib.call("smx_fused_moe_forward_noalloc", ptr(x), ptr(y2), _lib.SMX_F16, T, H, ptr(logits), _lib.SMX_F16,
                  E, k, 1, ptr(pool), pool.shape[0], pool.shape[1], ptr(slots), ptr(w), ptr(ids), stream_of(x))
    torch.cuda.synchronize()
    assert torch.equal(y, y2)
