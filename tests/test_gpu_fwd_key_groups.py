"""The three work splits of the bf16 block forward (1, 2 or 4 key groups per workgroup) at the edges of their tiles,
against the oracle on the same bf16 values.

Bound per element: rounding P to bf16 (relative 2^-9 each, and the row's sum is formed from the unrounded values) moves
the output by at most 2^-9 sum_j p_j |v_j|, storing it in bf16 by 2^-9 |out|; both are doubled for the fp32 sums and the
hardware exponential."""
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu

# B, Hq, Hkv such that launches of a few hundred rows take 4, 2 and 1 key groups
LAUNCHES = {4: (1, 3, 1), 2: (2, 64, 8), 1: (4, 64, 8)}
EDGES = [
    # Sq, Sc, D: rows around 32, 64, 128, 256, keys around 32, 64, 128, 256 and the rings' wrap
    (1, 1, 128), (31, 32, 128), (64, 33, 128), (65, 127, 64), (129, 128, 128), (130, 129, 40), (255, 257, 128),
    (257, 520, 64), (192, 700, 96), (33, 65, 72), (129, 257, 96),
]


def _compare(q, kv, scale, causal, tag):
    import mercury_artifact_amd as M

    k, v = kv[0].float(), kv[1].float()
    ro, rl = O.block_attention(q.float(), k, v, scale, causal=causal)
    amp, _ = O.block_attention(q.float(), k, v.abs(), scale, causal=causal)
    out, lse = M.attn_fwd_block(q.cuda(), kv[0].cuda(), kv[1].cuda(), scale, causal=causal)
    out, lse = out.float().cpu(), lse.cpu()
    assert torch.equal(torch.isinf(lse), torch.isinf(rl)), tag
    assert bool(((out - ro).abs() <= 2 ** -8 * (amp + ro.abs()) + 1e-6).all()), (tag, (out - ro).abs().max().item())
    seen = ~torch.isinf(rl)
    assert bool(((lse[seen] - rl[seen]).abs() <= 1e-5 * rl[seen].abs().clamp_min(1.0)).all()), tag


@pytest.mark.parametrize("groups", [4, 2, 1])
@pytest.mark.parametrize("Sq,Sc,D", EDGES)
def test_key_groups_at_tile_edges(groups, Sq, Sc, D):
    B, Hq, Hkv = LAUNCHES[groups]
    if groups == 1 and Sq * Sc > 140000:
        B = 2
    for causal in (False, True):
        tag = f"groups {groups} B{B} Hq{Hq} Sq{Sq} Sc{Sc} D{D} causal={causal}"
        print(tag, flush=True)
        g = torch.Generator().manual_seed(Sq * 1009 + Sc)
        q = torch.randn(B, Sq, Hq, D, generator=g).bfloat16()
        kv = torch.randn(2, B, Sc, Hkv, D, generator=g).bfloat16()
        _compare(q, kv, D ** -0.5, causal, tag)


@pytest.mark.parametrize("slope", [0.35, -0.35])
@pytest.mark.parametrize("causal", [False, True])
def test_key_groups_with_one_dominant_group(slope, causal):
    """Scores that climb or fall by a constant per key: the groups' reference scores and sums are far apart, and one
    group's part of the result vanishes beside another's."""
    B, Sq, Sc, H, D = 1, 96, 300, 2, 128
    g = torch.Generator().manual_seed(5)
    q = torch.zeros(B, Sq, H, D)
    q[..., 0] = 8.0
    kv = torch.randn(2, B, Sc, H, D, generator=g)
    kv[0, ..., 0] = slope / 8.0 * torch.arange(Sc)[None, :, None]
    _compare(q.bfloat16(), kv.bfloat16(), 1.0, causal, f"slope {slope} causal={causal}")


@pytest.mark.parametrize("launch", [4, 2, 1])
def test_a_key_of_nan_reaches_the_row_whatever_group_holds_it(launch):
    """A row that meets NaN gets an output of NaN and, as with one key group, an LSE of -inf; other rows see nothing."""
    import mercury_artifact_amd as M

    B, Hq, Hkv = LAUNCHES[launch]
    g = torch.Generator().manual_seed(11)
    q = torch.randn(B, 256, Hq, 128, generator=g).bfloat16()
    kv = torch.randn(2, B, 320, Hkv, 128, generator=g).bfloat16()
    clean, clean_lse = M.attn_fwd_block(q.cuda(), kv[0].cuda(), kv[1].cuda(), 0.1, causal=True)
    kv[0, :, 240] = float("nan")                  # hidden from the rows below 176
    out, lse = M.attn_fwd_block(q.cuda(), kv[0].cuda(), kv[1].cuda(), 0.1, causal=True)
    assert torch.equal(out[:, :176], clean[:, :176]) and torch.equal(lse[..., :176], clean_lse[..., :176])
    assert bool(out[:, 176:].isnan().all()) and bool((lse[..., 176:] == -torch.inf).all())
