"""The three work splits of the bf16 block forward (1, 2 or 4 key groups per workgroup) at the edges of their tiles,
against the oracle on the same bf16 values.

Bound per element: rounding P to bf16 (relative 2^-9 each, and the row's sum is formed from the unrounded values) moves
the output by at most 2^-9 sum_j p_j |v_j|, storing it in bf16 by 2^-9 |out|; both are doubled for the fp32 sums and the
hardware exponential."""
import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N

pytestmark = pytest.mark.gpu

# B, Hq, Hkv of a small, a larger and a large launch
LAUNCHES = {4: (1, 3, 1), 2: (2, 64, 8), 1: (4, 64, 8)}
EDGES = [
    # Sq, Sc, D: rows around 32, 64, 128, 256, keys around 32, 64, 128, 256 and the rings' wrap
    (1, 1, 128), (31, 32, 128), (64, 33, 128), (65, 127, 64), (129, 128, 128), (130, 129, 40), (255, 257, 128),
    (257, 520, 64), (192, 700, 96), (33, 65, 72), (129, 257, 96),
]
DEEP = [
    # five and more tiles for every key group, the last one whole, of one key, or short of one
    (65, 640, 64), (100, 641, 96), (129, 703, 128), (257, 385, 64), (161, 321, 40), (130, 447, 72), (33, 769, 104),
    (65, 673, 128),
]
# (B, Hq, Hkv) from few to many workgroups: the first that takes a given number of key groups is the launch of a case
HEADS = [(1, 3, 1), (1, 8, 8), (1, 20, 20), (1, 40, 8), (2, 36, 36), (2, 40, 8), (2, 48, 8), (2, 56, 8), (2, 64, 8),
         (2, 72, 72), (3, 64, 8), (4, 64, 8)]
# The rule never splits a few keys among many workgroups, nor leaves them in one group: some edges exist with four only.


def taken(B, Sq, Sc, Hq, Hkv, D, causal):
    """Key groups of a launch on contiguous K / V."""
    return N.lib().mhip_attn_fwd_plan(B, Sq, Sc, Hq, D, Hkv * D, Hkv * D, int(causal), N.MHIP_BF16)


def launch(groups, Sq, Sc, D, causal):
    return next((h for h in HEADS if taken(h[0], Sq, Sc, h[1], h[2], D, causal) == groups), None)


CASES = [(groups, Sq, Sc, D, causal) for groups in (4, 2, 1) for Sq, Sc, D in EDGES + DEEP for causal in (False, True)
         if launch(groups, Sq, Sc, D, causal)]


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
    """Three launch sizes with whatever split the rule gives them (the largest has one key group at most of the edges)."""
    B, Hq, Hkv = LAUNCHES[groups]
    if groups == 1 and Sq * Sc > 140000:
        B = 2
    for causal in (False, True):
        tag = f"{taken(B, Sq, Sc, Hq, Hkv, D, causal)} groups B{B} Hq{Hq} Sq{Sq} Sc{Sc} D{D} causal={causal}"
        print(tag, flush=True)
        g = torch.Generator().manual_seed(Sq * 1009 + Sc)
        q = torch.randn(B, Sq, Hq, D, generator=g).bfloat16()
        kv = torch.randn(2, B, Sc, Hkv, D, generator=g).bfloat16()
        _compare(q, kv, D ** -0.5, causal, tag)


@pytest.mark.parametrize("groups,Sq,Sc,D,causal", CASES)
def test_every_split_at_its_edges(groups, Sq, Sc, D, causal):
    B, Hq, Hkv = launch(groups, Sq, Sc, D, causal)
    tag = f"groups {groups} B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Sc{Sc} D{D} causal={causal}"
    print(tag, flush=True)
    g = torch.Generator().manual_seed(Sq * 1009 + Sc)
    q = torch.randn(B, Sq, Hq, D, generator=g).bfloat16()
    kv = torch.randn(2, B, Sc, Hkv, D, generator=g).bfloat16()
    _compare(q, kv, D ** -0.5, causal, tag)


RAMPS = [(groups, Sq, Sc, D) for groups, Sq, Sc in ((4, 161, 700), (2, 65, 641), (1, 129, 345)) for D in (64, 40, 96, 128)]


@pytest.mark.parametrize("rising", [True, False])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("groups,Sq,Sc,D", RAMPS)
def test_a_moving_reference_in_every_split(groups, Sq, Sc, D, causal, rising):
    """Scores that climb (or fall) by 20 binades per 64 keys: climbing ones outgrow the reference in every tile, so that O
    and the sums are rescaled and the tile's exponentials redone -- over packed P that the early pairs of the matrix phase
    have written -- in each of the main loops: 64, 96 and 128 columns, one, two and four key groups."""
    B, Hq, Hkv = launch(groups, Sq, Sc, D, causal)
    tag = f"ramp groups {groups} B{B} Hq{Hq} Hkv{Hkv} Sq{Sq} Sc{Sc} D{D} causal={causal} rising={rising}"
    print(tag, flush=True)
    g = torch.Generator().manual_seed(70 + D)
    q = torch.randn(B, Sq, Hq, D, generator=g) * 0.25
    kv = torch.randn(2, B, Sc, Hkv, D, generator=g)
    kv[0] *= 0.25
    scale = D ** -0.5
    ramp = torch.arange(Sc, dtype=torch.float32) / 64.0 * 20.0 / (scale * 1.4426950408889634)
    q[..., :16] = 2.0                                              # 16 columns x 2.0 x value
    kv[0, ..., :16] = ((ramp if rising else ramp.flip(0)) / 32.0)[None, :, None, None]
    _compare(q.bfloat16(), kv.bfloat16(), scale, causal, tag)


@pytest.mark.parametrize("slope", [0.35, -0.35])
@pytest.mark.parametrize("causal", [False, True])
def test_key_groups_with_one_dominant_group(slope, causal):
    """Scores that climb or fall by a constant per key: the groups' reference scores and sums are far apart, and one
    group's part of the result vanishes beside another's."""
    B, Sq, Sc, H, D = 1, 96, 300, 2, 128
    assert taken(B, Sq, Sc, H, H, D, causal) == 4
    g = torch.Generator().manual_seed(5)
    q = torch.zeros(B, Sq, H, D)
    q[..., 0] = 8.0
    kv = torch.randn(2, B, Sc, H, D, generator=g)
    kv[0, ..., 0] = slope / 8.0 * torch.arange(Sc)[None, :, None]
    _compare(q.bfloat16(), kv.bfloat16(), 1.0, causal, f"slope {slope} causal={causal}")


@pytest.mark.parametrize("groups", [4, 2, 1])
def test_a_key_of_nan_reaches_the_row_whatever_group_holds_it(groups):
    """A row that meets NaN gets an output of NaN and, as with one key group, an LSE of -inf; other rows see nothing."""
    import mercury_artifact_amd as M

    B, Hq, Hkv = launch(groups, 256, 320, 128, True)
    g = torch.Generator().manual_seed(11)
    q = torch.randn(B, 256, Hq, 128, generator=g).bfloat16()
    kv = torch.randn(2, B, 320, Hkv, 128, generator=g).bfloat16()
    clean, clean_lse = M.attn_fwd_block(q.cuda(), kv[0].cuda(), kv[1].cuda(), 0.1, causal=True)
    kv[0, :, 240] = float("nan")                  # hidden from the rows below 176
    out, lse = M.attn_fwd_block(q.cuda(), kv[0].cuda(), kv[1].cuda(), 0.1, causal=True)
    assert torch.equal(out[:, :176], clean[:, :176]) and torch.equal(lse[..., :176], clean_lse[..., :176])
    assert bool(out[:, 176:].isnan().all()) and bool((lse[..., 176:] == -torch.inf).all())
