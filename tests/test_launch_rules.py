"""What the sizes of the GPU tests make the launch rules choose (host functions: no GPU needed).  A test names the kernels
it is for; when a rule moves, these assertions say which kernels have been left without one."""
import pytest
import test_gpu_fwd_key_groups as G
from test_gpu_bwd_chunk import GROUPED, IN_TURN, JOINT, form, taken as bwd_plan

from mercury_artifact_amd import _native as N


def _columns(D):
    return 64 if D <= 64 else 96 if D <= 96 else 128


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("columns", [64, 96, 128])
@pytest.mark.parametrize("groups", [1, 2, 4])
def test_every_forward_split_has_its_cases(groups, columns, causal):
    """Edge cases with at least five tiles for every key group, whole and ragged, for each instantiation; and a ramp."""
    step = 64 if groups == 1 else 128                 # keys that all groups together take per tile (32 each with four)
    deep = [c for c in G.CASES if c[0] == groups and _columns(c[3]) == columns and c[4] == causal and c[2] > 4 * step]
    assert deep and any(c[1] % 32 and c[2] % step for c in deep)
    ramps = [r for r in G.RAMPS if r[0] == groups and _columns(r[3]) == columns]
    assert ramps and all(r[2] > 4 * step and G.launch(*r, causal) for r in ramps)


def test_forward_rule():
    plan = N.lib().mhip_attn_fwd_plan
    # rows too far apart for a tile put out of range by its 32-bit offset: one group
    assert plan(1, 256, 256, 4, 128, 512, 512, 0, N.MHIP_BF16) == 4
    assert plan(1, 256, 256, 4, 128, 1 << 21, 512, 0, N.MHIP_BF16) == plan(1, 256, 256, 4, 128, 512, 1 << 21, 0, N.MHIP_BF16) == 1
    assert plan(1, 4096, 4096, 32, 128, 4096, 4096, 0, N.MHIP_BF16) == 1
    assert plan(1, 256, 256, 4, 144, 512, 512, 0, N.MHIP_BF16) < 0 and plan(1, 256, 256, 4, 64, 512, 512, 0, N.MHIP_F32) < 0
    # nothing to do, nothing to see: any split does
    for Sq, Sc in ((0, 64), (64, 0)):
        assert plan(1, Sq, Sc, 4, 128, 512, 512, 1, N.MHIP_BF16) in (1, 2, 4)


def test_backward_rule():
    assert bwd_plan(1, 4096, 4096, 32, 32, 128, False) == (2, 1, 1)
    assert bwd_plan(1, 256, 256, 4, 4, 128, False) == (1, 1, 1)
    assert bwd_plan(1, 2048, 2048, 8, 1, 128, False)[2] > 1
    assert bwd_plan(1, 0, 64, 4, 4, 128, False) == bwd_plan(1, 64, 0, 4, 4, 128, False) == (2, 1, 1)
    assert bwd_plan(1, 64, 64, 4, 3, 128, False)[0] < 0


@pytest.mark.parametrize("columns", [64, 96, 128])
def test_carried_sums_are_tested_in_both_forms(columns):
    """First, middle and last chunk (three chunks or more) with one launch per pass on every column count."""
    steps = [c for c in IN_TURN if _columns(c[4]) == columns]
    assert any(c[0] >= 3 for c in steps) and all(bwd_plan(2, c[1], c[1], *c[2:], False)[0] == 2 for c in steps)
    assert any(_columns(c[4]) == columns and bwd_plan(2, c[1], c[1], *c[2:], False)[0] == 1 for c in JOINT)


def test_blocks_of_a_step_share_a_launch_of_up_to_eight_rounds():
    group = N.lib().mhip_attn_fwd_group
    assert group(1, 16384, 32, 8) == group(1, 8193, 32, 8) == 1               # more than four rounds by itself
    assert group(1, 8192, 32, 8) == 2 and group(1, 4096, 32, 8) == 4 and group(1, 2048, 32, 8) == 8
    assert group(1, 4096, 32, 7) == 4 and group(1, 4096, 32, 5) == 3          # 4 + 3, 3 + 2
    assert group(4, 512, 5, 8) == 8 and group(1, 256, 4, 4) == 4
    assert group(1, 16, 1, 64) == 16                                          # what an argument list holds
    assert group(1, 256, 4, 1) == 1 and group(1, 0, 4, 8) == group(0, 64, 4, 8) == 1
    assert group(1, 64, 0, 8) < 0 and group(1, 64, 4, 0) < 0 and group(-1, 64, 4, 1) < 0


def test_chunks_of_a_backward_step_go_together():
    """What the ring driver asks for, and the form of the call it then makes."""
    take = N.lib().mhip_attn_bwd_take
    assert take(1, 4096, 4096, 32, 32, 128, 8) == 8 and form(8, 1, 4096, 4096, 32, 32, 128) == (2, 1, 16)
    assert take(1, 1024, 1024, 32, 32, 128, 8) == 8 and form(8, 1, 1024, 1024, 32, 32, 128) == (1, 1, 32)
    assert take(1, 6000, 6000, 5, 5, 128, 8) == 4                             # 8 would be expected to gain 0.3 %
    assert take(4, 512, 512, 5, 5, 128, 8) == 8 and form(8, 4, 512, 512, 5, 5, 128) == (1, 1, 32)
    assert take(1, 512, 512, 4, 4, 128, 8) == 8 and form(8, 1, 512, 512, 4, 4, 128) == (1, 4, 32)
    assert take(1, 64, 64, 1, 1, 64, 40) == 14 and form(14, 1, 64, 64, 1, 1, 64) == (1, 1, 32)
    # shared query tiles: not for 4 us of a step that the host takes longer over, nor where the keys' workgroups take as long
    assert form(8, 1, 256, 256, 4, 4, 64) == (1, 8, 32) and form(3, 1, 700, 700, 8, 8, 128) == (1, 2, 32)
    assert form(8, 1, 128, 128, 16, 16, 128) == form(3, 2, 997, 997, 4, 2, 128) == form(2, 1, 564, 564, 8, 8, 80) == (1, 1, 32)
    assert form(2, 4, 319, 319, 32, 32, 64) == (2, 1, 32)                     # also where mhip_attn_bwd_group says 2
    assert form(8, 1, 2048, 2048, 32, 32, 64) == (2, 1, 32)                   # 64 columns keep the larger MFMA tiles
    assert take(1, 256, 256, 4, 4, 64, 1) == take(0, 64, 64, 4, 4, 64, 8) == take(1, 0, 64, 4, 4, 64, 8) == 1
    assert take(1, 64, 64, 4, 3, 64, 8) < 0 and take(1, 64, 64, 4, 4, 136, 8) < 0 and take(1, 64, 64, 4, 4, 64, 0) < 0
    assert form(17, 1, 64, 64, 4, 4, 64)[0] < 0 and form(0, 1, 64, 64, 4, 4, 64)[0] < 0 and form(1, 1, 64, 64, 4, 3, 64)[0] < 0
    for W, B, S, Hq, Hkv, D, group in GROUPED:
        assert take(B, S, S, Hq, Hkv, D, W) == group and form(group, B, S, S, Hq, Hkv, D)[0] == 1


def test_mfma_tiles_of_the_forward():
    tile = N.lib().mhip_attn_fwd_tile
    rows = [4096, 4096]
    assert [tile(8, 8, 1, 4096, 4096, 32, D, *rows, 0) for D in (64, 96, 128)] == [16, 16, 16]
    assert [tile(1, 1, 1, 4096, 4096, 32, D, *rows, 1) for D in (64, 96, 128)] == [32, 32, 16]
    assert [tile(1, 1, 1, 4096, 4096, 32, D, *rows, 0) for D in (64, 72, 96, 128)] == [32, 16, 16, 16]
    assert [tile(8, 1, 1, 4096, 4096, 32, D, *rows, 0) for D in (64, 96, 128)] == [32, 16, 16]       # chunk by chunk in one launch
    assert tile(8, 8, 1, 256, 256, 32, 128, *rows, 0) == 32 and tile(1, 1, 2, 256, 2048, 128, 128, *rows, 0) == 16
    assert tile(1, 1, 2, 256, 2048, 128, 96, *rows, 0) == 32                  # 32 key tiles: 64 from here on
    assert tile(1, 1, 1, 256, 256, 4, 128, *rows, 0) == 32                    # four key groups
    assert tile(0, 1, 1, 64, 64, 4, 128, *rows, 0) < 0 and tile(2, 3, 1, 64, 64, 4, 128, *rows, 0) < 0
    assert tile(2, 2, 1, 64, 64, 4, 128, *rows, 1) < 0 and tile(1, 1, 1, 64, 64, 4, 136, *rows, 0) < 0


def test_chunks_of_a_backward_step_share_a_launch():
    group = N.lib().mhip_attn_bwd_group
    assert group(1, 4096, 4096, 32, 32, 128, 8) == 1                          # 2048 workgroups by itself
    assert group(4, 512, 512, 5, 5, 128, 8) == group(1, 512, 512, 8, 1, 128, 8) == 8
    assert group(1, 1024, 1024, 32, 32, 128, 8) == 4                          # at most 2048 workgroups
    assert group(1, 64, 64, 1, 1, 64, 40) == 14                               # of at most 16: three launches
    assert group(1, 256, 256, 4, 4, 64, 1) == group(0, 64, 64, 4, 4, 64, 8) == group(1, 0, 64, 4, 4, 64, 8) == 1
    assert group(1, 64, 64, 4, 3, 64, 8) < 0 and group(1, 64, 64, 4, 4, 136, 8) < 0 and group(1, 64, 64, 4, 4, 64, 0) < 0


def test_runs_of_chunks_where_blocks_would_take_turns_on_the_cus():
    chain = N.lib().mhip_attn_fwd_chain
    for dtype in (N.MHIP_BF16, N.MHIP_E4M3):
        assert chain(1, 4096, 4096, 32, 128, 8, dtype) == chain(1, 2048, 2048, 32, 128, 8, dtype) == 8
        assert chain(1, 256, 256, 4, 64, 4, dtype) == chain(1, 512, 512, 8, 128, 16, dtype) == 1      # all side by side
        assert chain(1, 4096, 4096, 32, 128, 1, dtype) == chain(1, 4096, 0, 32, 128, 8, dtype) == chain(0, 64, 64, 4, 128, 8, dtype) == 1
        assert chain(1, 4096, 4096, 32, 128, 17, dtype) == 1                                          # more than a launch takes
        assert chain(1, 64, 64, 0, 128, 8, dtype) < 0 and chain(1, 64, 64, 4, 136, 8, dtype) < 0 and chain(1, 64, 64, 4, 64, 0, dtype) < 0
    assert chain(1, 1024, 1024, 32, 128, 8, N.MHIP_BF16) == 4             # 256 workgroups, and two results to fold
    assert chain(2, 1237, 1237, 16, 80, 8, N.MHIP_BF16) == 1              # 160 workgroups: any run leaves a ragged round
    assert chain(1, 64, 64, 4, 64, 8, N.MHIP_F32) < 0
