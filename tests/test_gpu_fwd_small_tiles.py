"""The bf16 forward on 16 x 16 MFMA tiles, which launches take that keep every CU busy for long: 256 workgroups of at least 32
key tiles (64 up to 96 columns; none but runs of chunks up to 64), causal launches of 512 and more.  Against the oracle on some of the
heads, with the bound of test_gpu_fwd_key_groups.py."""
import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N

pytestmark = pytest.mark.gpu
HEADS = 128          # of a batch of 2: 256 workgroups of up to 256 rows


def _check(q, kv, out, lse, scale, causal, tag, heads):
    G = q.shape[2] // kv.shape[3]
    for b, h in heads:
        one = [t[b:b + 1, :, h:h + 1].float() for t in (q, kv[0][:, :, h // G:h // G + 1].expand(-1, -1, q.shape[2], -1),
                                                        kv[1][:, :, h // G:h // G + 1].expand(-1, -1, q.shape[2], -1))]
        ro, rl = O.block_attention(*one, scale, causal=causal)
        amp, _ = O.block_attention(one[0], one[1], one[2].abs(), scale, causal=causal)
        o, l = out[b:b + 1, :, h:h + 1].float().cpu(), lse[b:b + 1, h:h + 1].cpu()
        assert torch.equal(torch.isinf(l), torch.isinf(rl)), tag
        assert bool(((o - ro).abs() <= 2 ** -8 * (amp + ro.abs()) + 1e-6).all()), (tag, (o - ro).abs().max().item())
        seen = ~torch.isinf(rl)
        assert bool(((l[seen] - rl[seen]).abs() <= 1e-5 * rl[seen].abs().clamp_min(1.0)).all()), tag


def _run(Sq, Sc, D, n, causal, ramp, tag):
    """n chunks as one result (n = 1: a lone block)."""
    B, H, Hkv, heads = (1, 32, 8, [(0, 0), (0, 31)]) if causal else (2, HEADS, 8, [(0, 0), (0, 77), (1, 127)])
    assert N.lib().mhip_attn_fwd_tile(n, n, B, Sq, Sc, H, D, Hkv * D, Hkv * D, int(causal)) == (16 if D > 64 or n > 1 else 32)
    print(tag, flush=True)
    g = torch.Generator().manual_seed(Sq * 1009 + Sc + D)
    q = torch.randn(B, Sq, H, D, generator=g)
    kv = torch.randn(2, B, Sc * n, Hkv, D, generator=g)
    scale = D ** -0.5
    if ramp:
        q, kv[0] = q * 0.25, kv[0] * 0.25
        level = torch.arange(Sc * n, dtype=torch.float32) / 64.0 * 20.0 / (scale * 1.4426950408889634)
        q[..., :16] = 2.0
        kv[0, ..., :16] = ((level if ramp > 0 else level.flip(0)) / 32.0)[None, :, None, None]
    q, kv = q.bfloat16(), kv.bfloat16()
    out = torch.full((1, B, Sq, H, D), 7.0, dtype=torch.bfloat16, device="cuda")
    lse = torch.full((1, B, H, Sq), 7.0, device="cuda")
    chunks = [kv[:, :, i * Sc:(i + 1) * Sc].contiguous().cuda() for i in range(n)]
    assert N.host.fwd_blocks(q.cuda(), chunks, n, scale, causal, None, None, None, out, lse, 0) is True
    torch.cuda.synchronize()
    _check(q, kv, out[0], lse[0], scale, causal, tag, heads)


@pytest.mark.parametrize("D,tiles", [(128, 32), (104, 33), (96, 64), (72, 64), (64, 64), (40, 65)])
@pytest.mark.parametrize("Sq,last", [(256, 64), (241, 1), (225, 63), (255, 17), (240, 33)])
def test_a_block_at_tile_edges(Sq, last, D, tiles):
    """The last tile whole, of one key, short of one, and ending inside and between its 16-key blocks; rows that end inside
    and between the 16-row blocks of the last wavefront."""
    _run(Sq, (tiles - 1) * 64 + last, D, 1, False, 0, f"small tiles Sq{Sq} Sc{(tiles - 1) * 64 + last} D{D}")


@pytest.mark.parametrize("D,n,Sc", [(128, 3, 700), (112, 2, 1024), (96, 5, 833), (80, 16, 255), (64, 4, 1025), (24, 2, 2048)])
def test_a_run_of_chunks(D, n, Sc):
    _run(250, Sc, D, n, False, 0, f"small tiles, run of {n} Sc{Sc} D{D}")


@pytest.mark.parametrize("Sq,Sc", [(4097, 4097), (4090, 4225), (4352, 4033)])
def test_under_the_causal_mask(Sq, Sc):
    """Rows that see every key, none, and keys up to a diagonal inside a 16-key block."""
    _run(Sq, Sc, 128, 1, True, 0, f"small tiles, causal Sq{Sq} Sc{Sc}")


@pytest.mark.parametrize("ramp", [1, -1])
@pytest.mark.parametrize("Sq,Sc,D,n,causal", [(241, 2100, 128, 1, False), (241, 4100, 96, 1, False), (241, 4100, 64, 1, False),
                                              (225, 800, 128, 3, False), (4100, 4100, 128, 1, True)])
def test_a_moving_reference(Sq, Sc, D, n, causal, ramp):
    """Scores that climb or fall by 20 binades per 64 keys, as in test_gpu_fwd_key_groups.py."""
    _run(Sq, Sc, D, n, causal, ramp, f"small tiles, ramp {ramp} Sq{Sq} Sc{Sc} D{D} n{n} causal={causal}")


def test_rows_move_their_references_on_their_own():
    """Only one row in 16 outgrows its reference, and only in one tile: the other rows of its lane keep theirs."""
    B, Sq, Sc, H, D = 2, 256, 2048, HEADS, 128
    assert N.lib().mhip_attn_fwd_tile(1, 1, B, Sq, Sc, H, D, 8 * D, 8 * D, 0) == 16
    g = torch.Generator().manual_seed(3)
    q, kv = torch.randn(B, Sq, H, D, generator=g), torch.randn(2, B, Sc, 8, D, generator=g)
    q[..., 0] = 0.0
    q[:, 5::16, :, 0] = 40.0
    kv[0, ..., 0] = 0.0
    kv[0, :, 1000, :, 0] = 40.0
    q, kv = q.bfloat16(), kv.bfloat16()
    out, lse = torch.empty(1, B, Sq, H, D, dtype=torch.bfloat16, device="cuda"), torch.empty(1, B, H, Sq, device="cuda")
    assert N.host.fwd_blocks(q.cuda(), [kv.cuda()], 1, D ** -0.5, False, None, None, None, out, lse, 0) is True
    torch.cuda.synchronize()
    _check(q, kv, out[0], lse[0], D ** -0.5, False, "own references", [(0, 3), (1, 100)])


def test_a_key_of_nan_reaches_the_rows_that_see_it():
    import mercury_artifact_amd as M

    assert N.lib().mhip_attn_fwd_tile(1, 1, 1, 4100, 4100, 32, 128, 1024, 1024, 1) == 16
    g = torch.Generator().manual_seed(11)
    q = torch.randn(1, 4100, 32, 128, generator=g).bfloat16().cuda()
    kv = torch.randn(2, 1, 4100, 8, 128, generator=g).bfloat16().cuda()
    clean, clean_lse = M.attn_fwd_block(q, kv[0], kv[1], 0.1, causal=True)
    kv[0, :, 3000] = float("nan")
    out, lse = M.attn_fwd_block(q, kv[0], kv[1], 0.1, causal=True)
    first = 2816          # rows of the workgroup that meets the key's tile see it as NaN x 0 only behind the diagonal
    assert torch.equal(out[:, :first], clean[:, :first]) and torch.equal(lse[..., :first], clean_lse[..., :first])
    assert bool(out[:, 3000:].isnan().all()) and bool((lse[..., 3000:] == -torch.inf).all())
