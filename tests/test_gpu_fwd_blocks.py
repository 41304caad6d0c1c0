"""Several block forwards of a step in one launch (mhip_attn_fwd_blocks) against the oracle, and which rings get them."""
import math

import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _loaded():
    N.lib()                    # the host module answers once it knows the library's entry points


def _inputs(n, B, Sq, Sc, Hq, Hkv, D, fp8):
    g = torch.Generator().manual_seed(n * 1000 + Sq + Sc)
    q = torch.randn(B, Sq, Hq, D, generator=g)
    chunks = [torch.randn(2, B, Sc, Hkv, D, generator=g) for _ in range(n)]
    if fp8:
        (qq, sq), made = O.quantize_e4m3(q), [O.quantize_e4m3(c) for c in chunks]
        scale = max(s for _, s in made)
        chunks = [(c / scale).clamp(-448, 448).to(torch.float8_e4m3fn) for c in chunks]
        return qq, chunks, sq, scale
    return q.bfloat16(), [c.bfloat16() for c in chunks], None, None


@pytest.mark.parametrize("n,B,Sq,Sc,Hq,Hkv,D,causal,fp8", [
    (1, 1, 64, 64, 1, 1, 128, False, False), (16, 1, 33, 70, 2, 1, 128, False, False), (4, 1, 256, 256, 4, 4, 64, False, False),
    (5, 2, 257, 130, 3, 3, 96, False, False), (3, 1, 100, 0, 2, 2, 64, False, False), (7, 2, 300, 200, 4, 2, 80, True, False),
    (4, 1, 512, 512, 8, 8, 128, True, False), (2, 1, 1024, 384, 32, 8, 128, False, False), (3, 1, 200, 300, 5, 5, 64, True, False),
    (4, 1, 256, 256, 4, 4, 128, False, True), (9, 1, 129, 200, 2, 1, 64, False, True), (4, 1, 512, 300, 8, 8, 96, True, True)])
def test_blocks_of_a_launch_match_the_oracle(n, B, Sq, Sc, Hq, Hkv, D, causal, fp8):
    """Every block of a launch, with ragged tiles, grouped heads and (batch, head) counts that do and do not divide over
    the XCDs, into places behind a first one that stays as it was.  bf16: one rounding of the result and of P, 2^-8 each
    of |out| <= max |v| < 5.5; e4m3: the bound of rounding P to e4m3 besides."""
    q, chunks, sq, sc = _inputs(n, B, Sq, Sc, Hq, Hkv, D, fp8)
    scale = D ** -0.5
    print(f"n{n} B{B} Sq{Sq} Sc{Sc} H{Hq}/{Hkv} D{D} causal={causal} fp8={fp8}", flush=True)
    outs = torch.full((n + 1, B, Sq, Hq, D), 7.0, dtype=torch.bfloat16, device="cuda")
    lses = torch.full((n + 1, B, Hq, Sq), 7.0, device="cuda")
    ds = [None] * 3 if not fp8 else [t.cuda().reshape(()) for t in (sq, sc, sc)]
    assert N.host.fwd_blocks(q.cuda(), [c.cuda() for c in chunks], 1, scale, causal, *ds, outs, lses, 1) is True
    torch.cuda.synchronize()
    assert (outs[0] == 7).all() and (lses[0] == 7).all()
    for i, c in enumerate(chunks):
        if fp8:
            ops = (O.dequantize(q, sq), O.dequantize(c[0], sc), O.dequantize(c[1], sc))
            bound = O.e4m3_p_rounding_bound(*ops, scale, causal=causal)
        else:
            ops, bound = (q.float(), c[0].float(), c[1].float()), 0.0
        ro, rl = O.block_attention(*ops, scale, causal=causal)
        got, lse = outs[i + 1].float().cpu(), lses[i + 1].cpu()
        assert ((got - ro).abs() - (bound + 2 ** -8 * ro.abs())).max().item() <= 2e-2, i
        assert torch.equal(torch.isinf(lse), torch.isinf(rl)), i
        seen = ~torch.isinf(rl)
        assert not seen.any() or ((lse[seen] - rl[seen]).abs() / rl[seen].abs().clamp_min(1.0)).max().item() <= 1e-3, i


def test_blocks_refuse_what_a_launch_cannot_take():
    """Chunks of another shape or layout, too many of them, places too few: left to the caller, nothing written."""
    q, chunks, _, _ = _inputs(3, 1, 64, 64, 2, 2, 64, False)
    q, chunks = q.cuda(), [c.cuda() for c in chunks]
    outs, lses = torch.full((3, 1, 64, 2, 64), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((3, 1, 2, 64), 7.0, device="cuda")

    def call(cs, first=0, q=q):
        return N.host.fwd_blocks(q, cs, 1, 0.1, False, None, None, None, outs, lses, first)

    strided = torch.empty(2, 1, 64, 2, 128, dtype=torch.bfloat16, device="cuda")[..., :64]
    assert call([]) is call(chunks, 1) is call(chunks, -1) is call(chunks * 6) is None
    assert call([chunks[0], chunks[1][:, :, :32]]) is call([chunks[0], strided]) is call([chunks[0], chunks[1].float()]) is None
    assert call([chunks[0], chunks[1].cpu()]) is call(chunks, q=q.float()) is None
    torch.cuda.synchronize()
    assert (outs == 7).all() and (lses == 7).all()
    assert call([strided] * 3) is True                                  # one layout for all, rows 256 bytes apart


@pytest.mark.parametrize("path", ["ring", "packed", "zigzag"])
@pytest.mark.parametrize("own_class", [False, True])
def test_only_rings_with_resident_chunks_get_grouped_launches(path, own_class):
    """A class derived from LocalRing may receive into a buffer it uses again, as this one does: its blocks are launched one
    by one, before the next hop overwrites their chunk.  Same results either way."""
    import mercury_artifact_amd as M
    from mercury_artifact_amd import flash_attn_interface as FI

    class OneBuffer(M.LocalRing):
        def send_recv(self, to, source, x, recv_tensor=None):
            got = super().send_recv(to, source, x)
            self.spare = getattr(self, "spare", None)
            if self.spare is None:
                self.spare = [torch.empty_like(got), torch.empty_like(got)]
            self.spare.reverse()
            return self.spare[0].copy_(got)

    q, chunks, _, _ = _inputs(4, 1, 130, 130, 2, 2, 64, False)
    q, chunks = q.cuda(), [c.cuda() for c in chunks]
    o, lse = torch.empty_like(q), torch.empty(1, 2, 130, device="cuda")
    step = {"ring": M.flash_attn_pack_kv, "packed": M.flash_attn_expose_reduce, "zigzag": M.zigzag_causal_pack_kv}[path]
    blocks, real = [], FI.attn_fwd_block
    FI.attn_fwd_block = lambda *a: blocks.append(1) or real(*a)
    try:
        step(q, chunks[2], o, lse, 0.125, ring=(OneBuffer if own_class else M.LocalRing)((4,), 2, chunks))
    finally:
        FI.attn_fwd_block = real
    torch.cuda.synchronize()
    # (zigzag at rank 2: the diagonal and, alone of its kind, the one chunk of a later rank have launches of their own)
    assert len(blocks) == (4 if own_class else {"ring": 0, "packed": 0, "zigzag": 2}[path])
    want, wl = torch.empty_like(o), torch.empty_like(lse)
    step(q, chunks[2], want, wl, 0.125, ring=M.LocalRing((4,), 2, chunks), deferred_merge=False)
    assert (o.float() - want.float()).abs().max().item() <= 2e-2 and (lse - wl).abs().max().item() <= 1e-3


@pytest.mark.parametrize("n,per,B,Sq,Sc,Hq,Hkv,D", [
    (2, 2, 1, 64, 64, 1, 1, 128), (16, 16, 1, 33, 1, 2, 1, 128), (5, 2, 2, 257, 65, 3, 3, 96), (5, 5, 1, 300, 257, 4, 2, 64),
    (3, 2, 1, 200, 320, 8, 8, 128), (7, 3, 1, 130, 200, 2, 2, 80), (4, 4, 1, 512, 512, 4, 4, 128), (9, 8, 2, 100, 130, 5, 5, 40),
    (6, 6, 1, 70, 448, 2, 1, 64), (8, 4, 1, 256, 383, 2, 2, 96)])
@pytest.mark.parametrize("ramp", [0.0, 30.0])
def test_chunks_of_one_result_match_the_oracle(n, per, B, Sq, Sc, Hq, Hkv, D, ramp):
    """Runs of chunks as one sequence of tiles: chunks of one tile to eight (fewer than, as many as and more than are requested
    ahead), ragged ends inside the sequence, a last run that is shorter; with a ramp the scores climb by 30 nats from the
    first chunk to the last, so that the reference of a row moves in later chunks.  Against attention over all keys of a
    run in fp32: one rounding of P and of the result."""
    q, chunks, _, _ = _inputs(n, B, Sq, Sc, Hq, Hkv, D, False)
    scale = D ** -0.5
    if ramp:
        q[..., :8] = 2.0
        for i, c in enumerate(chunks):
            c[0][..., :8] = ramp * i / max(n - 1, 1) / 16.0 / scale
    print(f"n{n} per{per} B{B} Sq{Sq} Sc{Sc} H{Hq}/{Hkv} D{D} ramp={ramp}", flush=True)
    runs = [chunks[i:i + per] for i in range(0, n, per)]
    outs = torch.full((len(runs) + 1, B, Sq, Hq, D), 7.0, dtype=torch.bfloat16, device="cuda")
    lses = torch.full((len(runs) + 1, B, Hq, Sq), 7.0, device="cuda")
    assert N.host.fwd_blocks(q.cuda(), [c.cuda() for c in chunks], per, scale, False, None, None, None, outs, lses, 0) is True
    torch.cuda.synchronize()
    assert (outs[-1] == 7).all() and (lses[-1] == 7).all()
    for i, run in enumerate(runs):
        k, v = torch.cat([c[0] for c in run], 1).float(), torch.cat([c[1] for c in run], 1).float()
        ro, rl = O.block_attention(q.float(), k, v, scale)
        got = outs[i].float().cpu()
        assert ((got - ro).abs() - 2 ** -8 * ro.abs()).max().item() <= 2e-2, i
        assert (got - ro).norm() <= 1e-2 * ro.norm(), i
        assert ((lses[i].cpu() - rl).abs() / rl.abs().clamp_min(1.0)).max().item() <= 1e-3, i


def test_a_run_of_chunks_needs_one_row_stride_and_no_mask():
    q, chunks, _, _ = _inputs(4, 1, 64, 64, 2, 2, 64, False)
    q, chunks = q.cuda(), [c.cuda() for c in chunks]
    outs, lses = torch.full((2, 1, 64, 2, 64), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((2, 1, 2, 64), 7.0, device="cuda")
    call = lambda per, causal, first=0: N.host.fwd_blocks(q, chunks, per, 0.1, causal, None, None, None, outs, lses, first)
    assert call(2, True) is call(0, False) is call(17, False) is call(2, False, 1) is call(1, False) is None
    torch.cuda.synchronize()
    assert (outs == 7).all() and (lses == 7).all()
    assert call(2, False) is True


@pytest.mark.parametrize("fp8,D", [(False, 64), (False, 128), (True, 128)])
def test_a_run_of_chunks_whose_rows_lie_at_one_place(fp8, D):
    """Row stride 0 (an expanded chunk): every chunk of the run is visited for all of its keys, bit for bit as where the same
    keys lie in memory."""
    g = torch.Generator(device="cuda").manual_seed(21)
    q = torch.randn(1, 300, 4, D, generator=g, device="cuda")
    one = [torch.randn(2, 1, 1, 4, D, generator=g, device="cuda") * (i + 1) for i in range(3)]
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    q, one, got = q.to(kind), [c.to(kind) for c in one], []
    descale = torch.ones((), device="cuda") if fp8 else None
    for chunks in ([c.expand(-1, -1, 200, -1, -1) for c in one], [c.expand(-1, -1, 200, -1, -1).contiguous() for c in one]):
        out, lse = torch.empty(1, 1, 300, 4, D, dtype=torch.bfloat16, device="cuda"), torch.empty(1, 1, 4, 300, device="cuda")
        assert N.host.fwd_blocks(q, chunks, 3, 0.125, False, descale, descale, descale, out, lse, 0) is True
        got.append((out, lse))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def test_the_only_result_of_a_step_goes_straight_out_unless_the_output_is_read():
    """Steps whose chunks all go into one result write the caller's tensors; an output that lies over the queries or over a
    chunk is written by a fold behind the launch instead."""
    import mercury_artifact_amd as M

    W, S, H, D = 2, 1024, 64, 128
    assert N.lib().mhip_attn_fwd_chain(1, S, S, H, D, W, N.MHIP_BF16) == W
    q, chunks, _, _ = _inputs(W, 1, S, S, H, H, D, False)
    want = None
    for over in ("nothing", "q", "chunk"):
        qd, dev = q.cuda(), [c.cuda() for c in chunks]
        o = {"nothing": torch.empty_like(qd), "q": qd, "chunk": dev[1][0]}[over]
        lse = torch.empty(1, H, S, device="cuda")
        M.flash_attn_pack_kv(qd, dev[0], o, lse, D ** -0.5, ring=M.LocalRing((W,), 0, dev))
        torch.cuda.synchronize()
        if want is None:
            want = o.clone(), lse.clone()
            ro, rl = O.block_attention(q.float(), *(torch.cat([c[i] for c in chunks], 1).float() for i in (0, 1)), D ** -0.5)
            assert (o.float().cpu() - ro).norm() <= 1e-2 * ro.norm()
        assert torch.equal(o, want[0]) and (lse - want[1]).abs().max().item() <= 1e-5, over


@pytest.mark.parametrize("n,per,B,Sq,Sc,Hq,Hkv,D", [
    (2, 2, 1, 64, 64, 1, 1, 128), (16, 16, 1, 33, 1, 2, 1, 128), (5, 2, 2, 257, 129, 3, 3, 96), (5, 5, 1, 300, 257, 4, 2, 64),
    (3, 3, 1, 200, 640, 4, 4, 128), (7, 3, 1, 130, 200, 2, 2, 80), (4, 2, 1, 130, 320, 130, 130, 128), (9, 8, 1, 130, 70, 130, 1, 64),
    (4, 4, 1, 130, 191, 130, 130, 96)])
def test_e4m3_chunks_of_one_result_match_the_oracle(n, per, B, Sq, Sc, Hq, Hkv, D):
    """The same for e4m3, with workgroups of four and (130 heads) of eight wavefronts."""
    q, chunks, sq, sc = _inputs(n, B, Sq, Sc, Hq, Hkv, D, True)
    scale = D ** -0.5
    runs = [chunks[i:i + per] for i in range(0, n, per)]
    print(f"e4m3 n{n} per{per} B{B} Sq{Sq} Sc{Sc} H{Hq}/{Hkv} D{D}", flush=True)
    assert N.lib().mhip_attn_fwd_plan(B * len(runs), Sq, Sc, Hq, D, D, D, 0, N.MHIP_E4M3) == (8 if Hq == 130 else 4)
    outs = torch.full((len(runs) + 1, B, Sq, Hq, D), 7.0, dtype=torch.bfloat16, device="cuda")
    lses = torch.full((len(runs) + 1, B, Hq, Sq), 7.0, device="cuda")
    ds = [t.cuda().reshape(()) for t in (sq, sc, sc)]
    assert N.host.fwd_blocks(q.cuda(), [c.cuda() for c in chunks], per, scale, False, *ds, outs, lses, 0) is True
    torch.cuda.synchronize()
    assert (outs[-1] == 7).all() and (lses[-1] == 7).all()
    for i, run in enumerate(runs):
        ops = [O.dequantize(q, sq)] + [torch.cat([O.dequantize(c[j], sc) for c in run], 1) for j in (0, 1)]
        ro, rl = O.block_attention(*ops, scale)
        bound = O.e4m3_p_rounding_bound(*ops, scale)
        got = outs[i].float().cpu()
        assert ((got - ro).abs() - (bound + 2 ** -8 * ro.abs())).max().item() <= 2e-3, i
        assert (got - ro).norm() <= 6e-2 * ro.norm(), i
        assert ((lses[i].cpu() - rl).abs() / rl.abs().clamp_min(1.0)).max().item() <= 1e-3, i


# row maxima of a run's chunks against those of the first one, in factors of 2
LEVELS = {"2 x -58": [0, -58, -116], "3 x -40": [0, -40, -80, -120], "4 x -45": [0, -45, -90, -135, -180],
          "7 x -17": [-17 * i for i in range(8)], "15 x -8": [-8 * i for i in range(16)], "2 x -70": [0, -70, -140],
          "7 x +17": [17 * i for i in range(8)], "fall, climb": [0, -58, -116, -30, 0, 3], "climb, fall": [-60, 0, 60, 2, -58, -118],
          "zigzag": [0, -50, 0, -50, 2, -59, 2, -59]}


def _levelled(name, B, Sq, Sc, Hq, D, fp8, scale):
    """Inputs whose scores lie around LEVELS[name] (natural units: times log 2), chunk by chunk: 16 columns of q are 4, and
    those of a chunk's keys alike."""
    levels = LEVELS[name]
    g = torch.Generator().manual_seed(len(levels) * 100 + Sq)
    q = torch.randn(B, Sq, Hq, D, generator=g)
    chunks = [torch.randn(2, B, Sc, Hq, D, generator=g) for _ in levels]
    q[..., :16] = 4.0
    for c, level in zip(chunks, levels):
        c[0][..., :16] = level * math.log(2) / scale / 64.0
    if not fp8:
        return q.bfloat16(), [c.bfloat16() for c in chunks], None, None, None
    top = [max(c[j].abs().max() for c in chunks) / 448.0 for j in (0, 1)]
    (qq, sq) = O.quantize_e4m3(q)
    return qq, [torch.stack([c[j] / top[j] for j in (0, 1)]).clamp(-448, 448).to(torch.float8_e4m3fn) for c in chunks], sq, *top


@pytest.mark.parametrize("name", LEVELS)
@pytest.mark.parametrize("B,Sq,Sc,Hq,D", [(1, 70, 200, 2, 128), (1, 130, 130, 130, 128), (1, 100, 300, 3, 64), (1, 33, 64, 2, 96)])
def test_e4m3_runs_of_chunks_whose_scores_fall_and_climb(name, B, Sq, Sc, Hq, D):
    """The reference of a row moves in both directions where a chunk begins, over a run by far more than fp32 has room for: the
    sum and O stay finite and what is left out is nothing.  With workgroups of four and (130 heads) of eight wavefronts.
    Bounds as above."""
    scale = D ** -0.5
    q, chunks, sq, sk, sv = _levelled(name, B, Sq, Sc, Hq, D, True, scale)
    n = len(chunks)
    print(f"e4m3 levels {name} B{B} Sq{Sq} Sc{Sc} H{Hq} D{D}", flush=True)
    assert N.lib().mhip_attn_fwd_plan(B, Sq, Sc, Hq, D, D, D, 0, N.MHIP_E4M3) == (8 if Hq == 130 else 4)
    out, lse = torch.empty(1, B, Sq, Hq, D, dtype=torch.bfloat16, device="cuda"), torch.empty(1, B, Hq, Sq, device="cuda")
    ds = [t.cuda().reshape(()) for t in (sq, sk, sv)]
    assert N.host.fwd_blocks(q.cuda(), [c.cuda() for c in chunks], n, scale, False, *ds, out, lse, 0) is True
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all() and torch.isfinite(lse).all()
    ops = [O.dequantize(q, sq)] + [torch.cat([O.dequantize(c[j], s) for c in chunks], 1) for j, s in ((0, sk), (1, sv))]
    ro, rl = O.block_attention(*ops, scale)
    bound = O.e4m3_p_rounding_bound(*ops, scale)
    got = out[0].float().cpu()
    assert ((got - ro).abs() - (bound + 2 ** -8 * ro.abs())).max().item() <= 2e-3
    assert (got - ro).norm() <= 6e-2 * ro.norm()
    assert ((lse[0].cpu() - rl).abs() / rl.abs().clamp_min(1.0)).max().item() <= 1e-3


@pytest.mark.parametrize("name", LEVELS)
@pytest.mark.parametrize("B,Sq,Sc,Hq,D", [(1, 70, 200, 2, 128), (1, 300, 65, 3, 64)])
def test_runs_of_chunks_whose_scores_fall_and_climb(name, B, Sq, Sc, Hq, D):
    """The same in bf16, where the reference only moves up: chunks far below it add nothing.  Bounds as above."""
    scale = D ** -0.5
    q, chunks, *_ = _levelled(name, B, Sq, Sc, Hq, D, False, scale)
    out, lse = torch.empty(1, B, Sq, Hq, D, dtype=torch.bfloat16, device="cuda"), torch.empty(1, B, Hq, Sq, device="cuda")
    assert N.host.fwd_blocks(q.cuda(), [c.cuda() for c in chunks], len(chunks), scale, False, None, None, None, out, lse, 0) is True
    torch.cuda.synchronize()
    ro, rl = O.block_attention(q.float(), *(torch.cat([c[j] for c in chunks], 1).float() for j in (0, 1)), scale)
    got = out[0].float().cpu()
    assert ((got - ro).abs() - 2 ** -8 * ro.abs()).max().item() <= 2e-2
    assert (got - ro).norm() <= 1e-2 * ro.norm()
    assert ((lse[0].cpu() - rl).abs() / rl.abs().clamp_min(1.0)).max().item() <= 1e-3


@pytest.mark.parametrize("fill", [float("-inf"), torch.finfo(torch.bfloat16).min])
@pytest.mark.parametrize("n,Sc,D", [(2, 200, 128), (3, 64, 64), (4, 100, 96)])
def test_a_run_that_begins_with_hidden_chunks(fill, n, Sc, D):
    """Keys of -inf or of the type's lowest value in every chunk but the last, whose scores are all far below zero: the
    attention over the last chunk.  (The scores are -inf: no product of q is negative, and lowest values add up to it.)  One
    rounding of P and of the result."""
    g = torch.Generator().manual_seed(n * 10 + D)
    q = (torch.rand(1, 130, 2, D, generator=g) + 0.5).bfloat16()
    chunks = [torch.randn(2, 1, Sc, 2, D, generator=g) for _ in range(n)]
    for c in chunks[:-1]:
        c[0] = fill
    scale = D ** -0.5
    chunks[-1][0] -= 200.0 / scale / D
    chunks = [c.bfloat16() for c in chunks]
    ro, rl = O.block_attention(q.float(), chunks[-1][0].float(), chunks[-1][1].float(), scale)
    assert rl.max() < -100
    out, lse = torch.empty(2, *q.shape, dtype=torch.bfloat16, device="cuda"), torch.empty(2, 1, 2, 130, device="cuda")
    assert N.host.fwd_blocks(q.cuda(), [c.cuda() for c in chunks], n, scale, False, None, None, None, out, lse, 0) is True
    assert N.host.fwd_blocks(q.cuda(), [torch.cat(chunks, 2).cuda()], 1, scale, False, None, None, None, out, lse, 1) is True
    torch.cuda.synchronize()
    for i in range(2):                   # the run, and its keys as one block (whose workgroups split them)
        assert ((lse[i].cpu() - rl).abs() / rl.abs()).max().item() <= 1e-3, i
        assert ((out[i].float().cpu() - ro).abs() - 2 ** -8 * ro.abs()).max().item() <= 2e-2, i


@pytest.mark.parametrize("hidden", [0, 1, 2])
@pytest.mark.parametrize("Sc,D", [(200, 128), (64, 64), (100, 96)])
@pytest.mark.parametrize("score", [-2.0 ** 70, -2.0 ** 127])
def test_rows_whose_every_score_is_very_low(score, hidden, Sc, D):
    """Finite scores near fp32's lowest number, alone or behind chunks of -inf: they count where nothing else does.  All of
    them are one power of two, whose product with the scale is exact, so P is 1 and the result the mean of V, rounded once."""
    g = torch.Generator().manual_seed(Sc + hidden)
    q = torch.zeros(1, 130, 2, D)
    q[..., 0] = 1.0
    chunks = [torch.randn(2, 1, Sc, 2, D, generator=g) for _ in range(hidden + 1)]
    for i, c in enumerate(chunks):
        c[0, ..., 0] = score if i == hidden else float("-inf")
    scale = D ** -0.5
    q, chunks = q.bfloat16().cuda(), [c.bfloat16() for c in chunks]
    ro = chunks[-1][1].float().mean(1, keepdim=True).expand(1, 130, 2, D)
    out, lse = torch.empty(2, 1, 130, 2, D, dtype=torch.bfloat16, device="cuda"), torch.empty(2, 1, 2, 130, device="cuda")
    run = [c.cuda() for c in chunks]
    assert N.host.fwd_blocks(q, run, len(run), scale, False, None, None, None, out, lse, 0) is True
    assert N.host.fwd_blocks(q, [torch.cat(run, 2)], 1, scale, False, None, None, None, out, lse, 1) is True
    torch.cuda.synchronize()
    for i in range(2):
        assert (lse[i].cpu() / (score * scale) - 1).abs().max().item() <= 1e-6, i
        assert ((out[i].float().cpu() - ro).abs() - 2 ** -8 * ro.abs()).max().item() <= 1e-5, i


@pytest.mark.parametrize("Sc,D", [(100, 128), (70, 64)])
def test_rows_that_see_no_key_at_a_very_large_scale(Sc, D):
    """Rows above the causal diagonal have no score at any scale: out = 0 and LSE = -inf."""
    import mercury_artifact_amd as M

    g = torch.Generator().manual_seed(Sc)
    q, k, v = (torch.randn(1, s, 2, D, generator=g).bfloat16().cuda() for s in (130, Sc, Sc))
    out, lse = M.attn_fwd_block(q, k, v, 2.0 ** 100, True)
    torch.cuda.synchronize()
    assert (out[:, :130 - Sc] == 0).all() and (lse[:, :, :130 - Sc] == -math.inf).all()


def test_a_ring_whose_chunks_are_one_stacked_tensor():
    """The chunks of all ranks as the first dimension of one tensor, in a step with one result and in one with several."""
    import mercury_artifact_amd as M

    for W, S, H, D in [(2, 1024, 64, 128), (4, 256, 4, 64)]:
        q, chunks, _, _ = _inputs(W, 1, S, S, H, H, D, False)
        q, stacked, got = q.cuda(), torch.stack(chunks).cuda(), []
        for held in (stacked, list(stacked.unbind(0))):
            o, lse = torch.empty_like(q), torch.empty(1, H, S, device="cuda")
            M.flash_attn_pack_kv(q, held[0], o, lse, D ** -0.5, ring=M.LocalRing((W,), 0, held))
            got.append((o, lse))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


def test_the_only_result_over_a_chunk_that_only_the_hop_knows():
    """A resident ring of one's own need not list its chunks: an output over one of them is written behind the launch."""
    import mercury_artifact_amd as M

    class Own(M.LocalRing):
        resident = True

        def __init__(self, mesh, rank, mine):
            super().__init__(mesh, rank)
            self.mine = mine

        def send_recv(self, to, source, x, recv_tensor=None):
            super().send_recv(to, source, x)
            return self.mine[self.current]

    W, S, H, D = 2, 1024, 64, 128
    q, chunks, _, _ = _inputs(W, 1, S, S, H, H, D, False)
    q, got = q.cuda(), []
    for over in (False, True):
        dev = [c.cuda() for c in chunks]
        o, lse = dev[1][1] if over else torch.empty_like(q), torch.empty(1, H, S, device="cuda")
        M.flash_attn_pack_kv(q, dev[0], o, lse, D ** -0.5, ring=Own((W,), 0, dev))
        got.append((o, lse))
    assert torch.equal(got[0][0], got[1][0]) and (got[0][1] - got[1][1]).abs().max().item() <= 1e-5


@pytest.mark.parametrize("path", ["ring", "packed", "zigzag", "backward"])
def test_a_ring_that_copies_holds_few_copies_at_a_time(path):
    """LocalRing(copy=True) hands out a copy per hop: a step holds the last block's, the next block's and the one that hop makes,
    however many chunks there are."""
    import mercury_artifact_amd as M

    W, S, H, D = 8, 256, 4, 128
    q, chunks, _, _ = _inputs(W, 1, S, S, H, H, D, False)
    q, chunks = q.cuda(), [c.cuda() for c in chunks]
    o, lse, dq, dkv = torch.empty_like(q), torch.zeros(1, H, S, device="cuda"), torch.empty_like(q), torch.empty_like(chunks[0])
    step = {"ring": M.flash_attn_pack_kv, "packed": M.flash_attn_expose_reduce, "zigzag": M.zigzag_causal_pack_kv,
            "backward": lambda q, kv, o, lse, scale, ring: M.flash_attn_backward(q, kv, o, lse, q, dq, dkv, scale, ring=ring)}[path]

    class Hops(M.LocalRing):             # hands over the chunks themselves, one by one
        pass

    def peak(ring):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        step(q, chunks[1], o, lse, 0.1, ring=ring)
        return torch.cuda.max_memory_allocated() - before

    one_by_one = peak(Hops((W,), 1, chunks))
    assert peak(M.LocalRing((W,), 1, chunks, copy=True)) <= one_by_one + 3 * chunks[0].numel() * 2


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("B,Sq,Sc,Hq,Hkv,D", [
    (1, 1, 1, 1, 1, 64), (1, 256, 256, 4, 4, 64), (1, 130, 300, 2, 1, 128), (2, 257, 130, 3, 3, 96), (1, 1000, 200, 72, 8, 128),
    (1, 1024, 257, 72, 72, 64), (1, 1024, 70, 72, 24, 96)])
def test_a_block_alone_and_beside_another_one(B, Sq, Sc, Hq, Hkv, D, fp8, causal):
    """A launch of one block has arguments and kernels of its own: bit for bit the block's result in a launch of two, for
    operands and places with gaps between their rows too."""
    q, chunks, sq, sc = _inputs(2, B, Sq, Sc, Hq, Hkv, D, fp8)
    print(f"alone B{B} Sq{Sq} Sc{Sc} H{Hq}/{Hkv} D{D} fp8={fp8} causal={causal}", flush=True)
    plans = [N.lib().mhip_attn_fwd_plan(k * B, Sq, Sc, Hq, D, Hkv * D, Hkv * D, int(causal), N.MHIP_E4M3 if fp8 else N.MHIP_BF16) for k in (1, 2)]
    assert plans[0] == plans[1]

    def gaps(t):
        wide = torch.zeros(*t.shape[:-1], D + 16, dtype=t.dtype, device="cuda")
        wide[..., :D] = t.cuda()
        return wide[..., :D]

    ds = [None] * 3 if not fp8 else [t.cuda().reshape(()) for t in (sq, sc, sc)]
    for form in (lambda t: t.cuda(), gaps):
        qd, dev = form(q), [form(c) for c in chunks]
        outs = form(torch.full((4, B, Sq, Hq, D), 7.0, dtype=torch.bfloat16))
        lses = torch.full((4, B, Hq, Sq), 7.0, device="cuda")
        assert N.host.fwd_blocks(qd, dev, 1, D ** -0.5, causal, *ds, outs, lses, 0) is True
        for i in (0, 1):
            assert N.host.fwd_blocks(qd, dev[i:i + 1], 1, D ** -0.5, causal, *ds, outs, lses, 2 + i) is True
        torch.cuda.synchronize()
        assert torch.equal(outs[:2], outs[2:]) and torch.equal(lses[:2], lses[2:]) and not (lses == 7).any()
