"""The carried sums of the backward ring step (mhip_attn_bwd_chunk): first, middle and last chunk, fp32 dK / dV, bf16
ones for the rank's own chunk, at ragged rows and head dimensions.

The kernels round P and dS to bf16 (relative 2^-9 each, random): rel-L2 of a gradient within 2^-8; the largest element
within 2^-8 of the sum of the magnitudes that enter it, for which 12 root mean squares are allowed here; bf16 results
add 2^-9.  Where the gradient is exactly zero (one key: dP = delta) the fp32 sums of D products of N(0,1) values, |dP| up
to 40, leave up to D 2^-24 40 in dS; 1e-4 is allowed absolutely."""
import ctypes

import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N

pytestmark = pytest.mark.gpu


def taken(B, Sq, Sc, Hq, Hkv, D, causal):
    """(launches of the two passes, workgroups per stationary tile of the dQ pass, of the dK / dV pass) of a block."""
    splits = (ctypes.c_int * 2)()
    return N.lib().mhip_attn_bwd_plan(B, Sq, Sc, Hq, Hkv, D, int(causal), splits), splits[0], splits[1]


def form(n, B, Sq, Sc, Hq, Hkv, D):
    """(launches, workgroups per query tile of the dQ pass, rows of its MFMA tiles) of a call over n chunks."""
    what = (ctypes.c_int * 2)()
    return N.lib().mhip_attn_bwd_chunks_plan(n, B, Sq, Sc, Hq, Hkv, D, 0, what), what[0], what[1]


def by_hops(W, rank, chunks):
    """A ring that makes no promise about its chunks: one launch (or one of each pass) for every chunk."""
    import mercury_artifact_amd as M

    class Hops(M.LocalRing):
        pass

    return Hops((W,), rank, chunks)


def _close(name, got, ref):
    got, ref = got.float().cpu(), ref.float()
    rms = ref.square().mean().sqrt()
    assert (got - ref).norm() <= 2 ** -8 * 1.5 * ref.norm() + 1e-4, (name, ((got - ref).norm() / ref.norm()).item())
    assert (got - ref).abs().max() <= 12 * 2 ** -8 * rms + 2 ** -8 * ref.abs().max() + 1e-4, name


JOINT = [(1, 300, 2, 2, 128), (2, 129, 4, 2, 64), (3, 257, 3, 1, 40), (4, 64, 2, 2, 128), (2, 400, 8, 1, 128), (2, 193, 4, 2, 96)]
# one launch per pass: from the second chunk on the dQ pass with eight wavefronts finds lse2 and delta prepared
IN_TURN = [(3, 130, 128, 128, 64), (3, 130, 128, 64, 88), (3, 130, 128, 128, 128), (2, 257, 128, 128, 40), (3, 257, 128, 128, 96),
           (2, 257, 128, 64, 128), (4, 65, 256, 256, 128)]


@pytest.mark.parametrize("W,S,Hq,Hkv,D", JOINT + IN_TURN)
@pytest.mark.parametrize("dq_dtype,keep", [(torch.bfloat16, True), (torch.float32, True), (torch.bfloat16, False)])
def test_backward_step_carries_the_sums(W, S, Hq, Hkv, D, dq_dtype, keep):
    """Chunk by chunk, and on a ring whose chunks may go together."""
    import mercury_artifact_amd as M

    print(f"W{W} S{S} Hq{Hq} Hkv{Hkv} D{D} {dq_dtype} keep={keep}", flush=True)
    B, rank, scale = 2, W - 1, D ** -0.5
    assert taken(B, S, S, Hq, Hkv, D, False)[0] == (2 if (W, S, Hq, Hkv, D) in IN_TURN else 1)
    g = torch.Generator().manual_seed(W * 1000 + S)
    q, dout = (torch.randn(B, S, Hq, D, generator=g).bfloat16() for _ in range(2))
    kvs = [torch.randn(2, B, S, Hkv, D, generator=g).bfloat16() for _ in range(W)]
    order = O.single_ring_order(rank, W)
    o, lse = O.ring_forward(q.float(), [c.float() for c in kvs], order, scale)
    rdq, rdkv = O.ring_backward(q.float(), [c.float() for c in kvs], order, o.bfloat16().float(), lse, dout.float(), scale)
    dev = [c.cuda() for c in kvs]
    for ring in (by_hops(W, rank, dev), M.LocalRing((W,), rank, dev)):
        dq = torch.full(q.shape, float("nan"), dtype=dq_dtype, device="cuda")
        dkv = torch.full_like(dev[rank], float("nan"))
        got = {} if keep else None
        M.flash_attn_backward(q.cuda(), dev[rank], o.bfloat16().cuda(), lse.cuda(), dout.cuda(), dq, dkv, scale, ring=ring,
                              dkv_chunks=got)
        torch.cuda.synchronize()
        _close("dq", dq, rdq)
        _close("own dkv", dkv, torch.stack(tuple(rdkv[rank])))
        if keep:
            assert torch.equal(got[rank], dkv.float())
        for c in range(W) if keep else ():
            assert got[c].dtype == torch.float32
            _close(f"dkv {c}", got[c], torch.stack(tuple(rdkv[c])))


# steps whose query tiles are shared, and some for which the third launch would cost more than it saves
SHARED = [(8, 130, 2, 2, 128), (7, 193, 3, 3, 96), (3, 700, 2, 2, 64), (6, 257, 1, 1, 72), (5, 385, 4, 2, 104), (8, 257, 2, 1, 40), (36, 129, 1, 1, 128)]
WHOLE = [(5, 200, 4, 2, 112), (8, 65, 2, 1, 40), (36, 64, 1, 1, 128)]


@pytest.mark.parametrize("W,S,Hq,Hkv,D", SHARED + WHOLE)
@pytest.mark.parametrize("dq_dtype", [torch.bfloat16, torch.float32])
def test_a_query_tile_shared_by_workgroups_of_a_step(W, S, Hq, Hkv, D, dq_dtype):
    """Steps of a few heads, whose chain of tiles over all chunks is shared by several workgroups: chunk counts that do and do
    not divide among them, ragged rows, and (36 chunks) launches that carry the sum on; twice the same bits."""
    import mercury_artifact_amd as M

    print(f"shared W{W} S{S} Hq{Hq} Hkv{Hkv} D{D} {dq_dtype}", flush=True)
    B, rank, scale = 1, 1, D ** -0.5
    together = N.lib().mhip_attn_bwd_take(B, S, S, Hq, Hkv, D, W)
    launches, shared_by, _ = form(together, B, S, S, Hq, Hkv, D)
    assert together == min(W, 12) and launches == 1 and (shared_by > 1) == ((W, S, Hq, Hkv, D) in SHARED)
    g = torch.Generator().manual_seed(W * 1000 + S)
    q, dout = (torch.randn(B, S, Hq, D, generator=g).bfloat16() for _ in range(2))
    kvs = [torch.randn(2, B, S, Hkv, D, generator=g).bfloat16() for _ in range(W)]
    order = O.single_ring_order(rank, W)
    o, lse = O.ring_forward(q.float(), [c.float() for c in kvs], order, scale)
    rdq, rdkv = O.ring_backward(q.float(), [c.float() for c in kvs], order, o.bfloat16().float(), lse, dout.float(), scale)
    dev, runs = [c.cuda() for c in kvs], []
    for _ in range(2):
        dq = torch.full(q.shape, float("nan"), dtype=dq_dtype, device="cuda")
        dkv, got = torch.full_like(dev[rank], float("nan")), {}
        M.flash_attn_backward(q.cuda(), dev[rank], o.bfloat16().cuda(), lse.cuda(), dout.cuda(), dq, dkv, scale,
                              ring=M.LocalRing((W,), rank, dev), dkv_chunks=got)
        torch.cuda.synchronize()
        runs.append(dq)
    assert torch.equal(*runs)
    _close("dq", dq, rdq)
    for c in range(W):
        _close(f"dkv {c}", got[c], torch.stack(tuple(rdkv[c])))


def _block(B, Sq, Sc, Hq, Hkv, D, causal, launches=1, shared=None):
    import mercury_artifact_amd as M

    plan = taken(B, Sq, Sc, Hq, Hkv, D, causal)
    assert plan[0] == launches and (shared is None or (max(plan[1:]) > 1) == shared)

    print(f"B{B} D{D} Sq{Sq} Sc{Sc} Hq{Hq} Hkv{Hkv} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(D * 1000 + Sq)
    q, dout = (torch.randn(B, Sq, Hq, D, generator=g).bfloat16() for _ in range(2))
    kv = torch.randn(2, B, Sc, Hkv, D, generator=g).bfloat16()
    scale = D ** -0.5
    o, lse = O.block_attention(q.float(), kv[0].float(), kv[1].float(), scale, causal=causal)
    refs = O.block_backward(dout.float(), q.float(), kv[0].float(), kv[1].float(), o.bfloat16().float(), lse, scale, causal=causal)
    dev = [x.cuda() for x in (dout, q, kv[0], kv[1], o.bfloat16(), lse)]
    dq = torch.full_like(dev[1], float("nan"))
    dkv = torch.full((2, *dev[2].shape), float("nan"), dtype=torch.bfloat16, device="cuda")
    delta = M.attn_bwd_block(*dev, dq, dkv[0], dkv[1], scale, causal=causal)
    torch.cuda.synchronize()
    for name, got, ref in zip(("dq", "dk", "dv"), (dq, dkv[0], dkv[1]), refs):
        _close(name, got, ref)
    want = (dout.float() * o.bfloat16().float()).sum(-1).transpose(1, 2)
    assert (delta.cpu() - want).abs().max() <= 1e-4
    # with an accumulator: the same dq, and the sum before its rounding (fp32 addition to 0.25: 2^-24 relative)
    acc, again = torch.full(dq.shape, 0.25, device="cuda"), torch.full_like(dq, float("nan"))
    M.attn_bwd_block(*dev, again, torch.empty_like(dkv[0]), torch.empty_like(dkv[1]), scale, causal=causal, dq_acc=acc)
    assert torch.equal(again, dq)
    assert bool(((acc - 0.25 - dq.float()).abs() <= 2 ** -8 * dq.float().abs() + 2 ** -22).all())


@pytest.mark.parametrize("D", [8, 56, 64, 72, 96, 104])
@pytest.mark.parametrize("Sq,Sc,Hq,Hkv,causal", [(1, 1, 2, 1, False), (65, 129, 4, 2, False), (257, 63, 2, 2, True),
                                                 (320, 400, 3, 3, True), (130, 700, 2, 1, False)])
def test_backward_block_on_narrow_heads(D, Sq, Sc, Hq, Hkv, causal):
    """Both sides of the lines between the 64-, 96- and 128-column kernels, ragged rows and keys, several turns of
    the tile ring; launches this small run both passes side by side."""
    _block(2, Sq, Sc, Hq, Hkv, D, causal)


@pytest.mark.parametrize("D", [64, 80, 128])
@pytest.mark.parametrize("Sq,Sc,causal", [(130, 129, False), (257, 64, True), (300, 385, True)])
def test_backward_block_in_two_launches(D, Sq, Sc, causal):
    """Enough heads to fill the chip with either pass: one launch each, dQ with eight wavefronts."""
    _block(2, Sq, Sc, 128, 128, D, causal, launches=2)


@pytest.mark.parametrize("D", [8, 24, 64])
@pytest.mark.parametrize("Sq,Sc,Hq,Hkv,causal", [(449, 385, 24, 24, False), (383, 577, 32, 8, False), (513, 512, 40, 20, True)])
def test_two_workgroups_on_a_cu(D, Sq, Sc, Hq, Hkv, causal):
    """64 columns: more workgroups than CUs, so that two of them share a CU's LDS; streams of more tiles than the tile ring
    has stages, with a last tile of 1, 63 or 64 rows."""
    _block(2, Sq, Sc, Hq, Hkv, D, causal, launches=taken(2, Sq, Sc, Hq, Hkv, D, causal)[0])


@pytest.mark.parametrize("D", [40, 88, 128])
@pytest.mark.parametrize("B,Sq,Sc,Hq,Hkv,causal", [(1, 321, 130, 8, 1, False), (1, 700, 777, 8, 1, True), (2, 513, 400, 12, 2, True),
                                                   (1, 130, 3000, 1, 1, False), (1, 3000, 130, 1, 1, True)])
def test_backward_block_with_shared_tiles(B, Sq, Sc, Hq, Hkv, causal, D):
    """Long chains of tiles on few workgroups (grouped heads, one head): their stationary tiles are shared and the sums
    added by the third launch."""
    _block(B, Sq, Sc, Hq, Hkv, D, causal, shared=True)


def test_partial_sums_stay_inside_the_workspace():
    """One workspace, sized with the first chunk, for chunks of other lengths and for both masks, among them launches that
    leave the most partial sums: nothing behind its end is written, and the results are those of a fresh one."""
    import mercury_artifact_amd as M
    B, Sq, Hq, Hkv, D = 1, 1000, 8, 1, 128
    g = torch.Generator(device="cuda").manual_seed(9)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    q, dout, kv = mk(B, Sq, Hq, D), mk(B, Sq, Hq, D), mk(2, B, 3000, Hkv, D)
    size = N.lib().mhip_attn_bwd_workspace_bytes(B, Sq, 64, Hq, Hkv, D)
    memory = torch.full((size + (32 << 20),), 0xA5, dtype=torch.uint8, device="cuda")
    for Sc, causal in ((64, False), (3000, False), (1000, True), (130, False), (2048, True)):
        print(f"Sc{Sc} causal={causal} {taken(B, Sq, Sc, Hq, Hkv, D, causal)}", flush=True)
        k, v = kv[0, :, :Sc], kv[1, :, :Sc]
        out, lse = M.attn_fwd_block(q, k, v, 0.1, causal=causal)
        want, got = (tuple(torch.empty_like(t) for t in (q, k, v)) for _ in range(2))
        M.attn_bwd_block(dout, q, k, v, out, lse, *want, 0.1, causal=causal)
        strides = [st for t in (q, k, got[1], got[0], out) for st in t.stride()[:3]]
        N.check(N.lib().mhip_attn_bwd_block(*map(N.ptr, (dout, q, k, v, out, lse, *got)), None, B, Sq, Sc, Hq, Hkv, D, *strides,
                                            0.1, int(causal), 0, N.ptr(memory), N.stream_of(q)), "mhip_attn_bwd_block")
        torch.cuda.synchronize()
        assert bool((memory[size:] == 0xA5).all())
        assert all(torch.equal(a, b) for a, b in zip(want, got))


@pytest.mark.parametrize("W", [1, 2])
@pytest.mark.parametrize("dq_over", ["q", "dout", "o"])
def test_backward_step_in_place(W, dq_over):
    """dq over q, dout or o and dkv over the own chunk: bit for bit the gradients that separate places receive."""
    import mercury_artifact_amd as M

    B, S, H, D = 1, 700, 4, 64
    g = torch.Generator(device="cuda").manual_seed(4)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    t = {"q": mk(B, S, H, D), "dout": mk(B, S, H, D), "o": mk(B, S, H, D)}
    chunks = [mk(2, B, S, H, D) for _ in range(W)]
    lse = M.attn_fwd_block(t["q"], chunks[0][0], chunks[0][1], 0.1)[1]
    want = torch.empty_like(t["q"]), torch.empty_like(chunks[0])
    M.flash_attn_backward(t["q"], chunks[0], t["o"], lse, t["dout"], *want, 0.1, ring=M.LocalRing((W,), 0, chunks))
    got = t[dq_over], chunks[0]
    M.flash_attn_backward(t["q"], chunks[0], t["o"], lse, t["dout"], *got, 0.1, ring=M.LocalRing((W,), 0, chunks))
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


GROUPED = [(8, 1, 64, 2, 2, 128, 8), (5, 2, 129, 4, 2, 64, 5), (3, 1, 300, 5, 1, 96, 3), (5, 1, 1024, 32, 32, 128, 5), (8, 2, 512, 5, 5, 128, 8), (7, 1, 257, 8, 8, 80, 7),
           (6, 2, 65, 3, 3, 40, 6), (16, 1, 200, 2, 1, 128, 16), (17, 1, 100, 2, 2, 64, 9)]


@pytest.mark.parametrize("W,B,S,Hq,Hkv,D,group", GROUPED)
@pytest.mark.parametrize("dq_dtype,keep", [(torch.bfloat16, True), (torch.float32, True), (torch.bfloat16, False)])
def test_backward_step_in_grouped_launches(W, B, S, Hq, Hkv, D, group, dq_dtype, keep):
    """Steps whose chunks share launches: one to three launches, chunks of one to eight tiles (the dQ pass changes chunks
    before, at and behind the tiles its prologue requests), ragged rows, grouped heads."""
    import mercury_artifact_amd as M

    print(f"grouped W{W} B{B} S{S} Hq{Hq} Hkv{Hkv} D{D} {dq_dtype} keep={keep}", flush=True)
    assert N.lib().mhip_attn_bwd_take(B, S, S, Hq, Hkv, D, W) == group and form(group, B, S, S, Hq, Hkv, D)[0] == 1
    rank, scale = W // 2, D ** -0.5
    g = torch.Generator().manual_seed(W * 1000 + S)
    q, dout = (torch.randn(B, S, Hq, D, generator=g).bfloat16() for _ in range(2))
    kvs = [torch.randn(2, B, S, Hkv, D, generator=g).bfloat16() for _ in range(W)]
    order = O.single_ring_order(rank, W)
    o, lse = O.ring_forward(q.float(), [c.float() for c in kvs], order, scale)
    rdq, rdkv = O.ring_backward(q.float(), [c.float() for c in kvs], order, o.bfloat16().float(), lse, dout.float(), scale)
    dev = [c.cuda() for c in kvs]
    dq = torch.full(q.shape, float("nan"), dtype=dq_dtype, device="cuda")
    dkv = torch.full_like(dev[rank], float("nan"))
    got = {} if keep else None
    M.flash_attn_backward(q.cuda(), dev[rank], o.bfloat16().cuda(), lse.cuda(), dout.cuda(), dq, dkv, scale,
                          ring=M.LocalRing((W,), rank, dev), dkv_chunks=got)
    torch.cuda.synchronize()
    _close("dq", dq, rdq)
    _close("own dkv", dkv, torch.stack(tuple(rdkv[rank])))
    for c in range(W) if keep else ():
        assert got[c].dtype == torch.float32
        _close(f"dkv {c}", got[c], torch.stack(tuple(rdkv[c])))

    dq1, dkv1, got1 = torch.empty_like(dq), torch.empty_like(dkv), {} if keep else None
    M.flash_attn_backward(q.cuda(), dev[rank], o.bfloat16().cuda(), lse.cuda(), dout.cuda(), dq1, dkv1, scale,
                          ring=by_hops(W, rank, dev), dkv_chunks=got1)
    _close("dq, chunk by chunk", dq1, rdq)
    _close("dkv, chunk by chunk", dkv1, torch.stack(tuple(rdkv[rank])))


@pytest.mark.parametrize("over", ["own chunk", "other chunk", "q"])
def test_grouped_gradients_over_operands(over):
    """dq or dkv over something a grouped launch reads: stored behind the launch, same values."""
    import mercury_artifact_amd as M

    W, B, S, H, D = 4, 1, 200, 4, 64
    assert N.lib().mhip_attn_bwd_take(B, S, S, H, H, D, W) == 4
    g = torch.Generator().manual_seed(3)

    def fresh():
        g.manual_seed(3)
        q, dout, o = (torch.randn(B, S, H, D, generator=g).bfloat16().cuda() for _ in range(3))
        chunks = [torch.randn(2, B, S, H, D, generator=g).bfloat16().cuda() for _ in range(W)]
        return q, dout, o, chunks, torch.full((B, H, S), 6.0, device="cuda")

    def step(q, dout, o, chunks, lse, dq, dkv):
        got = {}
        M.flash_attn_backward(q, chunks[1], o, lse, dout, dq, dkv, 0.125, ring=M.LocalRing((W,), 1, chunks), dkv_chunks=got)
        return dq.clone(), dkv.clone(), got

    t = fresh()
    want = step(*t, torch.empty_like(t[0]), torch.empty_like(t[3][1]))
    t = fresh()
    dq = t[0] if over == "q" else torch.empty_like(t[0])
    dkv = t[3][1] if over == "own chunk" else t[3][2] if over == "other chunk" else torch.empty_like(t[3][1])
    have = step(*t, dq, dkv)
    assert torch.equal(have[1], want[1]) and (have[0].float() - want[0].float()).abs().max() <= 2 ** -7 * want[0].float().abs().max()
    assert all(torch.equal(have[2][i], want[2][i]) for i in range(W))


def test_rows_past_the_end_are_no_other_heads():
    """A head whose dout is not finite leaves the next head's gradients alone, also in the ragged last tile of a long stream."""
    import mercury_artifact_amd as M

    B, S, H, D = 1, 330, 3, 64
    g = torch.Generator().manual_seed(8)
    q, dout, o = (torch.randn(B, S, H, D, generator=g).bfloat16().cuda() for _ in range(3))
    kv = torch.randn(2, B, S, H, D, generator=g).bfloat16().cuda()
    lse = torch.full((B, H, S), 6.0, device="cuda")
    grads = []
    for bad in (0.0, float("inf"), float("nan")):
        d = dout.clone()
        d[:, :, 1] = d[:, :, 1] + bad
        dq, dkv = torch.empty_like(q), torch.empty_like(kv)
        M.attn_bwd_block(d, q, kv[0], kv[1], o, lse, dq, dkv[0], dkv[1], 0.125)
        grads.append(torch.stack((dq, dkv[0], dkv[1]))[:, :, :, ::2])
    assert torch.isfinite(grads[0].float()).all()
    assert torch.equal(grads[1], grads[0]) and torch.equal(grads[2], grads[0])


def test_gradients_nobody_keeps_take_bounded_memory():
    """Without dkv_chunks the gradients of the other ranks' chunks are made and dropped: launches over several chunks hold
    32 MiB of them, whatever the step would have grouped."""
    import mercury_artifact_amd as M

    W, S, H, D = 8, 2048, 8, 128
    assert N.lib().mhip_attn_bwd_take(1, S, S, H, H, D, W) * 2 * S * H * D * 2 > 60 << 20
    g = torch.Generator(device="cuda").manual_seed(2)
    q, dout, o = (torch.randn(1, S, H, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    chunks = [torch.randn(2, 1, S, H, D, generator=g, device="cuda").bfloat16() for _ in range(W)]
    lse = torch.full((1, H, S), 9.0, device="cuda")
    dq, dkv = torch.empty_like(q), torch.empty_like(chunks[0])

    def peak(ring):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        M.flash_attn_backward(q, chunks[1], o, lse, dout, dq, dkv, D ** -0.5, ring=ring)
        return torch.cuda.max_memory_allocated() - before

    one_by_one = peak(by_hops(W, 1, chunks))         # one such gradient at a time
    assert peak(M.LocalRing((W,), 1, chunks)) <= one_by_one + (32 << 20)


@pytest.mark.parametrize("Hq,D,places,launches", [(64, 128, 2, []), (64, 128, 4, []), (64, 128, 8, [8]), (32, 64, 2, []), (32, 64, 5, [4, 4])])
def test_gradients_nobody_keeps_are_planned_for_the_places_there_are(Hq, D, places, launches, monkeypatch):
    """How many chunks share a launch is chosen among what there are places for, chunk by chunk included, and not cut down from
    what the whole step would have taken, which was chosen for more chunks to fill a launch with."""
    import mercury_artifact_amd as M
    from mercury_artifact_amd import ring as R

    W, S = 8, 64
    assert N.lib().mhip_attn_bwd_take(1, S, S, Hq, 1, D, W) == 8
    g = torch.Generator(device="cuda").manual_seed(6)
    q, dout, o = (torch.randn(1, S, Hq, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    chunks = [torch.randn(2, 1, S, 1, D, generator=g, device="cuda").bfloat16() for _ in range(W)]
    lse = torch.full((1, Hq, S), 6.0, device="cuda")
    taken_together, real = [], N.host.bwd_chunks
    monkeypatch.setattr(N.host, "bwd_chunks", lambda *a: (taken_together.append(len(a[2])), real(*a))[1])
    monkeypatch.setattr(R, "UNKEPT_BYTES", places * chunks[0].numel() * 2)
    grads = []
    for kept in (None, {}):
        dq, dkv = torch.empty_like(q), torch.empty_like(chunks[1])
        M.flash_attn_backward(q, chunks[1], o, lse, dout, dq, dkv, D ** -0.5, ring=M.LocalRing((W,), 1, chunks), dkv_chunks=kept)
        grads.append((dq, dkv))
    assert taken_together == launches + [8]
    # the same products summed in fp32 in another order, which can move a dS and a gradient to the next bf16 value
    for a, b in zip(*grads):
        assert (a.float() - b.float()).norm() <= 2 ** -8 * b.float().norm()
