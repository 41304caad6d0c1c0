"""The dQ pass on 16 x 16 MFMA tiles, which launches take that keep every CU busy for long: at least 218 workgroups of 256 query
rows in the last round of 256, 32 key tiles and more, causal launches of 512 workgroups.  Against the oracle on some of the
heads, with the bounds of test_gpu_bwd.py, whose oracle inputs (out, lse of the oracle's own forward) are used here too."""
import ctypes

import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N
from test_gpu_bwd import _check_grad
from test_gpu_bwd_chunk import by_hops

pytestmark = pytest.mark.gpu
H = 32


def _form(Sq, Sc, D, causal):
    """(launches, workgroups per query tile, rows of the dQ pass's MFMA tiles) of a block."""
    what = (ctypes.c_int * 2)()
    return N.lib().mhip_attn_bwd_chunks_plan(1, 1, Sq, Sc, H, H, D, int(causal), what), what[0], what[1]


def _run(Sq, Sc, D, causal, heads=(0, 31)):
    import mercury_artifact_amd as M

    assert _form(Sq, Sc, D, causal) == (2, 1, 16)
    print(f"small tiles, backward Sq{Sq} Sc{Sc} D{D} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(Sq * 1009 + Sc + D)
    q, dout = (torch.randn(1, Sq, H, D, generator=g).bfloat16() for _ in range(2))
    kv = torch.randn(2, 1, Sc, H, D, generator=g).bfloat16()
    out, lse, scale = torch.zeros_like(q), torch.zeros(1, H, Sq), D ** -0.5
    refs = {}
    for h in heads:
        one = [t[:, :, h:h + 1].float() for t in (q, kv[0], kv[1])]
        o, lse[:, h:h + 1] = O.block_attention(*one, scale, causal=causal)
        out[:, :, h:h + 1] = o.bfloat16()
        refs[h] = O.block_backward(dout[:, :, h:h + 1].float(), *one, out[:, :, h:h + 1].float(), lse[:, h:h + 1], scale, causal=causal)
    dev = [t.cuda() for t in (dout, q, kv, out, lse)]
    dq, dkv = torch.full_like(dev[1], 7.0), torch.full_like(dev[2], 7.0)
    delta = M.attn_bwd_block(dev[0], dev[1], dev[2][0], dev[2][1], dev[3], dev[4], dq, dkv[0], dkv[1], scale, causal=causal)
    torch.cuda.synchronize()
    for h, ref in refs.items():
        for name, got, want in zip(("dq", "dk", "dv"), (dq, dkv[0], dkv[1]), ref):
            _check_grad(f"{name} head {h}", got[:, :, h:h + 1], want)
        # 128 products of N(0,1) values summed in fp32 in another order: 128 ulps of sums around 11 is far above it
        want = (dout[:, :, h].float() * out[:, :, h].float()).sum(-1)
        assert (delta[:, h].cpu() - want).abs().max().item() <= 128 * 2 ** -23 * 16


@pytest.mark.parametrize("D", [128, 104, 96, 72])
@pytest.mark.parametrize("Sq,Sc", [(1793, 2048), (1791, 1985), (1809, 2047), (1777, 2000), (2048, 2081)])
def test_a_block_at_tile_edges(Sq, Sc, D):
    """Last tiles whole, of one row or key, short of one, and ending inside and between 16-row and 16-key blocks."""
    _run(Sq, Sc, D, False)


@pytest.mark.parametrize("Sq,Sc,D", [(4081, 4081, 128), (4090, 4225, 96), (4352, 4033, 128)])
def test_under_the_causal_mask(Sq, Sc, D):
    """Rows that see every key, none, and keys up to a diagonal inside a 16-key block."""
    _run(Sq, Sc, D, True, heads=(0, 17))


@pytest.mark.parametrize("Sq,Sc,D,causal", [(1793, 1985, 128, False), (1793, 2048, 96, False), (4081, 4081, 128, True), (4090, 4225, 96, True)])
def test_rows_prepared_by_an_earlier_chunk(Sq, Sc, D, causal):
    """lse2 and delta as an earlier chunk's call left them: a later call on them computes what one computes that works them out
    itself, bit for bit, alone, and as the first, a middle and the last chunk of a carried sum."""
    import mercury_artifact_amd as M

    assert _form(Sq, Sc, D, causal) == (2, 1, 16)
    print(f"prepared Sq{Sq} Sc{Sc} D{D} causal={causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(Sq + Sc + D)
    mk = lambda rows: torch.randn(1, rows, H, D, generator=g, device="cuda").bfloat16()
    q, dout, k, v, scale = mk(Sq), mk(Sq), mk(Sc), mk(Sc), D ** -0.5
    out, lse = M.attn_fwd_block(q, k, v, scale, causal=causal)
    want = [torch.empty_like(t) for t in (q, k, v)]
    M.attn_bwd_block(dout, q, k, v, out, lse, *want, scale, causal=causal)
    workspace = torch.empty(N.lib().mhip_attn_bwd_workspace_bytes(1, Sq, Sc, H, H, D), dtype=torch.uint8, device="cuda")
    acc = torch.full(q.shape, float("nan"), device="cuda")

    def call(first, last, prepared):
        dq, dk, dv = (torch.full_like(t, float("nan")) for t in (q, k, v))
        strides = [st for t in (q, k, dk, dq, out) for st in t.stride()[:3]]
        N.check(N.lib().mhip_attn_bwd_chunk(*map(N.ptr, (dout, q, k, v, out, lse)), N.ptr(dq), N.ptr(acc), first, last, prepared, N.ptr(dk),
                                            N.ptr(dv), None, None, 1, Sq, Sc, H, H, D, *strides, scale, int(causal), N.ptr(workspace),
                                            N.stream_of(q)), "mhip_attn_bwd_chunk")
        torch.cuda.synchronize()
        assert torch.equal(dk, want[1]) and torch.equal(dv, want[2])
        return dq

    for prepared in (0, 1):
        assert torch.equal(call(1, 1, prepared), want[0])
    call(1, 0, 1)
    once = acc.clone()
    assert torch.equal(once.bfloat16(), want[0])
    call(0, 0, 1)
    assert torch.equal(acc, once + once)
    assert torch.equal(call(0, 1, 1), (once + once + once).bfloat16())


@pytest.mark.parametrize("Sq,Sc,D", [(1793, 1985, 128), (1809, 2047, 96)])
def test_a_ring_that_hands_over_chunk_by_chunk(Sq, Sc, D):
    """The block's kernels from the second chunk on: prepared rows, a carried dQ, fp32 gradients of the chunks."""
    import mercury_artifact_amd as M

    W, rank, scale, heads = 3, 1, D ** -0.5, (0, 31)
    assert _form(Sq, Sc, D, False) == (2, 1, 16)
    print(f"small tiles, by hops Sq{Sq} Sc{Sc} D{D}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(Sq * 7 + Sc + D)
    q, dout = (torch.randn(1, Sq, H, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    chunks = [torch.randn(2, 1, Sc, H, D, generator=g, device="cuda").bfloat16() for _ in range(W)]
    out, lse = M.attn_fwd_block(q, torch.cat([c[0] for c in chunks], 1), torch.cat([c[1] for c in chunks], 1), scale)
    dq, dkv, kept = torch.full_like(q, float("nan")), torch.full_like(chunks[rank], float("nan")), {}
    M.flash_attn_backward(q, chunks[rank], out, lse, dout, dq, dkv, scale, ring=by_hops(W, rank, chunks), dkv_chunks=kept)
    torch.cuda.synchronize()
    assert torch.equal(kept[rank], dkv.float())
    for h in heads:
        one = lambda t: t[..., h:h + 1, :].float().cpu()
        rdq, rdkv = O.ring_backward(one(q), [one(c) for c in chunks], O.single_ring_order(rank, W), one(out), lse[:, h:h + 1].cpu(),
                                    one(dout), scale)
        _check_grad(f"dq head {h}", one(dq), rdq)
        for c in range(W):
            _check_grad(f"dkv {c} head {h}", one(kept[c]), torch.stack(tuple(rdkv[c])))


def test_the_same_bits_every_time():
    import mercury_artifact_amd as M

    g = torch.Generator(device="cuda").manual_seed(5)
    q, dout, k, v = (torch.randn(1, 2048, H, 128, generator=g, device="cuda").bfloat16() for _ in range(4))
    out, lse = M.attn_fwd_block(q, k, v, 0.1)
    first = None
    for _ in range(3):
        grads = [torch.empty_like(q) for _ in range(3)]
        M.attn_bwd_block(dout, q, k, v, out, lse, *grads, 0.1)
        first = first or grads
        assert all(torch.equal(a, b) for a, b in zip(first, grads))
