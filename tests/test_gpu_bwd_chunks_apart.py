"""Backward steps over several chunks with a launch of each pass over all of them, which steps take whose passes fill the chip by
themselves.  Against the chunk-by-chunk form of the same kernels and, on some heads, the oracle with the bounds of
test_gpu_bwd.py."""
import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N
from test_gpu_bwd import _check_grad
from test_gpu_bwd_chunk import by_hops, form

pytestmark = pytest.mark.gpu


# chunks of one to eight tiles (the dQ pass changes chunks before, at and behind the tiles its prologue requests), last tiles
# and chunks whole, of one row or key and short of one, grouped heads, each column count, 16 x 16 and 32 x 32 MFMA tiles
@pytest.mark.parametrize("B,Sq,Sc,Hq,Hkv,D,W", [(4, 500, 509, 32, 32, 128, 8), (4, 512, 258, 32, 32, 96, 12), (4, 300, 257, 64, 64, 64, 5),
                                                (8, 257, 449, 64, 32, 104, 4), (4, 513, 640, 64, 64, 40, 3), (4, 241, 64, 64, 64, 128, 16),
                                                (4, 256, 1, 64, 64, 72, 16), (8, 500, 193, 32, 32, 128, 19)])
@pytest.mark.parametrize("dq_dtype,keep", [(torch.bfloat16, True), (torch.float32, True), (torch.bfloat16, False)])
def test_a_step_with_a_launch_for_each_pass(B, Sq, Sc, Hq, Hkv, D, W, dq_dtype, keep):
    import mercury_artifact_amd as M

    print(f"apart B{B} Sq{Sq} Sc{Sc} Hq{Hq} Hkv{Hkv} D{D} W{W} {dq_dtype} keep={keep}", flush=True)
    together = N.lib().mhip_attn_bwd_take(B, Sq, Sc, Hq, Hkv, D, W)
    workgroups = B * Hq * -(-Sq // 128) + together * B * Hkv * -(-Sc // 128)
    assert together == min(W, 10 if W > 16 else 16) and workgroups > 4096         # more than both passes share a launch with
    small = D > 64 and together * -(-Sc // 64) >= 32                              # the dQ pass on 16 x 16 MFMA tiles
    assert form(together, B, Sq, Sc, Hq, Hkv, D) == (2, 1, 16 if small else 32)
    rank, scale = W // 2, D ** -0.5
    g = torch.Generator(device="cuda").manual_seed(W * 1000 + Sq)
    q, dout = (torch.randn(B, Sq, Hq, D, generator=g, device="cuda").bfloat16() for _ in range(2))
    chunks = [torch.randn(2, B, Sc, Hkv, D, generator=g, device="cuda").bfloat16() for _ in range(W)]
    order = O.single_ring_order(rank, W)
    heads, group = [(0, 0), (B - 1, Hq - 1)], Hq // Hkv
    out, lse = M.attn_fwd_block(q, torch.cat([c[0] for c in chunks], 1), torch.cat([c[1] for c in chunks], 1), scale)

    runs = []
    for ring in (M.LocalRing((W,), rank, chunks), M.LocalRing((W,), rank, chunks), by_hops(W, rank, chunks)):
        dq, dkv = torch.full(q.shape, float("nan"), dtype=dq_dtype, device="cuda"), torch.full_like(chunks[rank], float("nan"))
        kept = {} if keep else None
        M.flash_attn_backward(q, chunks[rank], out, lse, dout, dq, dkv, scale, ring=ring, dkv_chunks=kept)
        torch.cuda.synchronize()
        runs.append((dq, dkv, kept))
    assert torch.equal(runs[0][0], runs[1][0])
    # The same products summed in fp32; delta = rowsum(dout * out) may be added up in another order, which can move a dS to the
    # next bf16 value, and so can the sums a gradient: 2^-8 of each value at the very most.
    pairs = [("dq", runs[0][0], runs[2][0]), ("dkv", runs[0][1], runs[2][1])]
    for name, a, b in pairs + [(f"dkv {c}", runs[0][2][c], runs[2][2][c]) for c in range(W) if keep]:
        rel = ((a.float() - b.float()).norm() / b.float().norm()).item()
        assert rel <= 2 ** -8, (name, rel)
    for b, h in heads:
        one = lambda t: t[b:b + 1, :, h:h + 1].float().cpu()
        kv1 = [torch.stack([c[i][b:b + 1, :, h // group:h // group + 1] for i in range(2)]).float().cpu() for c in chunks]
        rdq, _ = O.ring_backward(one(q), kv1, order, one(out), lse[b:b + 1, h:h + 1].cpu(), one(dout), scale)
        _check_grad(f"dq {b} {h}", one(runs[0][0]), rdq)
