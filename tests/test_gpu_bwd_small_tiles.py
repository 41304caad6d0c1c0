"""The dQ pass on 16 x 16 MFMA tiles, which launches take that keep every CU busy for long: at least 218 workgroups of 256 query
rows in the last round of 256, 32 key tiles and more, causal launches of 512 workgroups.  Against the oracle on some of the
heads, with the bounds of test_gpu_bwd.py, whose oracle inputs (out, lse of the oracle's own forward) are used here too."""
import ctypes

import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N
from test_gpu_bwd import _check_grad

pytestmark = pytest.mark.gpu
H = 32


def _run(Sq, Sc, D, causal, heads=(0, 31)):
    import mercury_artifact_amd as M

    splits = (ctypes.c_int * 2)()
    assert N.lib().mhip_attn_bwd_plan(1, Sq, Sc, H, H, D, int(causal), splits) == 2
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
