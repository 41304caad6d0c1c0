"""Argument validation of the C ABI: every rejected call returns its error code before anything is launched,
so these run without a GPU (the pointers are never dereferenced)."""
import ctypes

import pytest

from mercury_artifact_amd import _native as N

OK, EINVAL, EDTYPE, EHEADDIM, EALIGN, EUNSUPPORTED = 0, -1, -2, -3, -4, -6
P = 0x10000           # a non-NULL, 16-byte aligned "pointer"


@pytest.fixture(scope="module")
def lib():
    return N.lib()


def _fwd(lib, q=P, k=P, v=P, out=P, lse=P, B=1, Sq=64, Sc=64, Hq=2, Hkv=2, D=128,
         strides=None, scale=0.1, mask=0, dtype=0, descales=(None, None, None)):
    if strides is None:
        strides = [Sq * Hq * D, Hq * D, D, Sc * Hkv * D, Hkv * D, D, Sc * Hkv * D, Hkv * D, D, Sq * Hq * D, Hq * D, D]
    return lib.mhip_attn_fwd_block(q, k, v, out, lse, B, Sq, Sc, Hq, Hkv, D, *strides, scale, mask, dtype,
                                   *descales, None)


def test_forward_rejects(lib):
    for bad in (0, 4, 100, 136, 256):
        assert _fwd(lib, D=bad) == EHEADDIM
    assert _fwd(lib, D=72, dtype=1) == EHEADDIM                 # e4m3: multiples of 16
    big64 = 1 << 19                                             # D = 64: spans of one (batch, head) stay below 1 GiB
    assert _fwd(lib, D=64, Sc=1024, strides=[64 * 128, 128, 64, 1024 * big64, big64, 64, 1024 * big64, big64, 64,
                                             64 * 128, 128, 64]) == EUNSUPPORTED
    assert _fwd(lib, Hq=3, Hkv=2) == EINVAL
    assert _fwd(lib, Sq=-1) == EINVAL
    assert _fwd(lib, scale=0.0) == EINVAL
    assert _fwd(lib, scale=float("inf")) == EINVAL
    assert _fwd(lib, scale=float("nan")) == EINVAL
    assert _fwd(lib, mask=2) == EINVAL
    assert _fwd(lib, dtype=7) == EDTYPE
    assert _fwd(lib, q=None) == EINVAL
    assert _fwd(lib, k=None) == EINVAL
    assert _fwd(lib, q=P + 8) == EALIGN
    s = [64 * 2 * 128, 2 * 128, 128] * 4
    s[1] += 4                                   # a row stride that breaks 16-byte alignment
    assert _fwd(lib, strides=s) == EALIGN
    big = 1 << 20                               # rows 2 MiB apart: 2048 of them span 4 GiB
    assert _fwd(lib, Sc=2048, strides=[64 * 256, 256, 128, 2048 * big, big, 128, 2048 * big, big, 128,
                                       64 * 256, 256, 128]) == EUNSUPPORTED
    assert _fwd(lib, dtype=1, descales=(P, P + 2, P)) == EALIGN    # descales are pointers to device floats
    # nothing to do: accepted without touching the pointers
    assert _fwd(lib, B=0) == OK
    assert _fwd(lib, Sq=0) == OK
    assert lib.mhip_error_string(EHEADDIM).startswith(b"head dimension")


def test_backward_rejects(lib):
    def bwd(B=1, Sq=64, Sc=64, Hq=2, Hkv=2, D=128, scale=0.1, mask=0, dq=P, ws=P, strides=None, dq_acc=None):
        if strides is None:
            strides = [Sq * Hq * D, Hq * D, D, Sc * Hkv * D, Hkv * D, D, Sc * Hkv * D, Hkv * D, D,
                       Sq * Hq * D, Hq * D, D, Sq * Hq * D, Hq * D, D]
        return lib.mhip_attn_bwd_block(P, P, P, P, P, P, dq, P, P, dq_acc, B, Sq, Sc, Hq, Hkv, D, *strides,
                                       scale, mask, 0, ws, None)

    for bad in (0, 4, 100, 136, 256):
        assert bwd(D=bad) == EHEADDIM
    assert bwd(Hq=5, Hkv=2) == EINVAL
    assert bwd(scale=-1.0) == EINVAL
    assert bwd(mask=3) == EINVAL
    assert bwd(dq=None) == EINVAL
    assert bwd(ws=None) == EINVAL
    assert bwd(dq=P + 4) == EALIGN
    assert bwd(strides=[64 * 256, 257, 128, 64 * 256, 256, 128, 64 * 256, 256, 128] + [64 * 256, 256, 128] * 2) == EALIGN
    assert bwd(strides=[64 * 256, 256, 128] * 3 + [64 * 256, 260, 128, 64 * 256, 256, 128]) == EALIGN     # dq rows
    assert bwd(Sq=4096, strides=[1 << 33, 1 << 21, 128, 64 * 256, 256, 128, 64 * 256, 256, 128]
               + [4096 * 256, 256, 128] * 2) == EUNSUPPORTED
    assert bwd(B=0) == OK
    assert lib.mhip_attn_bwd_workspace_bytes(2, 100, 64, 4, 2, 128) >= 2 * 2 * 4 * 100 * 4


@pytest.mark.parametrize("B,Sq,Hq", [(1, 64, 1), (1, 512, 8), (2, 1500, 12), (1, 4096, 32), (4, 512, 5)])
def test_one_backward_workspace_serves_every_chunk(lib, B, Sq, Hq):
    """A call does not say how large its workspace is, so a workspace kept over chunks of different lengths, for either
    mask, has to be large enough for all of them: the three row arrays and the largest partial sums."""
    sizes = {lib.mhip_attn_bwd_workspace_bytes(B, Sq, Sc, Hq, Hkv, D)
             for Sc in (0, 1, 64, 333, 1024, 4096, 65536) for Hkv in (1, Hq) for D in (8, 64, 96, 128)}
    assert sizes == {(B * Sq * Hq + 3) // 4 * 4 * 12 + (32 << 20)}
    assert lib.mhip_attn_bwd_workspace_bytes(B, 0, 64, Hq, 1, 64) == 0


def test_elementwise_rejects(lib):
    assert lib.mhip_flash_reduce(P, P, None, 8, 128, None) == EINVAL
    assert lib.mhip_flash_reduce(P, P + 4, P, 8, 128, None) == EALIGN
    assert lib.mhip_flash_reduce(P, P, P, -1, 128, None) == EINVAL
    assert lib.mhip_flash_reduce(P, P, P, 0, 128, None) == OK
    two = (ctypes.c_void_p * 2)(P, P)
    sb2 = (ctypes.c_int64 * 2)(8 * 4 * 128, 8 * 4 * 128)

    def many(outs=two, lses=two, sb=sb2, begin=None, n=2, fo=P, fl=P, D=128, st=(128 * 4, 128), B=1):
        return lib.mhip_lse_merge_many(outs, lses, sb, begin, n, fo, fl, B, 8, 4, D, *st, None)

    assert many(n=0) == EINVAL and many(n=65) == EINVAL
    assert many(fo=None) == EINVAL and many(outs=None) == EINVAL and many(sb=None) == EINVAL
    assert many(outs=(ctypes.c_void_p * 2)(P, None)) == EINVAL
    assert many(begin=(ctypes.c_int * 2)(0, 9)) == EINVAL and many(begin=(ctypes.c_int * 2)(-1, 0)) == EINVAL
    assert many(outs=(ctypes.c_void_p * 2)(P, P + 8)) == EALIGN
    assert many(st=(128 * 4 + 4, 128)) == EALIGN
    assert many(sb=(ctypes.c_int64 * 2)(4096, 4100)) == EALIGN
    assert many(D=44) == EUNSUPPORTED and many(D=264) == EUNSUPPORTED      # multiples of 8 up to 256
    assert many(B=0) == OK
    assert lib.mhip_tree_merge(P, None, P, 8, 128, 0, None) == EINVAL
    assert lib.mhip_tree_merge(P + 8, P, P, 8, 128, 1, None) == EALIGN
    assert lib.mhip_tree_merge(P, P, P, 0, 128, 1, None) == OK
    # overlapping operands: dst == src is the in-place form of the tree merge, any other overlap is refused;
    # the flat packed kernels take no overlap at all
    assert lib.mhip_tree_merge(P, P, P + 16, 8, 128, 1, None) == EINVAL
    assert lib.mhip_tree_merge(P + 16, P, P, 8, 128, 0, None) == EINVAL
    assert lib.mhip_flash_reduce(P, P + 0x100000, P, 8, 128, None) == EINVAL
    assert lib.mhip_flash_reduce(P + 0x100000, P, P + 16, 8, 128, None) == EINVAL
    assert lib.mhip_pack_reduce(P, P, P, P + 32, 1, 8, 2, 128, None) == EINVAL
    assert lib.mhip_pack_reduce(None, P, P, None, 1, 8, 2, 128, None) == EINVAL
    assert lib.mhip_pack_reduce(P + 4, P, P, P, 1, 8, 2, 128, None) == EALIGN
    assert lib.mhip_pack_reduce(None, P, P, P, 0, 8, 2, 128, None) == OK
    assert lib.mhip_grad_accumulate(None, P, None, 16, None) == EINVAL
    assert lib.mhip_grad_accumulate(None, P + 2, P, 16, None) == EALIGN
    assert lib.mhip_grad_accumulate(None, P, P, 0, None) == OK
    assert lib.mhip_unpack(P, None, P, 1, 8, 2, 128, None) == EINVAL
    assert lib.mhip_unpack(P, P + 8, P, 1, 8, 2, 128, None) == EALIGN
    assert lib.mhip_unpack(P, P, P, 1, 8, 2, 100, None) == EUNSUPPORTED
    assert lib.mhip_unpack(P, P, P, 0, 8, 2, 128, None) == OK
    assert lib.mhip_quantize_e4m3(P, 1, 64, P, P, P, None) == EDTYPE
    assert lib.mhip_quantize_e4m3(P, 2, -1, P, P, P, None) == EINVAL
    assert lib.mhip_quantize_e4m3(P, 2, 64, P, None, P, None) == EINVAL
    assert lib.mhip_quantize_e4m3(None, 2, 64, P, P, P, None) == EINVAL
    assert lib.mhip_quantize_e4m3(P + 4, 2, 64, P, P, P, None) == EALIGN


def test_forward_blocks_reject(lib):
    def blocks(ks=(P, P), vs=(P, P), n=2, o_sn=8192, out=P, per=1, mask=0):
        array = ctypes.c_void_p * 17
        return lib.mhip_attn_fwd_blocks(P, array(*ks) if ks else None, array(*vs) if vs else None, n, per, out, o_sn, P, 1, 64, 64, 1, 1, 128,
                                        *[8192, 128, 128] * 4, 0.1, mask, 0, None, None, None, None)

    assert blocks(per=0) == blocks(per=-1) == EINVAL and blocks(per=2, mask=1) == EUNSUPPORTED
    assert blocks(n=0) == blocks(n=17, ks=[P] * 17, vs=[P] * 17) == blocks(n=-1) == EINVAL
    assert blocks(ks=None) == blocks(vs=None) == blocks(ks=(P, 0)) == blocks(vs=(P, 0)) == blocks(out=None) == EINVAL
    assert blocks(ks=(P, P + 8)) == blocks(vs=(P, P + 8)) == blocks(o_sn=8196) == EALIGN


def test_backward_chunks_reject(lib):
    def chunks(n=3, ks=(P,) * 17, vs=(P,) * 17, dks=(P,) * 17, dvs=(P,) * 17, dk32s=(0,) * 17, dv32s=(0,) * 17, dout=P, q=P, out=P, lse=P,
               dq=P, acc=P, first=1, last=1, B=1, Sq=64, Sc=64, Hq=2, Hkv=2, D=128, k_ss=256, scale=0.1, workspace=P):
        lists = [None if x is None else (ctypes.c_void_p * 17)(*x) for x in (ks, vs, dks, dvs, dk32s, dv32s)]
        return lib.mhip_attn_bwd_chunks(dout, q, *lists[:2], n, out, lse, dq, acc, first, last, 0, *lists[2:], B, Sq, Sc, Hq, Hkv, D,
                                        Sq * 256, 256, 128, Sc * k_ss, k_ss, 128, *[Sc * 256, 256, 128] * 3, scale, workspace, None)

    def at(i, value, fill=P):
        return tuple(value if j == i else fill for j in range(17))

    assert chunks(n=0) == chunks(n=17) == chunks(n=-1) == EINVAL
    for name in ("ks", "vs", "dks", "dvs", "dk32s", "dv32s"):
        assert chunks(**{name: None}) == EINVAL
    for i in (0, 2):                     # the first element, which other checks see too, and one that only the list holds
        assert chunks(ks=at(i, 0)) == chunks(vs=at(i, 0)) == EINVAL
        assert chunks(dks=at(i, 0)) == chunks(dvs=at(i, 0)) == EINVAL                               # dk without dv, dv without dk
        assert chunks(dk32s=at(i, P, 0)) == chunks(dv32s=at(i, P, 0)) == EINVAL
        assert chunks(dks=at(i, 0), dvs=at(i, 0)) == EINVAL                                         # no place in either type
        for name in ("ks", "vs", "dks", "dvs"):
            assert chunks(**{name: at(i, P + 8)}) == EALIGN
        assert chunks(dk32s=at(i, P + 4, 0), dv32s=at(i, P, 0)) == chunks(dk32s=at(i, P, 0), dv32s=at(i, P + 4, 0)) == EALIGN
    assert chunks(first=0, acc=None) == chunks(first=0, last=0, acc=None) == chunks(last=0, acc=None) == EINVAL
    assert chunks(dq=None) == chunks(q=None) == chunks(dout=None) == chunks(out=None) == chunks(lse=None) == chunks(workspace=None) == EINVAL
    assert chunks(Hkv=0) == chunks(Hkv=3) == chunks(Sq=-1) == chunks(scale=0.0) == EINVAL
    assert chunks(D=132) == chunks(D=0) == EHEADDIM and chunks(k_ss=260) == EALIGN
    assert chunks(Sc=1 << 20, k_ss=1024) == EUNSUPPORTED                                            # a span of 2 GiB
    assert chunks(Sc=1 << 30, k_ss=0, Hq=16, Hkv=16, n=16) == EUNSUPPORTED                          # 2^31 workgroups
    assert chunks(B=0) == OK
