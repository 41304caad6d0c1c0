"""Fixed-schedule drivers of one rank's ring-attention step on one GPU.

Each driver has the argument list of the function Mercury generates from the template of the same
name (utils/flash_attn_dsl.py:127-180, 182-235, 237-291, 345-408; utils/attn_bwd_dsl.py:37-135) plus a
``ring`` keyword: the :class:`~mercury_artifact_amd.schedule.LocalRing` that stands in for the
neighbour exchange.  The body is the loop the code generator emits for that template
(mercury/backend/pytorch/codegen.py:264-355, 443-523): take the current KV chunk, start the hop for
the next one, run the block kernel, fold with ``update_out_and_lse``, and store after the last step.  A
forward driver's blocks go through ``_flash_attn_forward`` unless it would do nothing but call the kernel;
then they are written straight into places allocated once per step, and where a ring's chunks all lie in this GPU's
memory (``LocalRing.resident``), the blocks of several are launched together if one launch each is too small for the chip.

Two defaults of the forward drivers depart from the literal sequence without changing what is computed:
``deferred_merge=True`` keeps the bf16 block results of all chunks and folds them with ONE
``merge_many`` call after the last chunk (the fold is associative; every block output is read once
instead of the fp32 accumulator travelling through memory once per chunk; results agree with the chain
to fp32 rounding), and ``fused_epilogue=True`` lets the last merge of the chain write ``o`` / ``lse``
itself (bit-identical).  ``deferred_merge=False, fused_epilogue=False`` is the generated code's literal
sequence: ``update_out_and_lse`` per chunk, then ``o[...] = _out.to(o.dtype)``,
``lse[...] = _lse.squeeze(-1).transpose(1, 2)``.
"""
from __future__ import annotations

import warnings
from functools import lru_cache
from typing import Optional

import torch

from . import _native as N
from . import flash_attn_interface as _ops
from .flash_attn_interface import (_flash_attn_backward, _flash_attn_forward, aligned_rows, attn_bwd_block,
                                   attn_bwd_chunk)
from .merge import (MAX_MERGE_MANY, get_default_args, grad_accumulate, merge_into, merge_many, pack_block,
                    unpack_into, update_out_and_lse)
from .schedule import (LocalRing, n_dim_to_one_dim, n_ranks, one_dim_to_n_dim, reduce_buffer_route,
                       shift_tuple_element, zigzag_step)

MAX_GROUP = 16           # MHIP_MAX_GROUP: chunks of a launch
UNKEPT_BYTES = 32 << 20  # gradients that a launch over several chunks may make for nobody (or one chunk's, if that is more)

__all__ = ["flash_attn_pack_kv", "gqa_pack_kv", "flash_attn_pack_split_kv", "flash_attn_expose_reduce",
           "flash_attn_expose_reduce_q_ring",
           "flash_attn_backward", "zigzag_causal_pack_kv", "fp8_pack_split_kv", "quantize_e4m3"]


@lru_cache(maxsize=None)
def _hop_list(mesh_shape):
    total = n_ranks(mesh_shape)
    hops = []
    idx = [0] * len(mesh_shape)
    for _ in range(total):
        hops.append(next((d for d in range(len(mesh_shape)) if idx[d] + 1 != mesh_shape[d]), None))
        # advance the odometer (dimension 0 fastest)
        for d in range(len(mesh_shape)):
            idx[d] += 1
            if idx[d] < mesh_shape[d]:
                break
            idx[d] = 0
    return tuple(hops)


def _hops(ring: LocalRing):
    """The mesh dimension of the hop at every step in generated-loop order: innermost mesh dimension first, a hop on
    the next dimension when the inner loop wraps, None after the very last step."""
    return _hop_list(ring.mesh_shape)


@lru_cache(maxsize=None)
def _neighbour_ranks(mesh_shape, rank, dim):
    me = one_dim_to_n_dim(rank, mesh_shape)
    size = mesh_shape[dim]
    send_to = n_dim_to_one_dim(shift_tuple_element(me, dim, 1, size), mesh_shape)
    recv_from = n_dim_to_one_dim(shift_tuple_element(me, dim, -1, size), mesh_shape)
    return send_to, recv_from


def _neighbours(ring: LocalRing, dim: int):
    return _neighbour_ranks(ring.mesh_shape, ring.rank, dim)


def _block_forward(q, k, v, softmax_scale, dropout_p, causal, window_size, alibi_slopes, q_descale=None, k_descale=None,
                   v_descale=None, into=None):
    """(out, lse) of the block operator on the values a generated step passes it by keyword; ``into`` gives the two
    tensors to write (see :func:`_block_results`)."""
    if into is not None:
        return _ops.attn_fwd_block(q, k, v, softmax_scale, causal, q_descale, k_descale, v_descale, *into)
    outputs = _flash_attn_forward(q, k, v, dropout_p, softmax_scale, causal, window_size[0], window_size[1], 0.0, alibi_slopes,
                                  dropout_p > 0, q_descale, k_descale, v_descale)
    assert len(outputs) == 4
    return outputs[:2]


def _straight(q, kv, softmax_scale, dropout_p, causal, window_size, alibi_slopes, **descales) -> bool:
    """Whether the block operator would do nothing but call the kernel: nothing to report, nothing to record."""
    return bool(_ops.as_declared((softmax_scale, dropout_p), window_size, (causal,))
                and not (dropout_p or alibi_slopes is not None or window_size[0] != -1 or window_size[1] != -1)
                and q.dim() == 4 and N.host.undispatched(q, kv, *descales.values()))


def _result_places(n, q):
    """(outs, lses) for ``n`` block results over all rows of ``q``, from one allocation each."""
    B, Sq, Hq, D = q.shape
    return (torch.empty((n, B, Sq, Hq, D), dtype=torch.bfloat16, device=q.device),
            torch.empty((n, B, Hq, Sq), dtype=torch.float32, device=q.device))


def _block_results(n, q, kv, *args, **kwargs):
    """Places for the results of a step's ``n`` blocks over all rows of ``q``; None for every block where the operator has
    something to report or to record."""
    if not _straight(q, kv, *args, **kwargs):
        return [None] * n
    outs, lses = _result_places(n, q)
    return list(zip(outs.unbind(0), lses.unbind(0)))


def _resident(ring) -> bool:
    """Whether a step may take several chunks of the ring before it launches.  Not where every hop makes a copy: a step
    would hold as many of them as there are chunks, instead of the ones in use and the next."""
    return bool(type(ring).__dict__.get("resident")) and not getattr(ring, "copy", False)


class _Together:
    """Block forwards of one query tensor over ``n`` chunks of a ring whose chunks are all there, several to a launch
    (mhip_attn_fwd_group) and, where that is faster, a run of chunks to a result (mhip_attn_fwd_chain).  ``size``, the
    chunks of a launch, is 1 where every block goes its own way."""

    def __init__(self, n, q, kv, ring, softmax_scale, dropout_p, causal, window_size, alibi_slopes, q_descale=None, k_descale=None,
                 v_descale=None):
        self.size = self.per = 1
        if (n < 2 or not _resident(ring)
                or not _straight(q, kv, softmax_scale, dropout_p, causal, window_size, alibi_slopes, q_descale=q_descale,
                                 k_descale=k_descale, v_descale=v_descale)):
            return
        self.per = 1 if causal else N.host.fwd_chain(q, kv, n) or 1
        launches = -(-n // MAX_GROUP) if self.per > 1 else 0
        self.size = -(-n // launches) if launches else N.host.fwd_group(q, n) or 1
        self.q, self.args = q, (softmax_scale, causal, q_descale, k_descale, v_descale)
        self.results = n if self.per == 1 else sum(-(-min(self.size, n - at) // self.per) for at in range(0, n, self.size))

    def run(self, chunks, places=None):
        """The (out, lse) results over the step's chunks, in two lists or, all of them, as the tensors of ``places``."""
        outs, lses = places or _result_places(self.results, self.q)
        done, apart = 0, None                   # apart: results of launches whose chunks were not of one layout
        for at in range(0, len(chunks), self.size):
            part = chunks[at:at + self.size]
            if apart is None and N.host.fwd_blocks(self.q, part, self.per, *self.args, outs, lses, done) is True:
                done -= -len(part) // self.per
                continue
            if apart is None:
                apart = list(zip(outs[:done].unbind(0), lses[:done].unbind(0)))
            apart += [_ops.attn_fwd_block(self.q, c[0], c[1], *self.args) for c in part]
        return (outs, lses) if apart is None else ([r[0] for r in apart], [r[1] for r in apart])

    def step(self, chunks, o, lse):
        """The whole step: results and their fold.  A single result is written straight to ``o`` and ``lse`` if neither overlaps
        anything the launch reads."""
        places = None
        if self.results == 1:
            read = [t for t in (self.q, *chunks, *self.args[2:]) if t is not None]
            if N.host.apart(o, lse, *read) is True and N.host.apart(lse, *read) is True:
                places = o[None], lse[None]
        outs, lses = self.run(chunks, places)
        if (places and outs is places[0]) or N.host.merge_many(outs, lses, o, lse, None) is not None:
            return
        merge_many(list(outs), list(lses), o, lse)


@lru_cache(maxsize=256)
def _visits(mesh_shape, rank, held):
    """The chunks ``rank`` holds at the steps of a ring that starts with ``held``, and what everyone holds in the end."""
    ring = LocalRing(mesh_shape, rank)
    ring.held = list(held)
    seen = [ring.current]
    for hop in _hop_list(mesh_shape)[:-1]:
        seen.append(ring.hop(hop))
    return tuple(seen), ring.held


def _hop_methods():
    return LocalRing.send_recv, LocalRing.commit, LocalRing.wait, LocalRing.hop


_HOP = _hop_methods()       # as this package defines them: a wrapper put over one, on a ring or on the class, sees every hop


def _resident_chunks(ring, kv):
    """A step's chunks in visiting order, for a ring whose chunks are all there; leaves the ring where the hops would."""
    chunks = [_as_rows(kv)]
    if (type(ring) is LocalRing and ring.chunks is not None and not ring._committed
            and ring.__dict__.keys().isdisjoint(("send_recv", "commit", "wait", "hop")) and _hop_methods() == _HOP):  # nobody looks on
        seen, held = _visits(ring.mesh_shape, ring.rank, tuple(ring.held))
        chunks += [ring.chunks[i] for i in seen[1:]]
        ring.held = list(held)
        return chunks
    for step, hop in enumerate(_hops(ring)):
        if step > 0:
            ring.wait()
        if hop is not None:
            chunks.append(ring.send_recv(*_neighbours(ring, hop), chunks[-1]))
            ring.commit()
    return chunks


def _as_rows(t):
    """A chunk if the kernels take its rows as they are (alignment, 32-bit reach), else a copy."""
    return t if N.host.rows_fit(t) else t.contiguous()


_SIDE_STREAMS = {}


def _side_stream(device) -> "torch.cuda.Stream":
    """One extra stream per device (default priority), made on first use and kept."""
    key = torch.device(device).index if torch.device(device).index is not None else torch.cuda.current_device()
    if key not in _SIDE_STREAMS:
        _SIDE_STREAMS[key] = torch.cuda.Stream(device=key)
    return _SIDE_STREAMS[key]


def _ring_forward(q, kv, o, lse, softmax_scale, dropout_p, causal, window_size, alibi_slopes,
                  ring: LocalRing, fused_epilogue: bool, deferred_merge: bool, ring_divide: int = 1,
                  two_streams: bool = False, **extra):
    """The chunk loop of the forward templates.  ``ring_divide = k > 1`` is the schedule option of the same
    name (mercury/backend/pytorch/codegen.py:299-306): an outer loop over k sub-chunks of the KV rows wraps
    the ring loop, so the step makes k * W block calls on (Sq x Sc / k) blocks and every hop moves 1/k of a
    chunk.

    ``two_streams`` (with the deferred fold only, where the block launches do not depend on each other): every
    other block launch goes to a second stream, so that the tail of one launch (workgroups of its last round,
    drained pipelines) overlaps the head of the next; the fold waits for both.  The side stream starts behind
    everything queued on the current stream when the step begins, and a block launched there waits for the event
    recorded on the current stream right behind the hop that delivers its chunk (so for the hop's copy, not for the
    block launch that follows it on the current stream)."""
    blocks = []
    _out = None
    _lse = None
    _kv = None
    _next_kv = None
    steps = _hops(ring)
    ring_divide = int(ring_divide)
    Sc = kv.shape[2]
    if ring_divide < 1 or Sc % ring_divide:
        raise ValueError("ring_divide must divide the chunk's rows")
    if ring_divide > 1 and ring.chunks is None:
        raise ValueError("ring_divide needs a LocalRing that holds the chunks")
    sub = Sc // ring_divide
    n_blocks = len(steps) * ring_divide
    defer = (deferred_merge and n_blocks <= MAX_MERGE_MANY and o.dtype == torch.bfloat16
             and o.is_contiguous() and lse.is_contiguous())
    if deferred_merge and not defer:
        warnings.warn(f"ring step of {n_blocks} blocks into a {o.dtype} output: the one-pass fold takes at most "
                      f"{MAX_MERGE_MANY} blocks and writes contiguous bfloat16, so this step merges block by block "
                      "(same result, one pass over the fp32 accumulator per block)", RuntimeWarning, stacklevel=3)
    done = 0
    places = [None] * n_blocks
    # (a divided ring goes sub-chunk by sub-chunk whether its chunks are all there or not: the option is for rings that want
    # to hold little of other ranks' keys at a time)
    if defer and not two_streams and ring_divide == 1:
        together = _Together(n_blocks, q, kv, ring, softmax_scale, dropout_p, causal, window_size, alibi_slopes, **extra)
        if together.size > 1:
            together.step(_resident_chunks(ring, kv), o, lse)
            return
    if defer:
        places = _block_results(n_blocks, q, kv, softmax_scale, dropout_p, causal, window_size, alibi_slopes, **extra)
    main = side = None
    kv_ready = next_ready = None
    if two_streams and defer:
        main = torch.cuda.current_stream(q.device)
        side = _side_stream(q.device)
        side.wait_stream(main)
    for part in range(ring_divide):
        rows = slice(part * sub, (part + 1) * sub)
        part_ring = ring if ring_divide == 1 else \
            LocalRing(ring.mesh_shape, ring.rank, [c[:, :, rows] for c in ring.chunks], copy=ring.copy)
        for step, hop in enumerate(steps):
            if step == 0:
                _kv = kv if ring_divide == 1 else kv[:, :, rows]
                # (a subclass may send it, and transports want it in one piece)
                _kv = _as_rows(_kv) if type(ring) is LocalRing else _kv.contiguous()
                kv_ready = None
                if side is not None and part > 0:      # a copy above sits behind earlier launches
                    kv_ready = torch.cuda.Event()
                    kv_ready.record(main)
            else:
                part_ring.wait()
                _kv = _next_kv
                kv_ready = next_ready
            if hop is not None:
                send_to, recv_from = _neighbours(part_ring, hop)
                _next_kv = part_ring.send_recv(send_to, recv_from, _kv)
                part_ring.commit()
                next_ready = None
                if side is not None:                   # what the hop enqueued on the current stream ends here
                    next_ready = torch.cuda.Event()
                    next_ready.record(main)
            _k, _v = _kv.unbind(0)
            if side is not None and done % 2 == 1:
                if kv_ready is not None:
                    side.wait_event(kv_ready)
                _kv.record_stream(side)              # may have been allocated by the hop on the current stream
                with torch.cuda.stream(side):
                    block_out, block_lse = _block_forward(q, _k, _v, softmax_scale, dropout_p, causal, window_size,
                                                          alibi_slopes, into=places[done], **extra)
                for t in (block_out, block_lse):
                    t.record_stream(side if places[done] is not None else main)      # the stream it was not allocated under
            else:
                block_out, block_lse = _block_forward(q, _k, _v, softmax_scale, dropout_p, causal, window_size, alibi_slopes,
                                                      into=places[done], **extra)
            done += 1
            if defer:
                blocks.append((block_out, block_lse))
                if done == n_blocks:
                    if side is not None:
                        main.wait_stream(side)
                    merge_many([b[0] for b in blocks], [b[1] for b in blocks], o, lse)
                    return
                continue
            if fused_epilogue and done == n_blocks:
                # last merge writes o / lse directly (same arithmetic, two passes fewer)
                merge_into(_out, _lse, block_out, block_lse, None, None, o, lse)
                return
            _out, _lse = update_out_and_lse(_out, _lse, block_out, block_lse)
    o[:, :, :, :] = _out.to(o.dtype)
    lse[:, :, :] = _lse.squeeze(dim=-1).transpose(1, 2)


def flash_attn_pack_kv(q, kv, o, lse, softmax_scale, dropout_p=0, causal=False, window_size=(-1, -1),
                       alibi_slopes=None, deterministic=False, *, ring: LocalRing,
                       fused_epilogue: bool = True, deferred_merge: bool = True, ring_divide: int = 1,
                       two_streams: bool = False):
    """Single-ring forward step (template utils/flash_attn_dsl.py:127-180).  q (B,Sq,H,D), kv the
    rank's own (2,B,Sc,H,D), o (B,Sq,H,D) and lse (B,H,Sq) are written."""
    _ring_forward(q, kv, o, lse, softmax_scale, dropout_p, causal, window_size, alibi_slopes, ring,
                  fused_epilogue, deferred_merge, ring_divide, two_streams)


def gqa_pack_kv(q, kv, o, lse, softmax_scale, dropout_p=0, causal=False, window_size=(-1, -1),
                alibi_slopes=None, deterministic=False, *, ring: LocalRing, fused_epilogue: bool = True,
                deferred_merge: bool = True, ring_divide: int = 1):
    """GQA forward step (template utils/flash_attn_dsl.py:182-235): kv has Hkv heads, q has
    Hkv * HEADS_PER_GROUP; the block kernel maps q head h to kv head h // HEADS_PER_GROUP."""
    _ring_forward(q, kv, o, lse, softmax_scale, dropout_p, causal, window_size, alibi_slopes, ring,
                  fused_epilogue, deferred_merge, ring_divide)


def flash_attn_pack_split_kv(q, kv, o, lse, softmax_scale, dropout_p=0, causal=False,
                             window_size=(-1, -1), alibi_slopes=None, deterministic=False, *,
                             ring: LocalRing, fused_epilogue: bool = True, deferred_merge: bool = True,
                             ring_divide: int = 1):
    """Double-ring forward step (template utils/flash_attn_dsl.py:237-291): ``ring`` is built on the
    2-D mesh ``(inner, outer)``; the loop order and hops follow from the mesh shape."""
    if len(ring.mesh_shape) != 2:
        raise ValueError("the double ring needs a 2-D mesh (inner, outer)")
    _ring_forward(q, kv, o, lse, softmax_scale, dropout_p, causal, window_size, alibi_slopes, ring,
                  fused_epilogue, deferred_merge, ring_divide)


def _store_packed(buf, o, lse, fused: bool):
    """The stores after the managed reduction (utils/flash_attn_dsl.py:406-407): one kernel, or the literal
    torch expressions."""
    if fused and o.dtype == torch.bfloat16 and o.is_contiguous() and lse.is_contiguous() and o.shape[-1] % 8 == 0 \
            and 256 % (o.shape[-1] // 8) == 0:
        unpack_into(buf, o, lse)
        return
    o[:, :, :, :] = buf[..., :-1].to(o.dtype)
    lse[:, :, :] = buf[..., -1].transpose(1, 2)


def flash_attn_expose_reduce(q, kv, o, lse, softmax_scale, dropout_p=0, causal=False,
                             window_size=(-1, -1), alibi_slopes=None, deterministic=False, *,
                             ring: LocalRing, fused_epilogue: bool = True, deferred_merge: bool = True):
    """Managed-reduction form (template utils/flash_attn_dsl.py:345-408) with the KV ring: the reduction buffer
    ``(out | lse)`` stays on the rank, so with ``deferred_merge`` the bf16 block results are kept and folded by ONE
    ``merge_many`` call after the last chunk, straight into ``o`` and ``lse`` (results agree with the packed chain to fp32
    rounding).  Otherwise -- and with ``fused_epilogue=False``, the literal stores -- block results are packed and folded
    by ``flash_reduce`` chunk by chunk; pack and reduce run as one kernel."""
    buf = None
    _kv = None
    _next_kv = None
    hops = _hops(ring)
    blocks = []
    defer = (fused_epilogue and deferred_merge and len(hops) <= MAX_MERGE_MANY and o.dtype == torch.bfloat16
             and o.is_contiguous() and lse.is_contiguous())
    places = [None] * len(hops)
    if defer:
        together = _Together(len(hops), q, kv, ring, softmax_scale, dropout_p, causal, window_size, alibi_slopes)
        if together.size > 1:
            together.step(_resident_chunks(ring, kv), o, lse)
            return
        places = _block_results(len(hops), q, kv, softmax_scale, dropout_p, causal, window_size, alibi_slopes)
    for step, hop in enumerate(hops):
        if step == 0:
            _kv = kv.contiguous()
        else:
            ring.wait()
            _kv = _next_kv
        if hop is not None:
            send_to, recv_from = _neighbours(ring, hop)
            _next_kv = ring.send_recv(send_to, recv_from, _kv)
            ring.commit()
        _k, _v = _kv.unbind(0)
        block_out, block_lse = _block_forward(q, _k, _v, softmax_scale, dropout_p, causal, window_size, alibi_slopes,
                                              into=places[step])
        if defer:
            blocks.append((block_out, block_lse))
        else:
            buf = pack_block(block_out, block_lse, reduce_into=buf)
    if defer:
        merge_many([b[0] for b in blocks], [b[1] for b in blocks], o, lse)
        return
    _store_packed(buf, o, lse, fused_epilogue)


def flash_attn_expose_reduce_q_ring(qs, kvs, os_, lses, softmax_scale, dropout_p=0, causal=False,
                                    window_size=(-1, -1), alibi_slopes=None, deterministic=False, *,
                                    mesh_shape=None, fused_epilogue: bool = True):
    """The managed-reduction template (utils/flash_attn_dsl.py:345-408) scheduled as a ring over the
    *reduce buffer*: every rank keeps its KV shard, Q and the packed partial result ``(out | lse)``
    travel (codegen.py:116-190).  A rank's step is: block forward of the Q that just arrived against
    the local KV, ``buf = flash_reduce(arrived_partial, pack(block))`` (one fused kernel), send on;
    after the last step the buffer makes the write-back hop of ``get_src_dst_ranks``
    (mercury/backend/pytorch/utils.py:171-192) to the rank that owns its Q rows.

    What arrives at a rank was computed by the other ranks, so this driver runs ALL ranks of the mesh
    in lock step on the one GPU: ``qs[r]``, ``kvs[r]`` are rank r's shards, ``os_[r]`` / ``lses[r]``
    receive its result.  One rank's share of the work is 1 / world of the launches."""
    world = len(qs)
    mesh_shape = tuple(mesh_shape) if mesh_shape is not None else (world,)
    sends, home_of = reduce_buffer_route(mesh_shape)
    if len(home_of) != world or not (len(kvs) == len(os_) == len(lses) == world):
        raise ValueError("need one q, kv, o and lse per rank of the mesh")
    q_cur = list(qs)
    arrived = [None] * world
    home = [None] * world
    for step in range(world):
        buf = []
        for r in range(world):
            kv = kvs[r]
            block_out, block_lse = _block_forward(q_cur[r], kv[0], kv[1], softmax_scale, dropout_p, causal, window_size,
                                                  alibi_slopes)
            buf.append(pack_block(block_out, block_lse, reduce_into=arrived[r]))
        if step + 1 != world:
            q_next, arrived = [None] * world, [None] * world
            for r in range(world):
                q_next[sends[step][r]], arrived[sends[step][r]] = q_cur[r], buf[r]
            q_cur = q_next
        else:
            for r in range(world):
                home[home_of[r]] = buf[r]
    for r in range(world):
        _store_packed(home[r], os_[r], lses[r], fused_epilogue)


def zigzag_causal_pack_kv(q, kv, o, lse, softmax_scale, dropout_p=0, causal=True, window_size=(-1, -1),
                          alibi_slopes=None, deterministic=False, *, ring: LocalRing, deferred_merge: bool = True):
    """Causal forward step in the zigzag layout (rank r holds sequence blocks r and 2W-1-r).  Not in
    the reference, which only carries the ``slice_`` hook (utils/flash_attn_dsl.py:56,63-68); the
    three step classes are the diagonal (causal block), "first half of the chunk" and "second half
    of the Q rows" (merged through ``slice_``)."""
    if len(ring.mesh_shape) != 1:
        raise ValueError("zigzag runs on a 1-D ring")
    world = ring.world
    Sq = q.shape[1]
    if Sq % 2 or kv.shape[2] != Sq:
        raise ValueError("zigzag needs an even number of local rows and equal Q / KV shards")
    half = Sq // 2
    _out = _lse = _kv = _next_kv = None
    defer = (deferred_merge and world <= MAX_MERGE_MANY and o.dtype == torch.bfloat16
             and o.is_contiguous() and lse.is_contiguous())
    blocks = []
    kinds = [zigzag_step(ring.rank, step, world)[0] for step in range(world)]
    places, together, waiting = {}, {}, []
    how = (softmax_scale, dropout_p, causal, window_size, alibi_slopes)
    for kind, rows, keys in (("diag", q, kv), ("kv_first_half", q, kv[:, :, :half]), ("q_second_half", q[:, half:], kv)):
        n = kinds.count(kind)
        together[kind] = _Together(n if defer else 0, rows, keys, ring, softmax_scale, dropout_p, kind == "diag", window_size, alibi_slopes)
        grouped = together[kind].size > 1
        places[kind] = iter([None] * n if grouped or not defer or not n else _block_results(n, rows, keys, *how))
    for step, kind in enumerate(kinds):
        if step == 0:
            _kv = kv.contiguous()
        else:
            ring.wait()
            _kv = _next_kv
        if step + 1 != world:
            send_to, recv_from = _neighbours(ring, 0)
            _next_kv = ring.send_recv(send_to, recv_from, _kv)
            ring.commit()
        bq, bkv, sl = q, _kv, None
        if kind == "kv_first_half":
            bkv = _kv[:, :, :half]
        elif kind == "q_second_half":
            bq, sl = q[:, half:], (slice(None), slice(half, None))
        if together[kind].size > 1:
            waiting.append(bkv)
            if step + 1 == world or kinds[step + 1] != kind:
                blocks += [(*r, 0 if sl is None else half) for r in zip(*(list(t) for t in together[kind].run(waiting)))]
                waiting = []
            continue
        block_out, block_lse = _block_forward(bq, bkv[0], bkv[1], softmax_scale, dropout_p, kind == "diag", window_size,
                                              alibi_slopes, into=next(places[kind]))
        if defer:
            blocks.append((block_out, block_lse, 0 if sl is None else half))
            continue
        _out, _lse = update_out_and_lse(_out, _lse, block_out, block_lse, slice_=sl)
    if defer:
        merge_many([b[0] for b in blocks], [b[1] for b in blocks], o, lse, row_begin=[b[2] for b in blocks])
        return
    o[:, :, :, :] = _out.to(o.dtype)
    lse[:, :, :] = _lse.squeeze(dim=-1).transpose(1, 2)


def quantize_e4m3(x: torch.Tensor):
    """Per-tensor e4m3 quantisation through mhip_quantize_e4m3: scale s = amax / 448 (fp32; 1 for an all-zero
    tensor), x_q = round-to-nearest-even(clamp(x / s, -448, 448)) as ``torch.float8_e4m3fn``.  Returns
    ``(x_q, s)`` with ``s`` a 0-dim fp32 tensor on the device (the block kernel's descale).  fp32 or bf16
    input on the GPU."""
    done = N.host.quantize_e4m3(x)
    if done is not None:
        return done
    N.require_cuda(x)
    if x.dtype not in (torch.float32, torch.bfloat16):
        raise RuntimeError("quantize_e4m3 takes float32 or bfloat16")
    xc = x.contiguous()
    xq = torch.empty(xc.shape, dtype=torch.float8_e4m3fn, device=x.device)
    ws = torch.empty(2, dtype=torch.float32, device=x.device)          # [scale, scratch for the maximum]
    with torch.cuda.device(x.device):
        code = N.lib().mhip_quantize_e4m3(N.ptr(xc), N.MHIP_F32 if x.dtype == torch.float32 else N.MHIP_BF16,
                                          xc.numel(), N.ptr(xq), ws.data_ptr(), ws.data_ptr() + 4, N.stream_of(xc))
    N.check(code, "mhip_quantize_e4m3")
    return xq, ws[0]


def fp8_pack_split_kv(q, kv, o, lse, softmax_scale, q_descale, k_descale, v_descale, dropout_p=0,
                      causal=False, window_size=(-1, -1), alibi_slopes=None, deterministic=False, *,
                      ring: LocalRing, fused_epilogue: bool = True, deferred_merge: bool = True,
                      ring_divide: int = 1):
    """Forward step on e4m3 Q/K/V with per-tensor descales (not in the reference); any mesh."""
    _ring_forward(q, kv, o, lse, softmax_scale, dropout_p, causal, window_size, alibi_slopes, ring,
                  fused_epilogue, deferred_merge, ring_divide, q_descale=q_descale, k_descale=k_descale,
                  v_descale=v_descale)


def flash_attn_backward(q, kv, o, lse, dout, dq, dkv, softmax_scale, dropout_p=0, causal=False,
                        window_size=(-1, -1), alibi_slopes=None, deterministic=False, *,
                        ring: LocalRing, dkv_chunks: Optional[dict] = None, fused_accumulate: bool = True):
    """Backward ring step (template utils/attn_bwd_dsl.py:37-135 after ``shift`` on the KV axis):
    KV chunks arrive in ring order, each gets a block backward against the local q / o / lse / dout;
    dq accumulates in fp32 over the chunks (utils/attn_bwd_dsl.py:117-122) and is stored as
    ``dq.dtype`` at the end (131-132).  The fp32 dK/dV accumulator that travels with its chunk on a
    real ring has exactly one contribution per rank, so here each chunk's block gradient is kept in
    ``dkv_chunks[chunk id]`` (fp32) and the rank's own chunk is stored to ``dkv``.

    ``fused_accumulate=True`` (default) lets the block kernels do the sums: dq's carries over from chunk to chunk in
    fp32 (the sum sees the unrounded block gradients) and is written in q's type by the last one, and a chunk's dK/dV
    are written in fp32 where ``dkv_chunks`` asks for them: no pass over the gradients besides.  ``False`` is the literal
    sequence: block backward through ``_flash_attn_backward(**params)``, then ``torch.add`` on the bf16 block gradients.

    ``dq`` may lie over ``q``, ``dout`` or ``o`` and ``dkv`` over the own chunk: where a gradient's place overlaps what the
    launch that would write it reads, it is stored behind that launch."""
    if dropout_p != 0 or alibi_slopes is not None or tuple(window_size) != (-1, -1):
        fused_accumulate = False                # let the operator report what it does not support
    # operands of other layouts go through the block operator, which copies them where it has to
    carried = (fused_accumulate and aligned_rows(q, dout) and aligned_rows(o) and lse.is_contiguous()
               and q.shape == o.shape == dout.shape)
    write_dq = carried and aligned_rows(dq) and dq.shape == q.shape and N.host.apart(dq, q, dout, o, lse, kv)
    reduce_dq = None
    if not carried and fused_accumulate:
        reduce_dq = torch.zeros(q.shape, dtype=torch.float32, device=q.device)
    elif carried and not (write_dq and ring.world == 1):
        reduce_dq = torch.empty(q.shape, dtype=torch.float32, device=q.device)
    _kv = _next_kv = prepared = None
    own = ring.current
    group, waiting = 1, []
    if carried and _resident(ring):
        group = ring.world
        if dkv_chunks is None:
            # The other ranks' chunks' gradients need places all the same, and what a launch takes is chosen among as many as
            # there are places for: with fewer chunks another form can be the fastest, chunk by chunk among them (B4 H32/1
            # D128, 4 chunks of 6000 keys, places for two: 26.9 ms chunk by chunk, 28.3 two at a time).
            most = max(1, UNKEPT_BYTES // max(1, kv.numel() * kv.element_size()))
            group = -(-group // -(-group // most))          # in launches of one size
        group = N.host.bwd_group(q, kv, group) or 1
    for step, hop in enumerate(_hops(ring)):
        if step == 0:
            _kv = kv.contiguous()
        else:
            ring.wait()
            _kv = _next_kv
        chunk_id = ring.current
        if hop is not None:
            send_to, recv_from = _neighbours(ring, hop)
            _next_kv = ring.send_recv(send_to, recv_from, _kv)
            ring.commit()
        if carried:
            waiting.append((chunk_id, _kv))
            if len(waiting) < group and hop is not None:
                continue
            chunks = [c for _, c in waiting]
            if hop is None and write_dq and step > 0:
                write_dq = N.host.apart(dq, *chunks)
            block_dkvs, chunk_grads, staged = [], [], None
            for i, c in waiting:
                direct = (i == own and dkv.shape == c.shape and aligned_rows(dkv[0], dkv[1])
                          and N.host.apart(dkv, q, dout, o, lse, *chunks))
                block_dkv = chunk_grad = None
                if direct:
                    block_dkv = dkv
                elif i == own or dkv_chunks is None:
                    block_dkv = torch.empty(c.shape, dtype=c.dtype, device=c.device)
                    staged = block_dkv if i == own else staged
                if dkv_chunks is not None:
                    chunk_grad = dkv_chunks[i] = torch.empty(c.shape, dtype=torch.float32, device=c.device)
                block_dkvs.append(block_dkv)
                chunk_grads.append(chunk_grad)
            # rowsum(dout * o) and the scaled lse are the same for every chunk: worked out with the first one
            rows = [_as_rows(c) for c in chunks]
            first, last = step + 1 == len(chunks), bool(write_dq and hop is None)
            done = None
            if len(chunks) > 1:
                done = N.host.bwd_chunks(dout, q, rows, o, lse, dq if last else None, reduce_dq, first, last, block_dkvs,
                                         chunk_grads, softmax_scale, prepared)
                prepared = done if prepared is None else prepared
            for n, c in enumerate(rows if done is None else ()):
                _k, _v = c.unbind(0)
                usual = c.shape == kv.shape
                ws = attn_bwd_chunk(dout, q, _k, _v, o, lse, dq if write_dq else None, reduce_dq, first and n == 0,
                                    last and n + 1 == len(rows), block_dkvs[n], chunk_grads[n], softmax_scale,
                                    prepared if usual else None)
                prepared = ws if usual else prepared
            if staged is not None:
                dkv[...] = staged
            waiting = []
            continue
        block_dq = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        block_dkv = torch.empty(_kv.shape, dtype=kv.dtype, device=kv.device)
        if fused_accumulate:
            attn_bwd_block(dout, q, _kv[0], _kv[1], o, lse, block_dq, block_dkv[0], block_dkv[1], softmax_scale,
                           causal=False, deterministic=deterministic, dq_acc=reduce_dq)
            if dkv_chunks is not None:
                dkv_chunks[chunk_id] = grad_accumulate(None, block_dkv)
            if chunk_id == own:
                dkv[...] = block_dkv
            continue
        params = get_default_args(_flash_attn_backward).copy()
        params.update({
            "dout": dout, "q": q, "k": _kv[0], "v": _kv[1], "out": o, "softmax_lse": lse,
            "dq": block_dq, "dk": block_dkv[0], "dv": block_dkv[1],
            "softmax_scale": softmax_scale, "dropout_p": dropout_p, "causal": False,
            "deterministic": deterministic, "alibi_slopes": alibi_slopes,
        })
        if "window_size" in params:
            params.update({"window_size": window_size})
        else:
            params.update({"window_size_left": window_size[0], "window_size_right": window_size[1]})
        _flash_attn_backward(**params)
        reduce_dq = grad_accumulate(reduce_dq, block_dq)
        red = grad_accumulate(None, block_dkv)
        if dkv_chunks is not None:
            dkv_chunks[chunk_id] = red
        if chunk_id == own:
            dkv[...] = red.to(dkv.dtype)
    if not write_dq:
        dq[...] = reduce_dq.to(dq.dtype)
    if carried:
        N.host.written(dq, dkv)
