"""CPU-only checks of the host side: the C-ABI library loads and exports every symbol the header
declares, the operators expose the keyword surface the generated code relies on, the product's
schedule helpers agree with the oracle's (which is pinned by simulation), and the operators refuse
to run without a GPU instead of falling back."""
import ctypes
import os
import re

import pytest
import torch

import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    from mercury_artifact_amd import _native

    header = open(os.path.join(ROOT, "include", "mercury_hip.h")).read()
    declared = set(re.findall(r"\b(mhip_[a-z0-9_]+)\s*\(", header))
    assert declared and declared == set(_native.EXPORTED_SYMBOLS)
    handle = ctypes.CDLL(_native.LIB_PATH)
    for name in declared:
        assert hasattr(handle, name), name
    lib = _native.lib()
    assert lib.mhip_version() >= 1
    assert lib.mhip_error_string(0) == b"ok" and b"head dimension" in lib.mhip_error_string(-3)


def test_keyword_surface_of_the_block_operators():
    import mercury_artifact_amd as M

    fwd = M.get_default_args(M._flash_attn_forward)
    for key in ("q", "k", "v", "dropout_p", "softmax_scale", "causal", "window_size_left",
                "window_size_right", "softcap", "alibi_slopes", "return_softmax"):
        assert key in fwd
    assert list(fwd)[:11] == ["q", "k", "v", "dropout_p", "softmax_scale", "causal", "window_size_left",
                              "window_size_right", "softcap", "alibi_slopes", "return_softmax"]
    assert fwd["softcap"] == 0.0 and fwd["q"] is None and fwd["q_descale"] is None
    bwd = M.get_default_args(M._flash_attn_backward)
    for key in ("dout", "q", "k", "v", "out", "softmax_lse", "dq", "dk", "dv", "softmax_scale",
                "dropout_p", "causal", "deterministic", "alibi_slopes", "window_size_left",
                "window_size_right", "softcap", "rng_state"):
        assert key in bwd
    # plain functions work too, and the cached dict must be copied by callers
    def f(a, b=2, softcap=5.0):
        return a
    assert M.get_default_args(f) == {"a": None, "b": 2, "softcap": 0.0}
    ns = M.namespace()
    for name in ("_flash_attn_forward", "_flash_attn_backward", "get_default_args", "update_out_and_lse",
                 "flash_reduce", "one_dim_to_n_dim", "n_dim_to_one_dim", "shift_tuple_element",
                 "get_src_dst_ranks"):
        assert callable(ns[name])


def test_no_cpu_fallback():
    import mercury_artifact_amd as M

    q = torch.randn(1, 8, 1, 128).bfloat16()
    with pytest.raises(RuntimeError):
        M.attn_fwd_block(q, q, q, 0.1)
    with pytest.raises((RuntimeError, NotImplementedError)):
        M._flash_attn_forward(q=q, k=q, v=q, dropout_p=0, softmax_scale=0.1, causal=False,
                              window_size_left=-1, window_size_right=-1, softcap=0.0,
                              alibi_slopes=None, return_softmax=False)
    with pytest.raises(RuntimeError):
        M.update_out_and_lse(None, None, q, torch.zeros(1, 1, 8))
    with pytest.raises(RuntimeError):
        M.flash_reduce(torch.zeros(4, 129), torch.zeros(4, 129))
    with pytest.raises(RuntimeError):
        M.update_out_and_lse(None, None, q, torch.zeros(1, 1, 8), slice_=(slice(None),))


def test_index_helpers():
    import mercury_artifact_amd as M

    for shape in [(8,), (4, 2), (2, 2, 2), (3, 5)]:
        world = 1
        for s in shape:
            world *= s
        seen = set()
        for r in range(world):
            idx = M.one_dim_to_n_dim(r, shape)
            assert idx[0] == r % shape[0]                     # dimension 0 is the fastest digit
            assert M.n_dim_to_one_dim(idx, shape) == r
            seen.add(idx)
        assert len(seen) == world
    assert M.shift_tuple_element((0, 1), 0, -1, 4) == (3, 1)
    assert M.shift_tuple_element((3, 1), 0, 1, 4) == (0, 1)
    # single ring: source is rank-1, destination rank+1
    assert M.get_src_dst_ranks((2,), (8,), [0]) == (1, 3)
    # double ring (4, 2), ring dims [1, 0]: dim 0 shifts by 1, then dim 1 by the size of dim 0 (mod 2 -> 0)
    assert M.get_src_dst_ranks((0, 0), (4, 2), [1, 0]) == (3, 1)


@pytest.mark.parametrize("world", [1, 2, 4, 8])
def test_product_schedules_equal_oracle(world):
    import mercury_artifact_amd as M

    for r in range(world):
        assert M.single_ring_order(r, world) == O.single_ring_order(r, world)
        for step in range(world):
            assert M.zigzag_step(r, step, world) == O.zigzag_step(r, step, world)
        assert M.zigzag_blocks(r, world) == O.zigzag_blocks(r, world)
    assert M.ring_divide_order(world - 1, world, 2) == O.ring_divide_order(world - 1, world, 2)


@pytest.mark.parametrize("inner,outer", [(4, 2), (2, 2), (2, 4), (1, 3), (3, 1)])
def test_product_double_ring_equals_oracle(inner, outer):
    import mercury_artifact_amd as M

    for r in range(inner * outer):
        assert M.double_ring_order(r, inner, outer) == O.double_ring_order(r, inner, outer)


def test_local_ring_protocol_errors():
    import mercury_artifact_amd as M

    chunks = [torch.full((1,), float(i)) for i in range(4)]
    ring = M.LocalRing((4,), 1, chunks)
    with pytest.raises(RuntimeError):
        ring.wait()                                   # wait before commit
    got = ring.send_recv(2, 0, chunks[1])
    assert got.item() == 0.0                          # rank 1 receives rank 0's chunk
    ring.commit()
    with pytest.raises(RuntimeError):
        ring.commit()                                 # commit twice
    ring.wait()
    with pytest.raises(RuntimeError):
        ring.send_recv(3, 0, chunks[1])               # not a +1 / -1 hop
    with pytest.raises(ValueError):
        M.LocalRing((4,), 7)
    with pytest.raises(ValueError):
        M.LocalRing((4,), 0, chunks[:2])


def test_quantize_e4m3_has_no_cpu_path():
    import mercury_artifact_amd as M

    with pytest.raises(RuntimeError):
        M.quantize_e4m3(torch.randn(1000))


@pytest.mark.parametrize("mesh", [(4,), (8,), (4, 2), (2, 3), (2, 2, 2)])
def test_reduce_buffer_route_visits_every_rank_once_and_returns_home(mesh):
    """Follow every ringed reduce buffer by hand: it must be at a different rank at every step (so it
    folds in every KV shard exactly once) and the write-back hop must land it on the rank it started on."""
    import mercury_artifact_amd as M

    sends, home = M.reduce_buffer_route(mesh)
    world = len(home)
    assert len(sends) == world - 1
    for start in range(world):
        at, seen = start, [start]
        for s in range(world - 1):
            at = sends[s][at]
            seen.append(at)
        assert sorted(seen) == list(range(world))
        assert home[at] == start
    for s in range(world - 1):
        assert sorted(sends[s]) == list(range(world))        # a hop is a permutation of the ranks


def test_get_device_group_is_the_reference_grouping():
    """Ranks whose coordinates agree outside `dims` (mercury/backend/pytorch/utils.py:114-169), by brute force over
    the mesh; debug=True gives the rank tuple, otherwise a LocalGroup over the same ranks."""
    import itertools

    import mercury_artifact_amd as M

    for mesh_shape in [(4,), (2, 2), (4, 2), (2, 3, 2)]:
        world = 1
        for m in mesh_shape:
            world *= m
        for k in range(1, len(mesh_shape) + 1):
            for dims in itertools.combinations(range(len(mesh_shape)), k):
                for rank in range(world):
                    idx = M.one_dim_to_n_dim(rank, mesh_shape)
                    want = tuple(r for r in range(world)
                                 if all(M.one_dim_to_n_dim(r, mesh_shape)[d] == idx[d]
                                        for d in range(len(mesh_shape)) if d not in dims))
                    assert M.get_device_group(idx, mesh_shape, dims, debug=True) == want
                    group = M.get_device_group(idx, mesh_shape, dims)
                    assert group.ranks == want and group.ranks[group.rank] == rank and group.size() == len(want)
    with pytest.raises(ValueError):
        M.get_device_group((0, 0), (2, 2), (2,))
    # on one GPU the other ranks' operands have to come from somewhere
    group = M.get_device_group((1,), (4,), (0,))
    with pytest.raises(RuntimeError):
        group.operands(torch.zeros(1))
    with M.local_peers(lambda r: torch.full((1,), float(r))):
        assert [t.item() for t in group.operands(torch.full((1,), -1.0))] == [0.0, -1.0, 2.0, 3.0]


def test_debug_print_prefixes_the_rank(capsys):
    import mercury_artifact_amd as M

    M.namespace()["debug_print"]("x", 3)
    assert capsys.readouterr().out == "[Rank 0] x 3\n"


def test_local_mesh_replays_the_ring_protocol_of_all_ranks():
    """Every rank as a thread: what arrives hop by hop is the chunk order of LocalRing / the oracle; SendRecv misuse
    raises as in the reference; a rank waiting for a message nobody sends raises instead of hanging."""
    import mercury_artifact_amd as M
    import oracle as O

    inner, outer = 4, 2
    mesh = M.LocalMesh((inner, outer))

    def rank_fn(r):
        indices = M.one_dim_to_n_dim(mesh.dist.get_rank(), (inner, outer))
        seen = []
        for o in range(outer):
            for i in range(inner):
                if i == 0 and o == 0:
                    cur = torch.tensor([float(r)])
                    comm = mesh.SendRecv()
                else:
                    comm.wait()
                    cur = nxt
                seen.append(int(cur.item()))
                if i + 1 != inner:
                    to = M.n_dim_to_one_dim(M.shift_tuple_element(indices, 0, 1, inner), (inner, outer))
                    frm = M.n_dim_to_one_dim(M.shift_tuple_element(indices, 0, -1, inner), (inner, outer))
                    nxt = comm.send_recv(to, frm, cur)
                    comm.commit()
                elif o + 1 != outer:
                    to = M.n_dim_to_one_dim(M.shift_tuple_element(indices, 1, 1, outer), (inner, outer))
                    frm = M.n_dim_to_one_dim(M.shift_tuple_element(indices, 1, -1, outer), (inner, outer))
                    nxt = comm.send_recv(to, frm, cur)
                    comm.commit()
        return seen

    orders = mesh.run(rank_fn)
    for r in range(inner * outer):
        assert orders[r] == O.double_ring_order(r, inner, outer) == M.double_ring_order(r, inner, outer)

    small = M.LocalMesh((2,), timeout=0.5)

    def misuse(r):
        comm = small.SendRecv()
        with pytest.raises(RuntimeError, match="wait called before commit"):
            comm.wait()
        comm.send_recv(1 - r, 1 - r, torch.zeros(1))
        comm.commit()
        with pytest.raises(RuntimeError, match="commit called twice"):
            comm.commit()
        comm.wait()
        return small.dist.get_world_size()

    assert small.run(misuse) == [2, 2]

    def starved(r):
        comm = small.SendRecv()
        if r == 0:
            comm.send_recv(1, 1, torch.zeros(1))
            comm.commit()
            comm.wait()

    with pytest.raises(RuntimeError, match="waited"):
        small.run(starved)


def test_local_mesh_reports_the_first_failure_and_releases_the_waiting_ranks():
    """A rank that raises ends the whole run at once: the ranks waiting for its messages stop waiting (they do not sit
    out the time limit), and what run() raises is that rank's own exception, whichever rank index it had."""
    import time

    import mercury_artifact_amd as M

    mesh = M.LocalMesh((4,), timeout=30.0)

    def rank_fn(r):
        comm = mesh.SendRecv()
        if r == 3:
            time.sleep(0.2)                      # the others are waiting by now
            raise ValueError("rank 3 broke")
        comm.send_recv((r + 1) % 4, (r - 1) % 4, torch.zeros(1))
        comm.commit()
        comm.wait()                              # rank 0 waits for rank 3, which never sends
        return r

    begin = time.monotonic()
    with pytest.raises(ValueError, match="rank 3 broke"):
        mesh.run(rank_fn)
    assert time.monotonic() - begin < 5.0
    # the mesh is usable again afterwards: the messages of the failed run are gone, the barrier works
    def again(r):
        comm = mesh.SendRecv()
        got = comm.send_recv((r + 1) % 4, (r - 1) % 4, torch.full((1,), float(r + 10)))
        comm.commit()
        comm.wait()
        mesh.dist.barrier()
        return int(got.item())

    assert mesh.run(again) == [13, 10, 11, 12]


def test_host_module_built_after_the_import_is_found(monkeypatch):
    """A build from the package itself imports it first, without a host module: lib() looks again."""
    from mercury_artifact_amd import _native as N

    monkeypatch.setattr(N, "host", N._NoHost("not built"))
    monkeypatch.setattr(N, "_lib", None)
    N.lib()
    assert not isinstance(N.host, N._NoHost)
    # a module that is not there is reported, not passed over
    monkeypatch.setattr(N, "host", N._NoHost("not built"))
    monkeypatch.setattr(N, "_lib", None)
    monkeypatch.setattr(N, "_load_host", lambda: N._NoHost("not built"))
    with pytest.raises(RuntimeError, match="_mercury_host"):
        N.lib()


def test_host_module_of_another_abi_is_refused(monkeypatch):
    """Every entry point is there by name, but the module was compiled against another argument list."""
    from mercury_artifact_amd import _native as N

    bound = []

    class Stale:
        def bind(self, table):
            bound.append(table)
            return True

    for version in (N.ABI_VERSION - 1, N.ABI_VERSION + 1, None):
        stale = Stale()
        if version is not None:                    # a module from before there was a version has none
            stale.abi_version = version
        monkeypatch.setattr(N, "host", stale)
        monkeypatch.setattr(N, "_lib", None)
        with pytest.raises(RuntimeError, match=f"stale.*{version}"):
            N.lib()
    assert not bound
    monkeypatch.undo()
    assert N.host.abi_version == N.ABI_VERSION == N.lib().mhip_abi_version()


_NOT_THE_SCHEMAS = [("dropout_p", None), ("dropout_p", 0j), ("softmax_scale", "0.1"), ("softmax_scale", None), ("causal", "x"),
                    ("causal", []), ("window_size_left", None), ("window_size_right", -1.0), ("softcap", None)]


@pytest.mark.parametrize("name,value", _NOT_THE_SCHEMAS + [("return_softmax", "a"), ("q_descale", 1.0), ("alibi_slopes", 1)])
def test_forward_operator_refuses_what_its_schema_refuses(monkeypatch, name, value):
    _refuses(monkeypatch, "_flash_attn_forward", {"return_softmax": False, "alibi_slopes": None}, name, value)


@pytest.mark.parametrize("name,value", _NOT_THE_SCHEMAS + [("deterministic", "a"), ("rng_state", 1), ("alibi_slopes", 1)])
def test_backward_operator_refuses_what_its_schema_refuses(monkeypatch, name, value):
    t = torch.zeros(1, 2, 1, 8, dtype=torch.bfloat16)
    more = {k: t for k in ("dout", "out", "softmax_lse", "dq", "dk", "dv")}
    _refuses(monkeypatch, "_flash_attn_backward", {**more, "deterministic": False, "alibi_slopes": None}, name, value)


def _refuses(monkeypatch, op, more, name, value):
    """Also where the call would go past the dispatcher, which is where the schema is checked."""
    import mercury_artifact_amd.flash_attn_interface as I

    taken = []

    class Eager:
        undispatched = staticmethod(lambda *ts: all(t is None or isinstance(t, torch.Tensor) for t in ts))
        no_dropout = staticmethod(lambda q: (q, q))
        written = staticmethod(lambda *ts: None)

    monkeypatch.setattr(I.N, "host", Eager())
    monkeypatch.setattr(I, "attn_fwd_block", lambda *a: taken.append("f") or a[:2])
    monkeypatch.setattr(I, "attn_bwd_block", lambda *a: taken.append("b") or a[0])
    t = torch.zeros(1, 2, 1, 8, dtype=torch.bfloat16)
    args = {"q": t, "k": t, "v": t, "dropout_p": 0, "softmax_scale": 0.1, "causal": False, "window_size_left": -1,
            "window_size_right": -1, "softcap": 0.0, **more}
    getattr(I, op)(**args)
    assert len(taken) == 1                                   # as it should be, it needs no dispatcher
    with pytest.raises(RuntimeError, match="Expected a value of type"):
        getattr(I, op)(**{**args, name: value})
    assert len(taken) == 1


@pytest.mark.parametrize("values", [{"dropout_p": None}, {"softmax_scale": "0.1"}, {"causal": "x"}, {"window_size": (None, -1)},
                                    {"window_size": (-1, -1.0)}])
def test_drivers_leave_odd_arguments_to_the_operator(monkeypatch, values):
    import mercury_artifact_amd.ring as R

    class Eager:
        undispatched = staticmethod(lambda *ts: True)

    monkeypatch.setattr(R.N, "host", Eager())
    q = torch.zeros(1, 2, 1, 8, dtype=torch.bfloat16)
    args = {"softmax_scale": 0.1, "dropout_p": 0, "causal": False, "window_size": (-1, -1), "alibi_slopes": None}
    assert R._block_results(2, q, q, **args)[1] is not None
    assert R._block_results(2, q, q, **{**args, **values}) == [None, None]


@pytest.mark.parametrize("dtype,D,row_bytes,taken", [
    (torch.bfloat16, 128, 1 << 20, True), (torch.bfloat16, 128, 1 << 21, False), (torch.bfloat16, 64, (1 << 20) - 16, True),
    (torch.bfloat16, 64, 1 << 20, False), (torch.float8_e4m3fn, 128, 1 << 21, False), (torch.float8_e4m3fn, 96, 1 << 20, False),
    (torch.float8_e4m3fn, 96, 1 << 19, True), (torch.bfloat16, 128, 1032, False)])
def test_own_chunk_out_of_the_kernels_reach_is_copied(dtype, D, row_bytes, taken):
    """1024 rows of one layer of a packed cache: a view whose rows lie further apart than a 32-bit offset reaches (or do
    not start on 16 bytes) becomes a copy, as the driver's own chunk always did once."""
    from mercury_artifact_amd.ring import _as_rows

    row = row_bytes // dtype.itemsize
    chunk = torch.empty_strided((2, 1, 1024, 2, D), (1024 * row, 1024 * row, row, D, 1), dtype=dtype, device="meta")
    got = _as_rows(chunk)
    assert (got is chunk) == taken and (taken or got.is_contiguous())
    assert _as_rows(got) is got


@pytest.mark.parametrize("W", [1, 3])
@pytest.mark.parametrize("dq_over", ["", "q", "dout", "o", "half of q", "last chunk"])
@pytest.mark.parametrize("dkv_over", ["", "kv"])
def test_backward_step_in_place_writes_nothing_a_launch_still_reads(monkeypatch, W, dq_over, dkv_over):
    """Gradients that lie over operands: no launch writes what it (or another workgroup of it) reads, and they are stored
    all the same.  Without an overlap the launches store them directly."""
    import mercury_artifact_amd.ring as R
    from mercury_artifact_amd.schedule import LocalRing

    B, S, H, D = 1, 16, 2, 8
    memory = torch.zeros(2, B, 2 * S, H, D, dtype=torch.bfloat16)
    t = {"q": memory[0, :, :S], "dout": memory[1, :, S:], "o": torch.zeros(B, S, H, D, dtype=torch.bfloat16)}
    chunks = [torch.zeros(2, B, S, H, D, dtype=torch.bfloat16) for _ in range(W)]
    lse = torch.zeros(B, H, S)
    last_chunk = chunks[1 % W]                          # of rank 0's order 0, W - 1, ..., 1
    dq = {"": torch.zeros_like(t["o"]), "half of q": memory[0, :, S // 2: S // 2 + S], "last chunk": last_chunk[0]}.get(dq_over)
    dq = t[dq_over] if dq is None else dq
    dkv = chunks[0] if dkv_over else torch.zeros_like(chunks[0])
    direct = []

    def span(x):
        return x.data_ptr(), x.data_ptr() + x.numel() * x.element_size()          # (contiguous, all of them)

    def launch(dout, q, k, v, out, l, dq, acc, first, last, dkv, dkv32, scale, workspace=None):
        total = 1.0 if first else acc.max().item() + 1.0
        for written in [x for x in (dkv, dkv32, dq if last else None, None if last else acc) if x is not None]:
            for read in (dout, q, k, v, out, l):
                (a, b), (c, d) = span(written), span(read)
                assert b <= c or d <= a
        (dq if last else acc).fill_(total)
        dkv.fill_(7.0)
        direct.append((last, dkv.data_ptr()))
        return torch.empty(1, dtype=torch.uint8)

    monkeypatch.setattr(R, "attn_bwd_chunk", launch)
    R.flash_attn_backward(t["q"], chunks[0], t["o"], lse, t["dout"], dq, dkv, 0.1, ring=LocalRing((W,), 0, chunks))
    assert bool((dq == W).all())
    if not (dq_over == "last chunk" and dkv_over and W == 1):       # (dq over the place dkv is in)
        assert bool((dkv == 7).all())
    assert direct[-1][0] == (dq_over == "") and (direct[0][1] == dkv.data_ptr()) == (dkv_over == "")


@pytest.mark.parametrize("name", ["send_recv", "commit", "wait", "hop"])
@pytest.mark.parametrize("on", ["ring", "class"])
def test_a_wrapper_over_a_hop_sees_every_hop(monkeypatch, name, on):
    """A step that collects its chunks at once calls what is put over a ring's methods, on the ring or on its class, as a
    step that goes hop by hop does; the same chunks and the same places afterwards as with nothing put over them."""
    import mercury_artifact_amd.ring as R
    from mercury_artifact_amd.schedule import LocalRing

    chunks = [torch.full((2, 1, 8, 1, 8), float(i), dtype=torch.bfloat16) for i in range(8)]
    plain = LocalRing((4, 2), 5, chunks)
    want = R._resident_chunks(plain, chunks[5])
    ring, calls = LocalRing((4, 2), 5, chunks), []
    over, real = (ring, getattr(ring, name)) if on == "ring" else (LocalRing, getattr(LocalRing, name))
    monkeypatch.setattr(over, name, lambda *a, **kw: calls.append(1) or real(*a, **kw))
    got = R._resident_chunks(ring, chunks[5])
    assert len(calls) == 7 and ring.held == plain.held
    assert len(got) == 8 and all(a is b for a, b in zip(got[1:], want[1:])) and torch.equal(got[0], want[0])


def test_backward_step_without_the_host_modules_answers(monkeypatch):
    """A host module that declines every question: copies and staged stores, not a wrong call."""
    import mercury_artifact_amd.ring as R
    from mercury_artifact_amd.schedule import LocalRing

    class Declines:
        def __getattr__(self, name):
            return lambda *args: None

    def launch(dout, q, k, v, out, lse, dq, acc, first, last, dkv, dkv32, scale, workspace=None):
        assert type(first) is bool and last is False and acc is not None
        acc.fill_(3.0)
        dkv.fill_(7.0)
        return torch.empty(1, dtype=torch.uint8)

    monkeypatch.setattr(R.N, "host", Declines())
    monkeypatch.setattr(R, "attn_bwd_chunk", launch)
    q, kv = torch.zeros(1, 4, 1, 8, dtype=torch.bfloat16), torch.zeros(2, 1, 4, 1, 8, dtype=torch.bfloat16)
    dq, dkv = torch.zeros_like(q), torch.zeros_like(kv)
    R.flash_attn_backward(q, kv, q, torch.zeros(1, 1, 4), q, dq, dkv, 0.1, ring=LocalRing((1,), 0, [kv]))
    assert bool((dq == 3).all()) and bool((dkv == 7).all())


def test_documents_state_the_abi_version_and_every_entry_point():
    """The integration notes: their stub asserts the header's version, and their table names all the library exports."""
    import os
    import re

    from mercury_artifact_amd import _native as N

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    text = open(os.path.join(root, "INTEGRATION.md")).read()
    header = open(os.path.join(root, "include", "mercury_hip.h")).read()
    assert set(re.findall(r"mhip_abi_version\(\) == (\d+)", text) + re.findall(r"`MHIP_ABI_VERSION` \((\d+)\)", text)) == {str(N.ABI_VERSION)}
    assert re.findall(r"#define MHIP_ABI_VERSION (\d+)", header) == [str(N.ABI_VERSION)]
    assert f"\n * {N.ABI_VERSION}: " in header                      # what the value changed
    assert [name for name in N.EXPORTED_SYMBOLS if f"`{name}`" not in text] == []
