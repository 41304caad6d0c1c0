"""The compiled host module against the Python functions it stands in for: same results bit for bit where it takes a
call, the Python function's own handling or error where it does not, the registered operator wherever a mode, a
transform or autograd is at work."""
import ctypes

import pytest
import torch

import oracle as O
from mercury_artifact_amd import _native as N

pytestmark = pytest.mark.gpu


class _Absent:
    def __getattr__(self, name):
        return lambda *args: None


def _bits(x):
    if isinstance(x, (tuple, list)):
        return [_bits(y) for y in x]
    return x.contiguous().reshape(-1).view(torch.uint8).cpu()


def _same(a, b):
    if isinstance(a, list):
        return len(a) == len(b) and all(_same(x, y) for x, y in zip(a, b))
    return torch.equal(a, b)


def _data(B=2, Sq=70, Sc=90, Hq=4, Hkv=2, D=64):
    g = torch.Generator(device="cuda").manual_seed(3)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    return mk(B, Sq, Hq, D), mk(2, B, Sc, Hkv, D), mk(B, Sq, Hq, D)


def _calls():
    import mercury_artifact_amd as M

    q, kv, dout = _data()
    out, lse = M.attn_fwd_block(q, kv[0], kv[1], 0.1)
    wide = torch.zeros(2, 70, 4, 128, device="cuda", dtype=torch.bfloat16)
    wide[..., :64] = q
    B, S, H, D = q.shape
    acc, accl = torch.randn(B, S, H, D, device="cuda"), torch.randn(B, S, H, 1, device="cuda")
    q8, sc = M.quantize_e4m3(torch.randn(B, S, H, D, device="cuda"))

    def given():
        o, l = torch.empty_like(q), torch.empty(B, H, S, device="cuda")
        assert M.attn_fwd_block(q, kv[0], kv[1], 0.1, True, out=o, lse=l)[0] is o
        return o, l

    def backward(acc_too):
        dq, dkv = torch.empty_like(q), torch.empty_like(kv)
        dq_acc = torch.full(q.shape, 0.5, device="cuda") if acc_too else None
        d = M.attn_bwd_block(dout, q, kv[0], kv[1], out, lse, dq, dkv[0], dkv[1], 0.1, dq_acc=dq_acc)
        return [d, dq, dkv] + ([dq_acc] if acc_too else [])

    def fold(begins):
        o, l = torch.empty_like(q), torch.empty(B, H, S, device="cuda")
        sl = [0, 0] if begins is None else begins
        M.merge_many([out[:, b:].contiguous() for b in sl], [lse[:, :, b:].contiguous() for b in sl], o, l, begins)
        return o, l

    def merged(first, final):
        d = (None, None) if final else (torch.empty_like(acc), torch.empty_like(accl))
        f = (torch.empty_like(q), torch.empty(B, H, S, device="cuda")) if final else (None, None)
        M.merge_into(*((None, None) if first else (acc, accl)), out, lse, *d, *f)
        return [t for t in (*d, *f) if t is not None]

    return {
        "forward": lambda: M.attn_fwd_block(q, kv[0], kv[1], 0.1),
        "forward of a view, descale a Python number": lambda: M.attn_fwd_block(wide[..., :64], kv[0], kv[1], 0.1, q_descale=1.0),
        "forward into given tensors": given,
        "forward e4m3": lambda: M.attn_fwd_block(q8, q8, q8, 0.1, q_descale=sc, k_descale=sc, v_descale=sc),
        "operator": lambda: M._flash_attn_forward(q, kv[0], kv[1], 0.0, 0.1, True, -1, -1, 0.0, None, False)[:2],
        "backward": lambda: backward(False),
        "backward with accumulator": lambda: backward(True),
        "fold": lambda: fold(None),
        "fold of tails": lambda: fold([0, 33]),
        "first merge": lambda: merged(True, False),
        "merge": lambda: merged(False, False),
        "last merge": lambda: merged(False, True),
        "pack": lambda: M.pack_block(out, lse),
        "pack and reduce": lambda: M.pack_block(out, lse, torch.cat([acc, accl], -1)),
        "quantise": lambda: M.quantize_e4m3(acc),
        "quantise a view": lambda: M.quantize_e4m3(acc[:, :, 1:3]),
    }


def test_host_module_gives_the_python_functions_results(monkeypatch):
    calls = _calls()
    for name, call in calls.items():
        print(name, flush=True)
        fast = _bits(call())
        with monkeypatch.context() as m:
            m.setattr(N, "host", _Absent())
            slow = _bits(call())
        assert _same(fast, slow), name


def test_what_the_host_module_declines_is_reported_as_before():
    import mercury_artifact_amd as M

    q, kv, _ = _data()
    with pytest.raises(RuntimeError, match="GPU only"):
        M.attn_fwd_block(q.cpu(), kv[0], kv[1], 0.1)
    with pytest.raises(RuntimeError, match="dtype"):
        M.attn_fwd_block(q.half(), kv[0].half(), kv[1].half(), 0.1)
    with pytest.raises(RuntimeError, match="shape mismatch"):
        M.attn_fwd_block(q, kv[0][:, :3], kv[1], 0.1)
    with pytest.raises(RuntimeError, match="softmax scale"):
        M.attn_fwd_block(q, kv[0], kv[1], -1.0)
    with pytest.raises(RuntimeError, match="dropout"):
        M._flash_attn_forward(q, kv[0], kv[1], 0.5, 0.1, False, -1, -1, 0.0, None, False)
    with pytest.raises(RuntimeError):
        M._flash_attn_forward(q, kv[0])
    with pytest.raises(RuntimeError, match="final_out"):
        M.merge_many([q], [torch.zeros(2, 4, 70, device="cuda")], q.float(), torch.zeros(2, 4, 70, device="cuda"))


def test_the_operator_goes_through_the_dispatcher_where_something_watches():
    import mercury_artifact_amd as M
    from torch.utils._python_dispatch import TorchDispatchMode

    q, kv, _ = _data()
    args = (q, kv[0], kv[1], 0.0, 0.1, False, -1, -1, 0.0, None, False)
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), kw=None):
            seen.append(str(func))
            return func(*a, **(kw or {}))

    with Watch():
        M._flash_attn_forward(*args)
    assert any("mercury_amd._flash_attn_forward" in s for s in seen)
    out = M._flash_attn_forward(q.detach().requires_grad_(), *args[1:])[0]
    with torch.no_grad():
        plain = M._flash_attn_forward(q.detach().requires_grad_(), *args[1:])[0]
    assert torch.equal(out, plain) and not plain.requires_grad
    assert torch.ops.mercury_amd._flash_attn_forward(*args)[0].equal(plain)


def test_gradients_count_as_written():
    """The operator says that it writes dq, dk and dv; so does a call that goes past the dispatcher, and the driver."""
    import mercury_artifact_amd as M

    q, kv, dout = _data()
    out, lse = M.attn_fwd_block(q, kv[0], kv[1], 0.1)
    for mode in (torch.no_grad, torch.inference_mode):
        dq, dkv = torch.empty_like(q), torch.empty_like(kv)
        before = dq._version, dkv._version
        with mode():
            M._flash_attn_backward(dout, q, kv[0], kv[1], out, lse, dq, dkv[0], dkv[1], 0.0, 0.1, False, -1, -1, 0.0, None, False)
        assert dq._version > before[0] and dkv._version > before[1]
        before = dq._version, dkv._version
        with mode():
            M.flash_attn_backward(q, kv, out, lse, dout, dq, dkv, 0.1, ring=M.LocalRing((1,), 0, [kv]))
            inside = torch.empty_like(q)                 # an inference tensor keeps no count
            M._flash_attn_backward(dout, q, kv[0], kv[1], out, lse, inside, dkv[0], dkv[1], 0.0, 0.1, False, -1, -1, 0.0,
                                   None, False)
        assert dq._version > before[0] and dkv._version > before[1]


def _on_device(t, index):
    """``t``'s memory as a tensor that says it is on another GPU: nothing may touch it, so there need not be one."""
    class Head(ctypes.Structure):
        _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int), ("device_id", ctypes.c_int)]

    pointer = ctypes.pythonapi.PyCapsule_GetPointer
    pointer.restype, pointer.argtypes = ctypes.c_void_p, [ctypes.py_object, ctypes.c_char_p]
    capsule = torch.utils.dlpack.to_dlpack(t)
    Head.from_address(pointer(capsule, b"dltensor")).device_id = index
    return torch.utils.dlpack.from_dlpack(capsule)


def test_tensors_of_another_device_are_left_to_the_python_function():
    """The Python functions make the tensors' device current for the call; the host module declines."""
    q, kv, dout = (_on_device(t, 1) for t in _data(Sq=64, Sc=64, Hq=2))
    N.lib()
    assert q.device.index == 1 and torch.cuda.current_device() == 0
    k, v = kv.unbind(0)
    B, S, H, D = q.shape
    f32 = lambda *shape: _on_device(torch.zeros(shape, device="cuda"), 1)
    lse, acc, accl, packed = f32(B, H, S), f32(B, S, H, D), f32(B, S, H, 1), f32(B, S, H, D + 1)
    assert N.host.fwd_block(q, k, v, 0.1, False, None, None, None, None, None) is None
    assert N.host.bwd_block(dout, q, k, v, q, lse, dout, k, v, 0.1, False, False, None) is None
    assert N.host.bwd_chunk(dout, q, k, v, q, lse, dout, None, True, True, kv, None, 0.1, None) is None
    assert N.host.merge_into(None, None, q, lse, acc, accl, None, None) is None
    assert N.host.merge_many([q], [lse], dout, lse, None) is None
    assert N.host.pack_block(q, lse, None) is None
    assert N.host.unpack_into(packed, q, lse) is None
    assert N.host.quantize_e4m3(acc) is None


@pytest.mark.parametrize("code,error", [(-5, "kernel launch failed"), (-8, "runtime query failed"), (1, "unknown")])
def test_a_failed_launch_is_reported_once_and_not_repeated(code, error):
    """A launch that reports an error may have run all the same: a second one would add its dq to dq_acc again."""
    import mercury_artifact_amd as M

    q, kv, dout = _data()
    out, lse = M.attn_fwd_block(q, kv[0], kv[1], 0.1)
    table = {name: ctypes.cast(getattr(N.lib(), name), ctypes.c_void_p).value for name in N.EXPORTED_SYMBOLS}
    calls, stubs = [], {}
    for name in ("mhip_attn_fwd_block", "mhip_attn_bwd_block", "mhip_lse_merge_many"):
        stub = ctypes.CFUNCTYPE(*([N._SIGNATURES[name][0]] + N._SIGNATURES[name][1]))(lambda *a: calls.append(len(a)) or code)
        stubs[name] = (stub, ctypes.cast(stub, ctypes.c_void_p).value)
    dq, dkv, acc = torch.empty_like(q), torch.empty_like(kv), torch.zeros(q.shape, device="cuda")
    try:
        assert N.host.bind({**table, **{name: address for name, (_, address) in stubs.items()}})
        for name, call in (
                ("mhip_attn_fwd_block", lambda: M.attn_fwd_block(q, kv[0], kv[1], 0.1)),
                ("mhip_attn_fwd_block", lambda: M._flash_attn_forward(q, kv[0], kv[1], 0.0, 0.1, False, -1, -1, 0.0, None, False)),
                ("mhip_attn_bwd_block", lambda: M.attn_bwd_block(dout, q, kv[0], kv[1], out, lse, dq, dkv[0], dkv[1], 0.1, dq_acc=acc)),
                ("mhip_lse_merge_many", lambda: M.merge_many([out], [lse], torch.empty_like(q), torch.empty_like(lse)))):
            with pytest.raises(RuntimeError, match=f"{name}: .*{error}"):
                call()
    finally:
        assert N.host.bind(table)
    assert len(calls) == 4
    assert not acc.any()


def test_a_profiler_sees_the_operators():
    """The dispatcher is where a profiler hears of an operator: under one, plain calls and the drivers' blocks go there."""
    import mercury_artifact_amd as M
    from torch.profiler import ProfilerActivity, profile

    q, kv, dout = _data()
    fwd = lambda: M._flash_attn_forward(q, kv[0], kv[1], 0.0, 0.1, False, -1, -1, 0.0, None, False)
    out, lse = fwd()[:2]
    dq, dkv = torch.empty_like(q), torch.empty_like(kv)
    o, l = torch.empty_like(out), torch.empty_like(lse)
    with profile(activities=[ProfilerActivity.CPU]) as seen:
        again = fwd()
        M._flash_attn_backward(dout, q, kv[0], kv[1], out, lse, dq, dkv[0], dkv[1], 0.0, 0.1, False, -1, -1, 0.0, None, False)
        M.gqa_pack_kv(q, kv, o, l, 0.1, ring=M.LocalRing((3,), 0, [kv] * 3))
    counts = {e.key: e.count for e in seen.key_averages()}
    assert counts.get("mercury_amd::_flash_attn_forward") == 4 and counts.get("mercury_amd::_flash_attn_backward") == 1
    assert torch.equal(again[0], out) and torch.equal(again[1], lse)


def test_other_threads_run_while_a_launch_blocks():
    """A launch blocks while the queue is full.  poll(2) stands in for one here: called with the quantiser's arguments --
    (x, MHIP_BF16 = 0 descriptors, the number of elements as milliseconds, ...) -- it waits and touches nothing."""
    import threading
    import time

    x = torch.zeros(400, device="cuda", dtype=torch.bfloat16)
    table = {name: ctypes.cast(getattr(N.lib(), name), ctypes.c_void_p).value for name in N.EXPORTED_SYMBOLS}
    poll = ctypes.cast(ctypes.CDLL(None).poll, ctypes.c_void_p).value
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.wait(0.005):
            ticks.append(time.monotonic())

    thread = threading.Thread(target=tick)
    try:
        assert N.host.bind({**table, "mhip_quantize_e4m3": poll})
        thread.start()
        begin = time.monotonic()
        assert N.host.quantize_e4m3(x) is not None
        end = time.monotonic()
    finally:
        stop.set()
        assert N.host.bind(table)
    thread.join()
    assert end - begin >= 0.39
    assert sum(begin + 0.05 < t < end - 0.05 for t in ticks) >= 5


def test_named_tensors_are_refused_by_the_operator():
    import warnings

    import mercury_artifact_amd as M

    q, kv, _ = _data()
    M.attn_fwd_block(q, kv[0], kv[1], 0.1)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        named = q.refine_names("b", "s", "h", "d")
    with pytest.raises(RuntimeError, match="[Nn]amed"):
        M._flash_attn_forward(named, kv[0], kv[1], 0.0, 0.1, False, -1, -1, 0.0, None, False)
