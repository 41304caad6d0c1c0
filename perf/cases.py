"""What is measured: one rank's share of the attention steps this package exists for.

Every case is one rank's work between two exchanges of a sequence-parallel attention: block forwards or backwards
over the K/V chunks that visit the rank, with the merges that belong to them, called the way a program calls the
package -- through the ring drivers, through the names ``namespace()`` hands to generated code, or through the two
block operators.  ``LocalRing`` replays the neighbour exchange on the one GPU, so every kernel sees its real
per-rank shape.

Parameters of a case: ``path`` (which entry point), ``B`` batch, ``Sq`` local query rows, ``Sc`` rows of one K/V
chunk, ``Hq`` / ``Hkv`` heads, ``D`` head dimension, ``inner`` x ``outer`` mesh (their product is the number of
chunks), ``rank``, and options of a path: ``divide`` (sub-chunk loop), ``lazy`` (which merge generated code is
bound to), ``causal``.
"""
from __future__ import annotations

import math

import torch

import mercury_artifact_amd as M

DEVICE = "cuda:0"


def _case(path, B, Sq, Sc, Hq, Hkv, D, inner=1, outer=1, rank=0, divide=1, lazy=True, causal=False, **more):
    return dict(path=path, B=B, Sq=Sq, Sc=Sc, Hq=Hq, Hkv=Hkv, D=D, inner=inner, outer=outer, rank=rank,
                divide=divide, lazy=lazy, causal=causal, **more)


def listed():
    return [
        # The smallest ring of the test configurations: 4 heads of 64, 1024 tokens over 4 ranks.  A debugging or
        # unit-scale model; a step is four blocks of a few microseconds each, so launches and host work are what counts.
        _case("ring", 1, 256, 256, 4, 4, 64, 4, name="ring_small_d64"),
        # B4 S4096 H5 on 8 ranks: the shape of the ring tests, an ordinary short-sequence batch with an odd head count
        # that leaves most of the chip without a workgroup of 256 rows.
        _case("ring", 4, 512, 512, 5, 5, 128, 8, rank=3, name="ring_b4_h5"),
        # S8192 H32 on a 4 x 2 double ring, the double-ring benchmark's shape: mid-size blocks of 1024 x 1024.
        _case("ring", 1, 1024, 1024, 32, 32, 128, 4, 2, rank=5, name="double_ring_8k"),
        # The headline: S32768 H32 D128 on 8 ranks, blocks of 4096 x 4096.
        _case("ring", 1, 4096, 4096, 32, 32, 128, 8, name="ring_32k"),
        # The same step with every chunk cut in four (less memory for travelling chunks): 32 blocks of 4096 x 1024.
        _case("ring", 1, 4096, 4096, 32, 32, 128, 8, divide=4, name="ring_32k_divide4"),
        # Unchanged generated code, bound to namespace(): a batch of two uneven sequences (9896 tokens over 8 ranks),
        # grouped heads, a head dimension that is no power of two; rows and keys end inside a tile everywhere.
        _case("dropin", 2, 1237, 1237, 16, 8, 80, 8, rank=2, name="dropin_ragged_gqa"),
        # The managed reduction (packed out | lse buffers) at 2048 local rows.
        _case("packed", 1, 2048, 2048, 32, 32, 128, 8, rank=1, name="packed_reduce_16k"),
        # Causal training of a grouped-head model in the zigzag layout: B2, 32 / 8 heads, 65536 tokens over 8 ranks.
        _case("zigzag", 2, 8192, 8192, 32, 8, 128, 8, rank=3, name="zigzag_gqa_64k"),
        # Backward of the B4 H5 step: all chunk gradients are kept, as they travel on.
        _case("backward", 4, 512, 512, 5, 5, 128, 8, rank=3, name="backward_b4_h5"),
        # Backward of the headline step.
        _case("backward", 1, 4096, 4096, 32, 32, 128, 8, name="backward_32k"),
        # One layer's attention on one device, forward and backward through the block operators: causal, head
        # dimension 64, sequences of 1500 tokens.
        _case("block", 2, 1500, 1500, 12, 12, 64, causal=True, name="block_causal_d64"),
        # The long-context float8 step: S131072 on a 4 x 2 double ring; the rank quantises its own queries and then
        # visits 8 chunks of 16384 keys.  The largest case.
        _case("fp8", 1, 16384, 16384, 32, 32, 128, 4, 2, rank=5, name="fp8_double_ring_128k"),
    ]


# What a drawn case may cost: multiply-adds of the products of one pass (the largest listed case takes about as long
# as each of these at its type's rate) and the bytes of its chunks.
_MOST_FLOPS = {"fp8": 3.0e13, "backward": 6e12, "block": 6e12}
_MOST_CHUNK_BYTES = 2 << 30


def draw(rng):
    while True:
        path = rng.choice(["ring", "ring", "dropin", "packed", "zigzag", "backward", "backward", "block", "fp8"])
        B = rng.choice([1, 1, 1, 2, 2, 4])
        group = rng.choice([1, 1, 2, 4, 8])
        Hkv = rng.choice([1, 2, 3, 4, 5, 8, 8, 16, 32])
        Hq = Hkv * group
        D = rng.choice([64, 128, 128, 128, 16 * rng.randint(2, 8)])
        Sq = int(round(math.exp(rng.uniform(math.log(192), math.log(16384)))))
        size = rng.choice(["any", "round", "round"])
        if size == "round":
            Sq = max(256, Sq // 256 * 256)
        inner, outer = rng.choice([(2, 1), (4, 1), (4, 1), (8, 1), (2, 2), (4, 2)])
        divide, lazy, causal = 1, True, False
        Sc = Sq
        if path == "zigzag":
            outer, Sq = 1, Sq // 2 * 2
            Sc = Sq
        elif path == "block":
            inner = outer = 1
            causal = rng.random() < 0.5
            if not causal:
                Sc = max(64, int(Sq * rng.uniform(0.5, 2)))
        elif path == "ring":
            divide = rng.choice([1, 1, 2, 4])
            if Sc % divide:
                divide = 1
        elif path == "dropin":
            lazy = rng.random() < 0.7
        if Hq > 64:
            continue
        rank = rng.randrange(inner * outer)
        c = _case(path, B, Sq, Sc, Hq, Hkv, D, inner, outer, rank, divide, lazy, causal)
        if work(c)["flops"] <= _MOST_FLOPS.get(path, 1.2e13) and _chunk_bytes(c) <= _MOST_CHUNK_BYTES:
            return c


def _chunk_bytes(c):
    return 2 * c["B"] * c["Sc"] * c["Hkv"] * c["D"] * (1 if c["path"] == "fp8" else 2) * c["inner"] * c["outer"]


def _mesh(c):
    return (c["inner"], c["outer"]) if c["outer"] > 1 else (c["inner"],)


def _attention(q, chunks, scale):
    """Output (bf16) and log-sum-exp of attention over all chunks, in fp32 one head at a time: what the forward
    of a training step leaves for its backward."""
    B, Sq, Hq, D = q.shape
    group = Hq // chunks[0].shape[3]
    out = torch.empty_like(q)
    lse = torch.empty(B, Hq, Sq, dtype=torch.float32, device=q.device)
    for b in range(B):
        for h in range(Hq):
            k = torch.cat([c[0, b, :, h // group] for c in chunks]).float()
            v = torch.cat([c[1, b, :, h // group] for c in chunks]).float()
            s = (q[b, :, h].float() * scale) @ k.t().contiguous()
            lse[b, h] = torch.logsumexp(s, -1)
            out[b, :, h] = s.sub_(lse[b, h][:, None]).exp_() @ v
    return out, lse


def prepare(case, seed):
    c = dict(case)
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    B, Sq, Sc, Hq, Hkv, D = (c[k] for k in ("B", "Sq", "Sc", "Hq", "Hkv", "D"))
    W = c["inner"] * c["outer"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEVICE)

    s = {"case": c, "scale": D ** -0.5}
    if c["path"] == "fp8":
        # queries arrive in bf16 from the projection; the chunks come over the ring quantised, with one scale for
        # all keys and one for all values
        s["q"] = normal(B, Sq, Hq, D).bfloat16()
        s["k_scale"] = s["v_scale"] = torch.tensor(5.5 / 448.0, device=DEVICE)
        s["chunks"] = []
        for _ in range(W):
            x = normal(2, B, Sc, Hkv, D).div_(s["k_scale"]).clamp_(-448, 448)
            s["chunks"].append(x.to(torch.float8_e4m3fn))
            del x
    else:
        s["q"] = normal(B, Sq, Hq, D).bfloat16()
        s["chunks"] = [normal(2, B, Sc, Hkv, D).bfloat16() for _ in range(W)]
    if c["path"] in ("backward", "block"):
        s["dout"] = normal(B, Sq, Hq, D).bfloat16()
    if c["path"] == "backward":
        s["out"], s["lse"] = _attention(s["q"], s["chunks"], s["scale"])
        s["dq"] = torch.empty_like(s["q"])
        s["dkv"] = torch.empty_like(s["chunks"][c["rank"]])
    elif c["path"] != "block":
        s["out"] = torch.empty(B, Sq, Hq, D, dtype=torch.bfloat16, device=DEVICE)
        s["lse"] = torch.empty(B, Hq, Sq, dtype=torch.float32, device=DEVICE)
    if c["path"] == "dropin":
        s["names"] = M.namespace(lazy_merge=c["lazy"])
    return s


def _ring(s):
    c = s["case"]
    return M.LocalRing(_mesh(c), c["rank"], s["chunks"])


def _run_ring(s):
    c, mine = s["case"], s["chunks"][s["case"]["rank"]]
    step = M.flash_attn_pack_split_kv if c["outer"] > 1 else M.gqa_pack_kv if c["Hq"] != c["Hkv"] else M.flash_attn_pack_kv
    step(s["q"], mine, s["out"], s["lse"], s["scale"], ring=_ring(s), ring_divide=c["divide"])
    return s["out"], s["lse"]


def _forward_params(ns, q, k, v, scale, causal):
    params = ns["get_default_args"](ns["_flash_attn_forward"]).copy()
    params.update({"q": q, "k": k, "v": v, "dropout_p": 0, "softmax_scale": scale, "causal": causal,
                   "alibi_slopes": None, "return_softmax": False, "window_size_left": -1, "window_size_right": -1})
    return params


def _run_dropin(s):
    """The statements of a generated ring step, its names taken from ``namespace()``."""
    ns, c = s["names"], s["case"]
    out = lse = kv = next_kv = None
    comm = _ring(s)
    mesh = _mesh(c)
    at = ns["one_dim_to_n_dim"](c["rank"], mesh)
    inner, outer = c["inner"], c["outer"]
    for o in range(outer):
        for i in range(inner):
            if o == 0 and i == 0:
                kv = s["chunks"][c["rank"]].contiguous()
            else:
                comm.wait()
                kv = next_kv
            dim = 0 if i + 1 != inner else 1 if o + 1 != outer else None
            if dim is not None:
                to = ns["n_dim_to_one_dim"](ns["shift_tuple_element"](at, dim, 1, mesh[dim]), mesh)
                source = ns["n_dim_to_one_dim"](ns["shift_tuple_element"](at, dim, -1, mesh[dim]), mesh)
                next_kv = comm.send_recv(to, source, kv)
                comm.commit()
            outputs = ns["_flash_attn_forward"](**_forward_params(ns, s["q"], kv[0], kv[1], s["scale"], c["causal"]))
            block_out, block_lse, _, _ = outputs
            out, lse = ns["update_out_and_lse"](out, lse, block_out, block_lse)
    s["out"][:, :, :, :] = out.to(s["q"].dtype)
    s["lse"][:, :, :] = lse.squeeze(dim=-1).transpose(1, 2)
    return s["out"], s["lse"]


def _run_packed(s):
    M.flash_attn_expose_reduce(s["q"], s["chunks"][s["case"]["rank"]], s["out"], s["lse"], s["scale"], ring=_ring(s))
    return s["out"], s["lse"]


def _run_zigzag(s):
    M.zigzag_causal_pack_kv(s["q"], s["chunks"][s["case"]["rank"]], s["out"], s["lse"], s["scale"], ring=_ring(s))
    return s["out"], s["lse"]


def _run_backward(s):
    gradients = {}
    M.flash_attn_backward(s["q"], s["chunks"][s["case"]["rank"]], s["out"], s["lse"], s["dout"], s["dq"], s["dkv"],
                          s["scale"], ring=_ring(s), dkv_chunks=gradients)
    return s["dq"], s["dkv"], [gradients[i] for i in sorted(gradients)]


def _run_block(s):
    c, q, kv = s["case"], s["q"], s["chunks"][0]
    names = {"get_default_args": M.get_default_args, "_flash_attn_forward": M._flash_attn_forward}
    out, lse, _, _ = M._flash_attn_forward(**_forward_params(names, q, kv[0], kv[1], s["scale"], c["causal"]))
    dq, dkv = torch.empty_like(q), torch.empty_like(kv)
    params = M.get_default_args(M._flash_attn_backward).copy()
    params.update({"dout": s["dout"], "q": q, "k": kv[0], "v": kv[1], "out": out, "softmax_lse": lse, "dq": dq,
                   "dk": dkv[0], "dv": dkv[1], "dropout_p": 0, "softmax_scale": s["scale"], "causal": c["causal"],
                   "window_size_left": -1, "window_size_right": -1, "alibi_slopes": None, "deterministic": False})
    delta = M._flash_attn_backward(**params)
    return out, lse, dq, dkv, delta


def _run_fp8(s):
    q8, q_scale = M.quantize_e4m3(s["q"])
    M.fp8_pack_split_kv(q8, s["chunks"][s["case"]["rank"]], s["out"], s["lse"], s["scale"], q_scale, s["k_scale"],
                        s["v_scale"], ring=_ring(s))
    return s["out"], s["lse"]


_RUN = {"ring": _run_ring, "dropin": _run_dropin, "packed": _run_packed, "zigzag": _run_zigzag,
        "backward": _run_backward, "block": _run_block, "fp8": _run_fp8}


def run(state):
    return _RUN[state["case"]["path"]](state)


def work(case):
    B, Sq, Sc, Hq, Hkv, D = (case[k] for k in ("B", "Sq", "Sc", "Hq", "Hkv", "D"))
    W = case["inner"] * case["outer"]
    path = case["path"]
    product = 2.0 * B * Hq * Sq * Sc * D                  # one of the matrix products of one block
    q_bytes, lse_bytes = 2 * B * Sq * Hq * D, 4 * B * Hq * Sq
    chunk = 2 * B * Sc * Hkv * D                          # elements of one K/V chunk
    if path == "backward":
        # S, dP, dQ, dK, dV of every block; q, out, dout, lse and the chunks in, dq, dkv and the fp32 gradients of
        # the chunks out
        return {"flops": 5 * product * W, "bytes": 4 * q_bytes + lse_bytes + chunk * (2 * W + 2 + 4 * W)}
    if path == "block":
        visible = 0.5 if case["causal"] else 1.0
        return {"flops": 7 * product * visible, "bytes": 4 * q_bytes + 2 * lse_bytes + 4 * chunk}
    if path == "zigzag":
        return {"flops": product * (1.0 + (W - 1)), "bytes": 2 * q_bytes + lse_bytes + 2 * chunk * W}
    return {"flops": 2 * product * W, "bytes": 2 * q_bytes + lse_bytes + chunk * W * (1 if path == "fp8" else 2)}


def tolerance(case):
    # Against the same step in 64 bits (on a few of the shapes above): bf16 rel 2.1e-3 .. 2.9e-3 on every output,
    # largest difference 0.012 .. 0.016 of the root mean square; 0.02 .. 0.10 under the causal mask, where the first
    # rows see few keys and their gradients cancel.  float8 rounds the probabilities to three mantissa bits: rel 2.6e-2,
    # largest 0.14.  Four times that, the float8 rel kept near what one implementation shows.
    if case["path"] == "fp8":
        return {"rel": 3e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.4 if case["path"] == "block" else 0.08}
