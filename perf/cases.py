"""Performance cases of the device paths, through the C ABI and DeviceModel.

Every case is work that a program using this framework has the GPU do, on
buffers that are already in device memory: the gated delta rule forward and
BPTT (recurrent f32 form and chunked bf16 form), the decode step, the linear
projections with their gradients, the HashMoE block, the output head with its
cross-entropy, and two calls of a whole model (a training step and a decode
step).  Tensors are torch's; the library's calls run on torch's default
stream.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from asca_amd import _lib
from asca_amd.gpu import gpu
from asca_amd.model import DeviceModel

EPS = 1e-6  # RMSNorm epsilon of the model
LR, BETA1, BETA2, ADAM_EPS, WD = 3e-4, 0.9, 0.95, 1e-8, 0.01


def listed():
    return [
        # The smallest delta block: a unit-test-sized model; launches and the latency of the time loop.
        dict(name="delta_b4t128h4d32", kind="delta", B=4, T=128, H=4, dh=32),
        # The headline benchmark of the delta block: one layer of a byte model, forward and BPTT.
        dict(name="delta_b32t512h8d64", kind="delta", B=32, T=512, H=8, dh=64),
        # Wide heads and a ragged length in the recurrent f32 form (few units, a long time loop).
        dict(name="delta_b8t1000h8d128", kind="delta", B=8, T=1000, H=8, dh=128),
        # The chunked form on long bf16 sequences with wide heads, its largest use.
        dict(name="chunk_b8t4096h16d128c64", kind="chunk", B=8, T=4096, H=16, dh=128, C=64),
        # The chunked form at the head width of the training model, with a ragged last chunk.
        dict(name="chunk_b4t1000h8d64c64", kind="chunk", B=4, T=1000, H=8, dh=64, C=64),
        # Serving: one token for 512 concurrent sequences, states read and written once.
        dict(name="decode_n512h16d128", kind="decode", n=512, H=16, dh=128),
        # The fused q, k, v projection of the training model: y, then dx, dW, db.
        dict(name="linear_t16384k512n1536", kind="linear", T=16384, K=512, N=1536),
        # The same for a small batch and sizes that fill no tile.
        dict(name="linear_t1000k320n1000", kind="linear", T=1000, K=320, N=1000),
        # The HashMoE block of the training model (norm, routing, experts), forward and backward.
        dict(name="moe_t16384d512f1024e16", kind="moe", T=16384, d=512, dff=1024, E=16),
        # The output head of the training model: logits, cross-entropy, dW, dh.
        dict(name="head_t16384d512v256", kind="head", T=16384, d=512, V=256),
        # One whole training step of the byte model (143M parameters): forward, BPTT, AdamW.
        dict(name="train_d512l8b16t1024", kind="train", V=256, d=512, H=8, L=8, E=16, dff=1024, B=16, T=1024),
        # One token for 64 sequences through the same model: host ids in, host logits out.
        dict(name="step_d512l8n64", kind="step", V=256, d=512, H=8, L=8, E=16, dff=1024, n=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["delta", "delta", "chunk", "decode", "linear", "linear", "moe", "head", "train", "step"])
    while True:
        if kind == "delta":
            c = dict(B=_log(rng, 1, 32), T=_log(rng, 16, 1024), H=rng.choice([2, 4, 8, 16]),
                     dh=rng.choice([16, 32, 48, 64, 64, 96, 128]))
            ok = c["B"] * c["T"] * c["H"] * c["dh"] <= 32 * 512 * 8 * 64
        elif kind == "chunk":
            c = dict(B=_log(rng, 1, 8), T=_log(rng, 64, 4096), H=rng.choice([2, 4, 8, 16]),
                     dh=rng.choice([32, 64, 64, 128, 128]), C=rng.choice([32, 64, 64]))
            ok = c["B"] * c["T"] * c["H"] * c["dh"] <= 4 * 4096 * 8 * 128
        elif kind == "decode":
            c = dict(n=_log(rng, 1, 512), H=rng.choice([2, 4, 8, 16]), dh=rng.choice([32, 64, 128]))
            ok = True
        elif kind == "linear":
            c = dict(T=_log(rng, 64, 16384), K=_log(rng, 64, 1536), N=_log(rng, 64, 2048))
            ok = c["T"] * c["K"] * c["N"] <= 16384 * 512 * 2048
        elif kind == "moe":
            c = dict(T=_log(rng, 64, 16384), d=rng.choice([64, 128, 256, 384, 512]),
                     dff=rng.choice([128, 200, 256, 512, 1024]), E=rng.choice([4, 8, 16]))
            ok = True
        elif kind == "head":
            c = dict(T=_log(rng, 64, 16384), d=rng.choice([64, 128, 256, 384, 512]), V=_log(rng, 200, 4096))
            ok = c["T"] * c["V"] <= 16384 * 1024
        elif kind == "train":
            d = rng.choice([64, 128, 256, 384])
            c = dict(V=256, d=d, H=d // rng.choice([32, 64]), L=rng.choice([2, 4]), E=rng.choice([4, 8, 16]),
                     dff=2 * d, B=_log(rng, 1, 16), T=_log(rng, 32, 1024))
            ok = True
        else:
            d = rng.choice([64, 128, 256, 512])
            c = dict(V=256, d=d, H=d // rng.choice([32, 64]), L=rng.choice([2, 4, 8]), E=rng.choice([4, 8, 16]),
                     dff=2 * d, n=_log(rng, 1, 256))
            ok = True
        if ok:
            return dict(kind=kind, **c)


# ------------------------------------------------------------------ inputs


def _dev():
    if gpu() is None:
        raise RuntimeError("no GPU backend")
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(seed)


def _normal(g, *shape, scale=1.0, offset=0.0):
    return torch.randn(*shape, generator=g, device=g.device) * scale + offset


def _empty(*shape):
    return torch.empty(*shape, device=_dev())


def _tokens(g, n, V):
    return torch.randint(0, V, (n,), generator=g, device=g.device, dtype=torch.int32)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _ws(name, *args):
    n = C.c_size_t()
    _lib.call(name, *args, C.byref(n))
    return torch.empty(max(n.value, 4), dtype=torch.uint8, device=_dev())


def _unit(x, H, dh):
    """Per-head L2 normalisation: (normalised rows, norms)."""
    x3 = x.view(-1, H, dh)
    n = x3.norm(dim=2).clamp_min(1e-8)
    return (x3 / n[..., None]).reshape(x.shape).contiguous(), n.contiguous()


def _delta_inputs(g, rows, H, dh):
    """q, k normalised per head, v and dO ~ N(0,1), alpha = sigmoid(N(2,1)), beta = sigmoid(N(0,1))."""
    q, qn = _unit(_normal(g, rows, H * dh), H, dh)
    k, kn = _unit(_normal(g, rows, H * dh), H, dh)
    return dict(q=q, k=k, qn=qn, kn=kn, v=_normal(g, rows, H * dh),
                alpha=torch.sigmoid(_normal(g, rows, H, offset=2.0)), beta=torch.sigmoid(_normal(g, rows, H)),
                d_o=_normal(g, rows, H * dh))


def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("delta", "chunk"):
        x = _delta_inputs(g, case["B"] * case["T"], case["H"], case["dh"])
        if kind == "chunk":
            for n in ("q", "k", "v", "d_o"):
                x[n] = x[n].bfloat16()
        return x
    if kind == "decode":
        n, H, dh = case["n"], case["H"], case["dh"]
        gate = _normal(g, n, 2 * H)
        gate[:, :H] += 2.0
        return dict(states=_normal(g, n, H, dh, dh, scale=0.2), qkv=_normal(g, n, 3 * H * dh), gate=gate)
    if kind == "linear":
        T, K, N = case["T"], case["K"], case["N"]
        return dict(x=_normal(g, T, K), w=_normal(g, K, N, scale=K ** -0.5), b=_normal(g, N, scale=0.02),
                    dy=_normal(g, T, N, scale=1e-3))
    if kind == "moe":
        T, d, dff, E = case["T"], case["d"], case["dff"], case["E"]
        return dict(x=_normal(g, T, d), w1=_normal(g, d, E * dff, scale=d ** -0.5),
                    b1=_normal(g, E * dff, scale=0.02), w2=_normal(g, E * dff, d, scale=dff ** -0.5),
                    b2=_normal(g, d, scale=0.02), ids=_tokens(g, T, 256), dout=_normal(g, T, d, scale=1e-3))
    if kind == "head":
        T, d, V = case["T"], case["d"], case["V"]
        return dict(h=_normal(g, T, d), w=_normal(g, d, V, scale=d ** -0.5), tgt=_tokens(g, T, V))
    if kind == "train":
        B, T, V = case["B"], case["T"], case["V"]
        toks = _tokens(g, B * (T + 1), V).view(B, T + 1)
        return dict(ids=toks[:, :T].reshape(-1).contiguous(), tgt=toks[:, 1:].reshape(-1).contiguous(), g=g)
    return dict(ids=_tokens(g, case["n"], case["V"]), g=g)


class _Buffer:
    """A device buffer of the library as torch sees it (no copy)."""

    def __init__(self, ptr, n, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f4", data=(ptr, False), version=2)


def _view(ptr, n, owner):
    return torch.as_tensor(_Buffer(ptr, n, owner), device=_dev())


def _shapes(case):
    V, d, H, E, dff = case["V"], case["d"], case["H"], case["E"], case["dff"]
    s = [(V, d), (d, V)]
    for _ in range(case["L"]):
        s += [(d, 3 * d), (1, 3 * d), (d, 2 * H), (1, 2 * H), (d, d), (1, d), (d, E * dff), (1, E * dff),
              (E * dff, d), (1, d)]
    return s


def _offsets(case):
    """Tensors start at multiples of four floats of the flat buffers."""
    offs, at = [], 0
    for r, c in _shapes(case):
        offs.append(at)
        at += (r * c + 3) // 4 * 4
    return offs, at


def _init_params(case, g):
    """A flat parameter buffer with the model's initialisation: N(0, 1/fan_in) matrices, gate biases -2 and -1,
    other biases zero, embedding N(0, 0.02)."""
    offs, n = _offsets(case)
    flat = torch.zeros(n, device=g.device)
    for i, ((r, c), o) in enumerate(zip(_shapes(case), offs)):
        if r > 1:
            scale = 0.02 if i == 0 else (case["dff"] if (i - 2) % 10 == 8 and i >= 2 else case["d"]) ** -0.5
            flat[o:o + r * c].normal_(generator=g).mul_(scale)
        elif i >= 2 and (i - 2) % 10 == 3:
            flat[o:o + c // 2] = -2.0
            flat[o + c // 2:o + c] = -1.0
    return flat


def _init_states(case, g):
    H = case["H"]
    dh = case["d"] // H
    return _normal(g, case["L"] * case["n"] * H * dh * dh, scale=0.1)


def prepare(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    s = dict(case=dict(case), x=x)
    if kind == "delta":
        B, T, H, dh = (case[n] for n in ("B", "T", "H", "dh"))
        s.update(ws=_ws("asca_delta_ws_bytes", B, T, H, dh), o=_empty(B * T, H * dh),
                 d_qkv=_empty(B * T, 3 * H * dh), d_gate=_empty(B * T, 2 * H))
    elif kind == "chunk":
        B, T, H, dh, Cc = (case[n] for n in ("B", "T", "H", "dh", "C"))
        s.update(ws=_ws("asca_chunk_ws_bytes", B, T, H, dh, Cc))
        for n in ("o", "dq", "dk", "dv"):
            s[n] = _empty(B * T, H * dh)
        for n in ("dalpha", "dbeta"):
            s[n] = _empty(B * T, H)
    elif kind == "decode":
        s.update(o=_empty(case["n"], case["H"] * case["dh"]))
    elif kind == "linear":
        T, K, N = case["T"], case["K"], case["N"]
        s.update(y=_empty(T, N), dx=_empty(T, K), dw=_empty(K, N), db=_empty(N))
    elif kind == "moe":
        T, d, dff, E = case["T"], case["d"], case["dff"], case["E"]
        i32 = dict(dtype=torch.int32, device=_dev())
        s.update(expert=torch.empty(T, **i32), perm=torch.empty(T, **i32), offsets=torch.empty(E + 1, **i32),
                 rws=_ws("asca_hash_route_ws_bytes", T, E), xn=_empty(T, d), inv=_empty(T), out=_empty(T, d),
                 pre=_empty(T, dff), hidden=_empty(T, dff), dpre=_empty(T, dff), dxn=_empty(T, d), dx=_empty(T, d),
                 dw1=_empty(d, E * dff), db1=_empty(E * dff), dw2=_empty(E * dff, d), db2=_empty(d))
    elif kind == "head":
        T, d, V = case["T"], case["d"], case["V"]
        s.update(logits=_empty(T, V), dlogits=_empty(T, V), losses=_empty(T), dw=_empty(d, V), dh=_empty(T, d))
    else:
        m = DeviceModel(*(case[n] for n in ("V", "d", "H", "L", "E", "dff")))
        n = _offsets(case)[1]
        if n != m.n_floats:
            raise RuntimeError("the model's layout is not the documented one")
        _view(m._ptr["params"], n, m).copy_(_init_params(case, x["g"]))
        s["model"] = m
        if kind == "train":
            m.set_adamw(LR, BETA1, BETA2, ADAM_EPS, WD)
            ids, tgt = m.upload_batch(x["ids"].cpu().numpy().view("u4"), x["tgt"].cpu().numpy().view("u4"))
            s.update(ids=ids, tgt=tgt, grads=_view(m._ptr["grads"], n, m), params=_view(m._ptr["params"], n, m),
                     loss=_view(m._loss_buf().ptr, 1, m))
        else:
            st = m.new_decode_state(case["n"])
            view = _view(st.ptr, case["n"] * m.decode_state_floats(), st)
            view.copy_(_init_states(case, x["g"]))
            s.update(ids=x["ids"].cpu().numpy().view("u4"), st=st, states=view)
    return s


# --------------------------------------------------------------------- run


def _run_delta(s):
    c, x = s["case"], s["x"]
    dims = (c["B"], c["T"], c["H"], c["dh"], None)
    q, k, v, a, b = (_ptr(x[n]) for n in ("q", "k", "v", "alpha", "beta"))
    ws = _ptr(s["ws"])
    _lib.call("asca_delta_fwd", q, k, v, a, b, _ptr(s["o"]), ws, *dims)
    _lib.call("asca_delta_bwd_fused", q, k, v, a, b, _ptr(x["qn"]), _ptr(x["kn"]), _ptr(x["d_o"]), ws,
              _ptr(s["d_qkv"]), _ptr(s["d_gate"]), *dims)
    return {n: s[n] for n in ("o", "d_qkv", "d_gate")}


def _run_chunk(s):
    c, x = s["case"], s["x"]
    dims = (c["B"], c["T"], c["H"], c["dh"], c["C"], None)
    q, k, v, ws = _ptr(x["q"]), _ptr(x["k"]), _ptr(x["v"]), _ptr(s["ws"])
    outs = ("dq", "dk", "dv", "dalpha", "dbeta")
    _lib.call("asca_chunk_fwd", q, k, v, _ptr(x["alpha"]), _ptr(x["beta"]), _ptr(s["o"]), ws, *dims)
    _lib.call("asca_chunk_bwd", q, k, v, _ptr(x["d_o"]), ws, *(_ptr(s[n]) for n in outs), *dims)
    return {n: s[n] for n in ("o",) + outs}


def _run_decode(s):
    c, x = s["case"], s["x"]
    _lib.call("asca_delta_decode_step", _ptr(x["states"]), _ptr(x["qkv"]), _ptr(x["gate"]), _ptr(s["o"]), c["n"],
              c["H"], c["dh"], None)
    return {"o": s["o"], "states": x["states"]}


def _gemm(ta, tb, M, N, K, A, lda, B, ldb, out, bias=None):
    _lib.call("asca_gemm", ta, tb, M, N, K, 1.0, _ptr(A), lda, _ptr(B), ldb, 0.0, _ptr(out), N,
              None if bias is None else _ptr(bias), None)


def _run_linear(s):
    c, x = s["case"], s["x"]
    T, K, N = c["T"], c["K"], c["N"]
    _gemm(0, 0, T, N, K, x["x"], K, x["w"], N, s["y"], x["b"])
    _gemm(0, 1, T, K, N, x["dy"], N, x["w"], N, s["dx"])
    _gemm(1, 0, K, N, T, x["x"], K, x["dy"], N, s["dw"])
    _lib.call("asca_colsum", _ptr(x["dy"]), T, N, _ptr(s["db"]), 0, None)
    return {n: s[n] for n in ("y", "dx", "dw", "db")}


def _run_moe(s):
    c, x = s["case"], s["x"]
    T, d, dff, E = c["T"], c["d"], c["dff"], c["E"]
    _lib.call("asca_rmsnorm", _ptr(x["x"]), _ptr(s["xn"]), _ptr(s["inv"]), T, d, EPS, None)
    _lib.call("asca_hash_route", _ptr(x["ids"]), T, E, _ptr(s["expert"]), _ptr(s["perm"]), _ptr(s["offsets"]),
              _ptr(s["rws"]), None)
    _lib.call("asca_moe_fwd", _ptr(s["xn"]), _ptr(x["w1"]), _ptr(x["b1"]), _ptr(x["w2"]), _ptr(x["b2"]),
              _ptr(s["perm"]), _ptr(s["offsets"]), T, d, dff, E, _ptr(s["out"]), _ptr(s["pre"]), _ptr(s["hidden"]),
              None)
    _lib.call("asca_moe_bwd", _ptr(s["xn"]), _ptr(x["w1"]), _ptr(x["w2"]), _ptr(s["pre"]), _ptr(s["hidden"]),
              _ptr(s["perm"]), _ptr(s["offsets"]), _ptr(x["dout"]), T, d, dff, E, _ptr(s["dxn"]), _ptr(s["dw1"]),
              _ptr(s["db1"]), _ptr(s["dw2"]), _ptr(s["db2"]), _ptr(s["dpre"]), 0, None)
    _lib.call("asca_rmsnorm_bwd", _ptr(x["x"]), _ptr(s["dxn"]), _ptr(s["dx"]), T, d, EPS, None)
    return {n: s[n] for n in ("expert", "perm", "offsets", "out", "dx", "dw1", "db1", "dw2", "db2")}


def _run_head(s):
    c, x = s["case"], s["x"]
    T, d, V = c["T"], c["d"], c["V"]
    _gemm(0, 0, T, V, d, x["h"], d, x["w"], V, s["logits"])
    _lib.call("asca_cross_entropy", _ptr(s["logits"]), _ptr(x["tgt"]), T, V, _ptr(s["dlogits"]), _ptr(s["losses"]),
              None)
    _gemm(1, 0, d, V, T, x["h"], d, s["dlogits"], V, s["dw"])
    _gemm(0, 1, T, d, V, s["dlogits"], V, x["w"], V, s["dh"])
    return {n: s[n] for n in ("logits", "losses", "dw", "dh")}


def _run_train(s):
    c = s["case"]
    s["model"].train_step_dev(s["ids"], s["tgt"], c["B"], c["T"], sync=False)
    return {n: s[n] for n in ("loss", "grads", "params")}


def _run_step(s):
    return {"logits": s["model"].step(s["ids"], s["st"]), "states": s["states"]}


_RUN = dict(delta=_run_delta, chunk=_run_chunk, decode=_run_decode, linear=_run_linear, moe=_run_moe, head=_run_head,
            train=_run_train, step=_run_step)


def run(state):
    return _RUN[state["case"]["kind"]](state)


# -------------------------------------------------------------------- work


def _n_params(case):
    return sum(r * c for r, c in _shapes(case))


def work(case):
    kind = case["kind"]
    if kind in ("delta", "chunk"):
        # 7 dh^2 (forward) + 17 dh^2 (BPTT) flops per token-head; q, k, v, dO (f32 or bf16), the gates and, fused,
        # the norms in; o, dq, dk, dv and the gate gradients out.
        th, dh = case["B"] * case["T"] * case["H"], case["dh"]
        wide = 4 if kind == "delta" else 2
        return dict(flops=24 * dh * dh * th, bytes=th * (4 * dh * wide + 4 * dh * 4 + (24 if kind == "delta" else 16)))
    if kind == "decode":
        units, dh = case["n"] * case["H"], case["dh"]
        return dict(flops=7 * dh * dh * units, bytes=units * 4 * (2 * dh * dh + 4 * dh + 2))
    if kind == "linear":
        T, K, N = case["T"], case["K"], case["N"]
        return dict(flops=6 * T * K * N, bytes=4 * (2 * T * K + 2 * T * N + 2 * K * N + 2 * N))
    if kind == "moe":
        T, d, dff, E = case["T"], case["d"], case["dff"], case["E"]
        return dict(flops=12 * T * d * dff, bytes=4 * (4 * T * d + 4 * E * d * dff + 2 * E * dff + 2 * d + 3 * T))
    if kind == "head":
        T, d, V = case["T"], case["d"], case["V"]
        return dict(flops=6 * T * d * V, bytes=4 * (2 * T * d + 2 * d * V + T * V + 2 * T))
    d, H, L, dff, V = (case[n] for n in ("d", "H", "L", "dff", "V"))
    per_token = L * (2 * (4 * d * d + 2 * d * H + 2 * d * dff)) + 2 * d * V  # matrix products of one forward
    if kind == "train":
        toks = case["B"] * case["T"]
        return dict(flops=toks * (3 * per_token + L * 24 * H * (d // H) ** 2), bytes=4 * (8 * _n_params(case) + 2 * toks))
    n, dh = case["n"], d // H
    return dict(flops=n * (per_token + L * 7 * H * dh * dh),
                bytes=4 * (min(_n_params(case), n * per_token // 2) + 2 * n * L * H * dh * dh + n * (V + 1)))


# --------------------------------------------------------------- tolerance


def tolerance(case):
    return _TOL[case["kind"]]


# About four times the distance that the path shows from exact() (2-norms; f32 sums of a few thousand terms in all
# kinds, whole models through every layer): delta 2.1e-7, chunk 3.3e-7, decode 1.2e-7, linear 7.3e-7, moe 7.5e-7,
# head 4.2e-7, train 1.4e-6 (gradients), step 1.9e-6.  train's "max" is AdamW's: where a gradient is within rounding
# of zero, its first step of +-4e-4 may take the other sign, beside weights of about 0.05.
_TOL = dict(
    delta={"rel": 1e-6, "max": 1e-4},
    chunk={"rel": 1.5e-6, "max": 1e-4},
    decode={"rel": 5e-7, "max": 2e-5},
    linear={"rel": 3e-6, "max": 1e-4},
    moe={"rel": 3e-6, "max": 1e-4},
    head={"rel": 2e-6, "max": 1e-4},
    train={"rel": 8e-6, "max": 0.05},
    step={"rel": 8e-6, "max": 3e-4},
)


# ------------------------------------------------- the same in 64 bits


def _delta_fwd64(q, k, v, a, b, S=None, keep=0):
    """q, k, v (N, T, dh), a, b (N, T): o, the last state and every keep-th state."""
    N, T, dh = q.shape
    S = torch.zeros(N, dh, dh, dtype=q.dtype, device=q.device) if S is None else S
    o, kept = torch.empty_like(q), []
    for t in range(T):
        if keep and t % keep == 0:
            kept.append(S)
        kt, at, bt = k[:, t], a[:, t, None], b[:, t, None]
        u = bt * (v[:, t] - at * (kt[:, None, :] @ S)[:, 0])
        S = torch.baddbmm(at[:, :, None] * S, kt[:, :, None], u[:, None, :])
        o[:, t] = (q[:, t, None, :] @ S)[:, 0]
    return o, S, kept


def _delta_bwd64(q, k, v, a, b, do, kept, keep):
    N, T, dh = q.shape
    X = torch.zeros(N, dh, dh, dtype=q.dtype, device=q.device)
    dq, dk, dv, da, db = (torch.empty_like(x) for x in (q, k, v, a, b))
    for c in reversed(range(len(kept))):
        lo, hi = c * keep, min(T, c * keep + keep)
        _, last, S = _delta_fwd64(q[:, lo:hi], k[:, lo:hi], v[:, lo:hi], a[:, lo:hi], b[:, lo:hi], kept[c], 1)
        S.append(last)
        for t in reversed(range(lo, hi)):
            P, Sn = S[t - lo], S[t - lo + 1]
            qt, kt, vt, dot = q[:, t], k[:, t], v[:, t], do[:, t]
            at, bt = a[:, t, None], b[:, t, None]
            sk = (kt[:, None, :] @ P)[:, 0]
            w = vt - at * sk
            dq[:, t] = (Sn @ dot[:, :, None])[..., 0]
            X = torch.baddbmm(X, qt[:, :, None], dot[:, None, :])
            du = (kt[:, None, :] @ X)[:, 0]
            dsk = -at * bt * du
            dk[:, t] = (X @ (bt * w)[:, :, None] + P @ dsk[:, :, None])[..., 0]
            dv[:, t] = bt * du
            db[:, t] = (du * w).sum(1)
            da[:, t] = (X * P).sum((1, 2)) - (bt * du * sk).sum(1)
            X = torch.baddbmm(at[:, :, None] * X, kt[:, :, None], dsk[:, None, :])
    return dq, dk, dv, da, db


class _Delta64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, a, b):
        o, _, kept = _delta_fwd64(q, k, v, a, b, keep=64)
        ctx.save_for_backward(q, k, v, a, b)
        ctx.kept = kept
        return o

    @staticmethod
    def backward(ctx, do):
        return _delta_bwd64(*ctx.saved_tensors, do.contiguous(), ctx.kept, 64)


def _heads(x, B, T, H):
    """(B*T, H*w) rows -> (B*H, T, w)."""
    return x.double().view(B, T, H, -1).transpose(1, 2).reshape(B * H, T, -1).contiguous()


def _rows(x, B, T, H):
    return x.view(B, H, T, -1).transpose(1, 2).reshape(B * T, -1).contiguous()


def _exact_delta(case, x):
    B, T, H, dh = (case[n] for n in ("B", "T", "H", "dh"))
    q, k, v, do = (_heads(x[n], B, T, H) for n in ("q", "k", "v", "d_o"))
    a, b = (_heads(x[n], B, T, H)[..., 0] for n in ("alpha", "beta"))
    o, _, kept = _delta_fwd64(q, k, v, a, b, keep=64)
    dq, dk, dv, da, db = _delta_bwd64(q, k, v, a, b, do, kept, 64)
    if case["kind"] == "chunk":
        return {n: _rows(y, B, T, H) for n, y in
                (("o", o), ("dq", dq), ("dk", dk), ("dv", dv), ("dalpha", da), ("dbeta", db))}
    qn, kn = (_heads(x[n], B, T, H) for n in ("qn", "kn"))
    dq = (dq - q * (q * dq).sum(2, keepdim=True)) / qn
    dk = (dk - k * (k * dk).sum(2, keepdim=True)) / kn
    return {"o": _rows(o, B, T, H), "d_qkv": torch.cat([_rows(y, B, T, H) for y in (dq, dk, dv)], 1),
            "d_gate": torch.cat([_rows(y, B, T, H) for y in (da * a * (1 - a), db * b * (1 - b))], 1)}


def _decode64(S, qkv, gate, H, dh):
    n = qkv.shape[0]
    q, k, v = (t.reshape(n * H, dh) for t in qkv.double().view(n, 3, H, dh).unbind(1))
    q, k = (t / t.norm(dim=1, keepdim=True).clamp_min(1e-8) for t in (q, k))
    a, b = (torch.sigmoid(t.reshape(n * H, 1)) for t in gate.double().view(n, 2, H).unbind(1))
    S = S.double().reshape(n * H, dh, dh)
    u = b * (v - a * (k[:, None, :] @ S)[:, 0])
    S = torch.baddbmm(a[:, :, None] * S, k[:, :, None], u[:, None, :])
    return (q[:, None, :] @ S)[:, 0].reshape(n, H * dh), S.reshape(n, H, dh, dh)


def _route(ids, E):
    h = (ids.long() * 0x9E3779B1) & 0xFFFFFFFF
    h = h ^ (h >> 15)
    h = (h * 0x85EBCA6B) & 0xFFFFFFFF
    return (h ^ (h >> 13)) % E


def _rms(x):
    return x * torch.rsqrt(x.square().mean(1, keepdim=True) + EPS)


def _moe(xn, w1, b1, w2, b2, expert, E, dff):
    out = torch.zeros_like(xn)
    for e in range(E):
        rows = (expert == e).nonzero()[:, 0]
        cols = slice(e * dff, (e + 1) * dff)
        hid = torch.nn.functional.silu(xn[rows] @ w1[:, cols] + b1[cols])
        out = out.index_copy(0, rows, hid @ w2[cols] + b2)
    return out


def _exact_moe(case, x):
    E, dff = case["E"], case["dff"]
    expert = _route(x["ids"], E)
    p = {n: x[n].double().requires_grad_() for n in ("x", "w1", "b1", "w2", "b2")}
    out = _moe(_rms(p["x"]), p["w1"], p["b1"], p["w2"], p["b2"], expert, E, dff)
    dx, dw1, db1, dw2, db2 = torch.autograd.grad(out, [p[n] for n in ("x", "w1", "b1", "w2", "b2")],
                                                 x["dout"].double())
    return dict(expert=None, perm=None, offsets=None, out=out.detach(), dx=dx, dw1=dw1, db1=db1, dw2=dw2, db2=db2)


def _params64(case, flat):
    return [flat[o:o + r * c].view(r, c) for (r, c), o in zip(_shapes(case), _offsets(case)[0])]


def _layer(case, p, x, expert, delta):
    d, H = case["d"], case["H"]
    w_qkv, b_qkv, w_gate, b_gate, w_o, b_o, w1, b1, w2, b2 = p
    o = delta(x @ w_qkv + b_qkv, x @ w_gate + b_gate)
    x = x + o @ w_o + b_o
    return x + _moe(_rms(x), w1, b1[0], w2, b2[0], expert, case["E"], case["dff"])


def _exact_train(case, x):
    B, T, H, L = (case[n] for n in ("B", "T", "H", "L"))
    d = case["d"]
    dh = d // H
    flat = _init_params(case, x["g"]).double().requires_grad_()
    p = _params64(case, flat)
    ids, expert = x["ids"].long(), _route(x["ids"], case["E"])

    def delta(qkv, gate):
        q, k, v = (t.reshape(B, T, H, dh).transpose(1, 2).reshape(B * H, T, dh) for t in qkv.split(d, 1))
        q, k = (t / t.norm(dim=2, keepdim=True).clamp_min(1e-8) for t in (q, k))
        a, b = (torch.sigmoid(t).reshape(B, T, H).transpose(1, 2).reshape(B * H, T) for t in gate.split(H, 1))
        o = _Delta64.apply(q.contiguous(), k.contiguous(), v.contiguous(), a.contiguous(), b.contiguous())
        return _rows(o, B, T, H)

    h = p[0][ids]
    for l in range(L):
        h = _layer(case, p[2 + 10 * l:12 + 10 * l], h, expert, delta)
    logits = _rms(h) @ p[1]
    loss = torch.nn.functional.cross_entropy(logits, x["tgt"].long())
    g, = torch.autograd.grad(loss, flat)
    return dict(loss=loss.detach().view(1), grads=g, params=None)


def _exact_step(case, x):
    n, H, L, d = (case[k] for k in ("n", "H", "L", "d"))
    dh = d // H
    p = _params64(case, _init_params(case, x["g"]).double())
    states = _init_states(case, x["g"]).view(L, n, H, dh, dh)
    expert, new = _route(x["ids"], case["E"]), []
    h = p[0][x["ids"].long()]
    for l in range(L):
        def delta(qkv, gate):
            o, S = _decode64(states[l], qkv, gate, H, dh)
            new.append(S)
            return o

        h = _layer(case, p[2 + 10 * l:12 + 10 * l], h, expert, delta)
    return dict(logits=_rms(h) @ p[1], states=torch.stack(new).reshape(-1))


def exact(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    if kind in ("delta", "chunk"):
        return _exact_delta(case, x)
    if kind == "decode":
        o, S = _decode64(x["states"], x["qkv"], x["gate"], case["H"], case["dh"])
        return dict(o=o, states=S)
    if kind == "linear":
        X, w, b, dy = (x[n].double() for n in ("x", "w", "b", "dy"))
        return dict(y=X @ w + b, dx=dy @ w.t(), dw=X.t() @ dy, db=dy.sum(0))
    if kind == "moe":
        return _exact_moe(case, x)
    if kind == "head":
        h, w = x["h"].double(), x["w"].double()
        logits = h @ w
        losses = torch.nn.functional.cross_entropy(logits, x["tgt"].long(), reduction="none")
        dl = (torch.softmax(logits, 1) - torch.nn.functional.one_hot(x["tgt"].long(), case["V"])) / case["T"]
        return dict(logits=logits, losses=losses, dw=h.t() @ dl, dh=dl @ w.t())
    return _exact_train(case, x) if kind == "train" else _exact_step(case, x)
