"""Workloads of the library's main paths, for timing and for comparing results.

Each case goes through the public entry points (include/tlgemm.h, tltrain.h,
tldecode.h and the C host library, by way of tlgemm.py) the way a program that
uses them does:

  linear     one projection forward and backward (mm, mm_bt, mm_atb) on device
             buffers, any M, K, N
  gemv       the projections of one decode layer at M <= 8 as grouped launches
  host       the drop-in seam on host buffers, weights and gradients registered
  attention  causal GQA attention forward and backward of one layer
  moe        a top-1 mixture-of-experts FFN forward and backward (kept state)
  step       a whole training step: batch in, captured step, updated weights
  prefill    a prompt through the decoder: KV rings and logits
  generate   prefill and greedy tokens

Values are those of the models: activations and attention inputs ~ N(0, 1),
weights ~ N(0, 0.02^2), output gradients ~ N(0, 0.01^2), all fp32.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinylm-c_amd"))
import tlgemm  # noqa: E402

HEAD = 32                      # head_dim of every attention path
ROPE_BASE = 10000.0


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # the seam's self-test shape: odd everywhere, a few microseconds of work
        dict(name="linear_ragged", kind="linear", M=201, K=131, N=259),
        # one FFN projection of the m3 model at its training batch
        dict(name="linear_ffn", kind="linear", M=4096, K=256, N=768),
        # the head of the m8 model at its training batch: the largest projection
        dict(name="linear_head", kind="linear", M=8192, K=384, N=2048),
        # single-token decode of an m8 layer: latency and launches
        dict(name="gemv_m1", kind="gemv", M=1, D=384, KD=96, F=1024),
        # the -DUSE_HIP seam: activations cross PCIe on every call
        dict(name="host_ffn", kind="host", M=2048, K=128, N=384),
        # one m3 layer's attention at its training batch
        dict(name="attention_m3", kind="attention", B=16, T=256, H=8, KV=2, win=0, rope=True),
        # the m3-scale MoE layer with skewed experts
        dict(name="moe_m3", kind="moe", N=4096, D=256, F=768, E=4, tilt=1.0),
        # training steps: nano (launch bound), m3 (the usual size), m8 with MTP heads (the largest)
        dict(name="step_nano", kind="step", B=8, T=256, V=2048, D=128, L=1, H=4, KV=1, F=384, n_mtp=0, win=0),
        dict(name="step_m3", kind="step", B=16, T=256, V=2048, D=256, L=6, H=8, KV=2, F=768, n_mtp=0, win=0),
        dict(name="step_m8", kind="step", B=32, T=256, V=2048, D=384, L=8, H=12, KV=3, F=1024, n_mtp=2, win=0),
        # a long prompt into a full f32 ring, exact softmax
        dict(name="prefill_m8", kind="prefill", V=2048, D=384, L=8, H=12, KV=3, F=1024, W=256, n=250, f16=False,
             exact_exp=True),
        # chat-like greedy generation with the default f16 ring and fast exp
        dict(name="generate_m8", kind="generate", V=2048, D=384, L=8, H=12, KV=3, F=1024, W=256, n=16, gen=48,
             f16=True, exact_exp=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, q):
    return max(q, _log(rng, lo, hi) // q * q)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "gemv", "host", "attention", "attention", "moe", "step", "step",
                       "prefill", "generate"])
    if kind == "linear":
        q = rng.choice([1, 4, 4, 32])
        M, K, N = _log(rng, 2, 8192), _mult(rng, 24, 1536, q), _mult(rng, 24, 2048, q)
        return dict(kind=kind, M=M, K=K, N=N)
    if kind == "gemv":
        return dict(kind=kind, M=rng.randint(1, 8), D=_mult(rng, 64, 512, 4), KD=_mult(rng, 32, 128, 4),
                    F=_mult(rng, 96, 1536, 4))
    if kind == "host":
        return dict(kind=kind, M=_log(rng, 16, 2048), K=_log(rng, 24, 384), N=_log(rng, 24, 768))
    if kind == "attention":
        KV, g = rng.choice([1, 2, 3]), rng.choice([1, 2, 4, 4, 8])
        return dict(kind=kind, B=_log(rng, 1, 32), T=_log(rng, 9, 300), H=KV * g, KV=KV,
                    win=rng.choice([0, 0, rng.randint(5, 128)]), rope=g % 4 == 0)
    if kind == "moe":
        return dict(kind=kind, N=_log(rng, 64, 4096), D=_mult(rng, 32, 256, 4), F=_mult(rng, 64, 768, 4),
                    E=rng.randint(2, 8), tilt=rng.choice([0.0, 0.5, 1.0]))
    KV, g = rng.choice([1, 2, 3]), 4
    dims = dict(V=_mult(rng, 256, 2048, 8), D=KV * g * HEAD, L=rng.randint(1, 4), H=KV * g, KV=KV,
                F=_mult(rng, 96, 1024, 32))
    if kind == "step":
        return dict(kind=kind, B=_log(rng, 1, 16), T=_log(rng, 24, 256), n_mtp=rng.choice([0, 0, 1, 2]),
                    win=rng.choice([0, 0, 48]), **dims)
    n = _log(rng, 3, 256)
    dims.update(W=256, f16=rng.random() < 0.5, exact_exp=rng.random() < 0.5, n=n)
    if kind == "prefill":
        return dict(kind=kind, **dims)
    return dict(kind=kind, gen=_log(rng, 4, 64), **dims)


# --------------------------------------------------------------- plumbing --
_STREAM = None


def _own_stream(lib):
    """One stream of the program's own for every model: captures need one that
    is not the null stream, and calls on two streams would share the library's
    scratch."""
    global _STREAM
    if _STREAM is None:
        _STREAM = lib.tlg_stream_create()
    return _STREAM


def _lib():
    lib = tlgemm.load()
    lib.check(lib.tlg_init(0), "tlg_init")
    return lib


class _Mem:
    """Device memory that `owner` (a Train or Decode) frees when it goes."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(int(ptr), False), version=2)


def _view(owner, ptr, shape, typestr="<f4"):
    """A device buffer of `owner` as a tensor (no copy); the tensor keeps the owner alive."""
    t = torch.as_tensor(_Mem(owner, ptr, tuple(shape), typestr), device="cuda")
    t.owner = owner
    return t


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _model(c):
    return dict(V=c["V"], D=c["D"], L=c["L"], H=c["H"], KV=c["KV"], F=c["F"], T=c.get("T", c.get("W")),
                n_mtp=c.get("n_mtp", 0), win=c.get("win", 0), rope_base=ROPE_BASE)


def _layout(c):
    """(name, shape) of every tensor of the flat parameter buffer, in order."""
    D, KD, F = c["D"], c["KV"] * HEAD, c["F"]
    out = [("emb", (c["V"], D))]
    for l in range(c["L"]):
        out += [(f"{l}.an1", (D,)), (f"{l}.wq", (D, D)), (f"{l}.wk", (D, KD)), (f"{l}.wv", (D, KD)),
                (f"{l}.wo", (D, D)), (f"{l}.an2", (D,)), (f"{l}.w1", (D, F)), (f"{l}.w3", (D, F)), (f"{l}.w2", (F, D))]
    out.append(("nf", (D,)))
    return out + [(f"mtp{k}", (D, D)) for k in range(c.get("n_mtp", 0))]


def _params(c, seed):
    """The flat parameters a model starts from: N(0, 0.02^2), norm gains near 1."""
    g, parts = _gen(seed), []
    for name, shape in _layout(c):
        if len(shape) == 1:
            parts.append(1.0 + _normal(g, *shape, std=0.02))
        else:
            parts.append(_normal(g, *shape, std=0.02).reshape(-1))
    return torch.cat(parts)


def _unflatten(c, flat):
    out, at = {}, 0
    for name, shape in _layout(c):
        n = math.prod(shape)
        out[name] = flat[at:at + n].view(shape)
        at += n
    return out


def _tokens(c, count, seed):
    return np.random.default_rng(seed).integers(0, c["V"], count).astype(np.int32)


HYPER = (3e-4, 0.9, 0.95, 0.1)           # lr, b1, b2, weight decay


# ---------------------------------------------------------------- prepare --
def _inputs(c, seed):
    """The seeded inputs of a case (shared with exact())."""
    g, k = _gen(seed), c["kind"]
    if k == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return dict(X=_normal(g, M, K), W=_normal(g, K, N, std=0.02), dY=_normal(g, M, N, std=0.01))
    if k == "gemv":
        M, D, KD, F = c["M"], c["D"], c["KD"], c["F"]
        return dict(x=_normal(g, M, D), h=_normal(g, M, F), wq=_normal(g, D, D, std=0.02),
                    wk=_normal(g, D, KD, std=0.02), wv=_normal(g, D, KD, std=0.02), w1=_normal(g, D, F, std=0.02),
                    w3=_normal(g, D, F, std=0.02), w2=_normal(g, F, D, std=0.02))
    if k == "host":
        r, (M, K, N) = np.random.default_rng(seed), (c["M"], c["K"], c["N"])
        return dict(X=r.standard_normal((M, K), dtype=np.float32),
                    W=0.02 * r.standard_normal((K, N), dtype=np.float32),
                    dY=0.01 * r.standard_normal((M, N), dtype=np.float32))
    if k == "attention":
        R, D, KD = c["B"] * c["T"], c["H"] * HEAD, c["KV"] * HEAD
        return dict(q=_normal(g, R, D), k=_normal(g, R, KD), v=_normal(g, R, KD), dout=_normal(g, R, D, std=0.01))
    if k == "moe":
        N, D, F, E = c["N"], c["D"], c["F"], c["E"]
        x = _normal(g, N, D)
        x[:, 0] = 1.0                    # a constant feature: the router's bias towards low experts
        wr = _normal(g, D, E, std=0.05)
        wr[0] = c["tilt"] * torch.linspace(1.0, 0.0, E, device="cuda")
        return dict(x=x, fin=_normal(g, N, D), dout=_normal(g, N, D, std=0.01), wr=wr,
                    w1=_normal(g, E, D, F, std=0.02), w3=_normal(g, E, D, F, std=0.02),
                    w2=_normal(g, E, F, D, std=0.02))
    raise ValueError(k)


def _rope_tables(T):
    """cos / sin of the model's angles, which are fp32 products by definition."""
    inv = np.power(np.float32(ROPE_BASE), np.float32(-2.0) * np.arange(HEAD // 2, dtype=np.float32) / np.float32(HEAD))
    a = torch.from_numpy(np.arange(T, dtype=np.float32)[:, None] * inv).double()
    return a.cos(), a.sin()


def prepare(case, seed):
    lib, c, k = _lib(), case, case["kind"]
    st = torch.cuda.current_stream().cuda_stream
    s = dict(case=c, lib=lib, stream=st)
    if k in ("step", "prefill", "generate"):
        host = tlgemm.host()
        st = s["stream"] = _own_stream(lib)
        flat = _params(c, seed)
        torch.cuda.synchronize()
        if k == "step":
            t = s["train"] = host.train(_model(c), c["B"])
            s["np"] = t.np
            lib.check(lib.tlg_memcpy_d2d(t.buf(0), flat.data_ptr(), 4 * t.np, st), "weights")
            N = c["B"] * c["T"]
            s["batch"] = (_tokens(c, N, seed), _tokens(c, N, seed + 1),
                          _tokens(c, N * c["n_mtp"], seed + 2) if c["n_mtp"] else None)
            t.set_batch(*s["batch"], st)
            t.forward(st)                # sizes the library's scratch before the capture
            t.backward(st)
            t.graph_build(st)
            s["t"] = 0
        else:
            d = s["dec"] = host.decode(_model(c), W=c["W"], kv_f16=int(c["f16"]), exact_exp=int(c["exact_exp"]),
                                       maxpos=1024)
            d.upload(flat.cpu().numpy(), st)
            s["prompt"] = _tokens(c, c["n"], seed)
            if k == "generate":
                s["toks"] = torch.zeros(c["gen"], dtype=torch.int32, device="cuda")
        lib.check(lib.tlg_stream_sync(st), "sync")
        return s
    s.update(_inputs(c, seed))
    if k == "linear":
        s.update(Y=torch.empty(c["M"], c["N"], device="cuda"), dX=torch.empty(c["M"], c["K"], device="cuda"),
                 dW=torch.empty(c["K"], c["N"], device="cuda"))
    elif k == "gemv":
        M = c["M"]
        s.update({n: torch.empty(M, w, device="cuda") for n, w in
                  (("q", c["D"]), ("kk", c["KD"]), ("vv", c["KD"]), ("g", c["F"]), ("u", c["F"]), ("y", c["D"]))})
    elif k == "host":
        s.update(Y=np.empty((c["M"], c["N"]), np.float32), dX=np.empty((c["M"], c["K"]), np.float32),
                 dW=np.empty((c["K"], c["N"]), np.float32))
        s["reg"] = _Registered(lib, s["W"], s["dW"])
    elif k == "attention":
        R = c["B"] * c["T"]
        cs, sn = _rope_tables(c["T"])
        s.update(cs=cs.float().cuda(), sn=sn.float().cuda(), out=torch.empty_like(s["q"]),
                 lse=torch.empty(R, c["H"], device="cuda"), dq=torch.empty_like(s["q"]), dk=torch.empty_like(s["k"]),
                 dv=torch.empty_like(s["v"]))
    else:
        N, D, F, E = c["N"], c["D"], c["F"], c["E"]
        kb = lib.tlg_moe_keep_bytes(N, D, F, E)
        s.update(out=torch.empty(N, D, device="cuda"), dx=torch.empty(N, D, device="cuda"),
                 assign=torch.empty(N, dtype=torch.int32, device="cuda"), gate=torch.empty(N, device="cuda"),
                 rprobs=torch.empty(N, E, device="cuda"), keep=torch.empty(kb, dtype=torch.uint8, device="cuda"),
                 gwr=torch.empty_like(s["wr"]), gw1=torch.empty_like(s["w1"]), gw3=torch.empty_like(s["w3"]),
                 gw2=torch.empty_like(s["w2"]))
    return s


class _Registered:
    """Host buffers with a device mirror, as the seam's user keeps P and G."""

    def __init__(self, lib, *bufs):
        self.lib, self.bufs = lib, bufs
        for b in bufs:
            lib.check(lib.tlg_register(b.ctypes.data, b.nbytes), "tlg_register")

    def __del__(self):
        for b in self.bufs:
            self.lib.tlg_unregister(b.ctypes.data)


# -------------------------------------------------------------------- run --
def run(state):
    return _RUN[state["case"]["kind"]](state)


def _run_linear(s):
    lib, c, st = s["lib"], s["case"], s["stream"]
    M, K, N = c["M"], c["K"], c["N"]
    X, W, dY, Y, dX, dW = (s[n].data_ptr() for n in ("X", "W", "dY", "Y", "dX", "dW"))
    lib.mm(Y, X, W, M, K, N, st)
    lib.zero(dX, M * K, st)                     # the caller's memset before the accumulating backward
    lib.mm_bt(dX, dY, W, M, K, N, st)
    lib.zero(dW, K * N, st)
    lib.mm_atb(dW, X, dY, M, K, N, st)
    return [s["Y"], s["dX"], s["dW"]]


def _run_gemv(s):
    lib, c, st = s["lib"], s["case"], s["stream"]
    M, D, KD, F = c["M"], c["D"], c["KD"], c["F"]
    p = {n: s[n].data_ptr() for n in ("x", "h", "wq", "wk", "wv", "w1", "w3", "w2", "q", "kk", "vv", "g", "u", "y")}

    def mm(out, a, w, K, N):
        return dict(op="mm", C=p[out], M=M, K=K, N=N, A=[p[a]], B=[p[w]])

    lib.group([mm("q", "x", "wq", D, D), mm("kk", "x", "wk", D, KD), mm("vv", "x", "wv", D, KD)], st)
    lib.group([mm("g", "x", "w1", D, F), mm("u", "x", "w3", D, F)], st)
    lib.group([mm("y", "h", "w2", F, D)], st)
    return [s[n] for n in ("q", "kk", "vv", "g", "u", "y")]


def _run_host(s):
    lib, c = s["lib"], s["case"]
    M, K, N = c["M"], c["K"], c["N"]
    X, W, dY, Y, dX, dW = (s[n].ctypes.data for n in ("X", "W", "dY", "Y", "dX", "dW"))
    s["dX"].fill(0.0)
    s["dW"].fill(0.0)
    lib.check(lib.tlg_push(dW), "tlg_push")
    lib.tlg_sgemm_nn(Y, X, W, M, K, N)
    lib.tlg_sgemm_nt_acc(dX, dY, W, M, K, N)
    lib.tlg_sgemm_tn_acc(dW, X, dY, M, K, N)
    lib.check(lib.tlg_pull(dW), "tlg_pull")
    return [s["Y"], s["dX"], s["dW"]]


def _run_attention(s):
    lib, c, st = s["lib"], s["case"], s["stream"]
    q, k, v, dout, out, lse, dq, dk, dv, cs, sn = (
        s[n].data_ptr() for n in ("q", "k", "v", "dout", "out", "lse", "dq", "dk", "dv", "cs", "sn"))
    dims = (c["B"], c["T"], c["H"], c["KV"], HEAD, c["win"])
    if c["rope"]:
        lib.check(lib.tlg_dev_attn_fwd_rope(q, k, v, out, lse, *dims, cs, sn, st), "attn_fwd_rope")
        lib.check(lib.tlg_dev_attn_bwd_rope(q, k, v, out, lse, dout, dq, dk, dv, *dims, cs, sn, st), "attn_bwd_rope")
    else:
        lib.check(lib.tlg_dev_attn_fwd(q, k, v, out, lse, *dims, st), "attn_fwd")
        lib.check(lib.tlg_dev_attn_bwd(q, k, v, out, lse, dout, dq, dk, dv, *dims, st), "attn_bwd")
    return [s[n] for n in ("out", "lse", "dq", "dk", "dv")]


def _run_moe(s):
    lib, c, st = s["lib"], s["case"], s["stream"]
    N, D, F, E = c["N"], c["D"], c["F"], c["E"]
    p = {n: s[n].data_ptr() for n in ("x", "fin", "dout", "wr", "w1", "w3", "w2", "out", "dx", "assign", "gate",
                                      "rprobs", "keep", "gwr", "gw1", "gw3", "gw2")}
    for n in ("gwr", "gw1", "gw3", "gw2"):
        lib.zero(p[n], s[n].numel(), st)
    w = (p["wr"], p["w1"], p["w3"], p["w2"])
    lib.moe_fwd_keep(p["x"], p["fin"], p["out"], N, D, F, E, *w, p["assign"], p["gate"], p["rprobs"], p["keep"],
                     s["keep"].numel(), st)
    lib.moe_bwd_kept(p["x"], p["dout"], p["dx"], p["assign"], p["gate"], p["rprobs"], N, D, F, E, *w, p["gwr"],
                     p["gw1"], p["gw3"], p["gw2"], p["keep"], s["keep"].numel(), st)
    lib.check(lib.tlg_dev_gemm_flush(st), "tlg_dev_gemm_flush")
    return [s[n] for n in ("out", "assign", "gate", "rprobs", "dx", "gwr", "gw1", "gw3", "gw2")]


def _run_step(s):
    t, st = s["train"], s["stream"]
    s["t"] += 1
    t.set_batch(*s["batch"], st)
    t.set_hyper(*HYPER, s["t"], st)
    t.graph_step(st)
    return [_view(t, t.buf(1), (s["np"],)), _view(t, t.buf(0), (s["np"],))]


def _decoded(s, rows):
    """The logits' first `rows` rows and the written part of every layer's K and V ring."""
    d, c = s["dec"], s["case"]
    live, KD = min(c["n"] + c.get("gen", 0), c["W"]), c["KV"] * HEAD
    out = [_view(d, d.host.dll.tl_decode_logits(d.h), (rows, c["V"]))]
    for l in range(c["L"]):
        for kv in (0, 1):
            out.append(_view(d, d.host.dll.tl_decode_ring(d.h, l, kv), (live, KD), "<f2" if c["f16"] else "<f4"))
    return out


def _run_prefill(s):
    s["dec"].prime(s["prompt"], s["stream"])
    return _decoded(s, (s["case"]["n"] - 1) % 8 + 1)          # the rows of the last chunk


def _run_generate(s):
    d, c, st = s["dec"], s["case"], s["stream"]
    d.prime(s["prompt"], st)
    d.persist(c["gen"], st, s["toks"].data_ptr())
    return [s["toks"]] + _decoded(s, 1)


_RUN = dict(linear=_run_linear, gemv=_run_gemv, host=_run_host, attention=_run_attention, moe=_run_moe,
            step=_run_step, prefill=_run_prefill, generate=_run_generate)


# ------------------------------------------------------------------- work --
def _visible(T, win, first=0):
    return sum(min(t + 1, win) if win else t + 1 for t in range(first, T))


def work(case):
    c, k = case, case["kind"]
    if k in ("linear", "host"):
        M, K, N = c["M"], c["K"], c["N"]
        return dict(bytes=8.0 * (M * K + K * N + M * N), flops=6.0 * M * K * N)
    if k == "gemv":
        M, D, KD, F = c["M"], c["D"], c["KD"], c["F"]
        w = D * D + 2 * D * KD + 3 * D * F
        return dict(bytes=4.0 * (w + M * (3 * D + 2 * KD + 3 * F)), flops=2.0 * M * w)
    if k == "attention":
        R, D, KD, vis = c["B"] * c["T"], c["H"] * HEAD, c["KV"] * HEAD, c["B"] * _visible(c["T"], c["win"])
        # forward QK, PV; backward S, dP, dV, dQ, dK
        return dict(bytes=4.0 * R * (4 * D + 4 * KD + c["H"]), flops=14.0 * vis * c["H"] * HEAD)
    if k == "moe":
        N, D, F, E = c["N"], c["D"], c["F"], c["E"]
        w = D * E + 3 * E * D * F
        return dict(bytes=4.0 * (2 * w + N * (5 * D + E + 2)), flops=18.0 * N * D * F + 6.0 * N * D * E)
    D, KD, F, V, L = c["D"], c["KV"] * HEAD, c["F"], c["V"], c["L"]
    layer = 2 * D * D + 2 * D * KD + 3 * D * F
    np_ = V * D + L * (layer + 2 * D) + D + c.get("n_mtp", 0) * D * D
    if k == "step":
        N, mtp = c["B"] * c["T"], c["n_mtp"]
        mats = L * layer + V * D + mtp * (D * D + V * D)
        att = 14.0 * c["B"] * _visible(c["T"], c["win"]) * D * L
        return dict(bytes=4.0 * (7 * np_ + N * (2 + mtp)), flops=6.0 * N * mats + att)
    el = 2 if c["f16"] else 4
    rows = c["n"] + c.get("gen", 0)
    ring = 2.0 * el * L * KD
    passes = 1 + c.get("gen", 0)         # the prompt in one pass over the weights, then one for each token
    seen = ring * (c["n"] + sum(min(c["n"] + i, c["W"]) for i in range(c.get("gen", 0))))
    flops = 2.0 * rows * L * layer + 2.0 * V * D * passes + 4.0 * D * L * _visible(rows, c["W"])
    return dict(bytes=4.0 * (np_ - V * D) * passes + 4.0 * V * D * passes + seen, flops=flops)


# -------------------------------------------------------------- tolerance --
def tolerance(case):
    """About four times what the paths differ from fp64 (sums in other orders
    differ as much)."""
    k = case["kind"]
    if k in ("linear", "host"):
        return dict(rel=5e-6, max=5e-5)
    if k == "gemv":
        return dict(rel=1e-6, max=1e-5)
    if k == "attention":
        return dict(rel=2e-6, max=4e-5)
    if k == "moe":
        return dict(rel=4e-6, max=4e-5, differ=1e-3)
    if k == "step":                      # AdamW's early updates are +-lr whatever a gradient's size
        return dict(rel=4e-5, max=0.02)
    if case["f16"]:                      # an fp32 difference may round to the ring's next f16
        return dict(rel=1e-4, max=5e-3, differ=0.01)
    return dict(rel=4e-6, max=1e-4, differ=0.01)


# ------------------------------------------------------------------ exact --
def _rotate(x, cs, sn):
    a, b = x[..., :HEAD // 2], x[..., HEAD // 2:]
    return torch.cat([a * cs - b * sn, a * sn + b * cs], -1)


def _attend(q, k, v, c, T, rope=True):
    """q [B, T, H, 32], k / v [B, T, KV, 32] -> (out, base-2 log-sum-exp)."""
    if rope:
        cs, sn = (t.cuda()[None, :, None, :] for t in _rope_tables(T))
        q, k = _rotate(q, cs, sn), _rotate(k, cs, sn)
    g = c["H"] // c["KV"]
    k, v = (t.repeat_interleave(g, 2).transpose(1, 2) for t in (k, v))
    s = q.transpose(1, 2) @ k.transpose(2, 3) / math.sqrt(HEAD)
    i = torch.arange(T, device="cuda")
    hide = i[None, :] > i[:, None]
    if c.get("win", 0) > 0:
        hide = hide | (i[None, :] <= i[:, None] - c["win"])
    s = s.masked_fill(hide, -math.inf)
    lse = torch.logsumexp(s, -1).transpose(1, 2) / math.log(2.0)
    return (torch.softmax(s, -1) @ v).transpose(1, 2), lse


def _norm(x, g):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * g


def _forward(c, w, tok):
    """(final-norm rows [B, T, D], each layer's (rotated k, v)) of tokens [B, T]."""
    B, T = tok.shape
    x, kvs = w["emb"][tok], []
    cs, sn = (t.cuda()[None, :, None, :] for t in _rope_tables(T))
    for l in range(c["L"]):
        a = _norm(x, w[f"{l}.an1"])
        q = (a @ w[f"{l}.wq"]).view(B, T, c["H"], HEAD)
        k = _rotate((a @ w[f"{l}.wk"]).view(B, T, c["KV"], HEAD), cs, sn)
        v = (a @ w[f"{l}.wv"]).view(B, T, c["KV"], HEAD)
        kvs.append((k, v))
        o, _ = _attend(_rotate(q, cs, sn), k, v, c, T, rope=False)
        x = x + o.reshape(B, T, c["D"]) @ w[f"{l}.wo"]
        f = _norm(x, w[f"{l}.an2"])
        x = x + (torch.nn.functional.silu(f @ w[f"{l}.w1"]) * (f @ w[f"{l}.w3"])) @ w[f"{l}.w2"]
    return _norm(x, w["nf"]), kvs


def _exact_step(c, seed):
    N = c["B"] * c["T"]
    flat = _params(c, seed).double().requires_grad_(True)
    w = _unflatten(c, flat)
    tok, tgt = (torch.from_numpy(_tokens(c, N, seed + i)).long().cuda() for i in (0, 1))
    fn, _ = _forward(c, w, tok.view(c["B"], c["T"]))
    fn = fn.reshape(N, c["D"])
    loss = torch.nn.functional.cross_entropy(fn @ w["emb"].t(), tgt)
    if c["n_mtp"]:
        tm = torch.from_numpy(_tokens(c, N * c["n_mtp"], seed + 2)).long().cuda().view(c["n_mtp"], N)
        for h in range(c["n_mtp"]):
            hk = fn + torch.nn.functional.silu(fn @ w[f"mtp{h}"])
            loss = loss + 0.2 * 0.8 ** h * torch.nn.functional.cross_entropy(hk @ w["emb"].t(), tm[h])
    grad, = torch.autograd.grad(loss, flat)
    lr, _, _, wd = HYPER
    g = grad / max(1.0, float(grad.norm()))
    p = flat.detach()
    # AdamW's first step: both bias-corrected moments are those of this gradient
    return [grad, p - lr * (g / (g.abs() + 1e-8) + wd * p)]


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "step":
        return _exact_step(c, seed)
    if k in ("prefill", "generate"):
        if c["f16"] or not c["exact_exp"]:
            return None                  # the ring's rounding and the fast exponential are part of the result
        w = _unflatten(c, _params(c, seed).double())
        toks = _tokens(c, c["n"], seed).tolist()
        done = []
        for i in range(c.get("gen", 0) + 1):
            fn, kvs = _forward(dict(c, win=c["W"]), w, torch.tensor(toks, device="cuda")[None])
            row = fn[0, -1] @ w["emb"].t()
            toks.append(int(row.argmax()))
            done.append(toks[-1])
        n, KD = len(toks) - 1, c["KV"] * HEAD
        slot = torch.arange(n, device="cuda") % c["W"]
        rings = []
        for kk, vv in kvs:
            for t in (kk, vv):           # later positions replace the ones that had their slot
                ring = torch.zeros(min(n, c["W"]), KD, dtype=torch.float64, device="cuda")
                for at in range(0, n, c["W"]):
                    ring[slot[at:at + c["W"]]] = t[0].reshape(n, KD)[at:at + c["W"]]
                rings.append(ring)
        if k == "prefill":
            return [fn[0, -((n - 1) % 8 + 1):] @ w["emb"].t()] + rings
        # the last step decodes the token before the last one chosen
        return [torch.tensor(done[1:], dtype=torch.int32, device="cuda"), row[None]] + rings
    s = _inputs(c, seed)
    d = {n: (torch.from_numpy(v).cuda() if isinstance(v, np.ndarray) else v).double() for n, v in s.items()}
    if k in ("linear", "host"):
        return [d["X"] @ d["W"], d["dY"] @ d["W"].t(), d["X"].t() @ d["dY"]]
    if k == "gemv":
        return [d["x"] @ d["wq"], d["x"] @ d["wk"], d["x"] @ d["wv"], d["x"] @ d["w1"], d["x"] @ d["w3"],
                d["h"] @ d["w2"]]
    if k == "attention":
        B, T = c["B"], c["T"]
        q, kk, v = (d[n].view(B, T, h, HEAD).requires_grad_(True) for n, h in
                    (("q", c["H"]), ("k", c["KV"]), ("v", c["KV"])))
        out, lse = _attend(q, kk, v, c, T, c["rope"])
        grads = torch.autograd.grad(out, (q, kk, v), d["dout"].view_as(out))
        R = B * T
        return [out.detach().reshape(R, -1), lse.detach().reshape(R, -1)] + [t.reshape(R, -1) for t in grads]
    N, E = c["N"], c["E"]
    for n in ("x", "wr", "w1", "w3", "w2"):
        d[n].requires_grad_(True)
    p = torch.softmax(d["x"] @ d["wr"], -1)
    gate, e = p.max(-1)
    y = torch.zeros_like(d["fin"])
    for i in range(E):
        rows = (e == i).nonzero()[:, 0]
        xi = d["x"][rows]
        y = y.index_copy(0, rows, (torch.nn.functional.silu(xi @ d["w1"][i]) * (xi @ d["w3"][i])) @ d["w2"][i])
    out = d["fin"] + gate[:, None] * y
    share = torch.bincount(e, minlength=E).double() / N
    obj = (out * d["dout"]).sum() + 0.01 * E * (share * p.mean(0)).sum()
    gx, gwr, gw1, gw3, gw2 = torch.autograd.grad(obj, [d[n] for n in ("x", "wr", "w1", "w3", "w2")])
    return [out.detach(), e.int(), gate.detach(), p.detach(), gx, gwr, gw1, gw3, gw2]
