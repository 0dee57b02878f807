"""The workloads whose speed this package is judged by, through its public entry points.

Each case is a dict of plain values; `kind` names the entry point and what a program uses it
for, the rest are sizes and options.  `prepare` makes what such a program holds before the
call, `run` is one pass, `exact` the same outputs from plain torch in float64.

Kinds:
  gla_layer_decode  one decode step of a GLA layer, projections to normalised output
                    (fused_recurrent_gla_conv_norm_gate): a small serving batch, where launches
                    and latency count
  gla_decode        one decode step of the recurrence against a state cache
                    (fused_recurrent_gla): a full serving batch, bound by the state's bytes
  kda_decode        the same for KDA (fused_recurrent_kda)
  gla_fwd           chunk_gla without gradients: prefill of packed prompts or of a batch
  gla_recurrent     fused_recurrent_gla without gradients over whole sequences, state carried
                    in and out
  gla_train         chunk_gla forward and backward; with V = 2 K the head shape of a GLA layer
                    at its default expansion (expand_k 0.5, expand_v 1)
  simple_gla_train  chunk_simple_gla forward and backward over packed documents, one gate per
                    token or a constant decay per head
  kda_fwd           chunk_kda without gradients: prefill; "raw" takes the gate activation and
                    the q / k normalisation into the call, as a KDA layer does
  kda_train         chunk_kda forward and backward
  side_train        the ops around the recurrence in a layer: ShortConvolution and
                    FusedRMSNormGated, forward and backward
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pallas-kernel_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DT = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # decode of a GLA layer for a few users: one launch, its latency and the host path
        dict(name="gla_layer_decode_b8", kind="gla_layer_decode", B=8, H=16, K=128, V=128, W=4,
             dtype="bf16"),
        # decode of a full serving batch: the fp32 states in and out are nearly all the bytes
        dict(name="gla_decode_b256", kind="gla_decode", B=256, H=16, K=128, V=128, dtype="bf16"),
        dict(name="kda_decode_b64", kind="kda_decode", B=64, H=32, K=128, V=128, dtype="bf16"),
        # the smallest whole call: a short fp32 forward
        dict(name="gla_fwd_f32_b2", kind="gla_fwd", B=2, T=512, H=4, K=64, V=64, seqs=0,
             h0=False, dtype="f32"),
        # prefill of five prompts packed into one call, odd lengths
        dict(name="gla_prefill_packed", kind="gla_fwd", B=1, T=8191, H=16, K=128, V=128, seqs=5,
             h0=False, dtype="bf16"),
        # the recurrent mode of the layer over whole sequences
        dict(name="gla_recurrent_b16", kind="gla_recurrent", B=16, T=2048, H=8, K=128, V=128,
             h0=True, dtype="bf16"),
        # the training step at its usual size, states in and out of the graph
        dict(name="gla_train_b8", kind="gla_train", B=8, T=4096, H=16, K=128, V=128, seqs=0,
             h0=True, dtype="bf16"),
        # training of a layer whose value heads are twice as wide as its keys, ragged length
        dict(name="gla_train_wide", kind="gla_train", B=8, T=1000, H=8, K=128, V=256, seqs=0,
             h0=False, dtype="bf16"),
        # training over packed documents with one gate per token
        dict(name="simple_gla_train_packed", kind="simple_gla_train", T=16384, H=32, K=128, V=128,
             seqs=8, gate="token", dtype="bf16"),
        # prefill of one long prompt through a KDA layer's options, ragged length
        dict(name="kda_prefill_raw", kind="kda_fwd", B=1, T=5000, H=32, K=128, V=128, raw=True,
             h0=False, dtype="bf16"),
        # the largest: a KDA training step
        dict(name="kda_train_b4", kind="kda_train", B=4, T=8192, H=32, K=128, V=128, h0=False,
             dtype="bf16"),
        # the streams either side of the op in a training step
        dict(name="side_train_b8", kind="side_train", B=8, T=4096, H=16, V=128, W=4,
             dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case: kinds evenly, sizes over the logarithm of their range (B * T * H at most
    that of the largest listed case of the kind), head sizes as models have them, odd lengths."""
    kind = rng.choice(["gla_layer_decode", "gla_decode", "kda_decode", "gla_fwd", "gla_recurrent",
                       "gla_train", "gla_train", "simple_gla_train", "kda_fwd", "kda_train",
                       "side_train"])
    H = rng.choice([4, 8, 16, 32])
    K, V = rng.choice([(64, 64), (128, 128), (128, 128), (64, 128)])
    c = dict(kind=kind, H=H, K=K, V=V, dtype="bf16")
    if kind == "gla_layer_decode":
        c.update(B=_log_int(rng, 1, 256), H=rng.choice([4, 8, 16]), W=rng.choice([3, 4]))
    elif kind == "gla_decode":
        c.update(B=_log_int(rng, 1, 4096 // H))
    elif kind == "kda_decode":
        c.update(B=_log_int(rng, 1, 2048 // H))
    elif kind == "gla_fwd":
        c["dtype"] = rng.choice(["bf16", "bf16", "f32"])
        T = _log_int(rng, 100, 16384)
        seqs = rng.choice([0, 0, _log_int(rng, 2, 16)])
        B = 1 if seqs else _log_int(rng, 1, max(1, min(16, (1 << 19) // (T * H))))
        c.update(B=B, T=T, seqs=seqs, h0=rng.random() < 0.5)
    elif kind == "gla_recurrent":
        T = _log_int(rng, 100, 8192)
        c.update(B=_log_int(rng, 1, max(1, min(16, (1 << 18) // (T * H)))), T=T,
                 h0=rng.random() < 0.5)
    elif kind == "gla_train":
        c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "f32"])
        T = _log_int(rng, 100, 8192)
        seqs = rng.choice([0, 0, _log_int(rng, 2, 16)])
        B = 1 if seqs else _log_int(rng, 1, max(1, min(8, (1 << 18) // (T * H))))
        if rng.random() < 0.25:       # wide value heads, a batch that fills the card
            K, V, H, seqs = 128, 256, rng.choice([8, 16]), 0
            B = rng.choice([64 // H, 96 // H])
            T = _log_int(rng, 100, 2048)
        c.update(H=H, K=K, V=V, B=B, T=T, seqs=seqs, h0=rng.random() < 0.5)
    elif kind == "simple_gla_train":
        c.update(T=_log_int(rng, 500, 16384), seqs=rng.choice([0, 2, 5, 8, 16]),
                 gate=rng.choice(["token", "token", "head"]))
    elif kind == "kda_fwd":
        T = _log_int(rng, 100, 8192)
        c.update(B=_log_int(rng, 1, max(1, min(4, (1 << 18) // (T * H)))), T=T,
                 raw=rng.random() < 0.5, h0=rng.random() < 0.5)
    elif kind == "kda_train":
        T = _log_int(rng, 100, 8192)
        c.update(B=_log_int(rng, 1, max(1, min(4, (1 << 19) // (T * H)))), T=T,
                 h0=rng.random() < 0.5)
    else:
        T = _log_int(rng, 100, 4096)
        c.pop("K")
        c.update(B=_log_int(rng, 1, 8), T=T, W=rng.choice([3, 4]), H=rng.choice([4, 8, 16]))
    return c


# ---- inputs -------------------------------------------------------------------------------

def _cuts(case, seed):
    """Boundaries of the packed sequences (host ints, as a data loader hands them over)."""
    n = case.get("seqs", 0)
    if not n:
        return None
    T = case["T"]
    rng = random.Random(seed * 1000003 + 17)
    n = min(n, T)
    return [0] + sorted(rng.sample(range(1, T), n - 1)) + [T]


def _make(case, seed):
    """Every input tensor of a case (a dict), on the GPU."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = _DT[case["dtype"]]

    def n(*shape, std=1.0, dtype=torch.float32):
        x = torch.randn(*shape, generator=gen, device=dev)
        return (x * std if std != 1.0 else x).to(dtype)

    def u(*shape):
        return torch.rand(*shape, generator=gen, device=dev)

    kind, H, V = case["kind"], case["H"], case["V"]
    x = {}
    if kind == "side_train":
        B, T, D = case["B"], case["T"], H * V
        x.update(x=n(B, T, D, dtype=dt), dy=n(B, T, D), weight=n(D, 1, case["W"], std=0.5),
                 bias=n(D, std=0.1), o=n(B, T, H, V, dtype=dt), g=n(B, T, H, V, dtype=dt),
                 do=n(B, T, H, V, dtype=dt), nw=1 + n(V, std=0.1))
        return x
    K = case["K"]
    B, T = case.get("B", 1), case.get("T", 1)
    cu = _cuts(case, seed)
    N = B if cu is None else len(cu) - 1
    x["cu"] = cu
    kda = kind.startswith("kda")
    if kda and not case.get("raw"):
        x["q"], x["k"] = (F.normalize(n(B, T, H, K), dim=-1).to(dt) for _ in range(2))
    else:
        x["q"], x["k"] = n(B, T, H, K, dtype=dt), n(B, T, H, K, dtype=dt)
    x["v"] = n(B, T, H, V, dtype=dt)
    if kind == "simple_gla_train":
        if case["gate"] == "token":
            x["g"] = F.logsigmoid(n(B, T, H))
        else:                                     # RetNet's decays, 1 - 2^-5 to 1 - 2^-12
            x["gamma"] = torch.log1p(-torch.exp2(-5 - 7 * torch.arange(H, device=dev) / max(H - 1, 1)))
    elif case.get("raw"):
        # raw gates with A_log, dt_bias as they are initialised (step sizes 1e-3 to 1e-1)
        x["g"] = n(B, T, H, K, std=0.5, dtype=dt)
        x["A_log"] = torch.log(1 + 3 * u(H))
        step = torch.exp(math.log(1e-3) + u(H * K) * math.log(1e2))
        x["dt_bias"] = step + torch.log(-torch.expm1(-step))
    else:
        x["g"] = F.logsigmoid(n(B, T, H, K)) / 16
    if kda:
        x["beta"] = torch.sigmoid(n(B, T, H))
    if case.get("h0") or kind.endswith("decode"):
        x["h0"] = n(N, H, K, V, std=0.1)
    if kind.endswith("train"):
        x["do"] = n(B, T, H, V, dtype=dt)
        if case.get("h0"):
            x["dht"] = n(N, H, K, V, std=0.1)
    if kind == "gla_layer_decode":
        W = case["W"]
        x["conv_w"] = [n(H * d, W, std=0.5) for d in (K, K, V)]
        x["conv_c"] = [n(B, H * d, W) for d in (K, K, V)]
        x["og"], x["nw"] = n(B, T, H, V, dtype=dt), 1 + n(V, std=0.1)
    return x


_LEAVES = {"gla_train": ("q", "k", "v", "g", "h0"), "simple_gla_train": ("q", "k", "v", "g", "h0"),
           "kda_train": ("q", "k", "v", "g", "beta", "h0")}


def prepare(case, seed):
    x = _make(case, seed)
    kind = case["kind"]
    if kind == "side_train":
        from tops.modules import FusedRMSNormGated, ShortConvolution
        D = case["H"] * case["V"]
        conv = ShortConvolution(D, case["W"], bias=True, device="cuda")
        norm = FusedRMSNormGated(case["V"], device="cuda")
        with torch.no_grad():
            conv.weight.copy_(x["weight"])
            conv.bias.copy_(x["bias"])
            norm.weight.copy_(x["nw"])
        for k in ("x", "o", "g"):
            x[k].requires_grad_()
        x["conv"], x["norm"] = conv, norm
    for k in _LEAVES.get(kind, ()):
        if x.get(k) is not None:
            x[k].requires_grad_()
    return case, x


# ---- one pass -----------------------------------------------------------------------------

def run(state):
    case, x = state
    return _RUN[case["kind"]](x)


def _grads(x, names, o, ht):
    leaves = [x[n] for n in names if x.get(n) is not None]
    if x.get("dht") is not None:
        gr = torch.autograd.grad((o, ht), leaves, (x["do"], x["dht"]))
        return (o, ht) + gr
    return (o,) + torch.autograd.grad(o, leaves, x["do"])


def _run_gla_layer_decode(x):
    from tops.ops.gla import fused_recurrent_gla_conv_norm_gate
    with torch.no_grad():
        y, ht, caches = fused_recurrent_gla_conv_norm_gate(
            x["q"], x["k"], x["v"], x["conv_w"], None, x["conv_c"], "silu", x["g"], x["og"],
            x["nw"], initial_state=x["h0"], output_final_state=True)
    return (y, ht) + tuple(caches)


def _run_gla_decode(x):
    from tops.ops.gla import fused_recurrent_gla
    with torch.no_grad():
        return fused_recurrent_gla(x["q"], x["k"], x["v"], x["g"], initial_state=x["h0"],
                                   output_final_state=True)


def _run_kda_decode(x):
    from tops.ops.kda import fused_recurrent_kda
    with torch.no_grad():
        return fused_recurrent_kda(x["q"], x["k"], x["v"], x["g"], x["beta"], None, x["h0"], True)


def _run_gla_fwd(x):
    from tops.ops.gla import chunk_gla
    with torch.no_grad():
        return chunk_gla(x["q"], x["k"], x["v"], x["g"], initial_state=x.get("h0"),
                         output_final_state=True, cu_seqlens=x["cu"])


def _run_gla_recurrent(x):
    from tops.ops.gla import fused_recurrent_gla
    with torch.no_grad():
        return fused_recurrent_gla(x["q"], x["k"], x["v"], x["g"], initial_state=x.get("h0"),
                                   output_final_state=True)


def _run_gla_train(x):
    from tops.ops.gla import chunk_gla
    o, ht = chunk_gla(x["q"], x["k"], x["v"], x["g"], initial_state=x.get("h0"),
                      output_final_state=x.get("dht") is not None, cu_seqlens=x["cu"])
    return _grads(x, _LEAVES["gla_train"], o, ht)


def _run_simple_gla_train(x):
    from tops.ops.simple_gla import chunk_simple_gla
    o, _ = chunk_simple_gla(x["q"], x["k"], x["v"], x.get("gamma"), g=x.get("g"),
                            cu_seqlens=x["cu"])
    return _grads(x, _LEAVES["simple_gla_train"], o, None)


def _run_kda_fwd(x):
    from tops.ops.kda import chunk_kda
    opts = {}
    if "A_log" in x:
        opts = dict(A_log=x["A_log"], dt_bias=x["dt_bias"], use_gate_in_kernel=True,
                    use_qk_l2norm_in_kernel=True)
    with torch.no_grad():
        return chunk_kda(x["q"], x["k"], x["v"], x["g"], x["beta"], initial_state=x.get("h0"),
                         output_final_state=True, **opts)


def _run_kda_train(x):
    from tops.ops.kda import chunk_kda
    o, ht = chunk_kda(x["q"], x["k"], x["v"], x["g"], x["beta"], initial_state=x.get("h0"),
                      output_final_state=x.get("dht") is not None)
    return _grads(x, _LEAVES["kda_train"], o, ht)


def _run_side_train(x):
    conv, norm = x["conv"], x["norm"]
    y, _ = conv(x["x"])
    z = norm(x["o"], x["g"])
    gr = torch.autograd.grad((y, z), (x["x"], conv.weight, conv.bias, x["o"], x["g"], norm.weight),
                             (x["dy"], x["do"]))
    return (y, z) + gr


_RUN = {k[5:]: f for k, f in list(globals().items()) if k.startswith("_run_")}


# ---- what a pass cannot do without --------------------------------------------------------

def work(case):
    """Bytes: every input read once, every output written once.  Operations: the recurrence's
    own (per token and head 4 K V forward, 6 K V with the delta rule; the backward twice the
    forward)."""
    e = 2 if case["dtype"] == "bf16" else 4
    kind, H, V = case["kind"], case["H"], case["V"]
    B, T = case.get("B", 1), case.get("T", 1)
    R = B * T * H
    if kind == "side_train":
        # conv: x in, y out fp32; x, dy in, dx out.  norm: o, g in, z out; o, g, dz in, do, dg out
        conv = R * V * (e + 4) + R * V * (e + 4 + e)
        norm = R * V * 3 * e + R * V * 5 * e
        return {"bytes": conv + norm, "flops": R * V * (6 * case["W"] + 60)}
    K = case["K"]
    N = case["seqs"] if case.get("seqs") else B
    S = N * H * K * V * 4
    gate = {"token": 4, "head": 0}.get(case.get("gate"), (e if case.get("raw") else 4) * K)
    kda = kind.startswith("kda")
    ins = (2 * K + V) * e + gate + (4 if kda else 0)
    per_flops = (6 if kda else 4) * K * V
    if kind.endswith("train"):
        h = S if case.get("h0") else 0
        fwd = R * (ins + V * e) + 2 * h
        bwd = R * (ins + V * e) + R * ins + 2 * h
        return {"bytes": fwd + bwd, "flops": 3 * R * per_flops}
    h_in = S if (case.get("h0") or kind.endswith("decode")) else 0
    b = R * (ins + V * e) + h_in + S
    if kind == "gla_layer_decode":
        C = H * (2 * K + V)
        b += C * case["W"] * 4 + 2 * B * C * case["W"] * 4 + R * V * (e + 2)
    return {"bytes": b, "flops": R * per_flops}


def tolerance(case):
    """bf16 outputs: their own rounding, 1.7e-3 of the result against float64.  fp32 inputs run
    on bf16 hi + lo halves (the lo * lo term is left out, 6e-6).  The fused decode route keeps
    fp32 throughout (2e-7)."""
    if case["kind"] == "gla_layer_decode":
        return {"rel": 2e-6}
    if case["dtype"] == "f32":
        return {"rel": 4e-5}
    return {"rel": 7e-3}


# ---- float64 ------------------------------------------------------------------------------

_C = 64


def _d(t):
    return None if t is None else t.detach().double()


def _chunked(x, C=_C):
    """[B,T,H,D] -> [B,H,chunks,C,D], the end padded with zeros."""
    B, T, H, D = x.shape
    n = -(-T // C)
    x = F.pad(x, (0, 0, 0, 0, 0, n * C - T))
    return x.reshape(B, n, C, H, D).permute(0, 3, 1, 2, 4).contiguous()


def _flat(x, T):
    B, H, n, C, D = x.shape
    return x.permute(0, 2, 3, 1, 4).reshape(B, n * C, H, D)[:, :T]


def _gla64(q, k, v, g, h0, scale, beta=None):
    """The chunked recurrence of one batch of equally long sequences; with beta the delta rule.
    A zero token with a zero gate leaves the state as it is, so padding is harmless."""
    T = q.shape[1]
    q, k, v, G = _chunked(q * scale), _chunked(k), _chunked(v), _chunked(g).cumsum(-2)
    B, H, n, C, K = q.shape
    V = v.shape[-1]
    qg, kg = q * G.exp(), k * (-G).exp()
    A = torch.matmul(qg, kg.transpose(-1, -2).contiguous()).tril()
    if beta is not None:
        b = _chunked(beta[..., None])
        kb = k * G.exp()
        L = (torch.matmul(kb, kg.transpose(-1, -2).contiguous()) * b).tril(-1)
        eye = torch.eye(C, device=q.device, dtype=q.dtype)
        inv, P = eye - L, torch.matmul(L, L)          # (I + L)^-1, L nilpotent
        for i in range(5):
            inv = inv + torch.matmul(inv, P)
            P = torch.matmul(P, P) if i < 4 else P
        v, w = torch.matmul(inv, b * v), torch.matmul(inv, b * kb)
    end = G[..., -1, :].exp()
    S = torch.zeros(B, H, K, V, device=q.device, dtype=q.dtype) if h0 is None else h0
    kgT = kg.transpose(-1, -2).contiguous()
    os_ = []
    for c in range(n):
        vc = v[:, :, c]
        if beta is not None:
            vc = vc - torch.matmul(w[:, :, c], S)
        os_.append(torch.matmul(A[:, :, c], vc) + torch.matmul(qg[:, :, c], S))
        S = end[:, :, c, :, None] * (S + torch.matmul(kgT[:, :, c], vc))
    return _flat(torch.stack(os_, 2), T), S


def _seqs64(q, k, v, g, h0, scale, cu, beta=None):
    if cu is None:
        return _gla64(q, k, v, g, h0, scale, beta)
    os_, hs = [], []
    for i, (a, b) in enumerate(zip(cu[:-1], cu[1:])):
        o, h = _gla64(q[:, a:b], k[:, a:b], v[:, a:b], g[:, a:b],
                      None if h0 is None else h0[i:i + 1], scale,
                      None if beta is None else beta[:, a:b])
        os_.append(o)
        hs.append(h)
    return torch.cat(os_, 1), torch.cat(hs, 0)


def _rms64(o, g, w, eps=1e-5):
    return o * torch.rsqrt((o * o).mean(-1, keepdim=True) + eps) * w * F.silu(g)


def exact(case, seed):
    x = _make(case, seed)
    kind = case["kind"]
    if kind == "side_train":
        names = ("x", "weight", "bias", "o", "g", "nw")
        lv = {n: _d(x[n]).requires_grad_() for n in names}
        W, T = case["W"], case["T"]
        pre = lv["bias"]
        xp = F.pad(lv["x"], (0, 0, W - 1, 0))
        for j in range(W):
            pre = pre + xp[:, j:j + T] * lv["weight"][:, 0, j]
        y, z = F.silu(pre), _rms64(lv["o"], lv["g"], lv["nw"])
        gr = torch.autograd.grad((y, z), [lv[n] for n in names], (_d(x["dy"]), _d(x["do"])))
        return (y.detach(), z.detach()) + gr
    scale, cu = case["K"] ** -0.5, x["cu"]
    if kind == "gla_layer_decode":
        B, H = case["B"], case["H"]
        qkv, caches = [], []
        for t, w, c in zip((x["q"], x["k"], x["v"]), x["conv_w"], x["conv_c"]):
            c = torch.cat([_d(c)[..., 1:], _d(t).reshape(B, -1, 1)], -1)
            caches.append(c)
            qkv.append(F.silu((c * _d(w)).sum(-1)).reshape(B, 1, H, -1))
        o, ht = _gla64(*qkv, _d(x["g"]), _d(x["h0"]), scale)
        return (_rms64(o, _d(x["og"]), _d(x["nw"])), ht) + tuple(caches)
    train = kind.endswith("train")
    lv = {n: _d(x[n]) for n in ("q", "k", "v", "g", "beta", "h0") if x.get(n) is not None}
    if train:
        for t in lv.values():
            t.requires_grad_()
    q, k, v, g = lv["q"], lv["k"], lv["v"], lv.get("g")
    if kind == "simple_gla_train":
        g = _d(x["gamma"]).expand(q.shape[:3]) if g is None else g
        g = g[..., None].expand(q.shape)
    if case.get("raw"):
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        H, K = q.shape[2:]
        g = -_d(x["A_log"]).exp()[:, None] * F.softplus(g + _d(x["dt_bias"]).reshape(H, K))
    with torch.set_grad_enabled(train):
        o, ht = _seqs64(q, k, v, g, lv.get("h0"), scale, cu, lv.get("beta"))
    if not train:
        return o, ht
    leaves = [lv[n] for n in _LEAVES[kind] if n in lv]
    if x.get("dht") is not None:
        gr = torch.autograd.grad((o, ht), leaves, (_d(x["do"]), _d(x["dht"])))
        return (o.detach(), ht.detach()) + gr
    return (o.detach(),) + torch.autograd.grad(o, leaves, _d(x["do"]))
