"""The strip-specialised chunk sweep (gla_strip.hip) against the serial sweep
(gla_sweep.hip) and the float64 oracle.

bf16 chunk_gla calls with per-channel gates run on the strip kernel; TOPS_SWEEP_SERIAL=1 routes
the same calls to the serial kernel.  Both split every operand into the same bf16 hi + lo halves,
but they do not do the same arithmetic: the strip kernel decays the state as e (e S + Z~^T Y)
with e = 2^Gm, the serial one as 2^Gamma S + 2^(Gamma - Gm) Z~^T Y, the gate sums run over other
row segments, and the scale is applied elsewhere.  Each case runs forward + backward
(tops/ops/gla/chunk.py:1103-1199 and :1447-1509) under both schedules and checks
  * every output against the oracle at 2e-3 for bf16 (for tiny tensors the rounding floor of
    _gpu.out_bound), and
  * the two schedules against each other.  fp32 outputs (ht, dg, dh0): each is within 2.4e-6 to
    3.3e-6 of float64 (the 2^-17 of a hi + lo operand, and the gate sums), two independent
    errors differ by at most about 5e-6: 1e-5.  bf16 outputs (o, dq, dk, dv): an fp32 value that
    differs by 5e-6 rounds to the neighbouring bf16 value (2^-8 apart, mean step 5.6e-3) in one
    case of a thousand, sqrt(1e-3) 5.6e-3 = 1.8e-4 of the norm (1.0e-4 to 1.7e-4 measured): 1e-3.
Cases cover K of 32 / 64 / 128 (the kernel's three row splits), ragged T, varlen with
one-token sequences, h0 / dht, and the fp32 and paired checkpoint layouts (empty sequences:
the oracle rejects them, as tops/cpu does; other modules run them).  The default layout keeps
fp16 checkpoints, which only the strip kernel writes: test_gpu_ckpt16.py covers it.
"""
import os

import numpy as np
import pytest
import torch

from oracle import gla as O
from _inputs import gla_inputs
from _gpu import to_dev, seen, host, rel, out_bound

pytestmark = pytest.mark.gpu

CASES = [
    dict(B=2, T=300, H=3, K=128, V=128, seed=11, h0=True),
    dict(B=1, T=513, H=2, K=64, V=64, seed=12, h0=True),
    dict(B=2, T=200, H=2, K=32, V=96, seed=13),
    dict(B=1, T=700, H=2, K=128, V=64, seed=14, cu=[0, 1, 129, 130, 700], h0=True),
    dict(B=1, T=1000, H=4, K=128, V=128, seed=15, cu=[0, 1, 64, 65, 300, 1000], h0=True),
    dict(B=1, T=64, H=2, K=128, V=128, seed=16, h0=True),
    dict(B=1, T=1, H=2, K=128, V=128, seed=17, h0=True),
]


def _id(c):
    return "-".join(f"{k}{v}" for k, v in c.items() if k != "seed")


def _run(cfg, device, serial, layout="full32"):
    from tops.ops.gla import chunk_gla
    from tops.utils import set_checkpoint_layout, checkpoint_layout
    B, T, H, K, V = (cfg[x] for x in "BTHKV")
    cu = cfg.get("cu")
    n = len(cu) - 1 if cu else B
    d = gla_inputs(B, T, H, K, V, cfg["seed"], gate_div=16.0, h0=cfg.get("h0", False), N=n,
                   grads=True)
    bf = torch.bfloat16
    q, k, v = (to_dev(d[x], bf, device).requires_grad_() for x in "qkv")
    g = to_dev(d["g"], torch.float32, device).requires_grad_()
    h0 = to_dev(d["h0"], torch.float32, device)
    if h0 is not None:
        h0.requires_grad_()
    prev_env = os.environ.get("TOPS_SWEEP_SERIAL")
    prev_layout = checkpoint_layout()
    os.environ["TOPS_SWEEP_SERIAL"] = "1" if serial else "0"
    set_checkpoint_layout(layout)
    try:
        o, ht = chunk_gla(q, k, v, g, initial_state=h0, output_final_state=True,
                          cu_seqlens=cu)
        do = to_dev(d["do"], bf, device)
        dht = to_dev(d["dht"], torch.float32, device)
        torch.autograd.backward((o, ht), (do, dht))
        torch.cuda.synchronize()
    finally:
        set_checkpoint_layout(prev_layout)
        if prev_env is None:
            os.environ.pop("TOPS_SWEEP_SERIAL", None)
        else:
            os.environ["TOPS_SWEEP_SERIAL"] = prev_env
    out = dict(o=o, ht=ht, dq=q.grad, dk=k.grad, dv=v.grad, dg=g.grad,
               dh0=None if h0 is None else h0.grad)
    return d, out


@pytest.mark.parametrize("layout", ["full32", "paired"])
@pytest.mark.parametrize("cfg", CASES, ids=_id)
def test_pipe_vs_serial_and_oracle(cfg, layout, cuda_device):
    print(f"case {_id(cfg)} layout={layout}", flush=True)
    d, a = _run(cfg, cuda_device, serial=False, layout=layout)
    _, b = _run(cfg, cuda_device, serial=True, layout=layout)
    bf = torch.bfloat16
    s = {x: seen(d[x], bf) for x in ("q", "k", "v", "do")}
    K = cfg["K"]
    ro, rht = O.chunk_gla(s["q"], s["k"], s["v"], d["g"], initial_state=d.get("h0"),
                          output_final_state=True, chunk_size=64, cu_seqlens=cfg.get("cu"))
    rq, rk, rv, rg, rh0 = O.chunk_gla_bwd(s["q"], s["k"], s["v"], d["g"], K ** -0.5,
                                          d.get("h0"), s["do"], d["dht"], chunk_size=64,
                                          cu_seqlens=cfg.get("cu"))
    ref = dict(o=ro, ht=rht, dq=rq, dk=rk, dv=rv, dg=rg, dh0=rh0)
    for name, r in ref.items():
        if a[name] is None:
            continue
        x, y = host(a[name]), host(b[name])
        stored = a[name].dtype
        e = rel(x, r)
        bound = out_bound(r, bf, stored)
        assert e < bound, f"{name}: strip rel-err {e:.3e} vs oracle (bound {bound:.2e})"
        lim = 1e-3 if stored == bf else 1e-5
        ab = rel(x, y)
        assert ab <= lim, f"{name}: strip vs serial rel {ab:.3e} > {lim}"


@pytest.mark.parametrize("dt", [torch.float32, torch.float16], ids=["f32", "f16"])
def test_other_types_have_one_sweep(dt, cuda_device, monkeypatch):
    """fp32 and fp16 calls run on the strip kernel whatever TOPS_SWEEP_SERIAL says (the serial
    kernel has no per-channel-gate forward for them): the same bits either way."""
    from tops.ops.gla import chunk_gla
    d = gla_inputs(2, 200, 2, 64, 72, 5, gate_div=16.0, h0=True, grads=True)
    res = []
    for serial in ("0", "1"):
        monkeypatch.setenv("TOPS_SWEEP_SERIAL", serial)
        x = [to_dev(d[n], dt, cuda_device).requires_grad_() for n in "qkv"]
        x += [to_dev(d[n], torch.float32, cuda_device).requires_grad_() for n in ("g", "h0")]
        print(f"one sweep {dt} serial={serial}", flush=True)
        o, ht = chunk_gla(*x[:4], initial_state=x[4], output_final_state=True)
        gr = torch.autograd.grad((o, ht), x, (to_dev(d["do"], dt, cuda_device),
                                              to_dev(d["dht"], torch.float32, cuda_device)))
        res.append([o, ht, *gr])
    for a, b in zip(*res):
        assert torch.equal(a, b)
