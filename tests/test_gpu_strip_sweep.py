"""The strip-specialised chunk sweep (gla_strip.hip) at the edges of its tiles: channel blocks
of 32 with their remainders, 64-column value tiles with theirs, sequence lengths around one
and two 64-token chunks, both directions, against the float64 oracle
(tops/cpu/ops/gla/chunk.py:310-427, 551-607).  Tolerances: bf16 outputs 2e-3 (their own
rounding is 1.65e-3; tiny tensors as _gpu.out_bound), fp32 1e-4: every operand is a bf16 hi +
lo pair, whose dropped lo * lo term is 2^-16 relative per product.
"""
import pytest
import torch

from oracle import gla as O
from _inputs import gla_inputs
from _gpu import to_dev, seen, host, rel, out_bound

pytestmark = pytest.mark.gpu

CASES = [(T, K, V, dt) for dt in ("bf16", "f32")
         for T, K, V in ((1, 8, 8), (63, 40, 56), (64, 32, 64), (65, 64, 72), (127, 72, 128),
                         (128, 128, 120), (129, 104, 8), (200, 128, 128))]


@pytest.mark.parametrize("T,K,V,dt", CASES, ids=lambda x: str(x))
def test_strip_sweep_tile_edges(T, K, V, dt, cuda_device):
    from tops.ops.gla import chunk_gla
    dtype = {"bf16": torch.bfloat16, "f32": torch.float32}[dt]
    B, H = 2, 2
    d = gla_inputs(B, T, H, K, V, 900 + T, gate_div=4.0, h0=True, grads=True)
    x = {n: to_dev(d[n], dtype, cuda_device).requires_grad_() for n in "qkv"}
    x |= {n: to_dev(d[n], torch.float32, cuda_device).requires_grad_() for n in ("g", "h0")}
    print(f"strip sweep T={T} K={K} V={V} {dt}", flush=True)
    o, ht = chunk_gla(x["q"], x["k"], x["v"], x["g"], initial_state=x["h0"],
                      output_final_state=True)
    torch.autograd.backward((o, ht), (to_dev(d["do"], dtype, cuda_device),
                                      to_dev(d["dht"], torch.float32, cuda_device)))
    s = {n: seen(d[n], dtype) for n in ("q", "k", "v", "do")}
    ref = dict(zip(("o", "ht"), O.chunk_gla(s["q"], s["k"], s["v"], d["g"], initial_state=d["h0"],
                                            output_final_state=True, chunk_size=64)))
    ref |= dict(zip(("q", "k", "v", "g", "h0"),
                    O.chunk_gla_bwd(s["q"], s["k"], s["v"], d["g"], K ** -0.5, d["h0"], s["do"],
                                    d["dht"], chunk_size=64)))
    got = dict(o=o, ht=ht) | {n: t.grad for n, t in x.items()}
    with torch.no_grad():                      # the instance without checkpoints
        oi, hi = chunk_gla(*(x[n] for n in "qkvg"), initial_state=x["h0"], output_final_state=True)
    for n, a, r in [(n, got[n], ref[n]) for n in ref] + [("o inf", oi, ref["o"]), ("ht inf", hi, ref["ht"])]:
        e, lim = rel(host(a), r), out_bound(r, dtype, a.dtype)
        assert e < lim, f"{n}: rel-err {e:.3e} vs oracle (bound {lim:.2e})"
