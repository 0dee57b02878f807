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
# more than 128 value columns: fp32 checkpoints, of every chunk
CASES += [(T, K, V, dt) for dt in ("bf16", "f32")
          for T, K, V in ((65, 40, 144), (129, 128, 208), (200, 72, 256))]


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


KDA_CASES = [(T, K, V, dt) for dt in ("bf16", "f32")
             for T, K, V in ((1, 8, 8), (63, 40, 56), (65, 64, 72), (128, 72, 128),
                             (129, 128, 120), (200, 128, 64))]


@pytest.mark.parametrize("T,K,V,dt", KDA_CASES, ids=lambda x: str(x))
def test_strip_sweep_delta_rule_tile_edges(T, K, V, dt, cuda_device):
    """The delta-rule instances, forward (with checkpoints and without) and reverse, against
    the oracle (tops/cpu/ops/kda/naive.py:121-313, chunk_bwd.py:525-668); gate gradients
    against the scale of the k * dk terms they are differences of."""
    import numpy as np
    from oracle import kda as OK
    from _inputs import kda_inputs
    from tops.ops.kda import chunk_kda
    dtype = {"bf16": torch.bfloat16, "f32": torch.float32}[dt]
    B, H = 2, 2
    d = kda_inputs(B, T, H, K, V, 700 + T, gate_div=4.0, h0=True, grads=True)
    x = {n: to_dev(d[n], dtype, cuda_device).requires_grad_() for n in "qkv"}
    x |= {n: to_dev(d[n], torch.float32, cuda_device).requires_grad_() for n in ("g", "beta", "h0")}
    print(f"delta-rule strip sweep T={T} K={K} V={V} {dt}", flush=True)
    sc = K ** -0.5
    o, ht = chunk_kda(*(x[n] for n in ("q", "k", "v", "g", "beta")), scale=sc,
                      initial_state=x["h0"], output_final_state=True)
    torch.autograd.backward((o, ht), (to_dev(d["do"], dtype, cuda_device),
                                      to_dev(d["dht"], torch.float32, cuda_device)))
    with torch.no_grad():
        oi, hi = chunk_kda(*(x[n] for n in ("q", "k", "v", "g", "beta")), scale=sc,
                           initial_state=x["h0"], output_final_state=True)
    s = {n: seen(d[n], dtype) for n in ("q", "k", "v", "do")}
    a = (s["q"], s["k"], s["v"], np.float64(d["g"]), np.float64(d["beta"]))
    ro, rht = OK.chunk_kda(*a, sc, np.float64(d["h0"]), True)
    rq, rk, rv, rb, rg, rh0 = OK.chunk_kda_bwd(*a, sc, np.float64(d["h0"]), s["do"], np.float64(d["dht"]))
    pairs = [("o", o, ro), ("ht", ht, rht), ("o inf", oi, ro), ("ht inf", hi, rht),
             ("dq", x["q"].grad, rq), ("dk", x["k"].grad, rk), ("dv", x["v"].grad, rv),
             ("dbeta", x["beta"].grad, rb), ("dg", x["g"].grad, rg), ("dh0", x["h0"].grad, rh0)]
    for n, got, ref in pairs:
        ref = np.asarray(ref)
        err = np.linalg.norm(host(got) - ref)
        base = np.linalg.norm(s["k"] * rk) if n == "dg" else np.linalg.norm(ref)
        lim = out_bound(ref, dtype, torch.bfloat16 if n == "dg" and dt == "bf16" else got.dtype)
        assert err <= lim * max(base, np.linalg.norm(ref)), f"{n}: rel-err {err / base:.3e} (bound {lim:.2e})"


SIMPLE_CASES = [(T, K, V, gate) for gate in ("token", "head")
                for T, K, V in ((1, 8, 8), (63, 40, 56), (64, 32, 64), (65, 64, 72),
                                (127, 72, 128), (129, 104, 8), (200, 128, 128))]


@pytest.mark.parametrize("T,K,V,gate", SIMPLE_CASES, ids=lambda x: str(x))
def test_strip_sweep_token_gate_tile_edges(T, K, V, gate, cuda_device):
    """One gate per token, or a constant per head (bf16), against the oracle
    (tops/cpu/ops/simple_gla/chunk.py:53-129, 668-788), with checkpoints and without."""
    import numpy as np
    from _inputs import simple_gla_inputs
    from tops.ops.simple_gla import chunk_simple_gla
    bf, f32 = torch.bfloat16, torch.float32
    B, H = 2, 3
    d = simple_gla_inputs(B, T, H, K, V, 500 + T, h0=True, grads=True)
    x = {n: to_dev(d[n], bf, cuda_device).requires_grad_() for n in "qkv"}
    x["h0"] = to_dev(d["h0"], f32, cuda_device).requires_grad_()
    g = to_dev(d["g"], f32, cuda_device).requires_grad_()
    gam = to_dev(d["g_gamma"], f32, cuda_device)
    kw = dict(g=g) if gate == "token" else dict(g_gamma=gam)
    print(f"token-gate strip sweep T={T} K={K} V={V} {gate}", flush=True)

    def call():
        return chunk_simple_gla(x["q"], x["k"], x["v"], initial_state=x["h0"],
                                output_final_state=True, **kw)
    o, ht = call()
    torch.autograd.backward((o, ht), (to_dev(d["do"], bf, cuda_device),
                                      to_dev(d["dht"], f32, cuda_device)))
    with torch.no_grad():
        oi, hi = call()
    # the oracle of per-channel gates on the broadcast gate
    gfull = d["g"] if gate == "token" else np.broadcast_to(d["g_gamma"], d["g"].shape)
    gk = np.ascontiguousarray(np.broadcast_to(gfull[..., None], gfull.shape + (K,)))
    s = {n: seen(d[n], bf) for n in ("q", "k", "v", "do")}
    ro, rht = O.chunk_gla(s["q"], s["k"], s["v"], gk, initial_state=d["h0"],
                          output_final_state=True, chunk_size=64)
    rq, rk, rv, rg, rh0 = O.chunk_gla_bwd(s["q"], s["k"], s["v"], gk, K ** -0.5, d["h0"], s["do"],
                                          d["dht"], chunk_size=64)
    pairs = [("o", o, ro), ("ht", ht, rht), ("o inf", oi, ro), ("ht inf", hi, rht),
             ("dq", x["q"].grad, rq), ("dk", x["k"].grad, rk), ("dv", x["v"].grad, rv),
             ("dh0", x["h0"].grad, rh0)]
    for n, got, ref in pairs:
        e, lim = rel(host(got), ref), out_bound(ref, bf, got.dtype)
        assert e < lim, f"{n}: rel-err {e:.3e} vs oracle (bound {lim:.2e})"
    if gate == "token":
        # the sum of K per-channel gradients, each a difference of q dq and k dk terms
        err = np.linalg.norm(host(g.grad) - rg.sum(-1))
        scale = np.linalg.norm((np.abs(s["q"] * rq) + np.abs(s["k"] * rk)).sum(-1))
        assert err <= 1e-3 * scale, f"dg: {err / scale:.3e} of its terms"


# (B, H, K, V, dtype, packed boundaries), the tile the call takes, the factor of the heads whose
# call takes the tile after it (on 256 CUs)
NARROW = [((1, 2, 64, 128, "bf16", None), 16, (20, 32)), ((1, 2, 64, 8, "f32", None), 16, (65, 64)),
          ((1, 20, 64, 128, "bf16", None), 16, (2, 32)), ((1, 40, 64, 72, "f32", None), 16, (2, 64)),
          ((2, 33, 64, 128, "bf16", None), 64, None),
          ((2, 17, 128, 128, "bf16", None), 32, (2, 64)), ((2, 32, 32, 128, "f32", None), 32, (2, 64)),
          ((1, 65, 64, 64, "bf16", None), 32, (2, 64)), ((1, 40, 128, 120, "f32", None), 32, (2, 64)),
          ((1, 40, 32, 104, "bf16", None), 32, (2, 64)),
          ((1, 12, 64, 128, "bf16", [0, 1, 65, 130]), 32, (2, 64)),
          ((1, 12, 128, 72, "f32", [0, 64, 127, 130]), 16, (2, 64))]


@pytest.mark.parametrize("shape,bv,wider", NARROW, ids=lambda x: str(x))
def test_strip_sweep_delta_rule_narrow_tiles(shape, bv, wider, cuda_device):
    """The forward delta rule without checkpoints takes 16- or 32-column tiles while their
    workgroups are one round on the chip.  Every width, at the edges of the rule and with channel
    and value remainders, within the bounds of the oracle, and the same up to fp32 rounding as
    those heads in a call of more, which takes the next tile.  The widths are those of the
    launcher's rule, restated in addr_model.delta_tile."""
    import numpy as np
    from addr_model import delta_tile
    from oracle import kda as OK
    from _inputs import kda_inputs
    from tops.ops.kda import chunk_kda
    B, H, K, V, dt, cu = shape
    N = len(cu) - 1 if cu else B
    cus = torch.cuda.get_device_properties(cuda_device).multi_processor_count
    if cus == 256:
        assert delta_tile(H, N, V, False) == bv
        assert wider is None or delta_tile(H * wider[0], N, V, False) == wider[1]
    dtype = {"bf16": torch.bfloat16, "f32": torch.float32}[dt]
    T = 130
    d = kda_inputs(B, T, H, K, V, 40 + H, gate_div=4.0, h0=True, N=N)
    x = [to_dev(d[n], dtype, cuda_device) for n in "qkv"] + \
        [to_dev(d[n], torch.float32, cuda_device) for n in ("g", "beta")]
    h0 = to_dev(d["h0"], torch.float32, cuda_device)
    print(f"narrow tiles {shape} bv={bv}", flush=True)
    o, ht = chunk_kda(*x, initial_state=h0, output_final_state=True, cu_seqlens=cu)
    ins = [seen(d[n], dtype) for n in "qkv"] + [np.float64(d[n]) for n in ("g", "beta")]
    h64 = np.float64(d["h0"])
    if cu is None:
        ro, rht = OK.chunk_kda(*ins, K ** -0.5, h64, True)
    else:                                      # the oracle takes one sequence length
        parts = [OK.chunk_kda(*(t[:, lo:hi] for t in ins), K ** -0.5, h64[n:n + 1], True)
                 for n, (lo, hi) in enumerate(zip(cu, cu[1:]))]
        ro, rht = (np.concatenate(t, axis) for t, axis in zip(zip(*parts), (1, 0)))
    for n, got, ref in (("o", o, ro), ("ht", ht, rht)):
        e, lim = rel(host(got), ref), out_bound(ref, dtype, got.dtype)
        assert e < lim, f"{n}: rel-err {e:.3e} vs oracle (bound {lim:.2e})"
    if wider is None:
        return
    rep = [torch.cat([t] * wider[0], 2).contiguous() for t in x]
    ow, htw = chunk_kda(*rep, initial_state=torch.cat([h0] * wider[0], 1), output_final_state=True,
                        cu_seqlens=cu)
    # fp32 sums in the same order: the last bit of a state, one ulp of a rounded output
    assert rel(host(ow[:, :, :H]), host(o)) <= 1e-3 and rel(host(htw[:, :H]), host(ht)) <= 1e-5


def test_strip_sweep_gate_sum_precision(cuda_device):
    """Strong gates: the in-chunk gate sums reach 150 (log2 units), and the rounding of the sums
    shows in the final state beside the 2.4e-6 of the bf16 hi + lo operands.  Summed in log2
    units, as kda_prep and dq/dk/dg sum them, the state is 4.06e-6 off float64; summed in
    natural units and scaled afterwards (a rounding more per row and per total) 4.79e-6."""
    from tops.ops.gla import chunk_gla
    B, T, H, K = 4, 300, 32, 64
    gen = torch.Generator().manual_seed(77)
    q, k, v = (torch.randn(B, T, H, K, generator=gen).to(cuda_device, torch.bfloat16) for _ in range(3))
    g = -2 * torch.nn.functional.softplus(torch.randn(B, T, H, K, generator=gen)).to(cuda_device)
    h0 = torch.randn(B, H, K, K, generator=gen).to(cuda_device)
    print("gate sum precision", flush=True)
    _, ht = chunk_gla(q, k, v, g, initial_state=h0, output_final_state=True)
    S = h0.double()
    for t in range(T):
        S = S * g[:, t].double().exp()[..., None] + k[:, t].double()[..., None] * v[:, t].double()[..., None, :]
    err = float((ht.double() - S).norm() / S.norm())
    print(f"ht error {err:.3e}", flush=True)
    assert err < 4.35e-6, f"ht: {err:.3e} of float64"
