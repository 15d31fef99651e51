"""Products on operands as stored, on the hand-ordered tiles: row blocks of 256 and their remainders, of 128, ragged columns and odd slab
counts, an expert without rows; the same bits as with a transposed copy of the weight.  (The fourth and fifth shape take 256-row blocks for one of the two gradients: grouped_kn_large.)"""
import dataclasses

import numpy as np
import pytest

from oracle import binding as ob
from helpers import product_config, to_device
from test_gpu_backward import KIND, moe, routed_case  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [ob.BF16, ob.F16])
@pytest.mark.parametrize("shape", [(1, 64, 64, 2, 1), (520, 576, 320, 2, 1), (1100, 2112, 448, 2, 2), (1900, 2112, 1088, 8, 2), (2000, 1152, 2112, 8, 2), (400, 320, 1088, 70, 2)])
@pytest.mark.parametrize("gated", [False, True])
def test_data_gradients_on_weights_as_stored(moe, dtype, shape, gated):
    import torch
    import cuplayground_amd.api as api
    S, H, I, E, k = shape
    cfg, rng, count, offset = routed_case(S, H, I, E, k, dtype, seed=S, drop=0, skew=0.3)
    if gated:
        cfg = dataclasses.replace(cfg, act=ob.ACT_SWIGLU)
    R = int(count.sum())
    layer = moe.MoELayer(product_config(cfg))
    assert layer.gemm_kn_supported(H, I) == 2 and layer.gemm_kn_supported(I, H) == 2
    dev = lambda *s: to_device(ob.from_f32((rng.standard_normal(s) * 0.3).astype(np.float32), dtype), KIND[dtype])
    dcount, doff = to_device(count, "i32"), to_device(offset, "i32")
    rows = {n: dev(S * k, n) for n in (H, I)}
    u, g = dev(S * k, I), dev(S * k, I)
    for t in (rows[H], rows[I]):
        t[R:] = float("nan")                     # rows of no expert must not reach a result
    w_up, w_down = dev(E, I, H), dev(E, H, I)
    da = layer.expert_gemm_kn(rows[I], w_up, dcount, doff)
    assert torch.equal(da[:R], layer.expert_gemm(rows[I], api.transpose(w_up), None, dcount, doff, api.ACT_NONE)[:R])
    dh = layer.expert_gemm(rows[H], api.transpose(w_down), None, dcount, doff, api.ACT_NONE)
    want = layer.act_backward(dh, u, g if gated else None)
    du, dg = layer.expert_gemm_kn(rows[H], w_down, dcount, doff, u, g if gated else None)
    assert torch.equal(du[:R], want[0][:R]) and (not gated or torch.equal(dg[:R], want[1][:R]))
    # results in the place of the saved projections, as a caller short of memory may have them
    out = [u.clone(), g.clone()]
    rc = layer.L.moe_expert_gemm_kn(layer._h, api._ptr(rows[H]), api._ptr(w_down), api._ptr(out[0]), api._ptr(out[1] if gated else None), api._ptr(dcount),
                                    api._ptr(doff), I, H, api._ptr(out[0]), api._ptr(out[1] if gated else None), api._stream())
    assert rc == 0 and torch.equal(out[0][:R], want[0][:R]) and (not gated or torch.equal(out[1][:R], want[1][:R]))
    assert torch.equal(out[0][R:], u[R:])        # rows of no expert stay as they are


@pytest.mark.parametrize("dtype", [ob.BF16, ob.F16])
@pytest.mark.parametrize("shape", [(750, 2560, 1088, 5, 2), (2304, 2048, 1024, 24, 2), (700, 1152, 1920, 16, 4)])
def test_weight_gradients_on_rows_as_stored(moe, dtype, shape):
    """Workgroups with a tile each, with several in a row (and a ragged last round), and the 128 x 128 tiles (wgrad_large), experts
    without rows and with odd slab counts: the bits that the transposed copies give."""
    import torch
    S, H, I, E, k = shape
    cfg, rng, count, offset = routed_case(S, H, I, E, k, dtype, seed=S, drop=0, skew=0.2)
    count[1] += count[0]                         # an expert without rows
    offset[1], count[0] = offset[0], 0
    R = int(count.sum())
    layer, copies = moe.MoELayer(product_config(cfg)), moe.MoELayer(product_config(cfg), options={"grouped_tile": 1})
    dev = lambda *s: to_device(ob.from_f32(rng.standard_normal(s).astype(np.float32), dtype), KIND[dtype])
    dcount, doff = to_device(count, "i32"), to_device(offset, "i32")
    a, b = dev(S * k, H), dev(S * k, I)
    a[R:] = b[R:] = float("nan")
    for x, y in ((a, b), (b, a)):
        got, want = layer.expert_wgrad(x, y, dcount, doff), copies.expert_wgrad(x, y, dcount, doff)
        assert torch.equal(got, want) and not got[0].any() and got[-1].any()


@pytest.mark.parametrize("dtype", [ob.BF16, ob.F16])
@pytest.mark.parametrize("shape", [(1, 64, 64, 2, 1), (520, 576, 320, 2, 1), (1100, 2112, 448, 2, 2), (1900, 2112, 1088, 8, 2), (400, 320, 1088, 70, 2)])
def test_two_products_in_one_launch(moe, dtype, shape):
    """A SwiGLU layer's two projections of the same rows, and their data gradients: the bits of a launch each; also where an option asks
    for the 128 x 128 tile, which takes two."""
    import torch
    import cuplayground_amd.api as api
    S, H, I, E, k = shape
    cfg, rng, count, offset = routed_case(S, H, I, E, k, dtype, seed=S, drop=0, skew=0.3)
    cfg = dataclasses.replace(cfg, act=ob.ACT_SWIGLU)
    R = int(count.sum())
    layer, plain = moe.MoELayer(product_config(cfg)), moe.MoELayer(product_config(cfg), options={"grouped_tile": 0})
    dev = lambda *s: to_device(ob.from_f32((rng.standard_normal(s) * 0.3).astype(np.float32), dtype), KIND[dtype])
    dcount, doff = to_device(count, "i32"), to_device(offset, "i32")
    x, du, dg, w_up, w_gate = dev(S * k, H), dev(S * k, I), dev(S * k, I), dev(E, I, H), dev(E, I, H)
    for t in (x, du, dg):
        t[R:] = float("nan")
    for l in (layer, plain):
        for got, w in zip(l.expert_gemm_pair(x, w_up, w_gate, dcount, doff), (w_up, w_gate)):
            assert torch.equal(got[:R], l.expert_gemm(x, w, None, dcount, doff, api.ACT_NONE)[:R])
    for got, d, w in zip(layer.expert_gemm_kn_pair(du, dg, w_up, w_gate, dcount, doff), (du, dg), (w_up, w_gate)):
        assert torch.equal(got[:R], layer.expert_gemm_kn(d, w, dcount, doff)[:R])


@pytest.mark.parametrize("dtype", [ob.F32, ob.BF16, ob.F16])
@pytest.mark.parametrize("shape", [(1, 64, 64, 2, 1), (750, 2560, 1088, 5, 2), (2304, 2048, 1024, 24, 2), (700, 1152, 1920, 16, 4)])
def test_weight_gradients_in_one_launch(moe, dtype, shape):
    """One, two and three weight gradients a call: the bits of a call each, on the rows as they lie and (an option, fp32) from copies."""
    import torch
    S, H, I, E, k = shape
    cfg, rng, count, offset = routed_case(S, H, I, E, k, dtype, seed=S, drop=0, skew=0.2)
    R = int(count.sum())
    dev = lambda *s: to_device(ob.from_f32(rng.standard_normal(s).astype(np.float32), dtype), KIND[dtype])
    dcount, doff = to_device(count, "i32"), to_device(offset, "i32")
    x, dy, h, du = dev(S * k, H), dev(S * k, H), dev(S * k, I), dev(S * k, I)
    for t in (x, dy, h, du):
        t[R:] = float("nan")
    for options in ({}, {"grouped_tile": 1}):
        layer = moe.MoELayer(product_config(cfg), options=options)
        pairs = [(dy, h), (du, x), (h, x)]
        want = [layer.expert_wgrad(*p, dcount, doff) for p in pairs]
        for n in (1, 2, 3):
            assert all(torch.equal(g, w) for g, w in zip(layer.expert_wgrads(pairs[:n], dcount, doff), want))
