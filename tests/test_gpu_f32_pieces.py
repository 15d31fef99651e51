"""fp32 layers on bf16 pieces (csrc/ffn_f32_pieces.hip): no further from float64 than the fp32 matrix instructions, over both row block
heights and every epilogue, and those instructions themselves wherever a value is not held by three pieces."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# S, H, I, E, k, activation, capacity factor (0: none dropped), biases
SHAPES = {
    "relu_one_expert": (4500, 512, 2048, 1, 1, 0, 0.0, False),              # a ragged last row block
    "gelu_bias_drop": (4700, 640, 1920, 3, 1, 1, 0.9, True),                # ragged column tiles, odd slab counts a piece
    "swiglu_bias": (2600, 896, 1152, 2, 2, 2, 0.0, True),
    "relu_many_rounds": (9000, 256, 1024, 4, 2, 0, 1.0, False),
}


@pytest.fixture(scope="module")
def moe():
    import torch
    assert torch.cuda.is_available(), "these tests need the MI355X"
    import cuplayground_amd
    return cuplayground_amd


def _layers(moe, name):
    import torch
    S, H, I, E, k, act, cf, bias = SHAPES[name]
    cfg = moe.MoEConfig(capacity_factor=cf or 1.0, drop_tokens=int(cf > 0), expert_top_k=k, is_training=0, hidden_act=act, hidden_size=H,
                        intermediate_size=I, micro_batch=1, num_experts=E, sequence_len=S, torch_dtype=0, gate_fn=0, norm_topk_prob=0)
    pieces, tile = moe.MoELayer(cfg, options={}), moe.MoELayer(cfg, options={"f32_tile": 1}, ffn_mode=moe.api.FFN_TILED)
    assert pieces.workspace_bytes > tile.workspace_bytes + 6 * S * H          # the pieces have their place
    g = torch.Generator(device="cuda").manual_seed(S)
    rnd = lambda *s, std=0.05: torch.randn(*s, generator=g, device="cuda") * std
    w = {"gate_w": rnd(E, H), "w_up": rnd(E, I, H), "w_down": rnd(E, H, I)}
    if act == 2:
        w["w_gate"] = rnd(E, I, H)
    if bias:
        w.update(b_up=rnd(E, I), b_down=rnd(E, H), **({"b_gate": rnd(E, I)} if act == 2 else {}))
    return cfg, pieces, tile, rnd(S, H, std=1.0), w


def _float64(cfg, x, w, routing):
    import torch
    S, k, E = cfg.tokens, cfg.expert_top_k, cfg.num_experts
    out = torch.zeros(S, cfg.hidden_size, dtype=torch.float64, device="cuda")
    idx, slot, tw = (routing[n].reshape(S, k) for n in ("topk_idx", "slot", "topk_w"))
    d = lambda n, e: w[n][e].double() if n in w else 0.0
    for e in range(E):
        for r in range(k):
            m = ((idx[:, r] == e) & (slot[:, r] >= 0)).nonzero().flatten()
            rows = x[m].double()
            h = rows @ d("w_up", e).t() + d("b_up", e)
            if cfg.hidden_act == 2:
                h = torch.nn.functional.silu(rows @ d("w_gate", e).t() + d("b_gate", e)) * h
            else:
                h = torch.nn.functional.gelu(h) if cfg.hidden_act == 1 else torch.relu(h)
            out[m] += (h @ d("w_down", e).t() + d("b_down", e)) * tw[m, r:r + 1].double()
    return out


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_no_further_from_float64_than_the_fp32_tile(moe, name):
    cfg, pieces, tile, x, w = _layers(moe, name)
    routing = pieces.new_routing()
    got, other = pieces.forward(x, w, routing=routing), tile.forward(x, w)
    ref = _float64(cfg, x, w, routing)
    far = lambda o: ((o.double() - ref).norm() / ref.norm()).item()
    assert far(got) <= far(other) and far(got) < 1e-6, (far(got), far(other))
    assert ((got.double() - ref).abs().max() <= (other.double() - ref).abs().max() * 1.5)      # single values: the tails of two distributions
    pieces.close(), tile.close()


@pytest.mark.parametrize("kind", ["one_sign", "constant", "one_hot", "spread"])
@pytest.mark.parametrize("act", [0, 2])
def test_other_distributions_are_no_further_from_float64(moe, act, kind):
    """Sums of one sign, which an adder that truncates would show; equal terms; single terms, one rounding either way; magnitudes over 2^24."""
    import torch
    S, H, I = 4500, 1024, 2048
    cfg = moe.MoEConfig(capacity_factor=1.0, drop_tokens=0, expert_top_k=1, is_training=0, hidden_act=act, hidden_size=H, intermediate_size=I,
                        micro_batch=1, num_experts=1, sequence_len=S, torch_dtype=0, gate_fn=0, norm_topk_prob=0)
    pieces, tile = moe.MoELayer(cfg, options={}), moe.MoELayer(cfg, options={"f32_tile": 1}, ffn_mode=moe.api.FFN_TILED)
    assert pieces.workspace_bytes > tile.workspace_bytes + 6 * S * H
    g = torch.Generator(device="cuda").manual_seed(S + act)

    def values(*s, std=1.0):
        r = torch.randn(*s, generator=g, device="cuda") * std
        if kind == "spread":
            r *= torch.exp2(torch.randint(-12, 12, s, generator=g, device="cuda").float())
        return torch.full_like(r, 1.2345678 * std) if kind == "constant" else r.abs() if kind == "one_sign" else r
    x = values(S, H)
    if kind == "one_hot":
        t = torch.arange(S, device="cuda")
        x = torch.zeros_like(x).index_put_((t, t % H), x[t, t % H])
    w = {"gate_w": torch.zeros(1, H, device="cuda"), "w_up": values(1, I, H, std=0.05), "w_down": values(1, H, I, std=0.05)}
    if act == 2:
        w["w_gate"] = values(1, I, H, std=0.05)
    routing = pieces.new_routing()
    got, other = pieces.forward(x, w, routing=routing), tile.forward(x, w)
    ref = _float64(cfg, x, w, routing)
    far = lambda o: ((o.double() - ref).norm() / ref.norm()).item()
    assert far(got) <= far(other) and not torch.equal(got, other), (far(got), far(other))
    assert ((got.double() - ref).abs().max() <= (other.double() - ref).abs().max() * 1.5)
    pieces.close(), tile.close()


@pytest.mark.parametrize("what", ["x_inf", "x_nan", "w_huge", "h_huge"])
@pytest.mark.parametrize("name", ["gelu_bias_drop", "swiglu_bias"])
def test_values_that_pieces_do_not_hold(moe, name, what):
    """The whole call by the fp32 instructions, bit for bit (NaN in the same places)."""
    import torch
    cfg, pieces, tile, x, w = _layers(moe, name)
    if what == "x_inf":
        x[17, 5] = float("inf")
    elif what == "x_nan":
        x[cfg.tokens - 1, 0] = float("nan")
    elif what == "w_huge":
        w["w_down"][1, 3, 64] = 3e38
    else:      # operands that pieces hold, results of the up projection that they do not
        x *= 1e3
        w["w_up"] *= 1e21
    got, want = pieces.forward(x, w), tile.forward(x, w)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32)) or (torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num()))
    pieces.close(), tile.close()


@pytest.mark.parametrize("name,what", [(n, w) for n in ("gelu_bias_drop", "swiglu_bias") for w in ("w_tiny", "x_denormal", "h_tiny")] + [("swiglu_bias", "silu_tail")])
def test_small_values_are_held(moe, name, what):
    """However small a value is, it is held exactly: the call stays on pieces (the fp32 tile's bits are others), and is no further from
    float64.  A gate of -66 and less makes intermediate values below 2^-100 of ordinary tokens."""
    import torch
    cfg, pieces, tile, x, w = _layers(moe, name)
    if what == "w_tiny":
        w["w_up"][0, 7, 9] = 2.0 ** -101
        w["w_down"][:, 5] *= 2.0 ** -120
    elif what == "x_denormal":
        x[100, 11] = 1e-41
        x[:, 12] *= 2.0 ** -125
    elif what == "h_tiny":
        x *= 1e-15
        for n in ("w_up", "w_gate", "b_up", "b_gate", "b_down"):
            if n in w:
                w[n] *= 0.0 if n[0] == "b" else 1e15 if n == "w_gate" else 1e-20
        w["w_down"] *= 1e10
    else:
        w["b_gate"][:, ::3] = -torch.linspace(60.0, 90.0, w["b_gate"][:, ::3].shape[1], device="cuda")
    routing = pieces.new_routing()
    got, other = pieces.forward(x, w, routing=routing), tile.forward(x, w)
    ref = _float64(cfg, x, w, routing)
    far = lambda o: ((o.double() - ref).norm() / ref.norm()).item()
    assert ref.any() and far(got) <= far(other) and far(got) < 1e-6 and not torch.equal(got, other), (far(got), far(other))
    pieces.close(), tile.close()


def _same(got, want):
    import torch
    return torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(1.0, 2.0, 3.0), want.nan_to_num(1.0, 2.0, 3.0))


@pytest.mark.parametrize("what", ["down_infinite", "down_near_largest", "up_negative_infinite"])
def test_sums_that_overflow_on_pieces_only(moe, what):
    """Every operand is held by three pieces, but the pieces' products or their sums leave the range before those of the values do."""
    import torch
    cfg, pieces, tile, x, w = _layers(moe, "relu_one_expert")
    S, H = x.shape
    t, below = torch.arange(S, device="cuda"), 2.0 ** 64 * (1 - 2.0 ** -13)     # below: its first piece is 2^64
    x.zero_(), w["w_up"].zero_()
    j = torch.arange(H, device="cuda")
    if what == "up_negative_infinite":     # -2^128 (1 - 2^-12) and three times nearly 2^127: on pieces -inf, which ReLU turns into a zero
        for k in (1, 130, 260, 390):
            x[:, k], w["w_up"][0, :, k] = (-below, below) if k == 1 else (2.0 ** 63 * (1 - 2.0 ** -10), 2.0 ** 64)
        w["w_down"].fill_(2.0 ** -90)
    else:                                  # hidden column j is token column j
        w["w_up"][0, j, j] = 1.0
        x[t, t % H] = below if what == "down_near_largest" else 2.0 ** 70 * (1 + 2.0 ** -8 + 2.0 ** -12)
        w["w_down"][:] = below if what == "down_near_largest" else 2.0 ** 70 * 1.9989
        w["w_down"][:, ::2] *= -1
    got, want = pieces.forward(x, w), tile.forward(x, w)
    assert want.isinf().all() if what == "down_infinite" else want.isfinite().all() and want.any()
    assert _same(got, want)
    pieces.close(), tile.close()


def test_smallest_and_largest_magnitudes_that_pieces_hold(moe):
    """Tokens down to the denormal numbers against weights up to just below 2^76: all three pieces count."""
    import torch
    cfg, pieces, tile, x, w = _layers(moe, "relu_one_expert")
    x *= 2.0 ** -115
    x[:, ::5] *= 2.0 ** -15
    x[0, 0] = 2.0 ** -149
    w["w_up"] *= 2.0 ** 77
    w["w_up"].clamp_(-(2.0 ** 76 - 2.0 ** 52), 2.0 ** 76 - 2.0 ** 52)
    w["w_up"][0, 0, 0] = 2.0 ** 76 - 2.0 ** 52
    routing = pieces.new_routing()
    got, other = pieces.forward(x, w, routing=routing), tile.forward(x, w)
    ref = _float64(cfg, x, w, routing)
    far = lambda o: ((o.double() - ref).norm() / ref.norm()).item()
    assert far(got) <= far(other) and not torch.equal(got, other)
    pieces.close(), tile.close()


def test_schedules_options_and_traces_change_no_bits(moe):
    """The arithmetic is the plan's: every mode and way to combine, options of the queue and a trace leave a layer on pieces, and its two
    launches; the options that a handle reports make another like it."""
    import torch
    api = moe.api
    cfg, pieces, tile, x, w = _layers(moe, "gelu_bias_drop")
    want = pieces.forward(x, w)
    assert not torch.equal(want, tile.forward(x, w)) and tile.options["f32_tile"] == 1
    for options in ({}, {"combine": 0}, {"combine": 1}, {"combine": 2}, {"tail_round": 0}, {"row_chunk": 3}, {"queue_groups": 8}, {"queue_lag": 1}, {"blocks_per_cu": 1}):
        for mode in (api.FFN_AUTO, api.FFN_TILED, api.FFN_PERSISTENT):
            layer = moe.MoELayer(cfg, options=options, ffn_mode=mode)
            assert torch.equal(layer.forward(x, w), want) and layer.options["f32_tile"] == -1 and layer.ffn_mode == api.FFN_TILED, (options, mode)
            same = moe.MoELayer(cfg, options=layer.options, ffn_mode=layer.ffn_mode)
            assert torch.equal(same.forward(x, w), want)
            layer.close(), same.close()
    traced = moe.MoELayer(cfg, options={})
    traced.enable_task_trace(1 << 14)
    assert torch.equal(traced.forward(x, w), want) and len(traced.task_trace()) == 0
    queue = moe.MoELayer(cfg, options={"f32_tile": 1}, ffn_mode=api.FFN_PERSISTENT)      # where the queue, its reports and traces are
    queue.enable_task_trace(1 << 14)
    assert torch.equal(queue.forward(x, w), tile.forward(x, w)) and len(queue.task_trace()) > 0 and queue.queue_balance()["span_us"] > 0
    for l in (pieces, tile, traced, queue):
        l.close()


def test_replays_of_a_graph_change_over(moe):
    """One captured call on inputs that pieces hold and on others: every replay is the eager call."""
    import torch
    cfg, pieces, tile, x, w = _layers(moe, "relu_one_expert")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    out = torch.empty_like(x)
    with torch.cuda.stream(side):
        pieces.forward(x, w, out=out)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pieces.forward(x, w, out=out)
    clean = x.clone()
    for it in range(4):
        x.copy_(clean * (it + 1))
        if it % 2:
            x[3, 3] = float("inf")
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got, want = out.clone(), pieces.forward(x, w)
        assert torch.equal(got.nan_to_num(), want.nan_to_num()) and torch.equal(got.isnan(), want.isnan())
        assert bool(torch.isfinite(got).all()) == (it % 2 == 0)
    pieces.close(), tile.close()
