"""What the training layer hands to the kernels as raw addresses: the types must be the ones they read (no GPU needed: the
checks come before the first launch)."""
import pytest

torch = pytest.importorskip("torch")

from cuplayground_amd import api, training


def _cfg(**kw):
    c = dict(capacity_factor=1.0, drop_tokens=0, expert_top_k=2, hidden_act=api.ACT_GELU, hidden_size=64, intermediate_size=64,
             micro_batch=1, num_experts=4, sequence_len=8, torch_dtype=api.DTYPE_BF16, gate_fn=api.GATE_SIGMOID, norm_topk_prob=0)
    c.update(kw)
    return api.MoEConfig(**c)


def _module(cfg, monkeypatch, seen):
    """A MoE355Train without a handle, whose expert node only records what it is given."""
    m = training.MoE355Train.__new__(training.MoE355Train)
    torch.nn.Module.__init__(m)
    m.cfg, m.layer = cfg, None
    m.gate_w = torch.nn.Parameter(torch.randn(cfg.num_experts, cfg.hidden_size))
    m.w_up = m.w_down = torch.nn.Parameter(torch.zeros(1))
    m.w_gate = None
    idx = torch.arange(cfg.tokens * cfg.expert_top_k).reshape(cfg.tokens, cfg.expert_top_k) % cfg.num_experts
    tables = dict.fromkeys(("expert_count", "expert_offset", "token_indices", "pair_row"))
    monkeypatch.setattr(training.MoE355Train, "route", lambda self, x: (idx.int(), tables))
    monkeypatch.setattr(training._Experts, "apply", staticmethod(lambda *a: seen.append(a) or a[4].sum()))
    return m


@pytest.mark.parametrize("gate_fn", [api.GATE_SOFTMAX, api.GATE_SIGMOID])
@pytest.mark.parametrize("norm", [0, 1])
@pytest.mark.parametrize("autocast", [None, torch.bfloat16])
def test_gate_weights_reach_the_node_in_fp32(monkeypatch, gate_fn, norm, autocast):
    seen = []
    m = _module(_cfg(gate_fn=gate_fn, norm_topk_prob=norm), monkeypatch, seen)
    x = torch.randn(m.cfg.tokens, m.cfg.hidden_size)
    with torch.autocast("cpu", dtype=autocast or torch.bfloat16, enabled=autocast is not None):
        m(x).backward()
    assert seen[0][4].dtype == torch.float32 and seen[0][4].shape == (m.cfg.tokens, m.cfg.expert_top_k)
    assert m.gate_w.grad is not None and m.gate_w.grad.dtype == m.gate_w.dtype


@pytest.mark.parametrize("wrong", [torch.float16, torch.bfloat16, torch.float64])
def test_combine_refuses_weights_of_another_type(wrong):
    y, rows = torch.zeros(16, 64, dtype=torch.bfloat16), torch.zeros(8, 2, dtype=torch.int32)
    with pytest.raises(TypeError):
        api.combine(y, rows, torch.ones(8, 2, dtype=wrong))
    with pytest.raises(TypeError):
        api.combine(y, rows.long(), torch.ones(8, 2))
    with pytest.raises(ValueError):
        api.combine(y, rows, torch.ones(8, 1))


def test_row_passes_refuse_operands_of_another_type():
    layer = api.MoELayer.__new__(api.MoELayer)      # the checks need the layer's shape, not its handle
    layer.cfg, layer.S, layer.k, layer.H, layer.act_dtype, layer._h = _cfg(), 8, 2, 64, torch.bfloat16, None
    x, rows = torch.zeros(8, 64, dtype=torch.bfloat16), torch.zeros(16, 64, dtype=torch.bfloat16)
    tok, pairs, w = torch.zeros(16, dtype=torch.int32), torch.zeros(8, 2, dtype=torch.int32), torch.ones(8, 2)
    bad = [lambda: layer.dispatch_rows(x.float(), tok), lambda: layer.dispatch_rows(x, tok.long()),
           lambda: layer.act_forward(rows.half(), None, None, None), lambda: layer.act_forward(rows, rows.float(), None, None),
           lambda: layer.dispatch_backward(rows.float(), None, pairs), lambda: layer.dispatch_backward(rows, rows, pairs.long()),
           lambda: layer.combine_backward(x, rows, pairs, w.bfloat16()), lambda: layer.combine_backward(x.float(), rows, pairs, w),
           lambda: layer.combine_backward(x, rows.half(), pairs, w)]
    for call in bad:
        with pytest.raises(TypeError):
            call()
    for call in (lambda: layer.dispatch_rows(x[:7], tok), lambda: layer.combine_backward(x[:7], rows, pairs, w),
                 lambda: layer.act_forward(rows, rows[:15], None, None), lambda: layer.dispatch_backward(rows, rows[:15], pairs)):
        with pytest.raises(ValueError):
            call()


def test_router_passes_and_stored_weight_products_refuse_operands_they_would_read_past(monkeypatch):
    """Tables, the gradient buffer, results and weights of too few elements or another type: refused before the first launch."""
    layer = api.MoELayer.__new__(api.MoELayer)
    layer.cfg, layer.S, layer.k, layer.H, layer.E, layer.act_dtype, layer._h = _cfg(), 8, 2, 64, 4, torch.bfloat16, None
    monkeypatch.setattr(api.MoELayer, "router_grad_bytes", 768)
    bf16 = dict(dtype=torch.bfloat16)
    x, rows, gate_w = torch.zeros(8, 64, **bf16), torch.zeros(16, 64, **bf16), torch.zeros(4, 64, **bf16)
    pairs, w, router = torch.zeros(8, 2, dtype=torch.int32), torch.ones(8, 2), torch.zeros(768, dtype=torch.uint8)
    wkn, count = torch.zeros(4, 64, 64, **bf16), torch.zeros(4, dtype=torch.int32)

    def combine(**kw):
        a = dict(dout=x, y_rows=rows, pair_row=pairs, topk_w=w, topk_idx=pairs, logits=None, dy=rows, router_grad=router)
        return lambda: layer.combine_router_backward(**dict(a, **kw))

    def dispatch(**kw):
        a = dict(da_rows=rows, db_rows=None, pair_row=pairs, topk_idx=pairs, router_grad=router, gate_w=gate_w)
        return lambda: layer.dispatch_router_backward(**dict(a, **kw))

    def product(**kw):
        a = dict(a_rows=rows, w=wkn, expert_count=count, expert_offset=count)
        return lambda: layer.expert_gemm_kn(**dict(a, **kw))

    for call in (combine(dy=rows.float()), combine(router_grad=w), combine(topk_idx=pairs.long()), dispatch(pair_row=pairs.long()),
                 dispatch(topk_idx=pairs.long()), dispatch(router_grad=w), lambda: layer.gate_wgrad(x, w),
                 product(expert_count=count.long()), product(expert_offset=count.float())):
        with pytest.raises(TypeError):
            call()
    for call in (combine(dy=rows[:15]), combine(router_grad=router[1:]), combine(topk_idx=pairs[1:]), dispatch(pair_row=pairs[1:]),
                 dispatch(topk_idx=pairs[1:]), dispatch(router_grad=router[1:]), lambda: layer.gate_wgrad(x, router[1:]),
                 product(w=wkn[:3]), product(a_rows=rows[:, :32]), product(expert_count=count[:3]), product(expert_offset=count[:3])):
        with pytest.raises(ValueError):
            call()


def test_products_that_share_a_launch_refuse_operands_they_would_read_or_write_past(monkeypatch):
    """Tables, rows and weights of another type, of too few elements or of other columns: refused before the first launch."""
    layer = api.MoELayer.__new__(api.MoELayer)
    layer.cfg, layer.S, layer.k, layer.H, layer.E, layer.act_dtype, layer._h = _cfg(), 8, 2, 64, 4, torch.bfloat16, None

    def launched(*a):
        raise AssertionError("reached the launch")
    layer.L = type("L", (), dict.fromkeys(("moe_expert_gemm_pair", "moe_expert_gemm_kn_pair", "moe_expert_wgrads"), staticmethod(launched)))
    monkeypatch.setattr(api.MoELayer, "backward_scratch", lambda self: torch.zeros(16, dtype=torch.uint8))
    monkeypatch.setattr(api, "_stream", lambda: None)
    rows, w, count = torch.zeros(16, 64, dtype=torch.bfloat16), torch.zeros(4, 64, 64, dtype=torch.bfloat16), torch.zeros(4, dtype=torch.int32)

    def pair(a=rows, w0=w, w1=w, count=count, offset=count):
        return lambda: layer.expert_gemm_pair(a, w0, w1, count, offset)

    def kn_pair(a=rows, b=rows, w0=w, w1=w, count=count, offset=count):
        return lambda: layer.expert_gemm_kn_pair(a, b, w0, w1, count, offset)

    def wgrads(dy=rows, a=rows, count=count, offset=count):
        return lambda: layer.expert_wgrads([(rows, rows), (dy, a)], count, offset)

    for call in (pair(), kn_pair(), wgrads()):
        with pytest.raises(AssertionError):
            call()
    for f in (pair, kn_pair, wgrads):
        for call in (f(a=rows.half()), f(count=count.long()), f(offset=count.float())):
            with pytest.raises(TypeError):
                call()
        for call in (f(a=rows[:15]), f(count=count[:3]), f(offset=count[:3])):
            with pytest.raises(ValueError):
                call()
    for f in (pair, kn_pair):
        for call in (f(w1=w[:3]), f(a=rows.reshape(8, 128))):      # (as many elements, but results of 8 rows where 16 are written)
            with pytest.raises(ValueError):
                call()


class _RowsLayer:
    """The passes of the expert node as plain torch expressions (one expert, one rank): enough to run the node on the CPU."""
    fused_act_backward = False

    def dispatch_rows(self, x, tok):
        return x.clone()

    def expert_gemm(self, a, w, bias, count, offset, act, out=None):
        return out.copy_(a @ w[0].t())

    def act_forward(self, u, g, count, offset):
        return torch.relu(u) if g is None else torch.nn.functional.silu(g) * u

    def combine_backward(self, dout, y, pair_row, w, dy=None):
        return dy.copy_(dout * w), (dout * y).sum(1, keepdim=True)

    def act_backward(self, dh, u, g):
        with torch.enable_grad():
            args = [t.detach().requires_grad_(True) for t in (u, g) if t is not None]
            grads = torch.autograd.grad(self.act_forward(args[0], args[1] if g is not None else None, None, None), args, dh)
        return grads if g is not None else (grads[0], None)

    def dispatch_backward(self, da, db, pair_row):
        return da if db is None else da + db

    def expert_wgrad(self, dy, a, count, offset):
        return (dy.t() @ a).unsqueeze(0)


@pytest.mark.parametrize("swiglu", [False, True], ids=["relu", "swiglu"])
@pytest.mark.parametrize("needs", ["w", "x", "w_up", "w_gate", "w_down", "x w_up w_gate w_down w"])
def test_the_node_keeps_only_what_its_gradients_read(monkeypatch, swiglu, needs):
    """Rows, pre-activations, activations and weights stay alive until the backward only where a gradient that is asked for
    reads them; the gradients are torch's in every combination."""
    monkeypatch.setattr(api, "combine", lambda y, rows, w: y * w)
    monkeypatch.setattr(api, "transpose", lambda t: t.transpose(1, 2))
    S, H, I = 5, 4, 6
    g = torch.Generator().manual_seed(0)
    t = {n: torch.randn(*s, generator=g, dtype=torch.float64) for n, s in
         dict(x=(S, H), w_up=(1, I, H), w_gate=(1, I, H), w_down=(1, H, I), w=(S, 1)).items()}
    if not swiglu:
        t["w_gate"] = None
    want = [n for n in needs.split() if t[n] is not None]
    if not want:
        pytest.skip("the layer has no such matrix")
    for n in want:
        t[n].requires_grad_(True)
    saved = []
    with torch.autograd.graph.saved_tensors_hooks(lambda v: saved.append(tuple(v.shape)) or v, lambda v: v):
        out = training._Experts.apply(t["x"], t["w_up"], t["w_gate"], t["w_down"], t["w"], _RowsLayer(), None, None, None, None)
    wide = 0                                          # [S, I] buffers: u, g and h
    if {"x", "w_up", "w_gate"} & set(want):
        wide += 2 if swiglu else 1
    wide += "w_down" in want
    assert saved.count((S, I)) == wide
    assert saved.count((S, H)) == 1 + bool({"w_up", "w_gate"} & set(want))      # y, and the dispatched rows
    assert saved.count((1, I, H)) == (2 if swiglu else 1) * ("x" in want)
    dout = torch.randn(S, H, generator=g, dtype=torch.float64)
    got = torch.autograd.grad(out, [t[n] for n in want], dout)
    u = t["x"] @ t["w_up"][0].t()
    h = torch.relu(u) if not swiglu else torch.nn.functional.silu(t["x"] @ t["w_gate"][0].t()) * u
    ref = torch.autograd.grad(h @ t["w_down"][0].t() * t["w"], [t[n] for n in want], dout)
    for n, a, b in zip(want, got, ref):
        assert torch.allclose(a, b, rtol=1e-12, atol=1e-12), n


@pytest.mark.parametrize("extra", [0, 3])
def test_rows_behind_the_layers_tokens_get_zero_gradients(monkeypatch, extra):
    """A longer x is a longer buffer with the layer's tokens in front: the node takes those, the gradient has x's shape."""
    seen = []
    m = _module(_cfg(), monkeypatch, seen)
    monkeypatch.setattr(training._Experts, "apply", staticmethod(lambda *a: seen.append(a) or a[0].sum() + a[4].sum()))
    x = torch.randn(m.cfg.tokens + extra, m.cfg.hidden_size, requires_grad=True)
    m(x).backward()
    assert seen[0][0].shape == (m.cfg.tokens, m.cfg.hidden_size) and seen[0][0].data_ptr() == x.data_ptr()
    assert x.grad.shape == x.shape and (x.grad[:m.cfg.tokens] != 0).all() and not x.grad[m.cfg.tokens:].any()
