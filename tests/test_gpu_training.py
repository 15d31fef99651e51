"""The trainable layer built on the backward building blocks, against the same layer written in torch ops with fp32
parameters and torch's own autograd (forward values and every gradient)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def moe():
    import torch
    assert torch.cuda.is_available(), "these tests need the MI355X"
    import cuplayground_amd
    cuplayground_amd.load_library()
    return cuplayground_amd


def rel(a, b):
    a, b = a.detach().double(), b.detach().double()
    return float((a - b).abs().max() / b.abs().max().clamp(min=1e-30))


@pytest.mark.parametrize("act,dtype,drop,inter", [(2, 2, 0, 384), (1, 2, 1, 512), (0, 3, 0, 512), (2, 3, 1, 384), (0, 0, 0, 512),
                                                  (2, 0, 1, 384), (1, 1, 0, 512), (2, 2, 1, 512), (2, 3, 0, 512)])
def test_trainable_layer_matches_torch_autograd(moe, act, dtype, drop, inter):
    import torch
    from cuplayground_amd import training, torch_op
    cfg = moe.MoEConfig(capacity_factor=1.0, drop_tokens=drop, expert_top_k=2, hidden_act=act, hidden_size=256,
                        intermediate_size=inter, micro_batch=1, num_experts=6, sequence_len=700,
                        torch_dtype=dtype, gate_fn=0, norm_topk_prob=1, is_training=1)
    m = training.MoE355Train(cfg, init_std=0.05, seed=3)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").to(m.layer.act_dtype).requires_grad_(True)
    dout = torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").to(m.layer.act_dtype)
    # (the 16-bit cases' products take the weights as stored, with the activation's derivative in the epilogue; the branches of
    # layers that go by transposed copies give the same bits: the test below)
    assert m.layer.fused_act_backward == (dtype in (2, 3) and inter % 256 == 0)
    out = m(x)
    out.backward(dout)

    # the same layer in torch ops on fp32 copies of the same (16-bit valued) parameters, routing taken from the library
    idx, _ = m.route(x)
    xr = x.detach().float().requires_grad_(True)
    ps = {n: p.detach().float().requires_grad_(True) for n, p in m.named_parameters()}
    logits = xr @ ps["gate_w"].t()
    w = torch.softmax(logits, 1).gather(1, idx.long())
    w = w / w.sum(1, keepdim=True)
    ref = torch_op.torch_reference(xr, cfg, ps["gate_w"], ps["w_up"], ps.get("w_gate"), ps["w_down"], topk=(idx, w))
    ref.backward(dout.float())

    assert rel(out.float(), ref) <= {2: 1e-2, 3: 2e-3}.get(dtype, 2e-5)
    tol = {2: 2e-2, 3: 4e-3}.get(dtype, 1e-4)      # 16-bit gradients pass through two rounded products; fp32: summation order
    assert rel(x.grad.float(), xr.grad) <= tol
    for n, p in m.named_parameters():
        assert p.grad is not None and torch.isfinite(p.grad.float()).all(), n
        assert rel(p.grad.float(), ps[n].grad) <= tol, n
    if drop:                                # some pairs were dropped in this configuration: the test covers that path
        assert int((m.route(x)[1]["pair_row"] < 0).sum()) > 0


@pytest.mark.parametrize("tile", [1, 2])
@pytest.mark.parametrize("act,dtype,drop,inter", [(2, 2, 0, 384), (1, 2, 1, 512), (0, 3, 0, 512), (2, 3, 1, 384), (2, 2, 1, 512)])
def test_transposed_copies_and_operands_as_stored_give_the_same_step(moe, act, dtype, drop, inter, tile):
    """Large layers' gradients go by transposed copies of the weights and rows -- with the activation's derivative in the epilogue where
    the layer has that kernel, else as a pass of its own -- small ones' by the operands as stored.  Option grouped_tile takes a small
    layer the first way: the same sums in the same order, so the same bits."""
    import torch
    from cuplayground_amd import training
    cfg = moe.MoEConfig(capacity_factor=1.0, drop_tokens=drop, expert_top_k=2, hidden_act=act, hidden_size=256,
                        intermediate_size=inter, micro_batch=1, num_experts=6, sequence_len=700,
                        torch_dtype=dtype, gate_fn=0, norm_topk_prob=1, is_training=1)
    steps = []
    for options, stored in ((None, 2), ({"grouped_tile": tile}, 1)):
        m, g = training.MoE355Train(cfg, init_std=0.05, seed=3), torch.Generator(device="cuda").manual_seed(1)
        if options:
            m.layer = moe.MoELayer(cfg, options=options)
        for n, k in ((256, inter), (inter, 256)):
            assert m.layer.gemm_kn_supported(n, k) == stored
        assert m.layer.fused_act_backward == (inter % 256 == 0)
        x = torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").to(m.layer.act_dtype).requires_grad_(True)
        out = m(x)
        out.backward(torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").to(m.layer.act_dtype))
        steps.append([out.detach(), x.grad] + [p.grad for _, p in m.named_parameters()])
    assert all(torch.equal(a, b) for a, b in zip(*steps))


def test_e4m3_layers_are_refused(moe):
    from cuplayground_amd import training
    with pytest.raises(ValueError):
        training.MoE355Train(moe.MoEConfig(hidden_size=128, intermediate_size=128, micro_batch=1, sequence_len=128,
                                           torch_dtype=4))


@pytest.mark.parametrize("dtype", [0, 2, 3])
@pytest.mark.parametrize("S,H,I,E,k,act,cf", [(1, 64, 64, 2, 1, 0, 1.0), (37, 512, 128, 3, 2, 1, 0.6), (130, 576, 192, 5, 5, 2, 0.8),
                                              (513, 1088, 64, 8, 6, 2, 1.0)])
def test_row_passes_match_plain_torch(moe, S, H, I, E, k, act, cf, dtype):
    """Dispatch, activation, the adjoint of the dispatch and of the combine, over kept and dropped pairs: one rounding to
    the storage type behind fp32 arithmetic (2 ulp of it: the reference rounds the same fp64 value once)."""
    import torch
    cfg = moe.MoEConfig(capacity_factor=cf, drop_tokens=1, expert_top_k=k, hidden_act=act, hidden_size=H, intermediate_size=I,
                        micro_batch=1, num_experts=E, sequence_len=S, torch_dtype=dtype, gate_fn=0, norm_topk_prob=1)
    layer = moe.MoELayer(cfg)
    dt = layer.act_dtype
    g = torch.Generator(device="cuda").manual_seed(S + H)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(dt)

    idx = torch.stack([torch.randperm(E, generator=g, device="cuda")[:k] for _ in range(S)]).int()
    r = layer.route(idx)
    kept, pr = int(r["expert_count"].sum()), r["pair_row"].long()
    tok = r["token_indices"][:kept].long()
    eps = {0: 2e-6, 2: 2.0 ** -7, 3: 2.0 ** -10}[dtype]

    def close(a, b, scale=1.0):
        a, b = a.double(), b.double()
        return bool(((a - b).abs() <= eps * b.abs() + scale * (1e-6 if dtype else 2e-6)).all())

    x = normal(S, H)
    assert torch.equal(layer.dispatch_rows(x, r["token_indices"])[:kept], x[tok])
    u, gt = normal(S * k, I), normal(S * k, I) if act == 2 else None
    h = layer.act_forward(u, gt, r["expert_count"], r["expert_offset"])[:kept]
    ud = u[:kept].double()
    want = torch.nn.functional.silu(gt[:kept].double()) * ud if act == 2 else torch.nn.functional.gelu(ud) if act == 1 else torch.relu(ud)
    assert close(h, want)
    a, b = normal(S * k, H), normal(S * k, H)
    on = (pr >= 0).unsqueeze(-1).double()
    pick = lambda t: t.double()[pr.clamp(min=0)] * on
    assert close(layer.dispatch_backward(a, None, r["pair_row"]), pick(a).sum(1), scale=k)
    assert close(layer.dispatch_backward(a, b, r["pair_row"]), (pick(a) + pick(b)).sum(1), scale=2 * k)
    w = torch.rand(S, k, generator=g, device="cuda")
    dy, dw = layer.combine_backward(x, a, r["pair_row"], w)
    want_dy = torch.zeros(S * k, H, dtype=torch.float64, device="cuda")
    flat = pr.reshape(-1)
    want_dy[flat[flat >= 0]] = (w.double().unsqueeze(-1) * x.double().unsqueeze(1)).reshape(S * k, H)[flat >= 0]
    assert close(dy, want_dy)
    want_dw = (pick(a) * x.double().unsqueeze(1)).sum(-1)
    assert float((dw.double() - want_dw).abs().max()) <= 1e-6 * H       # fp32 sums of H products of order 1
    # operands that are not 16-byte aligned take the element-wise kernel, with the same dy
    pad = torch.zeros(S * H + 1, dtype=dt, device="cuda")
    pad[1:] = x.reshape(-1)
    dy2, dw2 = layer.combine_backward(pad[1:].view(S, H), a, r["pair_row"], w)
    assert torch.equal(dy2, dy) and float((dw2.double() - want_dw).abs().max()) <= 1e-6 * H


@pytest.mark.parametrize("norm", [0, 1])
def test_a_step_under_autocast_uses_its_gate_weights(moe, norm):
    """torch.autocast computes the router's logits, and with them a sigmoid's weights, in 16 bits: the step must be the one
    with exactly those weights, widened."""
    import torch
    from cuplayground_amd import training, torch_op
    cfg = moe.MoEConfig(capacity_factor=1.0, drop_tokens=0, expert_top_k=2, hidden_act=1, hidden_size=256, intermediate_size=128,
                        micro_batch=1, num_experts=5, sequence_len=301, torch_dtype=2, gate_fn=1, norm_topk_prob=norm, is_training=1)
    m = training.MoE355Train(cfg, init_std=0.05, seed=3)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").bfloat16()
    dout = torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").bfloat16()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = m(x)
        idx, _ = m.route(x)
        w = m.gate_weights(x, idx)
    out.backward(dout)
    ps = {n: p.detach().float() for n, p in m.named_parameters()}
    ref = torch_op.torch_reference(x.float(), cfg, ps["gate_w"], ps["w_up"], None, ps["w_down"], topk=(idx, w.detach().float()))
    assert rel(out.float(), ref) <= 1e-2
    for n, p in m.named_parameters():
        assert torch.isfinite(p.grad.float()).all() and float(p.grad.float().abs().max()) > 0, n


@pytest.mark.parametrize("act", [1, 2], ids=["gelu", "swiglu"])
@pytest.mark.parametrize("dtype", [2, 3], ids=["bf16", "fp16"])
def test_training_activation_is_the_fp32_function(moe, act, dtype):
    """Every finite value of the storage type (SwiGLU: as g, with u = 1) through moe_act_forward against torch's fp32 function
    rounded once.  Two evaluations of the function in fp32 differ by about 1e-7 of the value, a 2000th of fp16's spacing, so a
    result in a few thousand rounds the other way; the 5e-7 of an approximated erfc would move one in a hundred."""
    import torch
    cfg = moe.MoEConfig(capacity_factor=1.0, drop_tokens=0, expert_top_k=1, hidden_act=act, hidden_size=64, intermediate_size=64,
                        micro_batch=1, num_experts=2, sequence_len=1024, torch_dtype=dtype, gate_fn=0, norm_topk_prob=0)
    layer = moe.MoELayer(cfg)
    v = torch.arange(65536, dtype=torch.int32, device="cuda").to(torch.int16).view(layer.act_dtype).view(1024, 64)
    count = torch.tensor([1024, 0], dtype=torch.int32, device="cuda")
    offset = torch.tensor([0, 1024], dtype=torch.int32, device="cuda")
    u, g = (torch.ones_like(v), v) if act == 2 else (v, None)
    got = layer.act_forward(u, g, count, offset)
    f = v.float()
    want = (torch.nn.functional.silu(f) if act == 2 else torch.nn.functional.gelu(f)).to(layer.act_dtype)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    ok = torch.isfinite(want)
    assert torch.equal(got[~ok & ~torch.isnan(want)], want[~ok & ~torch.isnan(want)])
    tail = ok & (f < 0) & (f >= -4)                       # where 1 + erf cancels
    assert float((got != want)[tail].float().mean()) <= 1e-3
    assert float((got != want)[ok].float().mean()) <= 1e-3


@pytest.mark.parametrize("act,dtype,inter", [(2, 2, 384), (1, 3, 512), (0, 0, 384), (2, 0, 128)])
def test_a_layer_composed_of_the_projection_nodes_is_the_layer(moe, act, dtype, inter):
    """expert_linear and act_down with gather and combine as torch indexing against MoE355Train on the same weights: each is
    within the tolerance of test_trainable_layer_matches_torch_autograd of the same fp32 layer, so they are within twice that."""
    import torch
    from cuplayground_amd import training
    cfg = moe.MoEConfig(capacity_factor=0.9, drop_tokens=1, expert_top_k=2, hidden_act=act, hidden_size=256,
                        intermediate_size=inter, micro_batch=1, num_experts=5, sequence_len=333,
                        torch_dtype=dtype, gate_fn=0, norm_topk_prob=1, is_training=1)
    m = training.MoE355Train(cfg, init_std=0.05, seed=3)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").to(m.layer.act_dtype).requires_grad_(True)
    dout = torch.randn(cfg.tokens, cfg.hidden_size, generator=g, device="cuda").to(m.layer.act_dtype)
    leaves = dict(m.named_parameters(), x=x)

    def step(out):
        return out, dict(zip(leaves, torch.autograd.grad(out, leaves.values(), dout)))

    idx, r = m.route(x)
    count, offset, pairs = r["expert_count"], r["expert_offset"], r["pair_row"]
    x_rows = x.index_select(0, r["token_indices"].clamp(min=0).long())      # rows of no expert gather token 0 and are not used
    up = training.expert_linear(x_rows, m.w_up, m.layer, count, offset)
    gate = training.expert_linear(x_rows, m.w_gate, m.layer, count, offset) if act == 2 else None
    y = training.act_down(up, gate, m.w_down, m.layer, count, offset)
    picked = y[pairs.clamp(min=0).long()].float() * (pairs >= 0).unsqueeze(-1)
    composed, grads = step((picked * m.gate_weights(x, idx).unsqueeze(-1)).sum(1).to(x.dtype))
    out, want = step(m(x))
    assert int((pairs < 0).sum()) > 0
    assert rel(composed, out) <= 2 * {2: 1e-2, 3: 2e-3}.get(dtype, 2e-5)
    for n in leaves:
        assert rel(grads[n], want[n]) <= 2 * {2: 2e-2, 3: 4e-3}.get(dtype, 1e-4), n


@pytest.mark.parametrize("S,H,E,k,gate_fn,norm,dtype,drop", [
    (257, 320, 5, 3, 0, 1, 2, 1), (1, 64, 2, 1, 1, 0, 0, 0), (1, 64, 70, 8, 0, 1, 3, 0), (4100, 256, 16, 2, 0, 1, 2, 1),
    (300, 1024, 130, 6, 1, 1, 0, 1), (700, 448, 33, 4, 1, 1, 2, 0), (129, 576, 64, 16, 1, 0, 3, 1), (9000, 64, 8, 1, 0, 1, 0, 0)])
def test_router_gradients(moe, S, H, E, k, gate_fn, norm, dtype, drop):
    """The adjoint of the gate inside the combine's and the dispatch's, and the router's weight gradient, against float64."""
    import torch
    cfg = moe.MoEConfig(capacity_factor=0.8, drop_tokens=drop, expert_top_k=k, hidden_act=1, hidden_size=H, intermediate_size=64,
                        micro_batch=1, num_experts=E, sequence_len=S, torch_dtype=dtype, gate_fn=gate_fn, norm_topk_prob=norm)
    layer = moe.MoELayer(cfg)
    gen = torch.Generator(device="cuda").manual_seed(S + E)

    def rand(*shape):
        return torch.randn(*shape, generator=gen, device="cuda").to(layer.act_dtype)

    x, gate_w, y, dout = rand(S, H), rand(E, H) * H ** -0.5, rand(S * k, H), rand(S, H)
    idx, w, logits = layer.gate(x, gate_w, want_logits=True)
    rows = layer.route(idx)["pair_row"]
    dy, router = torch.empty_like(y), torch.empty(layer.router_grad_bytes, dtype=torch.uint8, device="cuda")
    layer.combine_router_backward(dout, y, rows, w, idx, logits if gate_fn and norm else None, dy, router)
    want_dy, dw = layer.combine_backward(dout, y, rows, w)
    assert torch.equal(dy[rows[rows >= 0].long()], want_dy[rows[rows >= 0].long()])

    # the gate in float64 from the kernel's own logits, its adjoint from the combine's fp32 gradients
    l64 = logits.double().requires_grad_(True)
    s = torch.softmax(l64, 1) if gate_fn == 0 else torch.sigmoid(l64)
    w64 = s.gather(1, idx.long())
    w64 = w64 / w64.sum(1, keepdim=True) if norm else w64
    w64.backward(dw.double())
    want = l64.grad.gather(1, idx.long())
    dl = router[:4 * S * k].view(torch.float32).view(S, k)
    # k products and sums of fp32 and the weights' own fp32 error: some tens of units of 2^-24 of the largest gradient of the token
    scale = dw.double().abs().amax(1, keepdim=True).clamp(min=1e-30) * (1.0 if not (gate_fn and norm) else k)
    assert float(((dl.double() - want).abs() / scale).max()) <= 64 * 2.0 ** -24

    # the sums: terms in fp32 (2^-24 of the sum of magnitudes for each of the terms one accumulator takes), then one rounding
    unit = {0: 2.0 ** -24, 1: 2.0 ** -24, 2: 2.0 ** -8, 3: 2.0 ** -11}[dtype]         # half a step of the stored type
    dense = torch.zeros(S, E, dtype=torch.float64, device="cuda").scatter_(1, idx.long(), dl.double())
    got, ref, mag = layer.gate_wgrad(x, router).double(), dense.t() @ x.double(), dense.t().abs() @ x.double().abs()
    tiny = 2.0 ** -24 if dtype == 3 else 0.0           # fp16 below its normal range
    assert bool(((got - ref).abs() <= unit * ref.abs() + (S / 4 + 68) * 2.0 ** -24 * mag + tiny).all())
    # the same sums from the packed rows, whatever the rows of no expert hold: a token without a row has no gradient to add
    packed = torch.full((S * k, H), float("nan"), dtype=layer.act_dtype, device="cuda")
    kept = (rows >= 0).nonzero()
    packed[rows[rows >= 0].long()] = x[kept[:, 0]]
    lost = (rows < 0).all(1)
    assert bool((dl[lost] == 0).all())
    x_kept = x.masked_fill(lost[:, None], 0)
    assert torch.equal(layer.gate_wgrad(packed, router, packed=True), layer.gate_wgrad(x_kept, router))
    a, b = rand(S * k, H), rand(S * k, H)
    got = layer.dispatch_router_backward(a, b, rows, idx, router, gate_w).double()
    part = torch.where((rows >= 0)[..., None], a[rows.clamp(min=0).long()].double() + b[rows.clamp(min=0).long()].double(), 0.0).sum(1)
    mag = torch.where((rows >= 0)[..., None], a[rows.clamp(min=0).long()].double().abs() + b[rows.clamp(min=0).long()].double().abs(), 0.0).sum(1)
    ref, mag = part + dense @ gate_w.double(), mag + dense.abs() @ gate_w.double().abs()
    assert bool(((got - ref).abs() <= unit * ref.abs() + (3 * k + 1) * 2.0 ** -24 * mag + tiny).all())


def test_a_softmax_over_all_experts_keeps_its_torch_gate(moe):
    """Not normalised over the chosen, each logit has a gradient: such a layer has no router kernels and says so."""
    import torch
    from cuplayground_amd import training
    cfg = moe.MoEConfig(expert_top_k=2, hidden_act=1, hidden_size=64, intermediate_size=64, micro_batch=1, num_experts=4,
                        sequence_len=32, torch_dtype=2, gate_fn=0, norm_topk_prob=0, is_training=1)
    m = training.MoE355Train(cfg, init_std=0.2)
    assert m.layer.router_grad_bytes == 0
    m(torch.randn(32, 64, device="cuda", dtype=torch.bfloat16)).float().sum().backward()
    assert bool((m.gate_w.grad.float().abs().sum(1) > 0).all())


@pytest.mark.parametrize("gate_fn", [0, 1], ids=["softmax", "sigmoid"])
def test_a_single_normalised_expert_keeps_its_torch_gate(moe, gate_fn):
    """Its weight is one, and the router's gradient the rounding of torch's w / w: the same bits as with gate weights of the
    caller's own, which are torch ops always."""
    import torch
    from cuplayground_amd import training

    class Own(training.MoE355Train):
        def gate_weights(self, x, idx):
            return super().gate_weights(x, idx)

    cfg = moe.MoEConfig(expert_top_k=1, hidden_act=1, hidden_size=128, intermediate_size=64, micro_batch=1, num_experts=4,
                        sequence_len=97, torch_dtype=0, gate_fn=gate_fn, norm_topk_prob=1, is_training=1)
    grads = []
    for kind in (training.MoE355Train, Own):
        m, g = kind(cfg, init_std=0.2, seed=2), torch.Generator(device="cuda").manual_seed(7)
        x = torch.randn(97, 128, generator=g, device="cuda", requires_grad=True)
        m(x).backward(torch.randn(97, 128, generator=g, device="cuda"))
        grads.append([x.grad] + [p.grad for _, p in m.named_parameters()])
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("dtype", [2, 3], ids=["bf16", "fp16"])
@pytest.mark.parametrize("gate_fn,norm", [(0, 1), (1, 0)], ids=["softmax", "sigmoid"])
def test_input_and_router_may_change_before_the_backward(moe, gate_fn, norm, dtype):
    """The layer's output added onto its input in place, and the router's weights stepped, between forward and backward: the
    gradients are those of the values that the forward read, to the bit."""
    import torch
    from cuplayground_amd import training
    cfg = moe.MoEConfig(expert_top_k=2, hidden_act=1, hidden_size=128, intermediate_size=64, micro_batch=1, num_experts=5,
                        sequence_len=131, torch_dtype=dtype, gate_fn=gate_fn, norm_topk_prob=norm, is_training=1)
    grads = []
    for change in (False, True):
        m, g = training.MoE355Train(cfg, init_std=0.2, seed=2), torch.Generator(device="cuda").manual_seed(7)
        assert m.layer.router_grad_bytes > 0
        x = torch.randn(131, 128, generator=g, device="cuda").to(m.layer.act_dtype).requires_grad_(True)
        dout = torch.randn(131, 128, generator=g, device="cuda").to(m.layer.act_dtype)
        h = x * 1
        y = m(h)
        if change:
            h += y
            with torch.no_grad():
                m.gate_w.mul_(0.5)
        else:
            h = h + y
        h.backward(dout)
        grads.append([x.grad] + [p.grad for _, p in m.named_parameters()])
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("act,dtype,gate_fn,norm,k", [(2, 2, 0, 1, 2), (1, 3, 1, 1, 3), (0, 2, 1, 0, 1), (2, 0, 0, 1, 2), (1, 2, 0, 0, 2)])
def test_saved_tensors_may_come_back_at_any_address(moe, act, dtype, gate_fn, norm, k):
    """Saved-tensor hooks that keep what a step saves as one odd element into a buffer of their own: the same gradients."""
    import torch
    from cuplayground_amd import training
    cfg = moe.MoEConfig(expert_top_k=k, hidden_act=act, hidden_size=128, intermediate_size=192, micro_batch=1, num_experts=5,
                        sequence_len=131, torch_dtype=dtype, gate_fn=gate_fn, norm_topk_prob=norm, is_training=1)
    m, g = training.MoE355Train(cfg, init_std=0.2, seed=2), torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(131, 128, generator=g, device="cuda").to(m.layer.act_dtype).requires_grad_(True)
    dout = torch.randn(131, 128, generator=g, device="cuda").to(m.layer.act_dtype)

    def pack(t):
        buf = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
        buf[1:] = t.detach().reshape(-1)
        return buf[1:].view(t.shape)

    grads = []
    for hooked in (False, True):
        x.grad = None
        m.zero_grad(set_to_none=True)
        if hooked:
            with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
                out = m(x)
        else:
            out = m(x)
        out.backward(dout)
        grads.append([x.grad] + [p.grad for _, p in m.named_parameters()])
    assert all(torch.equal(a, b) for a, b in zip(*grads))
