"""A trainable MoE layer over the backward building blocks of libmoe355 (fp32, tf32, bf16 and fp16 layers).

The reference declares a training knob (`is_training`, aristos_config.schema.json:20-23) that none of its code reads.
Here it has a consumer: `MoE355Train` runs the expert projections through `moe_expert_gemm` and gets their gradients
from `moe_expert_gemm` on the transposed weight or `moe_expert_gemm_kn` on the weight as stored (data gradient) and
`moe_expert_wgrad` (weight gradient).  Routing
decisions (top-k indices, slots, capacity drops) come from the library's router and are not differentiated; the gate
weights that scale the expert outputs are, by the router's own kernels (`_RoutedExperts`) or, where those do not exist, as
torch ops on the same logits formula, so the router's weight matrix and the tokens receive gradients through them.
Everything else -- dispatch, projections, activation, combine -- is one autograd node (`_Experts`, or that node with the
router) whose backward runs the library's adjoints; the data gradient of the down projection
carries the activation's derivative in its epilogue (either product; `moe_expert_gemm_act_backward`) where the layer has that kernel,
else `moe_expert_gemm` is followed by `moe_act_backward`.  `expert_linear` and `act_down` are the projections as nodes
of their own, for layers composed in torch.  There is no CPU path: every tensor lives on the GPU.
"""
from __future__ import annotations

import torch

from . import api


class _ExpertLinear(torch.autograd.Function):
    """rows[r] -> rows[r] . w[e(r)]^T over packed expert-major rows (rows of no expert give zeros)."""

    @staticmethod
    def forward(ctx, a_rows, w, layer, count, offset):
        a_rows = a_rows.contiguous()
        ctx.save_for_backward(a_rows, w, count, offset)
        ctx.layer = layer
        return layer.expert_gemm(a_rows, w, None, count, offset, api.ACT_NONE)

    @staticmethod
    def backward(ctx, dy):
        a_rows, w, count, offset = ctx.saved_tensors
        layer = ctx.layer
        dy = dy.contiguous()
        da = dw = None
        if ctx.needs_input_grad[0]:
            da = layer.expert_gemm(dy, api.transpose(w), None, count, offset, api.ACT_NONE)      # dA = dY . W
        if ctx.needs_input_grad[1]:
            dw = layer.expert_wgrad(dy, a_rows, count, offset)                                     # dW[e] = dY_e^T . A_e
        return da, dw, None, None, None


def expert_linear(a_rows, w, layer: api.MoELayer, expert_count, expert_offset):
    return _ExpertLinear.apply(a_rows, w, layer, expert_count, expert_offset)


class _ActDown(torch.autograd.Function):
    """(u rows, g rows or None) -> act(u, g) . w_down[e(r)]^T over packed expert-major rows."""

    @staticmethod
    def forward(ctx, u, g, w, layer, count, offset):
        act = layer.cfg.hidden_act
        if act == api.ACT_SWIGLU:
            h = torch.nn.functional.silu(g.float()) * u.float()
        elif act == api.ACT_GELU:
            h = torch.nn.functional.gelu(u.float())
        else:
            h = torch.relu(u.float())
        h = h.to(u.dtype)
        ctx.save_for_backward(u, g, h, w, count, offset)
        ctx.layer = layer
        return layer.expert_gemm(h, w, None, count, offset, api.ACT_NONE)

    @staticmethod
    def backward(ctx, dy):
        u, g, h, w, count, offset = ctx.saved_tensors
        layer = ctx.layer
        dy = dy.contiguous()
        w_t = api.transpose(w)                                                                     # [E, I, H]
        if layer.fused_act_backward:
            du, dg = layer.expert_gemm_act_backward(dy, w_t, u, g, count, offset)
        else:
            dh = layer.expert_gemm(dy, w_t, None, count, offset, api.ACT_NONE)                     # dH = dY . W_down
            du, dg = layer.act_backward(dh, u, g)
        dw = layer.expert_wgrad(dy, h, count, offset) if ctx.needs_input_grad[2] else None
        return du, dg, dw, None, None, None


def act_down(u_rows, g_rows, w_down, layer: api.MoELayer, expert_count, expert_offset):
    return _ActDown.apply(u_rows.contiguous(), None if g_rows is None else g_rows.contiguous(), w_down, layer,
                          expert_count, expert_offset)


def _aligned(t):
    """t, contiguous and at a 16-byte address (the row passes read 16 bytes at a time)."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _own(t, given):
    """What a node keeps of `given`, the caller's router weights, of which `t` is the aligned form: 16-bit ones as a copy, so that they may
    be stepped before the backward (as with gate weights in torch, which reads fp32 copies of them; fp32 ones autograd keeps itself, and
    refuses them once they are changed)."""
    return t.clone() if t.dtype != torch.float32 and t.data_ptr() == given.data_ptr() else t


def _unpacked(ctx):
    """The saved tensors as the kernels take them: a saved-tensor hook may hand back views at any address."""
    saved = ctx.saved_tensors
    for t in saved:
        if t is not None and (t.data_ptr() & 15 or not t.is_contiguous()):
            return [None if t is None else _aligned(t) for t in saved]
    return saved                       # (without hooks)


def _as_stored(layer, w):
    """Whether a data gradient [rows, K] . w[e] takes the weight w [E, K, N] as it is (else: a transposed copy)."""
    return isinstance(layer, api.MoELayer) and w.data_ptr() % 16 == 0 and layer.gemm_kn_supported(w.shape[2], w.shape[1]) == 2


def _expert_rows(x, w_up, w_gate, w_down, layer, token_indices, count, offset):
    """The packed rows of the expert side's forward pass: tokens, projections u and g, activation h, outputs y."""
    rows = layer.dispatch_rows(_aligned(x), token_indices)

    def product(a, w):
        out = torch.empty(a.shape[0], w.shape[1], dtype=a.dtype, device=a.device)
        return layer.expert_gemm(a, w, None, count, offset, api.ACT_NONE, out=out)

    if w_gate is None:
        u, g = product(rows, w_up), None
    elif isinstance(layer, api.MoELayer):
        u, g = layer.expert_gemm_pair(rows, w_up, w_gate, count, offset)
    else:
        u, g = product(rows, w_up), product(rows, w_gate)
    h = layer.act_forward(u, g, count, offset)
    return rows, u, g, h, product(h, w_down)


def _kept(needs, rows, u, g, h, w_up, w_gate, w_down, need_rows=False):
    """What of the forward pass the gradients that are asked for read (a step that trains the router alone reads y)."""
    need_x, need_up, need_gate, need_down = needs
    need_u = need_x or need_up or need_gate

    def kept(needed, t):
        return t if needed else None

    return (kept(need_up or need_gate or need_rows, rows), kept(need_u, u), kept(need_u, g), kept(need_down, h),
            kept(need_x, w_up), kept(need_x, w_gate), kept(need_u, w_down))


def _expert_gradients(layer, needs, dy, kept, count, offset):
    """(da rows, db rows or None, dw_up, dw_gate, dw_down), each None where it is not asked for."""
    rows, u, g, h, w_up, w_gate, w_down = kept
    need_x, need_up, need_gate, need_down = needs

    def product(a, w_t):
        out = torch.empty(a.shape[0], w_t.shape[1], dtype=a.dtype, device=a.device)
        return layer.expert_gemm(a, w_t, None, count, offset, api.ACT_NONE, out=out)

    da = db = dup = dgate = ddown = du = dg = None
    if need_x or need_up or need_gate:
        if _as_stored(layer, w_down):
            du, dg = layer.expert_gemm_kn(dy, w_down, count, offset, u, g)                         # dH = dY . W_down, times act'
        elif layer.fused_act_backward:
            du, dg = layer.expert_gemm_act_backward(dy, api.transpose(w_down), u, g, count, offset, du=torch.empty_like(u),
                                                    dg=None if g is None else torch.empty_like(g))
        else:
            du, dg = layer.act_backward(product(dy, api.transpose(w_down)), u, g)
        if need_x:
            def data_gradient(d, w):                                                               # dA = dU . W_up
                return layer.expert_gemm_kn(d, w, count, offset) if _as_stored(layer, w) else product(d, api.transpose(w))

            if g is not None and _as_stored(layer, w_up) and _as_stored(layer, w_gate):
                da, db = layer.expert_gemm_kn_pair(du, dg, w_up, w_gate, count, offset)
            else:
                da = data_gradient(du, w_up)
                db = None if g is None else data_gradient(dg, w_gate)
    asked = [p for need, p in ((need_down, (dy, h)), (need_up, (du, rows)), (need_gate, (dg, rows))) if need]      # dW[e] = dU_e^T . A_e
    if not asked:
        grads = iter(())
    elif isinstance(layer, api.MoELayer):
        grads = iter(layer.expert_wgrads(asked, count, offset))
    else:
        grads = iter([layer.expert_wgrad(d, a, count, offset) for d, a in asked])
    ddown, dup, dgate = (next(grads) if need else None for need in (need_down, need_up, need_gate))
    return da, db, dup, dgate, ddown


class _Experts(torch.autograd.Function):
    """(x [S,H], expert weights, topk_w [S,k]) -> the gate-weighted sum of the chosen experts' outputs.

    The whole expert side of a training step as one node over packed rows.  No result depends on the rows of no expert, so no
    buffer is cleared (the activation's derivative as a pass of its own computes on what lies there; nobody reads that), and
    dispatch, activation, combine and their adjoints are one pass each."""

    @staticmethod
    def forward(ctx, x, w_up, w_gate, w_down, topk_w, layer, token_indices, pair_row, count, offset):
        w_up, w_down, topk_w = w_up.contiguous(), w_down.contiguous(), topk_w.contiguous()
        w_gate = None if w_gate is None else w_gate.contiguous()
        rows, u, g, h, y = _expert_rows(x, w_up, w_gate, w_down, layer, token_indices, count, offset)
        ctx.save_for_backward(*_kept(ctx.needs_input_grad[:4], rows, u, g, h, w_up, w_gate, w_down), y, topk_w, pair_row, count, offset)
        ctx.layer = layer
        return api.combine(y, pair_row, topk_w)

    @staticmethod
    def backward(ctx, dout):
        *kept, y, topk_w, pair_row, count, offset = _unpacked(ctx)
        layer, needs = ctx.layer, ctx.needs_input_grad[:4]
        dy, dtopk = layer.combine_backward(_aligned(dout), y, pair_row, topk_w, dy=torch.empty_like(y))
        da, db, dup, dgate, ddown = _expert_gradients(layer, needs, dy, kept, count, offset)
        dx = layer.dispatch_backward(da, db, pair_row) if needs[0] else None
        return dx, dup, dgate, ddown, dtopk, None, None, None, None, None


class _RoutedExperts(torch.autograd.Function):
    """(x [S,H], expert weights, gate_w [E,H]) -> the layer's output: `_Experts` with the router inside the node.

    The gate weights are the routing kernel's own and their adjoint rides in passes that run anyway: the combine's adjoint, one
    wavefront a token, goes on to the logits' gradients; the dispatch's adds their product with the router's weight rows to the
    tokens' gradient in fp32; what is left is one pass over the tokens' packed rows for the router's weight gradient.  As torch ops the router took
    about 25 launches and fp32 copies of x.  A bf16 step, before and after: 919 -> 793 us (4096 tokens, 16 experts of
    2048 x 2048, GELU), 1238 -> 1127 us (3000 tokens, 16 of 2048 x 1408, top-4, SwiGLU), 650 -> 375 us for 300 tokens of the first,
    where launches are the time."""

    @staticmethod
    def forward(ctx, x, w_up, w_gate, w_down, gate_w, layer, grad_enabled):
        x, gate, w_up, w_down = _aligned(x), _aligned(gate_w), w_up.contiguous(), w_down.contiguous()
        w_gate = None if w_gate is None else w_gate.contiguous()
        c = layer.cfg
        need_x, need_gate_w = (grad_enabled and ctx.needs_input_grad[i] for i in (0, 4))
        want_logits = (need_x or need_gate_w) and c.gate_fn != api.GATE_SOFTMAX and bool(c.norm_topk_prob)
        idx, topk_w, *logits = layer.gate(x, gate, want_logits=want_logits)
        r = layer.route(idx)
        pair_row, count, offset = r["pair_row"], r["expert_count"], r["expert_offset"]
        rows, u, g, h, y = _expert_rows(x, w_up, w_gate, w_down, layer, r["token_indices"], count, offset)
        # (the router's gradients read the tokens from their packed rows: x itself is not kept, and may change before the backward)
        ctx.save_for_backward(*_kept(ctx.needs_input_grad[:4], rows, u, g, h, w_up, w_gate, w_down, need_rows=need_gate_w), y, topk_w, pair_row,
                              count, offset, _own(gate, gate_w) if need_x else None, idx, *logits)
        ctx.layer = layer
        return api.combine(y, pair_row, topk_w)

    @staticmethod
    def backward(ctx, dout):
        rows, u, g, h, w_up, w_gate, w_down, y, topk_w, pair_row, count, offset, gate_w, idx, *logits = _unpacked(ctx)
        layer, needs = ctx.layer, ctx.needs_input_grad[:4]
        dout, dy, router = _aligned(dout), torch.empty_like(y), None
        if needs[0] or ctx.needs_input_grad[4]:
            router = torch.empty(layer.router_grad_bytes, dtype=torch.uint8, device=y.device)
            layer.combine_router_backward(dout, y, pair_row, topk_w, idx, logits[0] if logits else None, dy, router)
        else:
            layer.combine_backward(dout, y, pair_row, topk_w, dy=dy)
        kept = rows, u, g, h, w_up, w_gate, w_down
        da, db, dup, dgate, ddown = _expert_gradients(layer, needs, dy, kept, count, offset)
        dx = layer.dispatch_router_backward(da, db, pair_row, idx, router, gate_w) if needs[0] else None
        dgate_w = layer.gate_wgrad(rows, router, packed=True) if ctx.needs_input_grad[4] else None
        return dx, dup, dgate, ddown, dgate_w, None, None


class MoE355Train(torch.nn.Module):
    """forward(x [S,H]) -> [S,H] with gradients for x, gate_w, w_up, w_gate and w_down."""

    def __init__(self, cfg: api.MoEConfig, init_std: float = 0.02, seed: int = 0):
        super().__init__()
        if cfg.torch_dtype == api.DTYPE_FP8:
            raise ValueError("the backward building blocks exist for fp32, tf32, bf16 and fp16 layers, not for e4m3 weights")
        self.cfg = cfg
        self.layer = api.MoELayer(cfg)
        dt = self.layer.act_dtype
        E, H, I = cfg.num_experts, cfg.hidden_size, cfg.intermediate_size
        g = torch.Generator(device="cpu").manual_seed(seed)

        def p(*shape):
            return torch.nn.Parameter((torch.randn(*shape, generator=g) * init_std).to(dt).cuda())

        self.gate_w, self.w_up, self.w_down = p(E, H), p(E, I, H), p(E, H, I)
        self.w_gate = p(E, I, H) if cfg.hidden_act == api.ACT_SWIGLU else None

    def route(self, x):
        """The library's routing decision for x (no gradient): top-k indices and the packed-row tables."""
        with torch.no_grad():
            idx, _ = self.layer.gate(x.detach(), self.gate_w.detach())
            return idx, self.layer.route(idx)

    def gate_weights(self, x, idx):
        """The weights of the chosen experts, differentiable, by the formula the router kernel uses."""
        c = self.cfg
        logits = x.float() @ self.gate_w.float().t()
        scores = torch.softmax(logits, dim=1) if c.gate_fn == api.GATE_SOFTMAX else torch.sigmoid(logits)
        w = scores.gather(1, idx.long())
        return w / w.sum(1, keepdim=True) if c.norm_topk_prob else w

    def _routed(self, x):
        """Whether the router's gradients have kernels for this call; else the gate weights are torch ops.  Not under autocast,
        which computes the logits in 16 bits, not with a route or gate weights of a subclass's own, and not for a softmax that is
        not normalised over the chosen experts (every logit has a gradient there).  A single expert's normalised weight is one and
        the router's gradient nothing but the rounding of w / w: it stays what the torch expression gives."""
        return (not (self.cfg.expert_top_k == 1 and self.cfg.norm_topk_prob) and isinstance(self.layer, api.MoELayer) and x.is_cuda and x.dim() == 2 and x.shape[0] >= self.cfg.tokens
                and x.shape[1] == self.cfg.hidden_size and x.dtype == self.gate_w.dtype == self.layer.act_dtype
                and getattr(self.route, "__func__", None) is _ROUTE and getattr(self.gate_weights, "__func__", None) is _GATE_WEIGHTS
                and not torch.is_autocast_enabled("cuda") and self.layer.router_grad_bytes > 0)

    def forward(self, x):
        c = self.cfg
        if self._routed(x):
            rows = x if x.shape[0] == c.tokens else x[:c.tokens]
            return _RoutedExperts.apply(rows, self.w_up, self.w_gate, self.w_down, self.gate_w, self.layer, torch.is_grad_enabled())
        idx, r = self.route(x)
        count, offset = r["expert_count"], r["expert_offset"]
        # fp32 whatever gate_weights computed in: the combine reads fp32 (under autocast the logits, and with them a sigmoid's
        # weights, are 16 bits wide); the cast is undone by autograd
        w = self.gate_weights(x, idx).float()
        rows = x if x.shape[0] == c.tokens else x[:c.tokens]      # rows behind the layer's tokens: zero gradients
        return _Experts.apply(rows, self.w_up, self.w_gate, self.w_down, w, self.layer, r["token_indices"], r["pair_row"],
                              count, offset)


_ROUTE, _GATE_WEIGHTS = MoE355Train.route, MoE355Train.gate_weights
