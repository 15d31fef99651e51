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
    for call in (lambda: layer.dispatch_rows(x[:7], tok), lambda: layer.combine_backward(x[:7], rows, pairs, w)):
        with pytest.raises(ValueError):
            call()
