"""The logits kernel whose workgroups take several tiles, and the selection by sixteen lanes a token: the bits of the other kernels."""
import pytest

pytestmark = pytest.mark.gpu


def _layer(S, H, E, k, gate_fn, norm, dtype, **options):
    import cuplayground_amd as moe
    cfg = moe.MoEConfig(capacity_factor=1.0, drop_tokens=0, expert_top_k=k, is_training=0, hidden_act=1, hidden_size=H, intermediate_size=64,
                        micro_batch=1, num_experts=E, sequence_len=S, torch_dtype=dtype, gate_fn=gate_fn, norm_topk_prob=norm)
    return moe.MoELayer(cfg, options=options)


def _inputs(S, H, E, dtype):
    import torch
    g = torch.Generator(device="cuda").manual_seed(S + E)
    dt = {2: torch.bfloat16, 3: torch.float16}[dtype]
    return (torch.randn(S, H, generator=g, device="cuda").to(dt), (torch.randn(E, H, generator=g, device="cuda") * 0.1).to(dt),
            torch.randn(E, generator=g, device="cuda") * 0.1)


# tiles per workgroup: one, several and a ragged last round, one step a tile, expert columns that end inside a tile
@pytest.mark.parametrize("dtype", [2, 3])
@pytest.mark.parametrize("S,H,E", [(2500, 512, 64), (20001, 512, 64), (9000, 1536, 40), (700, 1024, 300), (1, 512, 1), (33, 2048, 33)])
def test_logits_of_workgroups_that_stay(S, H, E, dtype):
    import torch
    x, w, b = _inputs(S, H, E, dtype)
    got, want = (_layer(S, H, E, 1, 0, 1, dtype, gate_mfma=m).gate(x, w, b, want_logits=True) for m in (1, 0))
    assert all(torch.equal(p, q) for p, q in zip(got, want))


@pytest.mark.parametrize("gate_fn,norm", [(0, 1), (0, 0), (1, 1)])
@pytest.mark.parametrize("S,E,k", [(1, 1, 1), (5, 16, 16), (77, 17, 3), (300, 33, 8), (1000, 64, 6), (19, 64, 16)])
def test_selection_by_rows_of_lanes(S, E, k, gate_fn, norm):
    """Against the wavefront's selection (moe_gate of a layer that has more experts, the rest of them out of reach)."""
    import torch
    x, w, b = _inputs(S, 512, E, 2)
    w[E // 2], b[E // 2] = w[0], b[0]                    # ties
    if S > 10:
        x[3, 5], x[7, 1], x[9] = float("nan"), float("inf"), 0.0
    rows = _layer(S, 512, E, k, gate_fn, norm, 2, gate_fused_topk=0).gate(x, w, b)
    far = torch.full((70,), -float("inf"), device="cuda")
    far[:E] = b
    wide = torch.zeros(70, 512, dtype=w.dtype, device="cuda")
    wide[:E] = w
    waves = _layer(S, 512, 70, k, gate_fn, norm, 2, gate_fused_topk=0).gate(x, wide, far)
    clean = torch.ones(S, dtype=torch.bool, device="cuda")
    if S > 10:
        clean[3] = clean[7] = False                      # there the experts out of reach are NaN too
        assert rows[0].min() >= 0 and rows[0].max() < E and rows[1][3].isnan().all()
    assert torch.equal(rows[0][clean], waves[0][clean]) and torch.equal(rows[1][clean], waves[1][clean])
