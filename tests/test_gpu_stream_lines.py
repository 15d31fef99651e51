"""The weight streamers where their weights are more than the memory-side cache holds (fetched once and not kept) against the same layer
where they are not: a layer of the same experts beside others that no token reaches has the same rows, and the same bits."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [2, 3, 4])
@pytest.mark.parametrize("act", [1, 2])
@pytest.mark.parametrize("S,H,I,k", [(20, 2048, 2176, 2), (40, 1536, 2048, 2), (70, 1536, 2176, 3)])
def test_cold_and_kept_weights_give_the_same_bits(S, H, I, k, act, dtype):
    import torch
    import cuplayground_amd as moe
    from cuplayground_amd import api

    g = torch.Generator(device="cuda").manual_seed(S + act)
    small = 8                                        # experts that tokens reach
    big = 112                                        # ... of that many in a layer whose weights are not kept
    adt = torch.float16 if dtype == 3 else torch.bfloat16
    x = torch.randn(S, H, generator=g, device="cuda").to(adt)
    mats = {"w_up": (I, H), "w_down": (H, I), **({"w_gate": (I, H)} if act == 2 else {})}
    w = {n: torch.randn(small, *s, generator=g, device="cuda") * 0.05 for n, s in mats.items()}
    gate = (torch.randn(small, H, generator=g, device="cuda") * 0.1).to(adt)
    hit = [min(S * k, E) * sum(a * b for a, b in mats.values()) * (1 if dtype == 4 else 2) for E in (small, big)]
    assert hit[0] <= 256 << 20 < hit[1]              # (stream_cold, csrc/stream_lines.hpp)
    outs = []
    for E in (small, big):
        cfg = moe.MoEConfig(capacity_factor=1.0, drop_tokens=0, expert_top_k=k, is_training=0, hidden_act=act, hidden_size=H, intermediate_size=I,
                            micro_batch=1, num_experts=E, sequence_len=S, torch_dtype=dtype, gate_fn=1, norm_topk_prob=1)
        d = {"gate_w": torch.zeros(E, H, dtype=adt, device="cuda"), "gate_bias": torch.full((E,), -float("inf"), device="cuda")}
        d["gate_w"][:small], d["gate_bias"][:small] = gate, 0.0
        for n, t in w.items():
            if dtype == 4:
                q, s = api.quantize_block128(t)
                d[n] = torch.zeros(E, *t.shape[1:], dtype=q.dtype, device="cuda")
                d["s" + n[1:]] = torch.zeros(E, *s.shape[1:], device="cuda")
                d[n][:small], d["s" + n[1:]][:small] = q, s
            else:
                d[n] = torch.zeros(E, *t.shape[1:], dtype=adt, device="cuda")
                d[n][:small] = t.to(adt)
        # (26 rows an expert: e4m3 layers of so many take the tile by themselves)
        outs.append(moe.MoELayer(cfg, options={"fp8_tile": 0} if dtype == 4 else None).forward(x, d))
    assert outs[0].isfinite().all() and outs[0].any()
    assert torch.equal(outs[0], outs[1])
