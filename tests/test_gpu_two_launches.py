"""The two launches of a 16-bit layer on row blocks and remainders (csrc/ffn_bf16_grouped.hip: grouped_task,
launch_ffn_split_16): every tile is taken once, by the same arithmetic as on the task queue, so the bits are the queue's."""
import numpy as np
import pytest

from oracle import binding as ob
from helpers import OUT_TOL, from_device, max_rel_err, product_config, upload_inputs
from test_gpu_layer import FFN_PERSISTENT, FFN_TILED, check_routing

pytestmark = pytest.mark.gpu

SHAPES = {
    # more experts than a wavefront has lanes, most of them with a few rows, some with none; one column tile and a ragged one
    "many_experts": (ob.Cfg(S=200, H=128, I=320, E=150, k=2, act=ob.ACT_SWIGLU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=0), False),
    # remainders of every kind, ragged columns, biases
    "ragged_gelu": (ob.Cfg(S=1531, H=448, I=704, E=9, k=3, act=ob.ACT_GELU, dtype=ob.F16, gate_fn=ob.GATE_SIGMOID, drop=0), True),
    "ragged_swiglu": (ob.Cfg(S=1100, H=320, I=448, E=5, k=2, act=ob.ACT_SWIGLU, dtype=ob.BF16, gate_fn=ob.GATE_SIGMOID, drop=0), True),
    # capacities that are no whole row blocks, and ones that are: 384 rows are a block and a full remainder
    "capped": (ob.Cfg(S=1536, H=256, I=256, E=8, k=2, act=ob.ACT_RELU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=1, capacity_factor=0.7), False),
    "capped_blocks": (ob.Cfg(S=1536, H=256, I=256, E=8, k=2, act=ob.ACT_GELU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=1, capacity_factor=1.0), False),
    "one_token": (ob.Cfg(S=1, H=256, I=512, E=4, k=1, act=ob.ACT_GELU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=0), False),
}


def _forward(cfg, dev, mode, tile):
    import torch
    import cuplayground_amd as moe
    layer = moe.MoELayer(product_config(cfg), ffn_mode=mode, options={"tile16": tile})
    routing = layer.new_routing()
    out = torch.full((cfg.S, cfg.H), float("nan"), dtype=layer.act_dtype, device="cuda")
    layer.forward(dev["x"], dev, out=out, routing=routing)
    torch.cuda.synchronize()
    layer.task_counts()
    res = {k: from_device(v) for k, v in routing.items()}
    res["out"] = from_device(out)
    layer.close()
    return res


@pytest.mark.parametrize("tile", [1, 2, 3])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_same_bits_as_the_queue(name, tile):
    cfg, bias = SHAPES[name]
    inp = ob.make_inputs(cfg, seed=5, with_bias=bias)
    want = ob.forward(cfg, inp)
    dev = upload_inputs(cfg, inp)
    got = _forward(cfg, dev, FFN_TILED, tile)
    check_routing(got, want)
    assert max_rel_err(ob.to_f32(got["out"], cfg.act_dtype), ob.to_f32(want["out"], cfg.act_dtype)) <= OUT_TOL[cfg.dtype]
    assert np.array_equal(got["out"], _forward(cfg, dev, FFN_PERSISTENT, tile)["out"])


@pytest.mark.parametrize("rows, experts, tokens, queue", [(64, 16, 512, False), (192, 64, 2048, False), (200, 64, 2134, True)])
def test_mode_that_is_chosen(rows, experts, tokens, queue):
    """Few rows per expert: two launches, also where there are many tasks; the queue's trace keeps it."""
    import cuplayground_amd as moe
    cfg = ob.Cfg(S=tokens, H=2048, I=1408, E=experts, k=6 if experts == 64 else 2, act=ob.ACT_SWIGLU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=0)
    layer = moe.MoELayer(product_config(cfg))
    assert (layer.ffn_mode == FFN_PERSISTENT) == queue
    if experts == 64:
        layer.enable_task_trace(1 << 10)
        assert layer.ffn_mode == FFN_PERSISTENT
        layer.disable_task_trace()
    layer.close()


@pytest.mark.parametrize("option", ["queue_groups", "queue_lag", "row_chunk", "blocks_per_cu", "tail_round", "queue_early"])
@pytest.mark.parametrize("rows, tile", [(94, 2), (160, 1)])
def test_options_of_the_queue_keep_it(rows, tile, option):
    """Any option of the queue that differs from what AUTO gives; a handle made from another one's options runs as that one does."""
    import cuplayground_amd as moe
    cfg = ob.Cfg(S=rows * 64 // 6, H=2048, I=1408, E=64, k=6, act=ob.ACT_SWIGLU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=0)
    layer = moe.MoELayer(product_config(cfg))
    assert layer.options["tile16"] == tile and layer.ffn_mode == FFN_TILED
    same = moe.MoELayer(product_config(cfg), options=layer.options)
    assert same.ffn_mode == FFN_TILED
    value = {"queue_groups": 2, "queue_lag": 1, "row_chunk": 3, "blocks_per_cu": layer.options["blocks_per_cu"] + 1, "tail_round": 0, "queue_early": 1}
    kept = moe.MoELayer(product_config(cfg), options={option: value[option]})
    assert (kept.ffn_mode == FFN_PERSISTENT) == (option != "queue_early" or tile == 1)      # (an option of the 256 x 256 tile)
    for l in (layer, same, kept):
        l.close()


@pytest.mark.parametrize("S,H,I,E,k,tile", [(900, 1984, 3008, 20, 3, 2), (1300, 1984, 3008, 20, 3, 2), (2300, 2048, 2048, 16, 2, 1), (1000, 320, 448, 5, 2, 2)])
def test_same_bits_whatever_blocks_the_rounds_choose(S, H, I, E, k, tile):
    """Layers planned on 128-row blocks whose launches take 256-row blocks and remainders, layers that keep the table's order, and
    ones on either side of the choice: an output is the same sum over k whichever tile holds it."""
    import torch
    import cuplayground_amd as moe
    cfg = ob.Cfg(S=S, H=H, I=I, E=E, k=k, act=ob.ACT_SWIGLU, dtype=ob.BF16, gate_fn=ob.GATE_SIGMOID, drop=0)
    g = torch.Generator(device="cuda").manual_seed(S)

    def normal(*shape):
        return (torch.randn(*shape, generator=g, device="cuda") * 0.02).bfloat16()

    dev = {"x": normal(S, H) * 50, "gate_w": normal(E, H), "w_up": normal(E, I, H), "w_gate": normal(E, I, H), "w_down": normal(E, H, I)}
    got = _forward(cfg, dev, FFN_TILED, tile)["out"]
    assert np.isfinite(ob.to_f32(got, cfg.act_dtype)).all()
    assert np.array_equal(got, _forward(cfg, dev, FFN_PERSISTENT, tile)["out"])


@pytest.mark.parametrize("E,k,H,I,rows,drop,queue", [(64, 6, 2048, 1408, 1434, 0, False), (64, 6, 2048, 1408, 1434, 1, True), (64, 6, 2048, 1408, 1024, 0, True),
                                                     (8, 2, 4096, 14336, 5734, 0, True), (32, 4, 2048, 2816, 2867, 0, True)])
def test_many_rounds_leave_the_queue_where_their_rows_stay_in_the_caches(E, k, H, I, rows, drop, queue):
    import cuplayground_amd as moe
    cfg = ob.Cfg(S=rows * E // k, H=H, I=I, E=E, k=k, act=ob.ACT_SWIGLU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=drop)
    layer = moe.MoELayer(product_config(cfg), allocate_workspace=False)
    assert (layer.ffn_mode == FFN_PERSISTENT) == queue
    layer.close()


def test_capped_layers_of_few_rows_keep_the_queue():
    import cuplayground_amd as moe
    for factor, queue in ((1.0, True), (2.0, False)):
        cfg = ob.Cfg(S=400, H=2048, I=1408, E=64, k=6, act=ob.ACT_SWIGLU, dtype=ob.BF16, gate_fn=ob.GATE_SOFTMAX, drop=1, capacity_factor=factor)
        layer = moe.MoELayer(product_config(cfg))
        assert (layer.ffn_mode == FFN_PERSISTENT) == queue
        layer.close()
