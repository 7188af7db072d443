"""The wide decode gate/up with fewer columns per workgroup: when the engine
takes it, and on the GPU each kernel at one round of items and (chosen by hand:
the rule takes them for one) at more than the 256 of a round, against the float64
oracle (the parity tests' bar, 2e-2) with the sorted format exact."""
import numpy as np
import pytest

from conftest import gpu_available
from netra_moe import engine
from netra_moe.config import MoEConfig

# (T, H, I, E, K, S) -> P
CASES = [
    ((17, 2048, 512, 256, 8, 1), 2), ((19, 2048, 512, 256, 8, 1), 2), ((21, 2048, 512, 256, 8, 1), 4),
    ((64, 2048, 512, 64, 4, 1), 2), ((40, 2048, 512, 32, 4, 0), 1),
    ((40, 1024, 1024, 24, 3, 1), 1), ((64, 1024, 1024, 48, 4, 1), 2), ((64, 1024, 1024, 200, 8, 1), 4),
    ((64, 4096, 256, 32, 4, 1), 1), ((64, 4096, 256, 300, 8, 1), 2),
    # experts of more than 16 rows: two and more tiles each
    ((32, 1024, 1024, 16, 8, 1), 1), ((48, 1024, 1024, 16, 8, 1), 2), ((64, 1024, 1024, 16, 8, 1), 2),
    ((40, 1024, 1024, 24, 8, 1), 1), ((64, 1024, 1024, 24, 8, 1), 2), ((64, 2048, 512, 24, 8, 1), 1),
    ((20, 2048, 512, 256, 8, 1), 2), ((64, 2048, 512, 64, 8, 1), 2), ((40, 2048, 512, 256, 4, 1), 4),
    ((60, 1024, 1024, 16, 15, 0), 2), ((60, 2048, 512, 16, 15, 0), 1), ((60, 2048, 512, 32, 12, 1), 2),
]
# (T, H, I, E, K, S), P: calls of more than one round of items
ROUNDS = [((64, 1024, 1024, 16, 8, 1), 1), ((64, 1024, 1024, 64, 8, 1), 2), ((64, 2048, 512, 64, 8, 1), 1),
          ((64, 2048, 512, 160, 8, 1), 2), ((64, 4096, 256, 160, 8, 1), 1)]


def config(shape, **kw):
    T, H, I, E, K, S = shape
    return MoEConfig(f"spread_t{T}_h{H}_e{E}", T=T, H=H, E=E, K=K, I=I, S=S, seed=1400 + T, **kw)


@pytest.mark.parametrize("shape,P", CASES)
def test_columns_per_workgroup(shape, P):
    cfg = config(shape)
    assert engine.ffn_wide_p(cfg) == P
    sym = engine.operations(cfg, "fused")[1]["symbol"]
    full = engine.FFN_WIDE_P[(cfg.H, cfg.I)]
    assert ("gate_up_down" in sym) or sym.endswith("_wide_gfx950" if P == full else f"_wide_p{P}_gfx950")


@pytest.mark.parametrize("T,E,K,S", [(64, 16, 8, 1), (64, 24, 8, 1), (40, 24, 8, 0), (64, 32, 15, 1), (17, 16, 2, 1),
                                     (64, 8, 8, 1), (3000, 16, 4, 1)])
def test_expected_tiles_counts_every_tile_of_an_expert(T, E, K, S):
    rng = np.random.default_rng(T * E + K)
    counts = np.stack([np.bincount(np.argsort(rng.random((T, E)), axis=1)[:, :K].ravel(), minlength=E)
                       for _ in range(400)])
    tiles = ((counts + 15) // 16).sum(1) + S * ((T + 15) // 16)
    assert engine.expected_tiles(config((T, 2048, 512, E, K, S))) == pytest.approx(tiles.mean(), rel=0.01)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("bias", ["none", "hot"])
@pytest.mark.parametrize("shape", [s for s, p in CASES if p < engine.FFN_WIDE_P[(s[1], s[2])]])
def test_against_the_oracle(shape, bias):
    against_the_oracle(config(shape, router_bias=bias))


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("shape,P", ROUNDS)
def test_several_rounds_of_items(shape, P, monkeypatch):
    monkeypatch.setattr(engine, "ffn_wide_p", lambda cfg: P)
    monkeypatch.setattr(engine, "down_variant", lambda cfg: "wide")
    cfg = config(shape)
    tiles = (against_the_oracle(cfg)["expert_counts"] + 15) // 16
    assert tiles.sum() * (cfg.I // 128) // P > engine.FFN_GRID[("gate_up", "wide")]


def against_the_oracle(cfg):
    import torch

    import oracle
    from moe_case import make_inputs, oracle_routing, run_gpu

    print(f"\n[spread] {cfg}", flush=True)
    dev = torch.device("cuda", 0)
    x, gpu_w, host = make_inputs(cfg, dev)
    got = run_gpu(cfg, x, gpu_w, dev, expose=("topk_ids", "sorted_ids"), repeats=2, path="fused")
    np.testing.assert_array_equal(got["runs"][0], got["runs"][1])
    ref = oracle_routing(cfg, host)
    np.testing.assert_array_equal(got["sorted_ids"], ref["sorted_ids"])
    out, _ = oracle.moe_tokens(ref["x_q"], ref["x_scale"], host["w13"], host["w13_scale"], host["w2"],
                               host["w2_scale"], ref["topk_ids"], ref["topk_weights"],
                               np.arange(cfg.T, dtype=np.int64), cfg.H, cfg.I)
    assert oracle.max_abs_rel(oracle.f32_from_bf16(got["out"]), out) <= 2e-2
    return ref
