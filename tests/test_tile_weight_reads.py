"""The tile path's choice of weight loads (moe_gemm_lds.hip, moe_gemm_tile.hip).

CPU: when a call takes the _cached kernels, by rows per expert and by the size
of the weights; the others load the weights of an expert with one block
(gate/up: one block pair) non-temporally. GPU: those against the _cached ones
(the same arithmetic: bit for bit) and the float64 oracle. Every token is on the
same experts (T rows each, and the shared expert), so T moves all of them across
the edges: one block, two, an absorbed tail of 1 and 16 rows, a pair of its own,
two pairs with a tail. Bars of the parity tests: the layer output within 2e-2 of the oracle,
bitwise equal on a second launch."""
import numpy as np
import pytest

from conftest import gpu_available
from netra_moe import engine
from netra_moe.config import MoEConfig


# (T, H, I, E, K, S) -> whether gate/up reads one-pair experts' W13 non-temporally
@pytest.mark.parametrize("shape,chooses", [
    ((512, 2048, 512, 256, 8, 1), True), ((4096, 2048, 512, 256, 8, 1), True), ((4097, 2048, 512, 256, 8, 1), False),
    ((1040, 2048, 512, 16, 4, 1), False), ((512, 2048, 512, 8, 2, 1), False), ((300, 2048, 512, 16, 4, 0), True)])
def test_gate_up_rule(shape, chooses):
    T, H, I, E, K, S = shape
    cfg = MoEConfig("rule", T=T, H=H, E=E, K=K, I=I, S=S)
    sym = next(o for o in engine.operations(cfg, "tile") if o["name"] == "moe.gate_up")["symbol"]
    assert sym == f"netra_moe_gate_up_lds_h{H}{'' if chooses else '_cached'}_gfx950"


# (T, H, I, E, K, S) -> whether down reads one-block experts' W2 non-temporally
@pytest.mark.parametrize("shape,chooses", [
    ((300, 2048, 512, 256, 8, 1), True), ((2560, 2048, 512, 256, 8, 1), True), ((2561, 2048, 512, 256, 8, 1), False),
    ((4096, 2048, 512, 256, 8, 1), False), ((300, 2048, 512, 32, 4, 0), True), ((300, 2048, 512, 31, 4, 0), False),
    ((1040, 2048, 512, 16, 4, 1), False), ((512, 2048, 512, 8, 2, 1), False), ((300, 512, 256, 256, 8, 0), True),
    ((300, 512, 256, 16, 2, 0), False), ((512, 512, 256, 64, 4, 1), False), ((300, 4096, 256, 32, 4, 1), True),
    ((300, 4096, 256, 16, 4, 1), False)])
def test_down_rule(shape, chooses):
    T, H, I, E, K, S = shape
    cfg = MoEConfig("rule", T=T, H=H, E=E, K=K, I=I, S=S)
    sym = next(o for o in engine.operations(cfg, "tile") if o["name"] == "moe.down")["symbol"]
    assert sym == f"netra_moe_down_rows_i{I}{'' if chooses else '_cached'}_gfx950"


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("T,H,I", [(t, 2048, 512) for t in (64, 65, 128, 129, 144, 145, 257, 272)]
                         + [(t, h, 256) for h in (512, 4096) for t in (64, 65, 130)]
                         + [(t, 1024, 1024) for t in (300, 700, 2000)])  # I 1024: down_tile, down_rows of 2 and 4 groups
def test_experts_of_every_block_count(T, H, I, monkeypatch):
    import torch

    import oracle
    from moe_case import make_inputs, oracle_routing, run_gpu, sample_tokens

    cfg = MoEConfig(f"reads_t{T}_h{H}", T=T, H=H, E=8, K=2, I=I, S=1, router_bias="hot", seed=1300 + T)
    print(f"\n[reads] {cfg}", flush=True)
    dev = torch.device("cuda", 0)
    x, gpu_w, host = make_inputs(cfg, dev)
    assert engine.weights_cached(cfg, "down") and engine.weights_cached(cfg, "gate_up")
    cached = run_gpu(cfg, x, gpu_w, dev, expose=("topk_ids",), repeats=2, path="tile")
    np.testing.assert_array_equal(cached["runs"][0], cached["runs"][1])
    monkeypatch.setattr(engine, "weights_cached", lambda cfg, op: False)
    got = run_gpu(cfg, x, gpu_w, dev, expose=("topk_ids",), repeats=2, path="tile")
    np.testing.assert_array_equal(got["runs"][0], got["runs"][1])
    np.testing.assert_array_equal(cached["out"], got["out"])
    ref = oracle_routing(cfg, host)
    np.testing.assert_array_equal(got["topk_ids"], ref["topk_ids"])
    tokens = sample_tokens(cfg, 64)
    out, _ = oracle.moe_tokens(ref["x_q"], ref["x_scale"], host["w13"], host["w13_scale"], host["w2"],
                               host["w2_scale"], ref["topk_ids"], ref["topk_weights"], tokens, cfg.H, cfg.I)
    assert oracle.max_abs_rel(oracle.f32_from_bf16(got["out"][tokens]), out) <= 2e-2
