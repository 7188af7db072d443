"""The tile path's choice of weight loads per expert (moe_gemm_lds.hip,
moe_gemm_tile.hip): at H 2048, I 512 an expert with one block pair (gate/up) or
one block (down) reads its weights non-temporally. Every token is on the same
experts (T rows each, and the shared expert), so T moves all of them across the
edges: one block, two, an absorbed tail of 1 and 16 rows, a pair of its own,
two pairs with a tail. Bars of the parity tests: the layer output within 2e-2
of the float64 oracle, bitwise equal on a second launch."""
import numpy as np
import pytest

from conftest import gpu_available
from netra_moe.config import MoEConfig


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("T,H,I", [(t, 2048, 512) for t in (64, 65, 128, 129, 144, 145, 257, 272)]
                         + [(t, 1024, 1024) for t in (300, 700, 2000)])  # I 1024: down_tile, down_rows of 2 and 4 groups
def test_experts_of_every_block_count(T, H, I):
    import torch

    import oracle
    from moe_case import make_inputs, oracle_routing, run_gpu, sample_tokens

    cfg = MoEConfig(f"reads_t{T}_h{H}", T=T, H=H, E=8, K=2, I=I, S=1, router_bias="hot", seed=1300 + T)
    print(f"\n[reads] {cfg}", flush=True)
    dev = torch.device("cuda", 0)
    x, gpu_w, host = make_inputs(cfg, dev)
    got = run_gpu(cfg, x, gpu_w, dev, expose=("topk_ids",), repeats=2, path="tile")
    np.testing.assert_array_equal(got["runs"][0], got["runs"][1])
    ref = oracle_routing(cfg, host)
    np.testing.assert_array_equal(got["topk_ids"], ref["topk_ids"])
    tokens = sample_tokens(cfg, 64)
    out, _ = oracle.moe_tokens(ref["x_q"], ref["x_scale"], host["w13"], host["w13_scale"], host["w2"],
                               host["w2_scale"], ref["topk_ids"], ref["topk_weights"], tokens, cfg.H, cfg.I)
    assert oracle.max_abs_rel(oracle.f32_from_bf16(got["out"][tokens]), out) <= 2e-2
