"""The wide decode gate/up with fewer columns per workgroup: when the engine
takes it, and on the GPU each kernel at one and several rounds of items against
the float64 oracle (the parity tests' bar, 2e-2) with the sorted format exact."""
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
]


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


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("bias", ["none", "hot"])
@pytest.mark.parametrize("shape", [s for s, p in CASES if p < engine.FFN_WIDE_P[(s[1], s[2])]])
def test_against_the_oracle(shape, bias):
    import torch

    import oracle
    from moe_case import make_inputs, oracle_routing, run_gpu

    cfg = config(shape, router_bias=bias)
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
