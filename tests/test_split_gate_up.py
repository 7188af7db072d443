"""The split gate/up (moe_gemm_split.hip): its dealing of chunks on the CPU,
and on the GPU the kernel against the path's general kernels and the oracle.

CPU: the kernel's own chunk table and shares (moe_split_table.h, compiled for
the host) against a restatement of the cut, covering every (16-row tile of an
expert, 128-column block of h) exactly once and keeping every chunk inside its
expert's rows, for drawn and extreme row counts and one to nine experts per
lane.

GPU, at the sizes where a tile count changes (hot: every token on the same
experts, T rows each): the layer output within the parity bar (2e-2) of the
float64 oracle, and h against the general kernel of the same path on the same
inputs: the row scales within one bf16 step (2^-7) and under 1% of the E4M3
codes different (two fp32 orders of the same sums; the bars of the parity
tests).
"""
import subprocess
from pathlib import Path

import numpy as np
import pytest

from conftest import REPO, gpu_available
from netra_moe import engine
from netra_moe.config import MoEConfig

RM, GRID = 4, engine.SPLIT_GRID


def chunks_of(counts):
    """(expert, first sorted row, tiles) of every chunk, in order."""
    out, block = [], 0
    for e, n in enumerate(counts):
        tiles = -(-n // 16)
        nc = -(-tiles // RM)
        for c in range(nc):
            t0, t1 = c * tiles // nc, (c + 1) * tiles // nc
            out.append((e, block * 64 + 16 * t0, t1 - t0))
        block += -(-n // 64)
    return out


@pytest.fixture(scope="module")
def host_table(tmp_path_factory):
    exe = tmp_path_factory.mktemp("split") / "table"
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", f"-I{REPO / 'netra-kernel_amd' / 'csrc' / 'kernels'}",
                    str(Path(__file__).with_name("split_table_host.cpp")), "-o", str(exe)], check=True)

    def run(counts, blocks, T):
        text = " ".join(map(str, [T, len(counts), RM, GRID, blocks, *counts]))
        lines = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.split("\n")[:-1]
        chunks = [tuple(map(int, ln.split())) for ln in lines if not ln.startswith("share")]
        return chunks, [tuple(map(int, ln.split()[1:])) for ln in lines if ln.startswith("share")]

    return run


@pytest.mark.parametrize("seed,experts,top", [(0, 257, 13), (1, 257, 70), (2, 513, 5), (3, 24, 416), (4, 1, 1),
                                              (5, 33, 64), (6, 513, 416), (7, 64, 17), (8, 65, 129), (9, 512, 1)])
def test_every_tile_and_column_block_is_dealt_once(seed, experts, top, host_table):
    rng = np.random.default_rng(seed)
    counts = rng.integers(0, top + 1, experts)
    counts[rng.integers(experts)] = top
    blocks = 4  # I = 512
    chunks, shares = host_table(counts, blocks, top)
    assert chunks == chunks_of(counts)
    seen = np.zeros((sum(-(-n // 64) for n in counts) * 4, blocks), np.int64)
    for lo, hi in shares:
        assert hi - lo - len(chunks) * blocks // GRID in (0, 1)
        for pos in range(lo, hi):
            e, row0, tiles = chunks[pos // blocks]
            assert 1 <= tiles <= RM
            base = 64 * sum(-(-n // 64) for n in counts[:e])
            assert base <= row0 and row0 + 16 * tiles <= base + 16 * -(-counts[e] // 16)
            seen[row0 // 16:row0 // 16 + tiles, pos % blocks] += 1
    want = np.zeros_like(seen)
    block = 0
    for n in counts:
        want[4 * block:4 * block + -(-n // 16)] = 1
        block += -(-n // 64)
    np.testing.assert_array_equal(seen, want)


def test_counts_beyond_the_tokens_are_clamped(host_table):
    chunks, _ = host_table([1 << 30, 3], 4, 20)
    assert chunks == chunks_of([20, 3])


@pytest.mark.parametrize("T,E,K,path,split", [(65, 256, 8, "stream", True), (416, 256, 8, "tile", True),
                                              (417, 256, 8, "tile", False), (512, 256, 8, "tile", False),
                                              (100, 24, 4, "stream", False)])
def test_rule_by_rows_per_expert(T, E, K, path, split):
    cfg = MoEConfig("rule", T=T, H=2048, E=E, K=K, I=512, S=1)
    assert engine.split_gate_up(cfg, path) == split
    sym = next(o for o in engine.operations(cfg, path) if o["name"] == "moe.gate_up")["symbol"]
    assert ("split" in sym) == split


# Calls that it slows (both ways, or more by skewed routing than it gains by uniform), and their neighbours
@pytest.mark.parametrize("T,E,K,S,path,split", [
    (80, 8, 1, 1, "stream", False), (100, 16, 2, 1, "stream", False), (100, 32, 4, 1, "stream", False),
    (128, 64, 4, 1, "stream", False), (100, 256, 4, 1, "stream", False), (128, 256, 4, 1, "stream", False),
    (129, 256, 4, 1, "stream", True), (65, 64, 8, 1, "stream", True), (128, 128, 8, 1, "stream", True),
    (65, 512, 10, 1, "stream", True), (256, 512, 10, 1, "stream", True), (65, 256, 8, 1, "stream", True),
    (256, 256, 8, 1, "stream", True), (257, 256, 8, 1, "tile", True), (416, 256, 8, 1, "tile", True),
    (400, 256, 4, 1, "tile", False), (1000, 256, 2, 1, "tile", False), (3000, 256, 1, 1, "tile", False),
    (300, 192, 6, 1, "tile", False), (416, 512, 10, 1, "tile", False)])
def test_rule_by_rows(T, E, K, S, path, split):
    cfg = MoEConfig("rule", T=T, H=2048, E=E, K=K, I=512, S=S)
    assert engine.split_gate_up(cfg, path) == split


GPU_CASES = {
    "t65": (dict(T=65, E=256, K=8, S=1), "stream"),
    "t1": (dict(T=1, E=256, K=8, S=1), "stream"),
    "t16_hot": (dict(T=16, E=256, K=8, S=1, router_bias="hot"), "stream"),
    "t17_hot": (dict(T=17, E=256, K=8, S=1, router_bias="hot"), "stream"),
    "t64_hot": (dict(T=64, E=256, K=8, S=0, router_bias="hot"), "stream"),
    "t65_hot": (dict(T=65, E=256, K=8, S=1, router_bias="hot"), "stream"),
    "t129_hot": (dict(T=129, E=128, K=4, S=1, router_bias="hot"), "tile"),
    "t40_e500": (dict(T=40, E=500, K=12, S=1), "tile"),
    "t70_e512": (dict(T=70, E=512, K=10, S=1), "stream"),
    "t333_zipf": (dict(T=333, E=256, K=8, S=1, router_bias="zipf1.1"), "tile"),
}


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("name", sorted(GPU_CASES))
def test_against_the_general_kernels_and_the_oracle(name, monkeypatch):
    import torch

    import oracle
    from moe_case import make_inputs, oracle_routing, run_gpu, sample_tokens

    shape, path = GPU_CASES[name]
    cfg = MoEConfig(f"split_{name}", H=2048, I=512, seed=1200 + len(name), **shape)
    print(f"\n[split] {cfg} path={path}", flush=True)
    dev = torch.device("cuda", 0)
    x, gpu_w, host = make_inputs(cfg, dev)
    expose = ("topk_ids", "sorted_ids", "h_q", "h_scale")
    assert engine.split_supported(cfg, path)  # whether or not the rule would take it
    with monkeypatch.context() as m:
        m.setattr(engine, "split_gate_up", lambda cfg, path: True)
        got = run_gpu(cfg, x, gpu_w, dev, expose=expose, repeats=2, path=path)
    with monkeypatch.context() as m:
        m.setattr(engine, "split_gate_up", lambda cfg, path: False)
        gen = run_gpu(cfg, x, gpu_w, dev, expose=expose, path=path)
    np.testing.assert_array_equal(got["runs"][0], got["runs"][1])
    np.testing.assert_array_equal(got["sorted_ids"], gen["sorted_ids"])
    rows = np.flatnonzero((got["sorted_ids"] & 0xFFFFFF) < cfg.T)
    if path == "stream":  # [tile][K block][2048] and [tile][K block][16]
        tile = lambda q: q.reshape(-1, cfg.I // 128, 2, 4, 16, 16).transpose(0, 4, 1, 3, 2, 5).reshape(-1, cfg.I)  # noqa: E731
        q0, q1 = tile(got["h_q"]), tile(gen["h_q"])
        s0, s1 = (r["h_scale"].transpose(0, 2, 1).reshape(-1, cfg.I // 128) for r in (got, gen))
    else:
        q0, q1, s0, s1 = got["h_q"], gen["h_q"], got["h_scale"], gen["h_scale"]
    assert np.max(np.abs(s0[rows] / s1[rows] - 1.0)) <= 2.0 ** -7
    assert np.mean(q0[rows] != q1[rows]) < 1e-2
    ref = oracle_routing(cfg, host)
    tokens = sample_tokens(cfg, 64)
    out, _ = oracle.moe_tokens(ref["x_q"], ref["x_scale"], host["w13"], host["w13_scale"], host["w2"],
                               host["w2_scale"], ref["topk_ids"], ref["topk_weights"], tokens, cfg.H, cfg.I)
    assert oracle.max_abs_rel(oracle.f32_from_bf16(got["out"][tokens]), out) <= 2e-2
