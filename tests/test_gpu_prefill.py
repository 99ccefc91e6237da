"""GPU parity of the prefill (tiled grouped-GEMM) expert path against the oracle.

The tiled MFMA kernels run for Q6_K layers whose hidden and intermediate
sizes are multiples of 256 when the call is in prefill mode (mode 2, or
mode 0 with more than 64 tokens). Tolerances are the MoE ones of
test_gpu_moe: max relative error 1e-2 (BF16 output, FP32 accumulation),
elementwise rtol/atol 1e-2, and at least 90 % of outputs bit-identical.
"""

import numpy as np
import pytest
import torch

from oracle import moe as oracle_moe
from q6moe.synth import moe_layer

from .test_gpu_moe import _oracle, _run, assert_moe_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,experts,top_k,hidden,inter", [
    (1, 4, 2, 256, 256),       # one partial tile per expert
    (40, 8, 3, 512, 256),      # partial tiles, several experts
    (300, 6, 2, 512, 512),     # experts with more than one 128-route tile
])
def test_prefill_matches_oracle(device, tokens, experts, top_k, hidden, inter):
    L = moe_layer(seed=100 + tokens, experts=experts, top_k=top_k, hidden=hidden, intermediate=inter,
                  tokens=tokens, bias_sigma=0.5, pack=False)
    got, _ = _run(L, device, mode=2)
    assert_moe_close(got, _oracle(L))


@pytest.mark.parametrize("qtype,down,hidden,inter", [
    ("Q6_K", "Q8_0", 512, 640),   # the Q6 checkpoint's mix; down K = 5 halves of 128
    ("Q8_0", "Q8_0", 384, 384),   # K of 3 halves for both projections
    ("Q4_K", "Q5_1", 512, 384),   # the Q4 checkpoint's mix
    ("Q4_K", "Q4_K", 256, 512),
    ("Q6_K", "Q5_1", 256, 128),   # down K of a single half
    ("Q8_0", "Q6_K", 640, 256),
    ("Q4_K", "Q8_0", 768, 640),
])
def test_tiled_prefill_format_mixes(device, qtype, down, hidden, inter):
    # Every format pair the tiled kernels take, with K not a multiple of 256
    # (odd counts of 128-wide K halves) and skewed routes (partial tiles of
    # every column-group count, experts over several 128-route tiles).
    L = moe_layer(seed=hidden + inter, experts=6, top_k=2, hidden=hidden, intermediate=inter, tokens=300,
                  qtype=qtype, down_qtype=down, bias_sigma=1.0, pack=False)
    got, ctx = _run(L, device, mode=2)
    assert_moe_close(got, _oracle(L))
    fn, tabs, x, ids, w, _ = ctx
    np.testing.assert_array_equal(got, fn(*tabs, x, ids, w).float().cpu().numpy())


def test_prefill_partial_tiles_of_every_width(device):
    # Top-1 routes assigned so that expert e holds counts[e] routes: partial
    # tiles of 1-32, 33-64, 65-96 and 97-128 routes (2, 4, 6 and 8 column
    # groups), exact multiples of 128 and a full tile plus a 1-route tail.
    counts = [1, 17, 32, 33, 50, 64, 65, 90, 96, 97, 113, 127, 128, 129, 256, 200]
    experts = len(counts)
    tokens = sum(counts)
    L = moe_layer(seed=23, experts=experts, top_k=1, hidden=256, intermediate=256, tokens=tokens, pack=False)
    ids = np.repeat(np.arange(experts, dtype=np.int32), counts)
    ids = np.random.default_rng(23).permutation(ids).reshape(tokens, 1)
    w = np.ones((tokens, 1), np.float32)
    got, _ = _run(L, device, mode=2, ids=ids, weights=w)
    assert_moe_close(got, _oracle(L, ids=ids, weights=w))


def test_prefill_and_decode_paths_agree(device):
    # Both paths are checked against the oracle; they share the routing and
    # the rounding boundaries, so they must also agree with each other.
    L = moe_layer(seed=21, experts=16, top_k=4, hidden=1024, intermediate=512, tokens=48, pack=False)
    pre, _ = _run(L, device, mode=2)
    dec, _ = _run(L, device, mode=1)
    want = _oracle(L)
    assert_moe_close(pre, want)
    assert_moe_close(dec, want)
    assert np.mean(pre == dec) >= 0.9


def test_prefill_duplicate_and_dead_routes(device):
    L = moe_layer(seed=22, experts=5, top_k=3, hidden=256, intermediate=256, tokens=200, pack=False)
    ids = L["ids"].copy()
    w = L["weights"].copy()
    ids[:50, 1] = ids[:50, 0]  # duplicated expert in a token: weights add
    w[60:70] = 0  # finished rows give exact zeros
    got, _ = _run(L, device, mode=2, ids=ids, weights=w)
    assert np.all(got[60:70] == 0)
    assert_moe_close(got, _oracle(L, ids=ids, weights=w))


def test_prefill_workload_full_size_sampled(device):
    # 4096 tokens, 128 experts, top-8, hidden 2048, intermediate 768, Q6_K,
    # skewed routing (per-expert logit bias N(0, 0.5)), seed 2. The GPU runs
    # the whole batch; each token's output depends only on its own routes,
    # so the oracle checks a seeded sample of 48 tokens, and a repeat run
    # must be bitwise identical.
    L = moe_layer(seed=2, tokens=4096, bias_sigma=0.5, pack=False)
    got, ctx = _run(L, device, mode=0)
    rows = np.sort(np.random.default_rng(7).choice(4096, 48, replace=False))
    want = oracle_moe.expert_ffn(L["gate"], L["up"], L["down"], L["x"][rows], L["ids"][rows],
                                 L["weights"][rows], types=("Q6_K",) * 3, hidden=2048, intermediate=768)
    assert_moe_close(got[rows], want)
    fn, tabs, x, ids, w, _ = ctx
    again = fn.with_mode(2)(*tabs, x, ids, w).float().cpu().numpy()
    np.testing.assert_array_equal(got, again)
    assert torch.isfinite(torch.from_numpy(got)).all()


def test_prefill_routing_wide_top_k(device):
    # Three routing chunks (256 + 256 + 88 tokens) with 24 routes per token:
    # the staged id/weight rows span several copy rounds per chunk, and the
    # duplicated, out-of-range and zero-weight entries go through the merge.
    L = moe_layer(seed=23, experts=48, top_k=24, hidden=256, intermediate=256, tokens=600, pack=False)
    ids = L["ids"].copy()
    w = L["weights"].copy()
    ids[::5, 2] = ids[::5, 0]
    ids[::7, 3] = 48 + 5
    w[100:110, :] = 0
    w[200:260, 5] = 0
    got, _ = _run(L, device, mode=2, ids=ids, weights=w)
    assert np.all(got[100:110] == 0)
    assert_moe_close(got, _oracle(L, ids=ids, weights=w))


def _q8_table(weights):
    """Q8_0 bytes [rows, blocks, 34] of exactly representable weights: scale 0.5, codes 2 * weights."""
    rows, width = weights.shape
    raw = np.zeros((rows, width // 32, 34), np.uint8)
    raw[..., :2] = np.array([0.5], np.float16).view(np.uint8)
    raw[..., 2:] = (2 * weights).astype(np.int8).view(np.uint8).reshape(rows, width // 32, 32)
    return raw


def test_tiled_q5_k_weights_are_exact(device):
    # One-hot tokens: every product sum has a single term, so no summation order
    # matters and the outputs show each decoded weight. Gate/up: a 1:1 down
    # projection passes the activations through, and the tiled kernel must agree
    # bit for bit with the decode-step one, whose decoder is checked on its own.
    # Down: one activation of 64 per token, y = RNE(64 * weight).
    from oracle.gguf import dequantize_rows
    from oracle.packed_q6 import bf16_round
    from q6moe.experts import expert_parallel

    rng = np.random.default_rng(55)

    def q5(rows, width):
        raw = rng.integers(0, 256, (rows, width // 256, 176), dtype=np.uint8)
        raw[..., :4] = rng.uniform(0.01, 0.05, (rows, width // 256, 2)).astype(np.float16).view(np.uint8)
        return raw

    H = I = 512
    eye = _q8_table(np.eye(H, dtype=np.float32))
    x = torch.eye(H, device=device, dtype=torch.bfloat16)
    ids = torch.zeros(H, 1, dtype=torch.int32, device=device)
    ones = torch.ones(H, 1, device=device, dtype=torch.bfloat16)
    fn = expert_parallel(None, gate_type="Q5_K", up_type="Q5_K", down_type="Q8_0", hidden=H, intermediate=I)
    tabs = fn.prepare(*(t.reshape(1, -1) for t in (q5(I, H), q5(I, H), eye)), device)
    for part in (slice(0, 256), slice(256, 512)):
        got = fn.with_mode(2)(*tabs, x[part], ids[part], ones[part])
        assert torch.equal(got, fn.with_mode(1)(*tabs, x[part], ids[part], ones[part])) and got.any()

    raw = q5(H, I)
    fn = expert_parallel(None, gate_type="Q8_0", up_type="Q8_0", down_type="Q5_K", hidden=H, intermediate=I)
    gate = _q8_table(np.eye(H, dtype=np.float32) * 32)  # g = 32, silu(g) = 32 exactly; u = 2
    tabs = fn.prepare(*(t.reshape(1, -1) for t in (gate, _q8_table(np.eye(H, dtype=np.float32) * 2), raw)), device)
    got = fn.with_mode(2)(*tabs, x, ids, ones).float().cpu().numpy()
    want = bf16_round(64 * bf16_round(dequantize_rows(raw, "Q5_K", I).reshape(H, I)).T)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("down,hidden,inter", [("Q5_K", 512, 256), ("Q8_0", 384, 640), ("Q5_1", 256, 384)])
def test_tiled_q5_k_layers(device, down, hidden, inter):
    L = moe_layer(seed=hidden + inter, experts=6, top_k=2, hidden=hidden, intermediate=inter, tokens=300,
                  qtype="Q5_K", down_qtype=down, bias_sigma=1.0, pack=False)
    got, _ = _run(L, device, mode=2)
    assert_moe_close(got, _oracle(L))


@pytest.mark.parametrize("qtype,down,hidden,inter", [("Q6_K", "Q8_0", 512, 640), ("Q8_0", "Q6_K", 384, 256),
                                                     ("Q4_K", "Q5_1", 512, 384), ("Q5_K", "Q5_K", 256, 256)])
def test_thin_tiles_of_every_width(device, qtype, down, hidden, inter):
    # Up to 48 routes per expert on average the tiles hold 64 routes: experts of
    # every column-group count, of exact multiples of 64 and one past them, and
    # idle ones, in every format.
    counts = [1, 31, 32, 33, 63, 64, 65, 128, 129, 0, 0, 0]
    experts, tokens = len(counts), sum(counts)
    assert tokens <= 48 * experts
    L = moe_layer(seed=hidden, experts=experts, top_k=1, hidden=hidden, intermediate=inter, tokens=tokens,
                  qtype=qtype, down_qtype=down, pack=False)
    ids = np.random.default_rng(9).permutation(np.repeat(np.arange(experts), counts)).astype(np.int32)[:, None]
    got, _ = _run(L, device, mode=2, ids=ids)
    assert_moe_close(got, _oracle(L, ids=ids))
    # the same tokens twice (over 48 routes per expert: tiles of 128)
    L2 = dict(L, x=np.concatenate([L["x"]] * 2), weights=np.concatenate([L["weights"]] * 2))
    twice, _ = _run(L2, device, mode=2, ids=np.concatenate([ids] * 2))
    np.testing.assert_array_equal(twice, np.concatenate([got, got]))


@pytest.mark.parametrize("qtype,down", [("Q4_K", "Q8_0"), ("Q6_K", "Q5_1"), ("Q5_K", "Q6_K"), ("Q8_0", "Q4_K"),
                                        ("Q6_K", "Q5_K")])
def test_thin_tiles_of_mixed_formats(device, qtype, down):
    # tiles of 64 routes with one projection of a format that keeps two waves per
    # SIMD, up to 36 routes per expert; the same tokens twice run in tiles of 128
    counts = [1, 16, 33, 64, 65, 129] + [0] * 5
    experts, tokens = len(counts), sum(counts)
    assert tokens <= 36 * experts < 48 * experts < 2 * tokens
    L = moe_layer(seed=tokens, experts=experts, top_k=1, hidden=512, intermediate=256, tokens=tokens, qtype=qtype,
                  down_qtype=down, pack=False)
    ids = np.random.default_rng(9).permutation(np.repeat(np.arange(experts), counts)).astype(np.int32)[:, None]
    got, _ = _run(L, device, mode=2, ids=ids)
    assert_moe_close(got, _oracle(L, ids=ids))
    L2 = dict(L, x=np.concatenate([L["x"]] * 2), weights=np.concatenate([L["weights"]] * 2))
    twice, _ = _run(L2, device, mode=2, ids=np.concatenate([ids] * 2))
    np.testing.assert_array_equal(twice, np.concatenate([got, got]))
