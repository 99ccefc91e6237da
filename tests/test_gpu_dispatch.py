"""Which kernels the size rules launch, read from a trace of the call: the lines
lie where the two sides measured alike, and a call on the wrong side of one
gives the same values, only later."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def q8_table(rng, experts, rows, width):
    raw = rng.integers(0, 256, (experts, rows, width // 32, 34), dtype=np.uint8)
    raw[..., :2] = np.array([0.001], np.float16).view(np.uint8)
    return raw


@pytest.mark.parametrize("inputs,tokens,tiled", [
    (3072, 64, False), (3072, 65, True),                       # up to 12 K blocks
    (3200, 65, False), (3200, 72, False), (3200, 73, True),    # more
])
def test_q8_matmul_kernel_by_size(device, kernels, inputs, tokens, tiled):
    from q6moe.compute import q8_matmul

    w = torch.from_numpy(q8_table(np.random.default_rng(1), 1, 256, inputs)[0]).to(device)
    x = torch.randn(tokens, inputs, device=device).to(torch.bfloat16)
    assert any("moe_pf_w8_kernel" in k for k in kernels(lambda: q8_matmul(x, w))) == tiled


@pytest.mark.parametrize("qtype,down,most", [
    ("Q6_K", "Q6_K", 48), ("Q8_0", "Q6_K", 48),                                         # both keep a third wave
    ("Q4_K", "Q8_0", 36), ("Q6_K", "Q5_1", 36), ("Q5_K", "Q8_0", 36), ("Q6_K", "Q4_K", 36),  # one of them
    ("Q4_K", "Q4_K", 0), ("Q5_K", "Q5_1", 0),                                           # neither
])
def test_tile_width_by_format_and_routes_per_expert(device, kernels, qtype, down, most):
    from q6moe.experts import expert_parallel
    from q6moe.synth import moe_layer

    E, H, I = 4, 256, 256
    L = moe_layer(seed=3, experts=E, top_k=1, hidden=H, intermediate=I, tokens=1, qtype=qtype, down_qtype=down,
                  pack=False)
    fn = expert_parallel(None, gate_type=qtype, up_type=qtype, down_type=down, hidden=H, intermediate=I).with_mode(2)
    tabs = fn.prepare(*(L[n].reshape(E, -1) for n in ("gate", "up", "down")), device)
    for per, thin in ((max(most, 1), most > 0), (most + 1, False)):
        tokens = E * per if thin else E * (per - 1) + 1
        x = torch.randn(tokens, H, device=device).to(torch.bfloat16)
        ids = (torch.arange(tokens, device=device, dtype=torch.int32) % E)[:, None]
        w = torch.ones(tokens, 1, device=device, dtype=torch.bfloat16)
        names = kernels(lambda: fn(*tabs, x, ids, w))
        for phase in ("moe_pf_gate_up_kernel<", "moe_pf_down_kernel<"):
            name, = [k for k in names if phase in k]
            assert (", 64>" in name, ", 128>" in name) == (thin, not thin), (per, name)


@pytest.mark.parametrize("tokens,mode,gated", [
    (3, 1, "moe_dec_gate_up_gated_kernel"), (3, 2, "moe_route_small_gated_kernel"),
    (257, 2, "moe_route_count_gated_kernel")])
def test_launches_without_a_gate_run_without_its_items(device, kernels, tokens, mode, gated):
    from q6moe.experts import expert_parallel, pack_experts
    from q6moe.synth import moe_layer

    L = moe_layer(seed=4, experts=4, top_k=2, hidden=256, intermediate=256, tokens=tokens, shared_intermediate=256,
                  pack=False)
    fn = expert_parallel(None, gate_type="Q6_K", up_type="Q6_K", down_type="Q6_K", hidden=256, intermediate=256)
    fn = fn.with_mode(mode)
    tabs = fn.prepare(*(L[n].reshape(4, -1) for n in ("gate", "up", "down")), device)
    sh = {n: pack_experts(L["shared"][n].reshape(1, -1), "Q6_K", 256, 256, device) for n in ("gate", "up", "down")}
    sh["intermediate"] = 256
    x = torch.from_numpy(L["x"]).to(device).to(torch.bfloat16)
    ids, w = torch.from_numpy(L["ids"]).to(device), torch.from_numpy(L["weights"]).to(device).to(torch.bfloat16)
    router = torch.ones(256, device=device, dtype=torch.bfloat16)
    scale = torch.ones(tokens, device=device, dtype=torch.bfloat16)
    for shared, gate in ((None, False), (sh, False), (dict(sh, scale=scale), False), (dict(sh, router=router), True)):
        assert any(gated in k for k in kernels(lambda: fn(*tabs, x, ids, w, shared=shared))) == gate  # noqa: B023


@pytest.mark.parametrize("qtype,down,experts,top_k,hidden,inter,shared,tokens,grouped", [
    # 2.5 routes per expert, both formats with three workgroups per CU
    ("Q8_0", "Q8_0", 128, 8, 1024, 512, 0, 39, False), ("Q8_0", "Q8_0", 128, 8, 1024, 512, 0, 40, True),
    # one of them: from 48 tokens
    ("Q4_K", "Q8_0", 128, 8, 1024, 512, 0, 47, False), ("Q4_K", "Q8_0", 128, 8, 1024, 512, 0, 48, True),
    # too few row blocks of down, below 16 routes per expert
    ("Q8_0", "Q8_0", 32, 4, 1024, 2048, 0, 64, False), ("Q8_0", "Q8_0", 8, 2, 1024, 8192, 0, 63, False),
    ("Q8_0", "Q8_0", 8, 2, 1024, 8192, 0, 64, True),
    # from 2^16, 1.5 routes per expert, one format or two, not with none
    ("Q8_0", "Q8_0", 256, 8, 1024, 256, 0, 47, False), ("Q8_0", "Q8_0", 256, 8, 1024, 256, 0, 48, True),
    ("Q4_K", "Q8_0", 256, 8, 1024, 256, 0, 47, False), ("Q4_K", "Q8_0", 256, 8, 1024, 256, 0, 48, True),
    ("Q4_K", "Q4_K", 256, 8, 1024, 256, 0, 63, False), ("Q4_K", "Q4_K", 256, 8, 1024, 256, 0, 64, True),
    # and 20 tokens
    ("Q8_0", "Q8_0", 256, 24, 1024, 256, 0, 19, False), ("Q8_0", "Q8_0", 256, 24, 1024, 256, 0, 20, True),
    # fewer routes per expert where the experts are large
    ("Q8_0", "Q8_0", 256, 13, 2048, 512, 0, 19, False), ("Q8_0", "Q8_0", 256, 13, 2048, 512, 0, 20, True),
    ("Q8_0", "Q8_0", 256, 13, 1024, 512, 0, 20, False), ("Q8_0", "Q4_K", 256, 13, 2048, 512, 0, 20, False),
    # few of many experts: the thin decode step's one launch
    ("Q8_0", "Q8_0", 1024, 8, 1024, 256, 0, 8, False),
    # with a shared expert
    ("Q8_0", "Q8_0", 256, 8, 1024, 256, 256, 48, False), ("Q8_0", "Q8_0", 256, 8, 1024, 256, 256, 49, True),
    ("Q8_0", "Q8_0", 128, 8, 1024, 512, 512, 55, False), ("Q8_0", "Q8_0", 128, 8, 1024, 512, 512, 56, True),
    ("Q4_K", "Q4_K", 256, 8, 1024, 256, 256, 63, False), ("Q4_K", "Q4_K", 256, 8, 1024, 256, 256, 64, True),
    ("Q8_0", "Q8_0", 1024, 2, 1024, 256, 256, 64, False), ("Q8_0", "Q8_0", 64, 8, 1024, 1024, 256, 64, False),
])
def test_default_family_by_size_and_format(device, kernels, qtype, down, experts, top_k, hidden, inter, shared, tokens,
                                           grouped):
    from q6moe.experts import expert_parallel, pack_experts

    block = {"Q8_0": (32, 34), "Q4_K": (256, 144)}

    def zeros(n, fmt, rows, width):  # which kernels run does not depend on the weights
        per, size = block[fmt]
        raw = torch.zeros(n, rows * (width // per) * size, dtype=torch.uint8, device=device)
        return pack_experts(raw, fmt, rows, width, device)

    def tables(n, rows):
        return zeros(n, qtype, rows, hidden), zeros(n, qtype, rows, hidden), zeros(n, down, hidden, rows)

    fn = expert_parallel(None, gate_type=qtype, up_type=qtype, down_type=down, hidden=hidden, intermediate=inter)
    tabs = tables(experts, inter)
    sh = dict(zip(("gate", "up", "down"), tables(1, shared)), intermediate=shared) if shared else None
    x = torch.randn(tokens, hidden, device=device).to(torch.bfloat16)
    ids = torch.rand(tokens, experts, device=device).topk(top_k).indices.to(torch.int32)
    w = torch.ones(tokens, top_k, device=device, dtype=torch.bfloat16)
    names = kernels(lambda: fn(*tabs, x, ids, w, shared=sh))
    assert any("moe_pf_gate_up_kernel" in k for k in names) == grouped
    assert any("moe_dec_" in k for k in names) != grouped


@pytest.mark.parametrize("inputs,tokens,tiled", [
    (640, 16, False), (640, 17, True), (648, 17, False), (768, 63, False), (768, 64, True), (2560, 63, False),
    (2560, 64, True)])
def test_projection_kernel_by_size(device, kernels, inputs, tokens, tiled):
    from oracle import packed_q6
    from q6moe import pack_q6
    from q6moe.kernel import q6_matmul

    p = pack_q6(packed_q6.fixture(64, inputs), inputs)
    data, scales = torch.from_numpy(p.data).to(device), torch.from_numpy(p.scales).to(device)
    x = torch.randn(tokens, inputs, device=device).to(torch.bfloat16)
    names = kernels(lambda: q6_matmul(x, data, scales, output_features=64))
    assert any("q6_tile_kernel" in k for k in names) == tiled
