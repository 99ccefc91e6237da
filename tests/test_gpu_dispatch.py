"""Which kernels the size rules launch, read from a trace of the call: the lines
lie where the two sides measured alike, and a call on the wrong side of one
gives the same values, only later."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def kernels(call):
    """Names of the kernels that ``call`` launches."""
    call()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as trace:
        call()
        torch.cuda.synchronize()
    names = [e.key for e in trace.key_averages() if "q6moe::" in e.key]
    assert names, "the trace holds no kernel of this library"
    return names


def launched(call, name):
    return any(name in k for k in kernels(call))


def q8_table(rng, experts, rows, width):
    raw = rng.integers(0, 256, (experts, rows, width // 32, 34), dtype=np.uint8)
    raw[..., :2] = np.array([0.001], np.float16).view(np.uint8)
    return raw


@pytest.mark.parametrize("inputs,tokens,tiled", [
    (3072, 64, False), (3072, 65, True),                       # up to 12 K blocks
    (3200, 65, False), (3200, 72, False), (3200, 73, True),    # more
])
def test_q8_matmul_kernel_by_size(device, inputs, tokens, tiled):
    from q6moe.compute import q8_matmul

    w = torch.from_numpy(q8_table(np.random.default_rng(1), 1, 256, inputs)[0]).to(device)
    x = torch.randn(tokens, inputs, device=device).to(torch.bfloat16)
    assert launched(lambda: q8_matmul(x, w), "moe_pf_w8_kernel") == tiled
