"""The few-token forward's 96-token tiles (65 to 96 tokens), bit for bit: with
one 1.0 per activation row every output is a dequantized weight, with two it
is their fp32 sum rounded once to bf16, whatever the order of the zeros."""
import pytest
import torch

from aethelstream_amd import gemm, nf4

pytestmark = pytest.mark.gpu


def _weight(n, k, seed, dq):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return nf4.quantize_weight(torch.randn(n, k, device="cuda", generator=g) * 0.02, 64,
                               double_quant=dq)


def _two_hot(m, k):
    """x [m, k] with two ones per row, and their columns."""
    i = torch.arange(m, device="cuda")
    a, b = i * 37 % k, (i * 37 + 1 + i % (k - 1)) % k
    a[-1], b[-1] = k - 1, 0
    x = torch.zeros(m, k, dtype=torch.bfloat16, device="cuda")
    x[i, a] = 1.0
    x[i, b] = 1.0
    return x, a, b


def _sum(w, a, b):
    t = nf4.dequant(w).float().t()
    return t[a] + t[b]


@pytest.mark.parametrize("m", [65, 80, 95, 96, 97])
@pytest.mark.parametrize("n,k", [(1, 64), (333, 1344), (1024, 4096)])
@pytest.mark.parametrize("dq", [False, True])
def test_fwd(m, n, k, dq):
    w = _weight(n, k, n + k, dq)
    x, a, b = _two_hot(m, k)
    ref = _sum(w, a, b).to(torch.bfloat16)
    print(f"m={m} n={n} k={k} dq={dq}", flush=True)
    assert torch.equal(gemm.linear_fwd(x, w), ref)
    assert torch.equal(gemm.linear_fwd(x, w, split_k=False), ref)
