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


# Hidden widths on both sides of the line between 32- and 64-column tiles (the
# wide ones with a ragged last tile).  fp32 silu on the gate sum: one bf16
# rounding of the output, 2^-8 at most, and the hardware exponential and
# reciprocal, a few fp32 ulps (below 1e-5).
@pytest.mark.parametrize("m", [33, 64, 65, 96, 100, 128])
@pytest.mark.parametrize("ff", [33, 8192, 8200, 20000])
@pytest.mark.parametrize("k,dq", [(64, True), (448, False), (1024, True)])
def test_swiglu_tile_widths(m, ff, k, dq):
    wg, wu = _weight(ff, k, 1, dq), _weight(ff, k, 2, dq)
    x, a, b = _two_hot(m, k)
    gate = _sum(wg, a, b).double()
    ref = gate * torch.sigmoid(gate) * _sum(wu, a, b).double()
    print(f"m={m} ff={ff} k={k} dq={dq}", flush=True)
    err = (gemm.linear_swiglu(x, wg, wu).double() - ref).abs()
    assert (err <= ref.abs() * (2.0 ** -8 + 1e-5)).all(), (err / ref.abs()).max().item()
