"""The few-token forward (m <= 128) against an fp64 product over the bf16
dequantized weights, at the edges of its token tiles (4, 16, 32, 64, 128 rows),
weight tiles (32 rows) and reduction steps (128 deep, k % 128 == 64 leaving
half a step; fewer steps than k-groups), for both absmax forms and block
sizes, grouped, SwiGLU, split over K slices or not, and unaligned outputs.

Tolerance: the output is one bf16 rounding of an fp32 sum.  bf16 keeps 8
significant bits, so rounding to nearest is off by at most 2^-8 of the value
(rel-L2 at most 2^-8 = 3.91e-3, about 1.7e-3 over many elements, more over
few) and the fp32 sum of k <= 13824 products adds below 1e-5: 3.92e-3.
SwiGLU rounds once too.
"""
import pytest
import torch

from aethelstream_amd import gemm, nf4

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 3.92e-3


def _weight(n, k, seed, dq, block=64):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return nf4.quantize_weight(torch.randn(n, k, device=DEV, generator=g) * 0.02, block,
                               double_quant=dq)


def _act(m, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)


def _ref(x, w):
    return x.double() @ nf4.dequant(w).double().t()


def _close(y, ref):
    assert torch.isfinite(y.float()).all()
    err = ((y.double() - ref).norm() / ref.norm()).item()
    assert err <= TOL, err


@pytest.mark.parametrize("m", [1, 2, 4, 5, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("n,k", [(1, 64), (31, 192), (96, 128), (130, 1088), (4096, 4096)])
@pytest.mark.parametrize("dq", [False, True])
def test_fwd_tile_edges(m, n, k, dq):
    w, x = _weight(n, k, n + k, dq), _act(m, k, m)
    ref = _ref(x, w)
    print(f"m={m} n={n} k={k} dq={dq}", flush=True)
    _close(gemm.linear_fwd(x, w), ref)
    _close(gemm.linear_fwd(x, w, split_k=False), ref)


@pytest.mark.parametrize("m", [1, 16, 20, 60, 100])
@pytest.mark.parametrize("block", [64, 128, 256])
def test_grouped_kinds_and_blocks(m, block):
    k = 2816 if block != 256 else 2816 // 256 * 256
    ns = [300, 64, 1025, 33]
    ws = [_weight(n, k, 7 + i, i % 2 == 0, block) for i, n in enumerate(ns)]
    x = _act(m, k, 3)
    print(f"m={m} block={block}", flush=True)
    for split in (True, False):
        for y, w in zip(gemm.linear_fwd_grouped(x, ws, split_k=split), ws):
            _close(y, _ref(x, w))


@pytest.mark.parametrize("m", [1, 16, 17, 64, 77, 128])
@pytest.mark.parametrize("ff,k", [(5, 64), (192, 320), (1000, 4096)])
@pytest.mark.parametrize("dq", [False, True])
def test_swiglu(m, ff, k, dq):
    wg, wu, x = _weight(ff, k, 1, dq), _weight(ff, k, 2, dq), _act(m, k, 5)
    print(f"m={m} ff={ff} k={k} dq={dq}", flush=True)
    gate = _ref(x, wg)
    _close(gemm.linear_swiglu(x, wg, wu), gate * torch.sigmoid(gate) * _ref(x, wu))


@pytest.mark.parametrize("m", [3, 24, 48, 128])
@pytest.mark.parametrize("dq", [False, True])
def test_one_hot_equals_dequantized_weight(m, dq):
    # 1.0 * W[n, j] added onto exact zeros: every output is a weight, bit for bit.
    n, k = 333, 1344
    w = _weight(n, k, 11, dq)
    j = torch.arange(m, device=DEV) * 37 % k
    j[-1] = k - 1
    x = torch.zeros(m, k, dtype=torch.bfloat16, device=DEV)
    x[torch.arange(m, device=DEV), j] = 1.0
    print(f"m={m} dq={dq}", flush=True)
    assert torch.equal(gemm.linear_fwd(x, w), nf4.dequant(w).t()[j])


@pytest.mark.parametrize("m", [5, 40])
def test_unaligned_output_and_special_values(m):
    n, k = 100, 192
    w, x = _weight(n, k, 21, True), _act(m, k, 22)
    y = gemm.linear_fwd(x, w)
    buf = torch.empty(m * n + 1, dtype=torch.bfloat16, device=DEV)
    off = buf[1:].view(m, n)
    gemm.linear_fwd(x, w, out=off)
    print(f"m={m}", flush=True)
    assert torch.equal(y, off)
    # A NaN or an infinity of one token stays in that token's row.
    x2 = x.clone()
    x2[1, k - 1] = float("nan")
    x2[2, 0] = float("inf")
    y2 = gemm.linear_fwd(x2, w)
    keep = [i for i in range(m) if i not in (1, 2)]
    assert torch.equal(y2[keep], y[keep])
    assert torch.isnan(y2[1]).all()
    col = nf4.dequant(w)[:, 0]
    assert torch.isinf(y2[2][col != 0]).all()


def test_split_slices_on_a_caller_workspace_are_deterministic():
    m, n, k = 50, 5120, 13824
    w, x = _weight(n, k, 31, True), _act(m, k, 32)
    need = gemm.fwd_workspace_bytes([n], m, k)
    assert need > 0
    buf = torch.full((need,), 0xff, dtype=torch.uint8, device=DEV)
    a = gemm.linear_fwd_grouped(x, [w], workspace=buf)[0]
    b = gemm.linear_fwd_grouped(x, [w])[0]
    print("split", flush=True)
    assert torch.equal(a, b)
    _close(a, _ref(x, w))
