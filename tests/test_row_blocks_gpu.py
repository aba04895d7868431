"""The tiled GEMMs at the edges of their row blocks: a launch takes 128, 256,
384 or 512 activation rows per tile by the number of tokens, output tiles and
reduction steps.  Forward (split-K or not), input gradient, their grouped and
summed forms and SwiGLU against an fp64 product over the bf16 dequantized
weights, at token counts on both sides of each block, with ragged output
widths, batched and per-step weight loads.

Tolerance: one bf16 rounding (at most 2^-8 = 3.91e-3 of a value) of an fp32
sum of up to 22016 products (below 1e-5): 3.92e-3.
"""
import pytest
import torch

from aethelstream_amd import gemm, nf4

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 3.92e-3


def _weight(n, k, seed, dq=True, block=64):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return nf4.quantize_weight(torch.randn(n, k, device=DEV, generator=g) * 0.02, block,
                               double_quant=dq)


def _act(m, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)


def _close(y, ref):
    assert torch.isfinite(y.float()).all()
    err = ((y.double() - ref).norm() / ref.norm()).item()
    assert err <= TOL, err


M = [129, 255, 256, 257, 384, 385, 512, 513, 700]


@pytest.mark.parametrize("m", M)
@pytest.mark.parametrize("n,k,dq", [(1000, 1024, True), (2050, 2048, False), (11008, 4096, True),
                                    (8192, 4096, True), (1500, 2112, True)])
def test_fwd(m, n, k, dq):
    w, x = _weight(n, k, 1, dq), _act(m, k, 2)
    ref = x.double() @ nf4.dequant(w).double().t()
    print(f"m={m} n={n} k={k}", flush=True)
    split = gemm.linear_fwd(x, w)
    whole = gemm.linear_fwd(x, w, split_k=False)
    _close(split, ref)
    _close(whole, ref)
    # The tokens' results do not depend on the row block they fall into.
    part = gemm.linear_fwd(x[:m - 1].contiguous(), w, split_k=False) if m > 129 else None
    if part is not None:
        assert torch.equal(part, whole[:m - 1])


@pytest.mark.parametrize("m", [1, 64, 128] + M)
@pytest.mark.parametrize("ns,k,dq", [([1024], 1024, True), ([2048, 512], 2048, False),
                                     ([11008, 11008], 4096, True), ([8192], 4096, True),
                                     ([1472, 64], 2112, True)])
def test_dgrad(m, ns, k, dq):
    ws = [_weight(n, k, 3 + i, dq) for i, n in enumerate(ns)]
    dys = [_act(m, n, 5 + i) for i, n in enumerate(ns)]
    ref = sum(d.double() @ nf4.dequant(w).double() for d, w in zip(dys, ws))
    print(f"m={m} ns={ns} k={k}", flush=True)
    _close(gemm.linear_dgrad_sum(dys, ws), ref)
    _close(gemm.linear_dgrad_sum(dys, ws, split_k=False), ref)


@pytest.mark.parametrize("m", M)
@pytest.mark.parametrize("ff,k,dq", [(1000, 1024, True), (5504, 4096, False), (1030, 2112, True)])
def test_swiglu(m, ff, k, dq):
    wg, wu, x = _weight(ff, k, 7, dq), _weight(ff, k, 8, dq), _act(m, k, 9)
    gate = x.double() @ nf4.dequant(wg).double().t()
    up = x.double() @ nf4.dequant(wu).double().t()
    print(f"m={m} ff={ff} k={k}", flush=True)
    _close(gemm.linear_swiglu(x, wg, wu), gate * torch.sigmoid(gate) * up)


@pytest.mark.parametrize("m", [200, 300, 600])
def test_block_128_and_mixed_kinds(m):
    k = 2048
    ws = [_weight(2000, k, 11, True, 128), _weight(640, k, 12, False), _weight(640, k, 13, True)]
    x = _act(m, k, 14)
    print(f"m={m}", flush=True)
    for y, w in zip(gemm.linear_fwd_grouped(x, ws), ws):
        _close(y, x.double() @ nf4.dequant(w).double().t())
