"""The weight gradient's two epilogues (through LDS for outputs that take 16-byte
stores, direct otherwise), bit for bit on small integers, whose sums are exact
in fp32: ragged rows and columns, an output 4 bytes off
alignment, a row stride that is no multiple of 16 bytes, and accumulation."""
import pytest
import torch

from aethelstream_amd import gemm

pytestmark = pytest.mark.gpu


def _ints(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-4, 5, shape, device="cuda", generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("m,n,k", [(33, 8, 256), (64, 256, 512), (100, 264, 520), (31, 520, 1024),
                                   (40, 136, 248), (96, 1000, 776), (200, 384, 2048)])
@pytest.mark.parametrize("offset", [0, 1])
def test_both_epilogues(m, n, k, offset):
    dy, x = _ints((m, n), 1), _ints((m, k), 2)
    ref = dy.float().t().contiguous() @ x.float()
    buf = torch.full((n * k + offset,), float("nan"), device="cuda")
    out = buf[offset:].view(n, k)
    print(f"m={m} n={n} k={k} offset={offset}", flush=True)
    gemm.linear_wgrad(dy, x, out)
    assert torch.equal(out, ref)
    gemm.linear_wgrad(dy, x, out, accumulate=True)
    assert torch.equal(out, 2 * ref)


def test_grouped_rows_stop_at_each_output():
    # Outputs that end inside a tile: rows past N stay untouched.
    m, k = 64, 768
    x = _ints((m, k), 3)
    ns = [264, 8, 248]
    dys = [_ints((m, n), 4 + n) for n in ns]
    bufs = [torch.full((n + 256, k), 7.0, device="cuda") for n in ns]
    outs = [b[:n] for b, n in zip(bufs, ns)]
    print("grouped", flush=True)
    for step in (1, 2):
        gemm.linear_wgrad_grouped(dys, x, outs, accumulate=step == 2)
        for dy, b, n in zip(dys, bufs, ns):
            assert torch.equal(b[:n], step * (dy.float().t().contiguous() @ x.float()))
            assert (b[n:] == 7.0).all()


# A ragged last column within the first and the second wave's half of a tile,
# and rows that are a multiple of 32, 16 and 8 floats (the store policies).
@pytest.mark.parametrize("k", [8, 136, 392, 768 + 32, 768 + 16, 768 + 248])
@pytest.mark.parametrize("m", [64, 2080])
def test_ragged_columns_stop_at_each_output(m, k):
    x = _ints((m, k), 3)
    ns = [264, 8, 248]
    dys = [_ints((m, n), 4 + n) for n in ns]
    bufs = [torch.full((n + 256, k), 7.0, device="cuda") for n in ns]
    print(f"m={m} k={k}", flush=True)
    for step in (1, 2):
        gemm.linear_wgrad_grouped(dys, x, [b[:n] for b, n in zip(bufs, ns)], accumulate=step == 2)
        for dy, b, n in zip(dys, bufs, ns):
            assert torch.equal(b[:n], step * (dy.float().t().contiguous() @ x.float()))
            assert (b[n:] == 7.0).all()


# More than 288 MiB of rows that are no multiple of 128 bytes: default stores
# up to 160 tokens, non-temporal ones beyond.
@pytest.mark.parametrize("m", [160, 161])
def test_large_outputs(m):
    dy, x = _ints((m, 10000), 5), _ints((m, 8200), 6)
    print(f"m={m}", flush=True)
    assert torch.equal(gemm.linear_wgrad(dy, x), dy.float().t().contiguous() @ x.float())
