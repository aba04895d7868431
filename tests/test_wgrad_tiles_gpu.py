"""The weight gradient's tile heights and tile orders, bit for bit on small
integers, whose sums are exact in fp32 (at most 4200 * 16 < 2^24): 256-row
tiles (full rounds in XCD blocks, partial ones in strips with a narrower last
strip), 128-row tiles in strips of 8, of 4 and of the whole width over several
rounds, in XCD blocks, and with one tile for a few of the compute units."""
import pytest
import torch

from aethelstream_amd import gemm

pytestmark = pytest.mark.gpu


def _ints(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-4, 5, shape, device="cuda", generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("m,ns,k", [
    (4200, (4088,), 4088),           # 256 rows, one full round
    (4200, (4088,), 7672),           # 256 rows, 1.9 rounds, strips 8 8 8 6
    (2080, (2000, 1000, 1088), 5112),  # 128 rows, strips of 4, products end inside tiles
    (1000, (4088,), 7672),           # 128 rows, 1.9 rounds, strips of 4
    (300, (4088, 8), 7672),          # strips of 8
    (20, (4088,), 7672),             # one strip of 30
    (2841, (7976,), 1080),           # one strip of 5
    (64, (8184,), 2048),             # one full round of two a CU
    (753, (7536,), 2048),            # 59 x 8 tiles: strips, not blocks of 59 x 1
    (1, (8,), 8), (65, (136,), 1288),
])
def test_tile_orders(m, ns, k):
    x = _ints((m, k), 1)
    dys = [_ints((m, n), 2 + i) for i, n in enumerate(ns)]
    outs = [torch.full((n, k), float("nan"), device="cuda") for n in ns]
    refs = [dy.float().t().contiguous() @ x.float() for dy in dys]
    print(f"m={m} ns={ns} k={k}", flush=True)
    for step in (1, 2):
        gemm.linear_wgrad_grouped(dys, x, outs, accumulate=step == 2)
        for out, ref in zip(outs, refs):
            assert torch.equal(out, step * ref)
