"""Quantize with power-of-two blocks from 8 to 512 elements (a block within one
wave's 512-element tile), bit for bit against the oracle: element counts at the
edges of blocks and tiles, unaligned buffers, quotients next to the code steps,
and blocks of zeros, tiny values, infinities and NaN."""
import numpy as np
import pytest
import torch

import oracle
from aethelstream_amd import nf4

pytestmark = pytest.mark.gpu
BLOCKS = [8, 16, 32, 128, 256, 512]


def _check(x: np.ndarray, bs: int, dev: torch.Tensor = None):
    dev = torch.from_numpy(x).cuda() if dev is None else dev
    r = nf4.quantize_nf4(dev, block_size=bs)
    torch.cuda.synchronize()
    pk, am = oracle.quantize_nf4(x, bs)
    np.testing.assert_array_equal(r.absmax.cpu().numpy().view(np.uint32), am.view(np.uint32))
    np.testing.assert_array_equal(r.packed.cpu().numpy(), pk)


@pytest.mark.parametrize("bs", BLOCKS)
@pytest.mark.parametrize("n", [1, 9, 511, 512, 513, 1030, 4099, 2048 * 4 + 100, 300001])
def test_counts(bs, n):
    print(f"bs={bs} n={n}", flush=True)
    _check(oracle.gen_normal(n + bs, n, 0.02), bs)


@pytest.mark.parametrize("bs", BLOCKS)
def test_unaligned_input(bs):
    x = oracle.gen_normal(bs, 5003, 0.02)
    buf = torch.empty(5004, device="cuda")
    buf[1:].copy_(torch.from_numpy(x))
    print(f"bs={bs}", flush=True)
    _check(x, bs, buf[1:])


@pytest.mark.parametrize("bs", BLOCKS)
def test_steps_and_special_blocks(bs):
    # One value of each block sets the absmax; the others sit within a few
    # ulps of the midpoints between codes times it.
    codes = nf4.NF4_CODES.numpy()
    mids = ((codes[1:] + codes[:-1]) / 2).astype(np.float32)
    rng = np.random.default_rng(bs)
    blocks = []
    for scale in (1.0, 0.0217, 3e-9, 7e37):
        for _ in range(12):
            q = rng.choice(mids, bs).astype(np.float32)
            b = q * np.float32(scale)
            b = (b.view(np.int32) + rng.integers(-3, 4, bs).astype(np.int32)).view(np.float32)
            b[rng.integers(bs)] = np.float32(scale)
            blocks.append(b)
    zero = np.zeros(bs, np.float32)
    blocks += [zero, zero + np.float32(1e-12)]
    for special in (np.inf, -np.inf, np.nan):
        b = oracle.gen_normal(5, bs, 0.02)
        b[bs // 2] = special
        blocks.append(b)
    print(f"bs={bs}", flush=True)
    _check(np.concatenate(blocks).astype(np.float32), bs)
