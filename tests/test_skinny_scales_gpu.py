"""A non-finite double-quant scale reaches only the weight rows whose blocks
use it.  The few-token forward runs reduction steps that lie past a wave's
part of K, and half steps where k % 128 == 64; their loads would otherwise
run on into the scale groups of later rows.

Sizes: fewer steps than k-groups (k = 64), half a step at the end (k = 192,
1344, 4160), parts of unequal length (k = 11008), with groups of 1 to 256
blocks, absmax blocks of 64 and 128."""
import pytest
import torch

from aethelstream_amd import gemm, nf4

pytestmark = pytest.mark.gpu

CASES = [(64, 64, 64, 1), (333, 192, 64, 1), (64, 1344, 64, 4), (64, 1344, 64, 256),
         (64, 1408, 128, 2), (4096, 4160, 64, 8), (4096, 11008, 64, 256)]


def _weight(n, k, block, group, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return nf4.quantize_weight(torch.randn(n, k, device="cuda", generator=g) * 0.02, block,
                               double_quant=True, dq_group=group)


def _poison(w, n, k, block, group, sel):
    """Sets the scales `sel` to infinities and NaNs; the rows that use one."""
    w.absmax_scale[sel[0::2]] = float("inf")
    w.absmax_scale[sel[1::2]] = float("nan")
    bad = torch.zeros(w.absmax_scale.numel(), dtype=torch.bool, device="cuda")
    bad[sel] = True
    return bad.repeat_interleave(group)[:n * k // block].view(n, -1).any(1)


@pytest.mark.parametrize("n,k,block,group", CASES)
@pytest.mark.parametrize("m", [1, 24, 100])
def test_other_rows_keep_their_values(n, k, block, group, m):
    w, up = (_weight(n, k, block, group, s) for s in (1, 2))
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(m, k, device="cuda", generator=g).to(torch.bfloat16)
    print(f"n={n} k={k} block={block} group={group} m={m}", flush=True)
    scales = w.absmax_scale.clone()
    for run in (lambda: gemm.linear_fwd(x, w), lambda: gemm.linear_swiglu(x, w, up)):
        w.absmax_scale.copy_(scales)
        clean = run()
        # Every seventh group, in seven rounds: each group is non-finite once.
        for first in range(7):
            w.absmax_scale.copy_(scales)
            sel = torch.arange(first, scales.numel(), 7, device="cuda")
            rows = _poison(w, n, k, block, group, sel)
            y = run()
            assert torch.equal(y[:, ~rows], clean[:, ~rows])
            assert not torch.isfinite(y[:, rows].float()).all(0).any()
