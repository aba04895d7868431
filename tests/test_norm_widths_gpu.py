"""RMSNorm at every row width class that stays in registers (4097 to 16384
elements by the 1024, whole and ragged last chunks) and at its edges: the rms
within fp32 rounding of the exact one (a tree over at most 64 terms per thread
and 256 threads, 2e-6), y bit for bit given that rms, NaN and infinity rows,
and nothing written past the last row."""
import numpy as np
import pytest
import torch

import oracle
from aethelstream_amd import norm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [4092, 4100, 5120, 5124, 6144, 7000, 8188, 8196, 9216, 11008, 12288,
                               12292, 13824, 16380, 16388])
def test_widths(d):
    m = 3
    x = oracle.gen_normal(d, m * d, 1.0).reshape(m, d)
    w = (1.0 + oracle.gen_normal(71, d, 0.1)).astype(np.float32)
    out = torch.full((m + 1, d), 7.0, dtype=torch.bfloat16, device="cuda")
    print(f"d={d}", flush=True)
    _, rms = norm.rms_norm_fwd(torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), out=out[:m])
    rms = rms.cpu().numpy()
    np.testing.assert_allclose(rms, np.sqrt((x.astype(np.float64) ** 2).mean(axis=1) + 1e-6),
                               rtol=2e-6, atol=0)
    want = oracle.f32_to_bf16_bits(((x / rms[:, None]).astype(np.float32) * w).astype(np.float32))
    np.testing.assert_array_equal(out[:m].view(torch.int16).cpu().numpy().view(np.uint16), want)
    assert (out[m] == 7.0).all()


def test_special_values_in_the_last_chunk():
    d = 5124
    x = torch.ones(3, d, device="cuda")
    x[0, -1] = float("nan")
    x[1, -1] = float("inf")
    y, rms = norm.rms_norm_fwd(x, torch.ones(d, device="cuda"))
    assert rms[0].isnan() and y[0].isnan().all()
    assert rms[1].isinf() and y[1, -1].isnan() and (y[1, :-1] == 0).all()
    assert (y[2] == 1).all()
