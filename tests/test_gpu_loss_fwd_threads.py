"""The cross-entropy forward on both sides of every change of threads per row
(by vocabulary, row count and row alignment) against the fp64 oracle."""
import numpy as np
import pytest
import torch

import kernelproblems_amd as kp
import oracle
from tests._util import to_u16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [8191, 8192, 16384, 16392, 24577, 32768])
@pytest.mark.parametrize("per_cu,more", [(2, -1), (2, 0), (2, 1), (3, 0), (3, 1), (4, 1), (6, 0), (6, 1)])
def test_both_sides(gpu, V, per_cu, more):
    M = per_cu * torch.cuda.get_device_properties(gpu).multi_processor_count + more
    print(f"[xent fwd threads] [{M},{V}]", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + V)
    x = torch.randn(M, V, generator=g, device=gpu, dtype=torch.bfloat16) * 2
    t = torch.randint(0, V, (M,), generator=g, device=gpu)
    t[::5] = -100
    loss, tw, lse = kp.cross_entropy_loss(x, t, return_lse=True)
    rows = torch.cat([torch.arange(0, M, 61), torch.tensor([M - 1])])
    _, _, want, _ = oracle.cross_entropy_fwd(to_u16(x[rows.to(gpu)]), t.cpu()[rows].numpy())
    np.testing.assert_allclose(lse.cpu()[rows].double().numpy(), want, rtol=2.0**-24, atol=2e-6)
    # the loss is the sum of lse - x_t over the rows that count: M fp32 lse of 2e-6 each
    keep = t != -100
    ref = (lse.double() - x.double().gather(1, t.clamp_min(0)[:, None]).view(-1))[keep].sum()
    assert float(tw) == int(keep.sum()) and float(loss) == pytest.approx(float(ref), rel=2e-6)
