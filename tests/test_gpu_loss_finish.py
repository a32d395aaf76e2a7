"""The loss's last launch at row counts around its 1024 threads and the four
rows each requests at a time: an exact count, and the fp64 sum of known rows."""
import pytest
import torch

import kernelproblems_amd as kp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 63, 65, 1023, 1024, 1025, 2047, 3072, 3073, 4095, 4096, 4097, 9001])
def test_sums(gpu, M):
    g = torch.Generator(device=gpu).manual_seed(M)
    x = torch.randn(M, 16, generator=g, device=gpu, dtype=torch.bfloat16)
    t = torch.randint(0, 16, (M,), generator=g, device=gpu)
    t[1::3] = -100
    loss, tw = kp.cross_entropy_loss(x, t, scale=0.5)
    keep = t != -100
    d = x.double()
    ref = 0.5 * (torch.logsumexp(d, -1) - d.gather(1, t.clamp_min(0)[:, None]).view(-1))[keep].sum()
    # fp32 exponentials per row, an fp64 sum rounded once
    assert float(tw) == int(keep.sum()) and float(loss) == pytest.approx(float(ref), rel=5e-7)
