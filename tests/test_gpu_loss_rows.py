"""GPU parity of the cross-entropy row kernels with the fp64 oracle at the
edges of their row shapes: vocabularies around every change of threads per row
and chunks per thread, odd ones and those below a chunk, rows at any 2-byte
address, targets in the first and the last (shared) chunk, all-negative and
masked rows, in-place gradients; and the forward's threads per row by row
count."""
import numpy as np
import pytest
import torch

import kernelproblems_amd as kp
import oracle
from tests._util import to_u16, ulp_bf16

pytestmark = pytest.mark.gpu

LOSS_RTOL = 2e-6  # fp32 exponentials and per-thread sums, fp64 row sums


def _inputs(M, V, gpu, pad=0, std=2.0):
    g = torch.Generator().manual_seed(M * 31 + V + pad)
    x = (torch.randn(M, V + pad, generator=g) * std).to(torch.bfloat16)
    t = torch.randint(0, V, (M,), generator=g)
    t[0], t[-1] = V - 1, 0
    if M > 2:
        t[1] = -100
        t[2] = max(0, V - 9)
    return x, t


def _check(x, t, gpu, gl=1 / 8192):
    """x: bf16 [M, V] on the GPU (any strides), t on the CPU."""
    out, loss, tw = kp.cross_entropy_forward_backward(x, t.to(gpu), gl, scale=gl, return_loss=True)
    eo, bad = oracle.cross_entropy_fwd_bwd(to_u16(x), t.numpy(), gl)
    u = ulp_bf16(to_u16(out), eo)
    assert bad == 0 and u.max() <= 1 and (u == 0).mean() > 0.998
    eloss, etw, else_, _ = oracle.cross_entropy_fwd(to_u16(x), t.numpy(), scale=gl)
    # each lse is within 2e-6 absolute (checked below), so the scaled sum of M of them within M * 2e-6 * gl
    # whatever its size: rows of one entry have loss 0
    slack = len(t) * 2e-6 * gl
    assert float(tw) == etw and float(loss) == pytest.approx(eloss, rel=LOSS_RTOL, abs=slack)
    loss2, tw2, lse = kp.cross_entropy_loss(x, t.to(gpu), scale=gl, return_lse=True)
    assert float(tw2) == etw and float(loss2) == pytest.approx(eloss, rel=LOSS_RTOL, abs=slack)
    np.testing.assert_allclose(lse.cpu().double().numpy(), else_, rtol=2.0**-24, atol=2e-6)
    return out


@pytest.mark.parametrize("V", [1, 7, 8, 9, 511, 512, 513, 1003, 4095, 4096, 4097, 16383, 16384, 16385, 32768, 50257, 65535,
                               65536, 65537, 98305, 131071, 131072, 131073])
def test_vocabularies(gpu, V):
    print(f"[xent rows] V={V}", flush=True)
    x, t = _inputs(5, V, gpu)
    _check(x.to(gpu), t, gpu)


@pytest.mark.parametrize("V", [600, 5000, 20000, 70001])
def test_unaligned_rows_and_in_place(gpu, V):
    x, t = _inputs(4, V, gpu, pad=11)
    xd = x.to(gpu)
    out = _check(xd[:, 3:3 + V], t, gpu)
    xi = xd[:, 3:3 + V].contiguous()
    r = kp.cross_entropy_forward_backward(xi, t.to(gpu), 1 / 8192, in_place=True)
    assert r.data_ptr() == xi.data_ptr() and torch.equal(r, out)


@pytest.mark.parametrize("M,V", [(2100, 1001), (600, 9001), (3, 40001), (520, 33000)])
def test_forward_threads_per_row(gpu, M, V):
    x, t = _inputs(M, V, gpu)
    loss, tw, lse = kp.cross_entropy_loss(x.to(gpu), t.to(gpu), return_lse=True)
    eloss, etw, else_, _ = oracle.cross_entropy_fwd(to_u16(x), t.numpy())
    assert float(tw) == etw and float(loss) == pytest.approx(eloss, rel=LOSS_RTOL)
    np.testing.assert_allclose(lse.cpu().double().numpy(), else_, rtol=2.0**-24, atol=2e-6)


@pytest.mark.parametrize("V", [1003, 5001, 70001])
def test_negative_masked_and_large_rows(gpu, V):
    """Rows with no value above zero (their order as integers is reversed), a
    row of -0.0, a row that is -inf but for its last element, and values
    whose lanes' maxima lie far apart."""
    x, t = _inputs(6, V, gpu)
    x[0] = -x[0].abs() - 1
    x[1] = -0.0
    x[2] = float("-inf")
    x[2, V - 1] = -3.0
    t[2] = V - 1
    x[3, : V // 2] = -200.0
    x[3, V // 2:] = 90.0
    x[4] = -1e4
    gl = 0.25
    out = kp.cross_entropy_forward_backward(x.to(gpu), t.to(gpu), gl)
    eo, _ = oracle.cross_entropy_fwd_bwd(to_u16(x), t.numpy(), gl)
    d = np.abs(out.cpu().double().numpy() - torch.from_numpy(eo.view(np.int16)).view(torch.bfloat16).double().numpy())
    # one bf16 unit, or where p - 1 cancels a few fp32 units of g
    assert ((ulp_bf16(to_u16(out), eo) <= 1) | (d <= 8 * 2.0**-24 * gl)).all()
