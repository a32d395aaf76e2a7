"""The chain's own zero fill (emb_zero_rows): tables whose rows are a part, one
and several blocks of 256 16-byte units, so that blocks straddle rows and end
past the share; every row bit for bit the embedding backward's of the same g,
into memory that held NaN."""
import pytest
import torch

from kernelproblems_amd import fused as F

pytestmark = pytest.mark.gpu

EPS = 1e-5


@pytest.mark.parametrize("V", [5, 1003])
@pytest.mark.parametrize("N,dtype", [(512, torch.bfloat16), (1536, torch.bfloat16), (2560, torch.bfloat16),
                                     (512, torch.float32), (1024, torch.float32), (8192, torch.float32)])
def test_untouched_rows(gpu, V, N, dtype):
    print(f"[chain zero rows] V={V} N={N} {dtype}", flush=True)
    M = 300
    g = torch.Generator(device=gpu).manual_seed(V + N)
    x, dy, res = (torch.randn(M, N, generator=g, device=gpu, dtype=torch.bfloat16) for _ in range(3))
    w = torch.randn(N, generator=g, device=gpu, dtype=torch.bfloat16) * 0.02 + 1
    ids = torch.randint(0, V, (M,), generator=g, device=gpu) // 3 * 3  # a third of the vocabulary
    dx, _ = F.rms_norm_backward([dy], [x], None, w, EPS, N, dx_residual=res, dw=None)
    want = F.embedding_dense_backward(dx, ids, V, out_dtype=dtype)
    junk = torch.full((V, N), float("nan"), dtype=dtype, device=gpu)
    del junk  # the allocator hands its memory to the call's table
    _, _, table = F.rms_norm_embedding_backward([dy], x, None, w, EPS, N, res, ids, V, want_y=False, out_dtype=dtype)
    bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
    assert torch.equal(table.view(bits), want.view(bits))
    assert not table[1::3].any()
