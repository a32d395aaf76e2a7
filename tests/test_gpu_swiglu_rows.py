"""The SwiGLU kernels' row forms, bit for bit against torch-ROCm eager: flat
runs whose element count is no multiple of a chunk, row-strided views of odd
widths (rows cut inside a chunk, at any 2-byte address), a size whose flat
backward takes four chunks per thread, and the forward in place."""
import pytest
import torch

import kernelproblems_amd as kp
from kernelproblems_amd import _lib as L

pytestmark = pytest.mark.gpu

# the last is past 6 * 2^20 chunks, where the flat backward takes four per thread
SHAPES = [(1, 8), (1, 9), (3, 15), (7, 5), (5, 43), (33, 1664), (100, 5461), (1, 100003), (1025, 4099), (12289, 4099)]


def _operands(gpu, kind, M, N, count):
    g = torch.Generator(device=gpu).manual_seed(M * 7 + N)
    r = lambda *s: torch.randn(*s, dtype=torch.bfloat16, device=gpu, generator=g) * 3  # noqa: E731
    if kind == "flat":
        return [r(M, N) for _ in range(count)]
    ab = r(M, 2 * N)  # the two halves of one projection's output
    return [ab[:, :N], ab[:, N:]] + [r(M, N + 3)[:, 1:1 + N] for _ in range(count - 2)]


@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("kind", ["flat", "halves"])
def test_bitwise_with_eager(gpu, kind, M, N):
    print(f"[swiglu rows] {kind} [{M},{N}]", flush=True)
    a, b, g, s = _operands(gpu, kind, M, N, 4)
    silu = torch.nn.functional.silu(a)
    da_ref = torch.ops.aten.silu_backward((g * b).contiguous(), a.contiguous())
    assert torch.equal(kp.swiglu(a, b), silu * b)
    assert torch.equal(kp.silu(a), silu)
    db, da = kp.swiglu_backward(g, s, b, a)
    assert torch.equal(db, g * s) and torch.equal(da, da_ref)
    h, db, da = kp.swiglu_forward_backward(a, b, g)
    assert torch.equal(h, silu * b) and torch.equal(db, g * silu) and torch.equal(da, da_ref)


@pytest.mark.parametrize("M,N", [(9, 1003), (1025, 4099)])
def test_forward_in_place_on_odd_rows(gpu, M, N):
    g = torch.Generator(device=gpu).manual_seed(1)
    base = torch.randn(M, N + 2, dtype=torch.bfloat16, device=gpu, generator=g)
    a, b = base[:, 1:1 + N], torch.randn(M, N, dtype=torch.bfloat16, device=gpu, generator=g)
    ref, edges = kp.swiglu(a, b), base[:, [0, -1]].clone()
    L.call("kp_swiglu_fwd_bf16", a.data_ptr(), N + 2, b.data_ptr(), N, a.data_ptr(), N + 2, M, N,
           torch.cuda.current_stream(gpu).cuda_stream)
    assert torch.equal(a, ref) and torch.equal(base[:, [0, -1]], edges)
