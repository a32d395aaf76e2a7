"""SwiGLU on row-strided views of rows past 2^32 columns, and of more chunks than
one launch numbers (rows in slabs): the ends of the rows and both sides of
column 2^32, bit for bit against torch-ROCm eager on the same slices."""
import pytest
import torch

import kernelproblems_amd as kp

pytestmark = pytest.mark.gpu

N = 2**32 + 4099  # the last chunk is cut by the row's end


def _ends(t):
    return [t[:, s] for s in (slice(0, 4096), slice(2**32 - 2048, 2**32 + 2048), slice(N - 2048, N))]


@pytest.mark.parametrize("rows", [2, 5])  # five rows: 2.7e9 chunks, slabs of three rows
def test_silu_of_rows_past_32_bit_columns(gpu, rows):
    x = torch.empty(rows, N + 5, dtype=torch.bfloat16, device=gpu).normal_(std=3.0)[:, :N]
    out = kp.silu(x)
    assert out.shape == x.shape
    for a, e in zip(_ends(out), _ends(x)):
        assert torch.equal(a, torch.nn.functional.silu(e))
