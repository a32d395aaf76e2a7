"""Calls of more rows than one launch has work-items for (2^32): the embedding
forward, RoPE at widths other than 128 and the fused loss take them in several
launches.  The ends of a slab and of the call against the same rows alone."""
import pytest
import torch

import kernelproblems_amd as kp

pytestmark = pytest.mark.gpu

SLAB = (2**32 - 1) // 256 * 4  # rows of one launch: a wave each, four to a block
ROWS = SLAB + 4099
ENDS = [slice(0, 64), slice(SLAB - 64, SLAB + 64), slice(ROWS - 64, ROWS)]


def test_embedding_rows_past_one_launch(gpu):
    table = torch.randn(509, 8, device=gpu).to(torch.bfloat16)
    ids = (torch.arange(ROWS, device=gpu, dtype=torch.int32) * 7) % 509
    out = kp.embedding(table, ids)
    for e in ENDS:
        assert torch.equal(out[e], table[ids[e].long()])


@pytest.mark.parametrize("pairing", ["half", "interleaved"])
def test_rope_positions_past_one_launch(gpu, pairing):
    x = torch.randn(4096, 16, device=gpu).to(torch.bfloat16).repeat(ROWS // 4096 + 1, 1)[:ROWS].view(1, ROWS, 1, 16)
    pos = (torch.arange(ROWS, device=gpu, dtype=torch.int32) % 1021).view(1, ROWS)
    out, _ = kp.rope(x, None, positions=pos, theta=1e4, pairing=pairing)
    for e in ENDS:
        part, _ = kp.rope(x[:, e], None, positions=pos[:, e], theta=1e4, pairing=pairing)
        assert torch.equal(out[:, e], part)


def test_loss_rows_past_one_launch(gpu):
    x = torch.randn(4096, 8, device=gpu).to(torch.bfloat16).repeat(ROWS // 4096 + 1, 1)[:ROWS]
    t = torch.arange(ROWS, device=gpu, dtype=torch.int32) % 8
    out = kp.cross_entropy_forward_backward(x, t, 1.0, ignore_index=-100, return_loss=False)
    for e in ENDS:
        part = kp.cross_entropy_forward_backward(x[e], t[e], 1.0, ignore_index=-100, return_loss=False)
        assert torch.equal(out[e], part)
