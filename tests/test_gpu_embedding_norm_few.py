"""Embedding -> RMSNorm of a few wide rows (a decode step's tokens): h, y and
rstd bit for bit those of embedding() then rms_norm(), on both sides of the row
count where the norm's layout changes, and ids outside the table."""
import pytest
import torch

import kernelproblems_amd as kp

pytestmark = pytest.mark.gpu

EPS = 1e-5


@pytest.mark.parametrize("D", [2048, 2560, 4096, 5120, 8192])
@pytest.mark.parametrize("T", [1, 16, "cus", "cus + 1"])
def test_bits_of_the_composition(gpu, T, D):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    T = {"cus": cus, "cus + 1": cus + 1}.get(T, T)
    print(f"[emb+rms few] T={T} D={D}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(T * 3 + D)
    table = torch.randn(997, D, generator=g, device=gpu, dtype=torch.bfloat16)
    w = torch.randn(D, generator=g, device=gpu, dtype=torch.bfloat16) * 0.02 + 1
    for dtype in (torch.int32, torch.int64):
        ids = torch.randint(0, 997, (T,), generator=g, device=gpu).to(dtype)
        h, y, r = kp.embedding_rms_norm(table, ids, w, EPS, return_h=True)
        emb = kp.embedding(table, ids)
        _, y2, r2 = kp.rms_norm([emb], w, EPS, D)
        assert torch.equal(h, emb) and torch.equal(r.view(-1), r2.view(-1)) and torch.equal(y, y2)
        assert torch.equal(kp.embedding_rms_norm(table, ids, w, EPS)[1], y)


def test_ids_outside_the_table(gpu):
    table = torch.randn(61, 4096, device=gpu, dtype=torch.bfloat16)
    w = torch.ones(4096, device=gpu, dtype=torch.bfloat16)
    ids = torch.tensor([5, 61, -1, 60], device=gpu)
    with pytest.raises(IndexError):
        kp.embedding_rms_norm(table, ids, w, EPS)
    kp.set_index_checking(False)
    try:
        h, y, _ = kp.embedding_rms_norm(table, ids, w, EPS, return_h=True)
    finally:
        kp.set_index_checking(True)
    assert not h[1:3].any() and not y[1:3].any() and torch.equal(h[[0, 3]], table[[5, 60]])
