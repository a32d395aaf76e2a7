"""GPU parity of RoPE at head widths other than 128 (one wave per position for
widths of whole chunks, one pair per lane for the rest) and at any alignment:
both pairings, theta and table angles, conjugate, fp32 outputs, transposed and
offset views, more units than a wave takes in one round, out-of-range
positions, and rotations in place.  Reference: fp64 on the same fp32 angles."""
import pytest
import torch

import kernelproblems_amd as kp
from kernelproblems_amd import _lib as L
from tests._util import assert_bf16_close, to_u16

pytestmark = pytest.mark.gpu

THETA, ROWS = 10000.0, 512


def _reference(x, cos, sin, pairing):
    x = x.double()
    if pairing == "half":
        a, b = x.chunk(2, -1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)


def _angles(gpu, D, pos, table, conj):
    if table is not None:
        f = table[pos.clamp(0, ROWS - 1)][:, :, None, :]
        cos, sin = f.real.double(), f.imag.double()
        ok = ((pos >= 0) & (pos < ROWS))[:, :, None, None].double()
        cos, sin = cos * ok, sin * ok
    else:
        inv = (THETA ** (-torch.arange(0, D, 2, device=gpu, dtype=torch.float64) / D)).float()
        a = (pos.float()[..., None] * inv).double()[:, :, None, :]
        cos, sin = a.cos(), a.sin()
    return cos, -sin if conj else sin


@pytest.mark.parametrize("D", [2, 6, 8, 16, 40, 64, 72, 80, 96, 112, 256, 512])
@pytest.mark.parametrize("pairing", ["half", "interleaved"])
@pytest.mark.parametrize("layout", ["contiguous", "heads_first", "offset"])
def test_widths(gpu, D, pairing, layout):
    print(f"[rope widths] D={D} {pairing} {layout}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(D)
    r = lambda *s: torch.randn(*s, generator=g, device=gpu, dtype=torch.bfloat16)  # noqa: E731
    for B, S, Hq, Hk in ((2, 17, 5, 3), (1, 9, 32, 8), (3, 5, 1, 0)):
        def make(H):
            if layout == "heads_first":
                return r(B, H, S, D).transpose(1, 2)
            if layout == "offset":
                return r(B, S, H, D + 3)[..., 1:1 + D]
            return r(B, S, H, D)
        q, k = make(Hq), make(Hk) if Hk else None
        pos = torch.randint(0, ROWS, (B, S), generator=g, device=gpu)
        table = torch.randn(ROWS, D // 2, generator=g, device=gpu, dtype=torch.complex64)
        for use_table, conj, dt in ((False, False, torch.bfloat16), (True, True, torch.bfloat16), (True, False, torch.float32),
                                    (False, True, torch.float32)):
            out = kp.rope(q, k, positions=pos, theta=None if use_table else THETA, freqs_cis=table if use_table else None,
                          pairing=pairing, conj=conj, q_dtype=dt, k_dtype=dt)
            cos, sin = _angles(gpu, D, pos, table if use_table else None, conj)
            for x, o in zip((q, k), out):
                if x is None:
                    continue
                ref = _reference(x, cos, sin, pairing)
                # each output is a sum of two products, |a| + |b| at most sqrt(2) times the pair's length
                mag = _reference(x.abs(), cos.abs(), -sin.abs(), pairing).abs().max()
                if dt == torch.float32:
                    # fp32 sine and cosine (a few units of 2^-24), one product, one fma
                    assert float((o.double() - ref).abs().max()) <= 2.0**-21 * float(mag)
                else:
                    assert_bf16_close(to_u16(o), to_u16(ref.to(torch.bfloat16)), what="rope", max_ulp=1, min_exact=0.98,
                                      ulp_abs_slack=2.0**-21 * float(mag))


@pytest.mark.parametrize("D", [64, 96, 256])
@pytest.mark.parametrize("pairing", ["half", "interleaved"])
def test_out_of_range_positions_are_zero(gpu, D, pairing):
    g = torch.Generator(device=gpu).manual_seed(D)
    q = torch.randn(1, 6, 4, D, generator=g, device=gpu, dtype=torch.bfloat16)
    table = torch.randn(ROWS, D // 2, generator=g, device=gpu, dtype=torch.complex64)
    pos = torch.tensor([[0, ROWS, 5, -1, ROWS - 1, 7]], device=gpu)
    kp.set_index_checking(False)
    try:
        out, _ = kp.rope(q, freqs_cis=table, positions=pos, pairing=pairing)
    finally:
        kp.set_index_checking(True)
        with pytest.raises(IndexError):
            kp.check_indices()
    cos, sin = _angles(gpu, D, pos, table, False)
    assert not out[0, [1, 3]].any()
    assert_bf16_close(to_u16(out), to_u16(_reference(q, cos, sin, pairing).to(torch.bfloat16)), what="rope", max_ulp=1,
                      ulp_abs_slack=2.0**-21 * 8)


@pytest.mark.parametrize("D,H", [(64, 8), (96, 40), (256, 24)])
@pytest.mark.parametrize("pairing", [L.KP_ROPE_HALF, L.KP_ROPE_INTERLEAVED])
def test_in_place_through_the_abi(gpu, D, H, pairing):
    """The output may be the input: the same bits as out of place, also where a
    position's heads take several rounds of a wave."""
    import ctypes as C
    g = torch.Generator(device=gpu).manual_seed(D)
    B, S = 2, 301
    x = torch.randn(B, S, H, D, generator=g, device=gpu, dtype=torch.bfloat16)
    ref, _ = kp.rope(x, theta=THETA, pairing="half" if pairing == L.KP_ROPE_HALF else "interleaved")
    st = (C.c_int64 * 3)(*x.stride()[:3])
    L.call("kp_rope_bf16", x.data_ptr(), x.data_ptr(), H, st, st, None, None, 0, None, None, B, S, D, None, 0, 0, 0, pairing,
           THETA, None, 0, 0, 0, 0, None, torch.cuda.current_stream(gpu).cuda_stream)
    assert torch.equal(x, ref)
